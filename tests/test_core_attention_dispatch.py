"""CoreAttention.forward runs the sparse_attention_bias that the object has: the
class's own, a subclass's, one set on the instance or patched into the class."""
import types

import pytest
import torch

from neutrongt_amd import CoreAttention


def _mark(value):
    def sparse_attention_bias(self, q, k, v, edge_index, attn_bias, kv_ext=None,
                              interleave_grads=False):
        return torch.full((q.shape[1], q.shape[2], q.shape[3]), value), "score"
    return sparse_attention_bias


@pytest.mark.parametrize("where", ["subclass", "instance", "instance_method", "class"])
def test_an_overridden_sparse_attention_bias_runs(monkeypatch, where):
    cls, fn = CoreAttention, _mark(3.0)
    if where == "subclass":
        cls = type("Sub", (CoreAttention,), {"sparse_attention_bias": fn})
    core = cls(16, 0.0, 2)
    if where == "instance":
        core.sparse_attention_bias = lambda *a, **kw: fn(core, *a, **kw)
    elif where == "instance_method":
        core.sparse_attention_bias = types.MethodType(fn, core)
    elif where == "class":
        monkeypatch.setattr(CoreAttention, "sparse_attention_bias", fn)
    q = torch.zeros(1, 5, 2, 8)
    x, score = core(q, q, q, None, torch.zeros(2, 3, dtype=torch.long), "sparse")
    assert x.shape == (1, 5, 16) and bool((x == 3.0).all()) and score == "score"
