"""Shapes at the edges of the encoder's projections, with a stand-in core."""
import pytest
import torch
from torch import nn

from neutrongt_amd.encoder import EncoderLayer
from neutrongt_amd.linear import WgradLinear, project


class _Core(nn.Module):
    def forward(self, q, k, v, attn_bias, edge_index, attn_type):
        assert q.dim() == 4
        return (q + k + v).flatten(2), None


def _layer():
    layer = EncoderLayer(16, 16, 0.0, 0.0, 2)
    layer.self_attention.local_attn = _Core()
    return layer


@pytest.mark.parametrize("n", [0, 1, 3])
def test_a_window_of_any_size_passes(n):
    x = torch.randn(1, n, 16, requires_grad=True)
    y, _, (k, v) = _layer()(x, torch.zeros(2, 0, dtype=torch.long), "sparse")
    assert y.shape == (1, n, 16) and k.shape == v.shape == (1, n, 2, 8)
    y.sum().backward()
    assert x.grad.shape == x.shape


def test_project_views_empty_rows_as_heads():
    lins = [WgradLinear(16, 24) for _ in range(3)]
    assert [t.shape for t in project(torch.zeros(2, 0, 16), *lins, heads=4)] == [(2, 0, 4, 6)] * 3


def test_rows_without_a_batch_dimension_are_refused():
    with pytest.raises(ValueError):
        _layer()(torch.randn(3, 16), torch.zeros(2, 0, dtype=torch.long), "sparse")
