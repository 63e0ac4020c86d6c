"""The encoder layers' C++ autograd nodes (ngt_autograd.so) against the Python
autograd.Functions: the same casts, GEMMs and kernels in the same order, so
every output and gradient agrees bit for bit."""
import pytest
import torch

from neutrongt_amd import AdjacencyCache, _lib
from neutrongt_amd.encoder import EncoderLayer, GTEncoderLayer, WindowGraphormer
from neutrongt_amd.layernorm import FusedLayerNorm, add_dropout_layernorm
from neutrongt_amd.linear import WgradLinear, project
from tests._util import random_coo

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(monkeypatch, fn):
    """fn() through the C++ nodes and through the Python Functions."""
    out = []
    for python in (False, True):
        with monkeypatch.context() as m:
            if python:
                m.setattr(_lib, "node_ext", lambda: None)
                m.setattr(_lib, "autograd_ext", lambda: None)
            else:
                assert _lib.node_ext() is not None  # else Python would face Python
            torch.manual_seed(11)
            out.append(fn())
            torch.cuda.synchronize()
    assert len(out[0]) == len(out[1])
    for i, (a, b) in enumerate(zip(*out)):
        assert (a is None) == (b is None), i
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


def _params(mod):
    g = torch.Generator().manual_seed(5)
    with torch.no_grad():
        for p in mod.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.2)
    return mod.to(DEV).train()


@pytest.mark.parametrize("cls,n,hidden,H,dropout,ext_rows", [
    (EncoderLayer, 1, 8, 1, 0.0, 0),       # a window of one node
    (EncoderLayer, 333, 64, 8, 0.3, 0),    # one row chunk
    (EncoderLayer, 4501, 96, 4, 0.0, 90),  # row chunks and a remainder, related keys
    (GTEncoderLayer, 2100, 32, 4, 0.2, 0),
])
def test_block_matches_python_nodes(monkeypatch, cls, n, hidden, H, dropout, ext_rows):
    print(f"case {cls.__name__} n={n} hidden={hidden} H={H} p={dropout} ext={ext_rows}", flush=True)
    g = torch.Generator().manual_seed(n)
    mod = _params(cls(hidden, hidden, dropout, 0.5, H))
    x0 = torch.randn(1, n, hidden, generator=g).bfloat16().to(DEV)
    gy = torch.randn(1, n, hidden, generator=g).bfloat16().to(DEV)
    ei = torch.from_numpy(random_coo(n, n + ext_rows, 6 * n, seed=n)).to(DEV)
    ext = None
    if ext_rows:
        ext = tuple(torch.randn(ext_rows, H, hidden // H, generator=g).bfloat16().to(DEV)
                    for _ in range(2))

    def run():
        mod.self_attention.local_attn.adjacency_cache = AdjacencyCache()
        x = x0.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, score, (k, v) = mod(x, ei, "sparse", ext)
        grads = torch.autograd.grad(y, (x, *mod.parameters()), gy.to(y.dtype), allow_unused=True)
        return [y.detach(), score, k.detach(), v.detach(), *grads]

    _both(monkeypatch, run)


def test_model_matches_python_nodes(monkeypatch):
    n = 1500
    g = torch.Generator().manual_seed(2)
    model = _params(WindowGraphormer(2, 4, 100, 32, 47, attention_dropout_rate=0.5))
    x = torch.randn(n, 100, generator=g).to(DEV)
    ei = torch.from_numpy(random_coo(n, n, 5 * n, seed=8)).to(DEV)

    def run():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, scores = model(x, ei)
        return [y.detach(), *scores, *torch.autograd.grad(y.square().sum(), model.parameters())]

    _both(monkeypatch, run)


def test_parts_of_the_gradients_match_python_nodes(monkeypatch):
    """Unused outputs, frozen inputs, layers without a bias, strided and
    misaligned operands, an unused sum or norm."""
    g = torch.Generator().manual_seed(9)
    lins = [_params(WgradLinear(16, w, bias=b)) for w, b in ((24, True), (24, False), (8, True))]
    ln = _params(FusedLayerNorm(16))
    drop = torch.nn.Dropout(0.4)
    wide = torch.randn(3, 40, 33, generator=g).to(DEV)

    def run():
        res = []
        for x0 in (wide[..., 1:17], wide[0, :, :16].bfloat16()):
            for need in (True, False):
                x = x0.detach().requires_grad_(need)
                with torch.autocast("cuda", dtype=torch.bfloat16):
                    for used in ((0, 1, 2), (2,), (0, 1)):
                        ys = project(x, *lins)
                        loss = sum(ys[i].float().square().sum() for i in used)
                        ps = [p for l in lins for p in l.parameters()] + ([x] if need else [])
                        res += torch.autograd.grad(loss, ps, allow_unused=True)
                    ys = project(x, *lins, heads=8)
                    res += [y.detach() for y in ys]
                    y = lins[0](x)
                    res += [y.detach(), *torch.autograd.grad(
                        y[..., ::2].float().sum(), [lins[0].bias] + ([x] if need else []))]
                    z = ln(x)
                    res += [z.detach(), *torch.autograd.grad(z.sum(), [ln.weight])]
                    other = torch.ones_like(x).requires_grad_(True)
                    for pick in (0, 1):
                        out = add_dropout_layernorm(x, other, ln, drop)
                        res += [o.detach() for o in out]
                        res += torch.autograd.grad(out[pick].double().square().sum(),
                                                   [other] + ([ln.bias] if pick else []))
        return res

    _both(monkeypatch, run)


def test_the_layers_run_as_cpp_nodes():
    """Under bf16 autocast every layer's output comes from a C++ node."""
    print("case cpp nodes", flush=True)
    lins, ln = [_params(WgradLinear(16, 16)) for _ in range(3)], _params(FusedLayerNorm(16))
    x = torch.randn(1, 5, 16, device=DEV, requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        outs = [lins[0](x), *project(x, *lins, heads=2), ln(x),
                *add_dropout_layernorm(x, x, ln, torch.nn.Dropout(0.5))]
    for y, node in zip(outs, ["Linear"] + 3 * ["Projection3"] + ["LayerNorm"] + 2 * ["AddLayerNorm"]):
        name = y.grad_fn.name()
        assert "CppNode" in name and node in name, name


@pytest.mark.parametrize("python", [False, True])
def test_batched_gradients_of_layers_without_a_bias(monkeypatch, python):
    """torch.autograd.grad(is_grads_batched=True): weight and input gradients over a
    batch of output gradients, as one at a time."""
    print(f"case batched gradients python={python}", flush=True)
    if python:
        monkeypatch.setattr(_lib, "node_ext", lambda: None)
    lins = [_params(WgradLinear(16, 24, bias=False)) for _ in range(3)]
    x = torch.randn(50, 16, device=DEV, requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y, ys = lins[0](x), project(x, *lins)
    for out, ins in ((y, [x, lins[0].weight]), (ys[1], [x, lins[1].weight])):
        g = torch.randn(3, *out.shape, device=DEV).bfloat16()
        got = torch.autograd.grad(out, ins, g, is_grads_batched=True, retain_graph=True)
        for i in range(3):
            for a, b in zip(got, torch.autograd.grad(out, ins, g[i], retain_graph=True)):
                assert (a[i].double() - b.double()).norm() <= 2e-3 * b.double().norm()
