"""fp32 dense attention where its products change: fp32 MFMAs on the matrices
themselves up to 2^25 scores (2^22 at d = 64) or 128 rows on one side, bf16
pieces above."""
import math

import pytest
import torch

from neutrongt_amd import dense_attention
from tests._util import relerr

pytestmark = pytest.mark.gpu


def _run(n_q, n_k, H, d, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + n_q + d)
    q, k, v, go = (torch.randn(n, H, d, device="cuda", generator=g) for n in (n_q, n_k, n_k, n_q))
    t = [w.requires_grad_(True) for w in (q, k, v)]
    x, _ = dense_attention(*t)
    got = (x.detach(), *torch.autograd.grad(x, t, go))
    # dS = p (dP - D) keeps an error of 2^-22 |dP| where the two cancel (a query
    # with nearly all its weight on one key): so much in each row of dq and dk
    top = [w.detach().norm(dim=-1).max().item() for w in (q, k, v, go)]
    floor = 2.0 ** -22 * math.sqrt(d * H) * top[3] * top[2]
    floors = (0.0, floor * top[1] * math.sqrt(n_q), floor * top[0] * math.sqrt(n_k), 0.0)
    Q, K, V = (w.detach().double().transpose(0, 1).contiguous().requires_grad_(True) for w in t)
    y = torch.softmax((Q * math.sqrt(d)) @ K.transpose(1, 2).contiguous(), -1) @ V
    ref = (y, *torch.autograd.grad(y, (Q, K, V), go.double().transpose(0, 1).contiguous()))
    return got, [r.detach().transpose(0, 1) for r in ref], floors


# Logits of up to about d^1.5 are rounded to 24 bits and exp() turns that into a
# relative error of p: 1.5e-6 at d = 8 to 2e-5 at d = 64.
@pytest.mark.parametrize("n_q,n_k,H,d", [(2048, 2048, 8, 8), (2048, 2049, 8, 8), (1023, 1025, 32, 24),
                                         (1025, 1024, 32, 24), (724, 724, 8, 64), (724, 725, 8, 64),
                                         (1, 3, 1, 16), (4100, 33, 2, 32),
                                         # one side of 128 rows and of 129; few queries: more splits
                                         (33000, 128, 8, 24), (33000, 129, 8, 24), (128, 33000, 8, 16),
                                         (129, 33000, 8, 16), (40, 16000, 2, 32), (1000, 16000, 1, 8)])
def test_both_sides_of_the_rule(n_q, n_k, H, d):
    print(f"case dense few n_q={n_q} n_k={n_k} H={H} d={d}", flush=True)
    got, ref, floors = _run(n_q, n_k, H, d)
    for name, a, b, floor in zip(("x", "dq", "dk", "dv"), got, ref, floors):
        if n_q > 1:
            floor = 0.0  # many queries: the cancelling ones do not show
        assert (a.double() - b).norm() < (3e-7 * d + 1e-6) * b.norm() + floor, name


@pytest.mark.parametrize("tiles", [1, 2])
def test_piece_gradients_round_with_the_forward(monkeypatch, tiles):
    """The dK/dV pass's scores round as the forward's, so dV (3.2e-6 when they did
    not) has the error of the one-pass kernels, 1.3e-6, and dK 2.2e-6 (3.3e-6)."""
    monkeypatch.setenv("NGT_DENSE_F32_TILES", str(tiles))
    print(f"case dense pieces d=16 tiles={tiles}", flush=True)
    got, ref, _ = _run(406, 406, 8, 16)
    assert relerr(got[3], ref[3]) < 1.8e-6 and relerr(got[2], ref[2]) < 2.7e-6


@pytest.mark.parametrize("what,value", [("v", float("inf")), ("q", float("nan")), ("v", 3.4e38)])
def test_pieces_hand_special_values_to_the_fp32_products(monkeypatch, what, value):
    """As without pieces: finite, infinite and NaN elements are the same."""
    t = {n: torch.randn(70, 2, 8, device="cuda", generator=torch.Generator("cuda").manual_seed(i))
         for i, n in enumerate("qkv")}
    t[what][3, 1, 0] = value
    print(f"case dense pieces special {what}={value}", flush=True)
    x, _ = dense_attention(t["q"], t["k"], t["v"])
    monkeypatch.setenv("NGT_DENSE_F32_TILES", "2")
    y, _ = dense_attention(t["q"], t["k"], t["v"])
    assert torch.equal(x[:, 1].isnan(), y[:, 1].isnan())
    assert torch.equal(x[:, 1].isinf(), y[:, 1].isinf())
    assert relerr(y[:, 0], x[:, 0].double()) < 1e-6
