"""GPU tests of ngt_wgrad_bf16: dW = dY^T X and db = column sums of dY of a
bf16 linear layer from one pass over its rows.

The bf16 products are exact in fp32, so the only error is that of fp32 sums:
at most 2,560 terms in a chain and then the splits, below 1e-6 in the 2-norm."""
import pytest
import torch

from neutrongt_amd import _lib
from neutrongt_amd.linear import (WgradLinear, _fused, _grads, _library_weight_grad, colsum_bf16,
                                  linear_grads)
from tests._util import relerr

pytestmark = pytest.mark.gpu


# rows around a stage (64 and 128), a split and the chain limit; widths around the
# 8-column patches, both tiles and the narrowest (below 8: two-byte loads)
@pytest.mark.parametrize("K,n_out,n_in", [
    (0, 8, 8), (1, 1, 1), (3, 7, 9), (63, 64, 64), (64, 65, 65), (65, 128, 129), (127, 47, 64),
    (129, 64, 47), (257, 130, 100), (1000, 6, 768), (2561, 128, 128), (10007, 192, 64),
    (5121, 257, 72), (3000, 2304, 768), (131072 * 3 + 5, 9, 17)])
def test_wgrad_matches_fp64(K, n_out, n_in):
    print(f"case wgrad K={K} n_out={n_out} n_in={n_in}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + 3 * n_out + n_in)
    x = torch.randn(K, n_in, device="cuda", generator=g).to(torch.bfloat16)
    dy = torch.randn(K, n_out, device="cuda", generator=g).to(torch.bfloat16)
    dw, db = linear_grads(x, dy, True)
    assert dw.shape == (n_out, n_in) and dw.dtype == db.dtype == torch.float32
    if K == 0:
        assert not dw.any() and not db.any()
        return
    assert relerr(dw, dy.double().t() @ x.double()) < 1e-6
    assert relerr(db, dy.double().sum(0)) < 1e-6
    again, none = linear_grads(x, dy, False)
    assert none is None and torch.equal(again, dw)  # a fixed order, with the bias or without


@pytest.mark.parametrize("n_out,n_in", [(64, 64), (47, 100), (136, 256), (5, 3)])
def test_any_two_byte_alignment_gives_the_same_bits(n_out, n_in):
    print(f"case wgrad alignment {n_out} {n_in}", flush=True)
    K = 300
    g = torch.Generator(device="cuda").manual_seed(n_out)
    flat = torch.randn(2, K * 256 + 8, device="cuda", generator=g).to(torch.bfloat16)
    x, dy = flat[0, 1:1 + K * n_in].view(K, n_in), flat[1, 3:3 + K * n_out].view(K, n_out)
    assert x.data_ptr() % 4 == 2
    a, b = linear_grads(x, dy, True), linear_grads(x.clone(), dy.clone(), True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_infinities_and_nan_stay_in_their_row_and_column():
    print("case wgrad special values", flush=True)
    K, n_out, n_in = 500, 47, 70
    x = torch.ones(K, n_in, device="cuda", dtype=torch.bfloat16)
    dy = torch.ones(K, n_out, device="cuda", dtype=torch.bfloat16)
    x[7, 69], dy[499, 46] = float("inf"), float("nan")
    dw, db = linear_grads(x, dy, True)
    ref = dy.double().t() @ x.double()
    assert torch.equal(dw.isnan(), ref.isnan()) and torch.equal(dw.isinf(), ref.isinf())
    assert db[:46].eq(K).all() and db[46].isnan()


@pytest.mark.parametrize("K,n_out,n_in,fused", [
    (1999, 1536, 768, False), (2000, 1536, 768, True), (1000, 768, 768, True),
    (32768, 768, 768, False), (16000, 2304, 768, True), (24000, 2304, 768, False),
    (4000, 3072, 1024, False), (32768, 47, 768, True), (131072, 47, 768, False)])
def test_both_routes_agree_at_the_rule(K, n_out, n_in, fused):
    print(f"case wgrad rule {K} {n_out} {n_in}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(K, n_in, device="cuda", generator=g).to(torch.bfloat16)
    dy = torch.randn(K, n_out, device="cuda", generator=g).to(torch.bfloat16)
    with torch.no_grad():
        assert _fused(x, dy) == fused
        dw, db = _grads(x, dy, True, True)
        assert relerr(dw, _library_weight_grad(x, dy).double()) < 2e-6
        assert relerr(db, colsum_bf16(dy).double()) < 2e-6
    # the layer's node takes the same route
    lin = WgradLinear(n_in, n_out).cuda()
    assert _lib.node_ext() is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = lin(x)
    gw, gb = torch.autograd.grad(y, (lin.weight, lin.bias), dy)
    assert torch.equal(gw, dw) and torch.equal(gb, db)
