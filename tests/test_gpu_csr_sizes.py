"""GPU tests of the window CSR build where its sorts change: the merge sort below
16,384 edges, small radix tiles up to 1,200,000, large ones above, merge sorts
under graph capture, and one sort by (dst, src) where both fit 32 bits."""
import ctypes as C

import numpy as np
import pytest
import torch

from neutrongt_amd import WindowAdjacency, _lib
from oracle import graph as OG

pytestmark = pytest.mark.gpu


def _edges(n_q, n_k, E, seed):
    rng = np.random.default_rng(seed)
    return np.stack([(rng.random(E) ** 3 * n_k).astype(np.int64), rng.integers(0, n_q, E)])


def _check(adj, ei, n_q, n_k, chunk, small):
    ref = OG.csr_from_coo(ei[0], ei[1], n_q, n_k)
    for name, want in ref.items():
        np.testing.assert_array_equal(getattr(adj, name).cpu().numpy()[: want.shape[0]], want, name)
    oq, ok = OG.row_orders(ref["rowptr"], ref["t_rowptr"], n_q, n_k)
    np.testing.assert_array_equal(adj.order_q.cpu().numpy()[: oq.shape[0]], oq)
    np.testing.assert_array_equal(adj.order_k.cpu().numpy()[: ok.shape[0]], ok)
    for side, rp in (("q", ref["rowptr"]), ("k", ref["t_rowptr"])):
        for kind, want in zip(("items_", "splits_", "packed_"), OG.work_items(rp, chunk, small)):
            got = getattr(adj, kind + side).cpu().numpy()[: want.shape[0]]
            np.testing.assert_array_equal(got, want, kind + side)


@pytest.mark.parametrize("n_q,n_k,E", [(3000, 3000, 16384), (3000, 3000, 16385), (257, 4000, 20481),
                                       (4000, 257, 262144), (32768, 32768, 1200000),
                                       (32768, 40000, 1200001), (65535, 65535, 70000),
                                       (65535, 65536, 70000), (1, 90000, 30000)])
def test_csr_at_the_sorts_edges(n_q, n_k, E):
    print(f"case csr n_q={n_q} n_k={n_k} E={E}", flush=True)
    ei = _edges(n_q, n_k, E, E)
    _check(WindowAdjacency(torch.from_numpy(ei).cuda(), n_q, n_k, 128, 16), ei, n_q, n_k, 128, 16)


@pytest.mark.parametrize("n_q,n_k,E", [(2000, 2300, 50000), (600000, 600001, 50000)])
def test_csr_build_replayed_from_a_graph(n_q, n_k, E):
    """Each replay rebuilds the arrays from the edges that the buffer holds then;
    the second case's row sort, both sides together, is longer than 1,048,576."""
    chunk, small = 128, 16
    print(f"case csr captured n_q={n_q} n_k={n_k} E={E}", flush=True)
    buf = torch.from_numpy(_edges(n_q, n_k, E, 0)).cuda()
    adj = WindowAdjacency(buf.clone(), n_q, n_k, chunk, small)
    lib, nb = _lib.load(), C.c_size_t()
    _lib.check(lib.ngt_csr_workspace_bytes(E, n_q, n_k, C.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        _lib.check(lib.ngt_csr_build(buf.data_ptr(), adj.ptr(), ws.data_ptr(), nb.value,
                                     _lib.stream_ptr(buf.device)))
    for seed in range(1, 5):
        ei = _edges(n_q, n_k, E, seed)
        buf.copy_(torch.from_numpy(ei))
        adj.mem.fill_(-7)
        ws.fill_(0xEE)
        graph.replay()
        torch.cuda.synchronize()
        _check(adj, ei, n_q, n_k, chunk, small)
