"""The top-k sum with the reduction over the ranks behind it, against the same steps one by one: the same bits."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


# one rank, one token; more ranks than loads in flight and a remainder of them; one to 32 rows a token; a piece of a window, a
# window and a piece, several
@pytest.mark.parametrize("W,m,topk,hidden", [(1, 1, 1, 8), (1, 5, 9, 520), (2, 3, 2, 512), (4, 1, 4, 1032), (8, 33, 8, 4096), (9, 7, 17, 264), (16, 2, 32, 1544)])
def test_like_the_steps_one_by_one(cuda, W, m, topk, hidden):
    from triton_dist import _lib
    from triton_dist.kernels.amd import moe_weighted_combine
    from triton_dist.kernels.amd.gemm_reduce_scatter import ring_reduce_after_scatter
    announce("combine and reduce W=%d m=%d topk=%d hidden=%d" % (W, m, topk, hidden))
    g = torch.Generator(device="cuda").manual_seed(W * hidden + topk)
    M = W * m
    rows = torch.randn((M * topk, hidden), generator=g, device=cuda).to(torch.bfloat16)
    weight = torch.rand((M, topk), generator=g, device=cuda)
    peers = torch.randn((M, hidden), generator=g, device=cuda).to(torch.bfloat16)
    index = torch.arange(M * topk, dtype=torch.int32, device=cuda).view(M, topk)
    y = moe_weighted_combine(None, rows, None, index, weight, from_slots=False)
    for rank in {0, W // 2, W - 1}:
        partials, sums, out = peers.clone(), torch.full_like(y, -3.0), torch.empty((m, hidden), dtype=torch.bfloat16, device=cuda)
        _lib.call("tdist_moe_combine_reduce", rows.data_ptr(), weight.data_ptr(), M, topk, hidden, rank, W, partials.data_ptr(), sums.data_ptr(),
                  out.data_ptr(), _lib.stream_ptr())
        own = slice(rank * m, (rank + 1) * m)
        want = peers.clone()
        want[own] = y[own]
        assert torch.equal(partials, want)
        assert torch.equal(out, ring_reduce_after_scatter(rank, W, want, None))
        want = y.clone()
        want[own] = -3.0
        assert torch.equal(sums, want)
