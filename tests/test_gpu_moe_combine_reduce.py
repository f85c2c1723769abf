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


def _layer(cuda, mpr=3, world=2, hidden=264):
    from triton_dist.kernels.amd import create_moe_rs_context
    g = torch.Generator().manual_seed(mpr)
    logits = [torch.randn((mpr, 4), generator=g).to(cuda) for _ in range(world)]
    ctx = create_moe_rs_context(None, 0, world, world, world * mpr, hidden, 4, 2, torch.bfloat16, torch.bfloat16, cuda, 128, logits[0], {1: logits[1]})
    ctx.set_peer_partials({1: torch.randn((mpr, hidden), generator=g).to(cuda)})
    a = torch.randn((world * mpr * 2, 192), generator=g).bfloat16().to(cuda)
    return ctx, a, torch.randn((4, 192, hidden), generator=g).bfloat16().to(cuda)


def test_what_the_layer_refuses_of_a_context(cuda):
    """Buffers that the one launch cannot take, as the copy into a slice and the reduction behind it refused them."""
    from triton_dist.kernels.amd import moe_reduce_rs
    announce("moe reduce-rs: replaced buffers and types")
    for make in (lambda b: torch.zeros((b.shape[0], b.shape[1] + 8), dtype=b.dtype, device=b.device)[:, :-8], lambda b: b[:-1]):
        ctx, a, b = _layer(cuda)
        ctx.rs_buffers[0] = make(ctx.rs_buffers[0])
        with pytest.raises(NotImplementedError):
            moe_reduce_rs(0, 2, 2, a, b, ctx)
    ctx, a, b = _layer(cuda)
    with pytest.raises(TypeError):
        moe_reduce_rs(0, 2, 2, a.float(), b.float(), ctx)


def test_a_world_that_does_not_divide_the_tokens(cuda):
    """Whole slices are reduced; the tokens behind them are nobody's."""
    from triton_dist.kernels.amd import moe_reduce_rs, moe_weighted_combine
    from triton_dist.kernels.amd.gemm_reduce_scatter import ring_reduce_after_scatter
    announce("moe reduce-rs: 6 tokens by 4 ranks")
    ctx, a, b = _layer(cuda)
    for rank in (0, 3):
        partials = ctx.rs_buffers[0].normal_().clone()
        got = moe_reduce_rs(rank, 4, 4, a, b, ctx)
        index = torch.arange(12, dtype=torch.int32, device=cuda).view(6, 2)
        y = moe_weighted_combine(None, ctx.final_output_buffer[:12], None, index, ctx.topk_weight_f32, from_slots=False)
        partials[rank] = y[rank]
        assert got.shape == (1, 264) and torch.equal(got, ring_reduce_after_scatter(rank, 4, partials[:4], None))
