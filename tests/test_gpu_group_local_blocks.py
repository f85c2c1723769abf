"""Grouped GEMMs with every rank's rows at hand: row blocks without rank segments, walked several at a time, against the
fp32 oracle (exact on integer-valued inputs) and against the flag-gated form in segmented blocks."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu


def _case(world, mpr, K, N, E, topk, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    shards = [torch.randint(-2, 3, (mpr, K), generator=g).float().to(dtype) for _ in range(world)]
    w = torch.randint(-2, 3, (E, K, N), generator=g).float().to(dtype)
    return shards, w, golden.random_distinct_experts(world * mpr, E, topk, g)


def _context(cuda, shards, w, ids, rank, E):
    from triton_dist.kernels.amd import create_ag_group_gemm_intra_node_context
    a, b = shards[rank].to(cuda), w.to(cuda)
    ctx = create_ag_group_gemm_intra_node_context(None, a, b, ids.to(cuda), E, max_M=len(shards) * a.shape[0], rank=rank,
                                                  num_ranks=len(shards))
    ctx.set_peer_shards({r: s.to(cuda) for r, s in enumerate(shards) if r != rank})
    ctx.workspace_tensors[rank].view(torch.uint8).fill_(0x7B)   # stale rows must never reach C
    return ctx, a, b


# one entry; blocks of one row; 129 rows for one expert; columns that end inside a tile, are no multiple of 8 and span more
# than one XCD's worth of tiles; last groups of one to three row blocks; a ragged K, one K tile, no whole 64 bytes of K
@pytest.mark.parametrize("block", [128, 256])
@pytest.mark.parametrize("dtype,world,mpr,K,N,E,topk", [
    (torch.bfloat16, 2, 1, 256, 256, 4, 1), (torch.bfloat16, 2, 3, 192, 264, 64, 2), (torch.float16, 3, 43, 256, 40, 1, 1),
    (torch.bfloat16, 4, 150, 512, 2312, 6, 3), (torch.float16, 4, 301, 200, 4100, 5, 2), (torch.float8_e4m3fn, 4, 130, 384, 1288, 7, 2),
    (torch.float8_e4m3fn, 8, 96, 208, 8200, 3, 2), (torch.bfloat16, 2, 257, 64, 520, 4, 2), (torch.bfloat16, 2, 64, 40, 136, 4, 2)])
def test_exact_and_like_the_gated_form(cuda, monkeypatch, block, dtype, world, mpr, K, N, E, topk):
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, allgather_group_gemm
    announce("local blocks %s block %d W=%d m=%d K=%d N=%d E=%d topk=%d" % (dtype, block, world, mpr, K, N, E, topk))
    monkeypatch.setattr(allgather_group_gemm, "_row_block", lambda *a: block)
    shards, w, ids = _case(world, mpr, K, N, E, topk, dtype, seed=K + N)
    ctx, a, b = _context(cuda, shards, w, ids, world - 1, E)
    esz = a.element_size()
    if K * esz % 64 != 0 and K * esz <= 128:
        from triton_dist import _lib
        with pytest.raises(_lib.TdistError):   # refused in either form
            ag_group_gemm_intra_node(a, b, ctx)
        return
    c = ag_group_gemm_intra_node(a, b, ctx)
    ctx.check_status()
    want = golden.ag_group_gemm_fp32(shards, w, ids)
    assert torch.equal(c.float().cpu(), want.to(c.dtype).float())
    ctx.local_blocks = None
    ctx.workspace_tensors[world - 1].view(torch.uint8).fill_(0x11)
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx), c)
    ctx.check_status()


def test_routing_changed_in_the_context_and_shards_off_16_bytes(cuda):
    """Blocks that no longer stand for the context's routing, and shards the gather does not take, go through the flags."""
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, sort_topk_ids_align_block_size
    announce("local blocks given up")
    world, mpr, K, N, E, topk, rank = 2, 70, 256, 264, 4, 2, 0
    shards, w, ids = _case(world, mpr, K, N, E, topk, torch.bfloat16, seed=3)
    ctx, a, b = _context(cuda, shards, w, ids, rank, E)
    other = golden.random_distinct_experts(world * mpr, E, topk, torch.Generator().manual_seed(8))
    new = sort_topk_ids_align_block_size(other.to(cuda), E, world, mpr, ctx.BLOCK_M)
    ctx.sorted_topk_ids, ctx.aligned_expert_ids, ctx.aligned_barrier_ids, ctx.rank_block_num, ctx.aligned_num_tokens = new
    want = golden.ag_group_gemm_fp32(shards, w, other).bfloat16()
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), want)
    ctx, a, b = _context(cuda, shards, w, ids, rank, E)
    for t, src in zip((ctx.sorted_topk_ids, ctx.aligned_expert_ids, ctx.aligned_barrier_ids, ctx.aligned_num_tokens),
                      (new[0], new[1], new[2], new[4])):
        t.copy_(src)                                                           # in place
    ctx.first_block = 0
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), want)
    ctx, a, b = _context(cuda, shards, w, ids, rank, E)
    off = torch.empty(mpr * K + 4, dtype=torch.bfloat16, device=cuda)[4:].view(mpr, K)   # 8 bytes past a boundary
    off.copy_(shards[1].to(cuda))
    ctx.set_peer_shards({1: off})
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), golden.ag_group_gemm_fp32(shards, w, ids).bfloat16())
    ctx.check_status()
