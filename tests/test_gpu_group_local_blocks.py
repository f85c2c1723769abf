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
    from triton_dist import _lib
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, allgather_group_gemm
    announce("local blocks %s block %d W=%d m=%d K=%d N=%d E=%d topk=%d" % (dtype, block, world, mpr, K, N, E, topk))
    monkeypatch.setattr(allgather_group_gemm, "_join_plan", lambda n, e, _: (block, (n + e * (block - 1)) // block))
    shards, w, ids = _case(world, mpr, K, N, E, topk, dtype, seed=K + N)
    ctx, a, b = _context(cuda, shards, w, ids, world - 1, E)
    esz = a.element_size()
    if K * esz % 64 != 0 and K * esz <= 128:
        with pytest.raises(_lib.TdistError):   # refused in either form
            ag_group_gemm_intra_node(a, b, ctx)
        return
    with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, 0 if block == 256 else 4):   # (the large tile of so many rows)
        c = ag_group_gemm_intra_node(a, b, ctx)
    ctx.check_status()
    assert {blocks.block_size for blocks in ctx.joined.values()} == {block}
    want = golden.ag_group_gemm_fp32(shards, w, ids)
    assert torch.equal(c.float().cpu(), want.to(c.dtype).float())
    ctx.gather_rows = False
    ctx.workspace_tensors[world - 1].view(torch.uint8).fill_(0x11)
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx), c)
    ctx.check_status()


def test_routing_changed_in_the_context_and_shards_off_16_bytes(cuda):
    """Blocks are joined from what the context holds when the call runs: replaced, rewritten in place, rewritten through the
    C entry point, or with the experts of the blocks alone exchanged. Shards the gather does not take go through the flags."""
    from triton_dist import _lib
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, sort_topk_ids_align_block_size
    announce("joined blocks of another routing")
    world, mpr, K, N, E, topk, rank = 2, 70, 256, 264, 4, 2, 0
    shards, w, ids = _case(world, mpr, K, N, E, topk, torch.bfloat16, seed=3)
    ctx, a, b = _context(cuda, shards, w, ids, rank, E)
    other = golden.random_distinct_experts(world * mpr, E, topk, torch.Generator().manual_seed(8))
    other_d = other.to(cuda)
    new = sort_topk_ids_align_block_size(other_d, E, world, mpr, ctx.BLOCK_M)
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
    ws = _lib.zeroed_scratch(_lib.load().tdist_moe_align_workspace_bytes(other.numel(), E, world), cuda)
    _lib.call("tdist_moe_align_block_size", other_d.data_ptr(), 0 if other_d.dtype == torch.int32 else 1, other.numel(), E, world,
              mpr * topk, ctx.BLOCK_M, ctx.sorted_topk_ids.data_ptr(), ctx.sorted_topk_ids.numel(), ctx.aligned_expert_ids.data_ptr(),
              ctx.aligned_barrier_ids.data_ptr(), ctx.rank_block_num.data_ptr(), ctx.aligned_num_tokens.data_ptr(), ws.data_ptr(),
              ws.numel(), _lib.stream_ptr())                                   # by pointer: no version counter sees it
    ctx.first_block = 0
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), want)
    for by_replacing in (True, False):
        ctx, a, b = _context(cuda, shards, w, ids, rank, E)
        if by_replacing:
            ctx.aligned_expert_ids = (ctx.aligned_expert_ids + 1) % E          # every block to the next expert
        else:
            ctx.aligned_expert_ids.add_(1).remainder_(E)
        assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), golden.ag_group_gemm_fp32(shards, w, (ids + 1) % E).bfloat16())
    ctx, a, b = _context(cuda, shards, w, ids, rank, E)
    off = torch.empty(mpr * K + 4, dtype=torch.bfloat16, device=cuda)[4:].view(mpr, K)   # 8 bytes past a boundary
    off.copy_(shards[1].to(cuda))
    ctx.set_peer_shards({1: off})
    assert torch.equal(ag_group_gemm_intra_node(a, b, ctx).cpu(), golden.ag_group_gemm_fp32(shards, w, ids).bfloat16())
    ctx.check_status()


def test_contexts_made_in_inference_mode_and_rerouted_between_replays(cuda):
    """Both halves of the layer with contexts made under torch.inference_mode (whose tensors count no versions), captured, and
    replayed after the routing's tensors have been rewritten."""
    from triton_dist.kernels.amd import (ag_group_gemm_intra_node, create_moe_rs_context, moe_reduce_rs,
                                         sort_topk_ids_align_block_size)
    announce("joined blocks, inference mode and graph")
    world, mpr, K, N, E, topk, rank = 2, 70, 256, 264, 4, 2, 1
    shards, w, ids = _case(world, mpr, K, N, E, topk, torch.bfloat16, seed=5)
    H = 256
    g = torch.Generator().manual_seed(6)
    down = torch.randint(-1, 2, (E, N, H), generator=g).bfloat16()
    down_d = down.to(cuda).transpose(1, 2).contiguous().transpose(1, 2)
    logits = [torch.randn((mpr, E), generator=g).to(cuda) for _ in range(world)]
    with torch.inference_mode():
        w_kn = w.transpose(1, 2).contiguous().transpose(1, 2)   # contiguous along K: read as it lies
        ctx, a, _ = _context(cuda, shards, w, ids, rank, E)
        b = w_kn.to(cuda)
        assert b.stride(1) == 1
        rs = create_moe_rs_context(None, rank, world, world, world * mpr, H, E, topk, torch.bfloat16, torch.bfloat16, cuda, 128,
                                   logits[rank], {0: logits[0]})
        rs.topk_weight_f32.fill_(1.0)
        pre = rs.precompute_ctx
        stream = torch.cuda.Stream()
        ctx.group_gemm_stream = None
        ag_group_gemm_intra_node(a, b, ctx)   # (sizes, LDS reservations)
        moe_reduce_rs(rank, world, world, torch.zeros((world * mpr * topk, N), dtype=torch.bfloat16, device=cuda), down_d, rs)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            h = ag_group_gemm_intra_node(a, b, ctx)
            y = moe_reduce_rs(rank, world, world, h, down_d, rs)
        for seed in (11, 12):
            other = golden.random_distinct_experts(world * mpr, E, topk, torch.Generator().manual_seed(seed))
            new = sort_topk_ids_align_block_size(other.to(cuda), E, world, mpr, 128)
            for t, src in zip((ctx.sorted_topk_ids, ctx.aligned_expert_ids, ctx.aligned_num_tokens), (new[0], new[1], new[4])):
                t.copy_(src)
            for t, src in zip((pre.full_sorted_token_ids, pre.full_token_expert_ids, pre.full_num_tokens_post_padded_list), (new[0], new[1], new[4])):
                t.copy_(src)
            graph.replay()
            torch.cuda.synchronize()
            up = golden.ag_group_gemm_fp32(shards, w, other).bfloat16()
            assert torch.equal(h.cpu(), up)
            flat = other.reshape(-1)
            rows = torch.stack([up[i].float() @ down[flat[i]].float() for i in range(flat.numel())]).bfloat16().float()
            sums = rows.view(-1, topk, H).sum(1)[rank * mpr:(rank + 1) * mpr].bfloat16()   # (the other rank's partial is zero)
            assert torch.equal(y.cpu(), sums)


# one entry; blocks that are full, short and of one row; an expert without rows; more experts than entries; a block size that is
# no whole number of waves; more blocks than waves in the grid; experts that come back in a later block
@pytest.mark.parametrize("entries,E,world,block,out_block", [(2, 4, 1, 128, 128), (1000, 3, 4, 128, 256), (3000, 7, 4, 128, 192), (20000, 7, 4, 128, 192), (64, 40, 2, 128, 128), (4000, 64, 8, 128, 256),
                                                             (640, 5, 2, 96, 128), (20000, 9, 8, 32, 256), (300, 512, 4, 256, 128)])
def test_joined_blocks_are_the_sort_without_segments(cuda, monkeypatch, entries, E, world, block, out_block):
    from triton_dist import _lib
    from triton_dist.kernels.amd import allgather_group_gemm as g, sort_topk_ids_align_block_size
    announce("join blocks of %d entries, %d experts, %d segments, %d -> %d rows" % (entries, E, world, block, out_block))
    monkeypatch.setattr(g, "_join_plan", lambda n, e, _: (out_block, (n + e * (out_block - 1)) // out_block))
    gen = torch.Generator().manual_seed(entries)
    ids = torch.randint(0, E, (entries, 1), generator=gen, dtype=torch.int32).to(cuda)
    ids[:entries // 3] = int(ids[0])   # a crowded expert
    sorted_ids, experts, _, _, padded = sort_topk_ids_align_block_size(ids, E, world, entries // world, block)
    def join():
        blocks = g.joined_row_blocks({}, sorted_ids, experts, padded, block, entries, E, 256, 256, _lib.stream_ptr())
        assert blocks.block_size == out_block
        n = blocks.num_blocks
        return blocks.memory.split((n * out_block, n, n, 1))
    got = join()
    want = sort_topk_ids_align_block_size(ids, E, 1, entries, out_block)
    total = int(want[4])
    assert int(got[3]) == total
    assert torch.equal(got[0][:total], want[0][:total]) and torch.equal(got[1][:total // out_block], want[1][:total // out_block])
    assert int(got[2][:total // out_block].abs().sum()) == 0
    # blocks in another order, each with its expert: the same sets, experts in order
    used = int(padded) // block
    order = torch.randperm(used, generator=gen).to(cuda)
    sorted_ids[:used * block] = sorted_ids[:used * block].view(used, block)[order].view(-1)
    experts[:used] = experts[:used][order]
    moved = join()
    assert int(moved[3]) == total and torch.equal(moved[1][:total // out_block], got[1][:total // out_block])
    for e in range(E):
        pick = got[1][:total // out_block] == e
        assert torch.equal(moved[0][:total].view(-1, out_block)[pick].reshape(-1).sort().values, got[0][:total].view(-1, out_block)[pick].reshape(-1).sort().values)


def test_what_the_join_refuses(cuda):
    from triton_dist import _lib
    lib = _lib.load()
    p = torch.zeros(64, dtype=torch.int32, device=cuda).data_ptr()
    call = lambda blocks, size, experts: lib.tdist_moe_join_blocks(p, p, p, blocks, size, 4, experts, 128, p, 128, p, p, p, None)
    assert call(1, 513, 4) == call(1, 128, 4097) == call(50000, 128, 4) == _lib.TDIST_ERR_UNSUPPORTED
    assert call(0, 128, 4) == call(1, 0, 4) == call(1, 128, 0) == _lib.TDIST_ERR_INVALID
