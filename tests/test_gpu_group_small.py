"""The grouped GEMM on the small tiles: blocks of 64 and 128 rows with 128 columns, whole or in pieces of K, exactly as the oracle has
it (whole numbers small enough for every sum); and the large tiles in the blocks that are chosen where no estimate has them."""
import pytest
import torch

from oracle import golden
from tests import test_gpu_group_local_blocks as local_blocks
from tests.conftest import announce

pytestmark = pytest.mark.gpu


# one row; fewer rows than experts; one to three blocks an expert with a row more and less than a block; columns that end inside a
# tile, are no multiple of 8 and span several XCDs' tiles; a ragged K, less than one K tile, more pieces of K than K tiles
@pytest.mark.parametrize("dtype,world,mpr,K,N,E,topk", [
    (torch.bfloat16, 2, 1, 256, 256, 4, 1), (torch.bfloat16, 2, 3, 1192, 264, 64, 2), (torch.float16, 3, 43, 256, 40, 1, 1),
    (torch.bfloat16, 2, 64, 72, 136, 1, 1), (torch.float16, 2, 65, 2048, 1288, 2, 2), (torch.bfloat16, 4, 150, 1024, 2312, 6, 3),
    (torch.float8_e4m3fn, 4, 130, 1040, 1288, 7, 2), (torch.float8_e4m3fn, 2, 5, 4096, 513, 3, 2), (torch.float16, 16, 2, 520, 4100, 5, 4)])
@pytest.mark.parametrize("tile", [5, 6])
@pytest.mark.parametrize("pieces", [None, 0, 2, 8])
def test_small_tiles_exact(cuda, tile, pieces, dtype, world, mpr, K, N, E, topk):
    from triton_dist import _lib
    from triton_dist.kernels.amd import ag_group_gemm_intra_node
    announce("grouped small %s tile %d pieces %s W=%d m=%d K=%d N=%d E=%d topk=%d" % (dtype, tile, pieces, world, mpr, K, N, E, topk))
    shards, w, ids = local_blocks._case(world, mpr, K, N, E, topk, dtype, seed=K + N)
    ctx, a, b = local_blocks._context(cuda, shards, w, ids, world - 1, E)
    with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, tile), _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_SPLIT_K, pieces):
        c = [ag_group_gemm_intra_node(a, b, ctx) for _ in range(2)]
    ctx.check_status()
    assert {blocks.block_size for blocks in ctx.joined.values()} == {64 if tile == 5 else 128}
    want = golden.ag_group_gemm_fp32(shards, w, ids).to(c[0].dtype).float()
    for got in c:   # (the second on the counters that the first left behind)
        assert torch.equal(got.float().cpu(), want)


# experts of enough row blocks that an XCD goes down 2, 4 and 8 of them before the next column, the last group shorter
@pytest.mark.parametrize("mpr,E", [(141, 1), (600, 1), (600, 2), (601, 3)])
@pytest.mark.parametrize("tile", [5, 6])
def test_walk_down_several_row_blocks(cuda, tile, mpr, E):
    test_small_tiles_exact(cuda, tile, None, torch.bfloat16, 4, mpr, 256, 1288, E, 1)


@pytest.mark.parametrize("block", [128, 256])
@pytest.mark.parametrize("dtype,world,mpr,K,N,E,topk", [(torch.bfloat16, 4, 150, 512, 2312, 6, 3), (torch.float16, 2, 3, 192, 264, 64, 2),
                                                        (torch.float8_e4m3fn, 8, 96, 208, 8200, 3, 2)])
def test_large_tiles_in_blocks_without_an_estimate(cuda, monkeypatch, block, dtype, world, mpr, K, N, E, topk):
    from triton_dist.kernels.amd import allgather_group_gemm
    monkeypatch.setattr(allgather_group_gemm, "_block_plan", lambda *_: None)
    local_blocks.test_exact_and_like_the_gated_form(cuda, monkeypatch, block, dtype, world, mpr, K, N, E, topk)


def test_what_the_small_blocks_refuse(cuda):
    """Blocks of 64 rows are for calls without flags: the gated entry points refuse them as before."""
    from triton_dist import _lib
    from triton_dist.kernels.amd import allgather_group_gemm as g
    from triton_dist.kernels.amd import sort_topk_ids_align_block_size
    ids = torch.randint(0, 4, (64, 1), device=cuda)
    a, b, c = torch.zeros((64, 256), dtype=torch.bfloat16, device=cuda), torch.zeros((4, 256, 256), dtype=torch.bfloat16, device=cuda), torch.zeros(
        (64, 256), dtype=torch.bfloat16, device=cuda)
    rows, experts, segments, _, padded = sort_topk_ids_align_block_size(ids, 4, 1, 64, 64)
    with pytest.raises(_lib.TdistError):
        g.group_gemm_gated(a, None, 0, b, c, rows, experts, segments, padded, 64, 64, 1, 64, 0, None, 0)
    lib = _lib.load()
    assert lib.tdist_group_gemm_row_block(0, 4, 256, 512, 0) == 0
    # from few rows to many the block only grows
    sizes = [lib.tdist_group_gemm_row_block(n, 8, 4096, 4096, 1 << 26) for n in (1, 64, 512, 2048, 16384)]
    assert sizes == sorted(sizes) and sizes[0] == 64 and sizes[-1] == 256
