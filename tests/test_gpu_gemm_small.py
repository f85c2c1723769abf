"""The GEMM tiles for shapes that do not fill the chip (64 x 128 and 128 x 128, several workgroups to a tile along K) and
the first K tile of the large ones where K is no whole number of 128 bytes: exact on integer-valued inputs, at edges of
tiles and of K, from operands whose every byte around the rows is a NaN."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


def poisoned(rows, k, dtype, g, cuda):
    """[rows, k] integer-valued, a view of a tensor whose other elements are NaN."""
    full = torch.full((rows + 2, k + 64), float("nan"))
    full[1:-1, :k] = torch.randint(-2, 3, (rows, k), generator=g).float()
    return full.to(dtype).to(cuda)[1:-1, :k]


@pytest.mark.parametrize("tile,pieces", [(5, 1), (5, 2), (5, 8), (5, 16), (6, 1), (6, 4), (0, 0), (1, 0), (2, 0), (3, 0), (4, 0), (0, 1), (4, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
def test_each_tile_with_ragged_k(cuda, switches, dtype, tile, pieces):
    from triton_dist import _lib
    from triton_dist.kernels.amd import gated_gemm
    ws = _lib.new_split_k_workspace(cuda)
    switches(_lib.TDIST_DEBUG_GEMM_TILE, tile)
    switches(_lib.TDIST_DEBUG_GEMM_SPLIT_K, pieces)
    esz = 1 if dtype == torch.float8_e4m3fn else 2
    out_dtype = torch.float16 if dtype == torch.float16 else torch.bfloat16
    for M, N, k_bytes in ((1, 8, 128), (63, 129, 16), (64, 128, 256), (129, 260, 144), (300, 1000, 1008), (2050, 520, 4112)):
        announce("gemm tile %d pieces %d %s %dx%d K bytes %d" % (tile, pieces, dtype, M, N, k_bytes))
        g = torch.Generator().manual_seed(M + N)
        a, b = poisoned(M, k_bytes // esz, dtype, g, cuda), poisoned(N, k_bytes // esz, dtype, g, cuda)
        want = (a.float() @ b.float().t()).to(out_dtype)
        for _ in range(2):   # (twice on one workspace: the counters are left at zero)
            c = torch.full((M, N), float("nan"), dtype=out_dtype, device=cuda)
            gated_gemm(a, None, 0, b, c, None, 0, 0, 1, sk_workspace=ws)
            torch.cuda.synchronize()
            assert torch.equal(c, want)


# the ring of two, three, four or six stages (whether the tiles fill the chip twice chooses) filled in part, just filled and gone round,
# with a whole and a ragged first K tile; pieces of one to four K tiles whose last is shorter
@pytest.mark.parametrize("tile", [5, 6])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("M,N,pieces", [(130, 200, 1), (130, 200, 3), (130, 200, 7), (2300, 2200, 1)])
def test_every_number_of_k_tiles(cuda, switches, dtype, tile, M, N, pieces):
    from triton_dist import _lib
    from triton_dist.kernels.amd import gated_gemm
    announce("gemm small tile %d %s %dx%d pieces %d, K tiles 1 to 14" % (tile, dtype, M, N, pieces))
    ws = _lib.new_split_k_workspace(cuda)
    switches(_lib.TDIST_DEBUG_GEMM_TILE, tile)
    switches(_lib.TDIST_DEBUG_GEMM_SPLIT_K, pieces)
    esz = 1 if dtype == torch.float8_e4m3fn else 2
    g = torch.Generator().manual_seed(M + pieces)
    for k_bytes in [128 * n for n in range(1, 15)] + [128 * n + 48 for n in range(1, 14, 3)]:
        a, b = poisoned(M, k_bytes // esz, dtype, g, cuda), poisoned(N, k_bytes // esz, dtype, g, cuda)
        c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=cuda)
        gated_gemm(a, None, 0, b, c, None, 0, 0, 1, sk_workspace=ws)
        assert torch.equal(c, (a.float() @ b.float().t()).to(torch.bfloat16)), k_bytes


@pytest.mark.parametrize("coherent", [0, 1])
def test_pieces_meet_in_the_l2_and_through_memory_alike(cuda, switches, coherent):
    from triton_dist import _lib
    from triton_dist.kernels.amd import gated_gemm
    announce("gemm small tiles, coherent exchange %d" % coherent)
    ws = _lib.new_split_k_workspace(cuda)
    switches(_lib.TDIST_DEBUG_GEMM_TILE, 5)
    switches(_lib.TDIST_DEBUG_GEMM_SPLIT_K, 4)
    switches(_lib.TDIST_DEBUG_GEMM_SK_COHERENT, coherent)
    g = torch.Generator().manual_seed(3)
    a, b = poisoned(200, 4096, torch.bfloat16, g, cuda), poisoned(1536, 4096, torch.bfloat16, g, cuda)
    want = (a.float() @ b.float().t()).to(torch.bfloat16)
    for _ in range(3):
        c = torch.full((200, 1536), float("nan"), dtype=torch.bfloat16, device=cuda)
        gated_gemm(a, None, 0, b, c, None, 0, 0, 1, sk_workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(c, want)


@pytest.mark.parametrize("tile", [5, 6])
def test_scatter_and_scales(cuda, switches, tile):
    """The scatter to the owners' buffers and the e4m3 scales (powers of two: exact)."""
    from triton_dist import _lib
    from triton_dist.kernels.amd import create_gemm_rs_intra_node_context, gemm_rs_intra_node
    announce("gemm_rs on the small tile %d" % tile)
    switches(_lib.TDIST_DEBUG_GEMM_TILE, tile)
    W, rank, M, N, K = 4, 1, 512, 512, 768
    g = torch.Generator().manual_seed(tile)
    a = torch.randint(-2, 3, (M, K), generator=g).float().to(torch.float8_e4m3fn).to(cuda)
    b = torch.randint(-2, 3, (N, K), generator=g).float().to(torch.float8_e4m3fn).to(cuda)
    rs = (2.0 ** torch.randint(-2, 3, (M, ), generator=g)).to(cuda)
    cs = (2.0 ** torch.randint(-2, 3, (N, ), generator=g)).to(cuda)
    ctx = create_gemm_rs_intra_node_context(M, N, torch.bfloat16, rank, W, None)
    gemm_rs_intra_node(a, b, ctx, row_scale=rs, col_scale=cs)
    torch.cuda.synchronize()
    want = ((a.float() @ b.float().t()) * rs[:, None] * cs[None, :]).to(torch.bfloat16)
    for o in range(W):
        assert torch.equal(ctx.scatter_bufs[o][rank * M // W:(rank + 1) * M // W], want[o * M // W:(o + 1) * M // W])
