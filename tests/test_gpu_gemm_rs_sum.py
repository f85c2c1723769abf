"""tdist_gemm_rs, the product and the sum of this rank's rows in one launch on the small tiles: the sum and every owner's buffer against the
ordered reduction of what the buffers hold, bit for bit."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu


def partials(shape, dtype, g):
    """Other ranks' rows: normal values, among them both zeros and infinities of one sign to a column."""
    x = torch.randn(shape, generator=g)
    x[0, ::7], x[-1, 1::5], x[shape[0] // 2, 2::9], x[1, ::11] = -0.0, 0.0, float("inf"), float("-inf")
    return x.to(dtype)


# tiles of 64 and 128 rows whole and in pieces of K (one launch), and the large ones (two); 1 to 16 ranks: 1, 2, and what one batch of
# seven slices leaves over; one row tile per rank and several; columns that end inside a tile and inside its 128-byte lines
@pytest.mark.parametrize("tile,pieces", [(5, 1), (5, 4), (6, 1), (6, 2), (2, 0), (None, None)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("world,rank,m_per,N", [(1, 0, 128, 256), (2, 1, 384, 264), (3, 0, 128, 512), (8, 7, 256, 200), (8, 3, 128, 1024), (9, 4, 128, 72),
                                                (16, 5, 128, 328), (17, 16, 128, 128)])
def test_sum_beside_the_product(cuda, switches, dtype, tile, pieces, world, rank, m_per, N):
    from triton_dist import _lib
    announce("gemm_rs in one launch: tile %s pieces %s %s world %d rank %d, %d rows each, %d columns" % (tile, pieces, dtype, world, rank, m_per, N))
    switches(_lib.TDIST_DEBUG_GEMM_TILE, tile)
    switches(_lib.TDIST_DEBUG_GEMM_SPLIT_K, pieces)
    M, K = world * m_per, 1040
    out_dtype = torch.float16 if dtype == torch.float16 else torch.bfloat16
    g = torch.Generator().manual_seed(M + N)
    a, b = [torch.randint(-2, 3, (n, K), generator=g).float().to(dtype).to(cuda) for n in (M, N)]
    want = (a.float() @ b.float().t()).to(out_dtype)
    scales = None, None
    if dtype == torch.float8_e4m3fn and m_per == 128:
        scales = [(2.0 ** torch.randint(-2, 3, (n, ), generator=g)).to(cuda) for n in (M, N)]
        want = (want.float() * scales[0][:, None] * scales[1]).to(out_dtype)
    ws = _lib.new_split_k_workspace(cuda)
    for _ in range(2):
        bufs = [torch.full((M, N), 7.0, dtype=out_dtype, device=cuda) for _ in range(world)]
        for r in range(world):
            bufs[rank][r * m_per:(r + 1) * m_per] = partials((m_per, N), out_dtype, g).to(cuda)
        before = [t.clone() for t in bufs]
        table = torch.tensor([t.data_ptr() for t in bufs], dtype=torch.int64, device=cuda)
        out = torch.full((m_per, N), float("nan"), dtype=out_dtype, device=cuda)
        _lib.call("tdist_gemm_rs", _lib.dtype_code(dtype), a.data_ptr(), K, b.data_ptr(), K, table.data_ptr(), bufs[rank].data_ptr(), out.data_ptr(),
                  M, N, K, _lib.ptr(scales[0]), _lib.ptr(scales[1]), rank, world, *_lib.workspace_args(ws), _lib.stream_ptr(None))
        torch.cuda.synchronize()
        at = slice(rank * m_per, (rank + 1) * m_per)
        for o in range(world):
            before[o][at] = want[o * m_per:(o + 1) * m_per]
            assert torch.equal(bufs[o].view(torch.int16), before[o].view(torch.int16)), o
        total = golden.reduce_slices_ordered(bufs[rank].cpu().view(world, m_per, N), (rank + 1) % world)
        nan = total.isnan()
        assert torch.equal(out.cpu().isnan(), nan)
        assert torch.equal(out.cpu().masked_fill(nan, 0).view(torch.int16), total.masked_fill(nan, 0).view(torch.int16))


def test_replays_of_a_graph_add_up_what_the_buffers_hold_then(cuda, switches):
    from triton_dist import _lib
    from triton_dist.kernels.amd import create_gemm_rs_intra_node_context, gemm_rs_intra_node
    announce("gemm_rs in one launch, captured")
    switches(_lib.TDIST_DEBUG_GEMM_TILE, 6)
    W, rank, M, N, K = 4, 2, 1024, 512, 256
    g = torch.Generator().manual_seed(1)
    a, b = [torch.randn((n, K), generator=g).to(torch.bfloat16).to(cuda) for n in (M, N)]
    ctx = create_gemm_rs_intra_node_context(M, N, torch.bfloat16, rank, W, None)
    gemm_rs_intra_node(a, b, ctx)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = gemm_rs_intra_node(a, b, ctx)
    for _ in range(3):
        ctx.set_peer_partials({r: torch.randn((M // W, N), generator=g).to(torch.bfloat16).to(cuda) for r in range(W) if r != rank})
        a.copy_(torch.randn((M, K), generator=g))
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, gemm_rs_intra_node(a, b, ctx))
        stored = ctx.scatter_bufs[rank].cpu().view(W, M // W, N)
        assert torch.equal(got.cpu().view(torch.int16), golden.reduce_slices_ordered(stored, (rank + 1) % W).view(torch.int16))
