"""The all-gather GEMM and the grouped GEMM of rows that are read where they lie, against the same product of the gathered rows: one
kernel and one order of sums, so the bits are the same, for every tile, at shards shorter and longer than a tile, and where the
shards are too far apart or too many and are gathered after all."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


def scattered(cuda, g, W, shape, dtype):
    """W shards in memory in another order than the ranks', with room between them."""
    raw = [None] * W
    for r in sorted(range(W), key=lambda r: (r * 7 + 3) % W):
        x = torch.randn(shape, generator=g).to(torch.bfloat16 if dtype == torch.float8_e4m3fn else dtype).to(dtype)
        room = torch.empty(x.numel() * x.element_size() + 4096, dtype=torch.uint8, device=cuda)
        raw[r] = room[256:256 + x.numel() * x.element_size()].view(dtype).view(shape)
        raw[r].copy_(x)
    return raw


def product(cuda, shards, b, tile, scales=(None, None)):
    """(rows where they lie, gathered rows)"""
    from triton_dist import _lib
    from triton_dist.kernels.amd.all_gather_gemm import ag_gemm_intra_node, create_ag_gemm_intra_node_context, gated_gemm
    W, (m, K) = len(shards), shards[0].shape
    out = torch.bfloat16 if b.dtype == torch.float8_e4m3fn else b.dtype
    ctx = create_ag_gemm_intra_node_context(W * m, b.shape[0], K, b.dtype, out, W // 2, W, None, M_PER_CHUNK=m, ragged_chunks=True)
    ctx.set_peer_shards({r: s for r, s in enumerate(shards) if r != W // 2})
    ctx.workspace_tensors[W // 2].view(torch.uint8).fill_(0x7B)
    full = torch.cat([s.view(torch.uint8) for s in shards]).view(b.dtype)
    want = torch.empty((W * m, b.shape[0]), dtype=out, device=cuda)
    with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, tile):
        got = ag_gemm_intra_node(shards[W // 2], b, False, ctx, row_scale=scales[0], col_scale=scales[1])
        gated_gemm(full, None, 0, b, want, None, 0, 0, W, row_scale=scales[0], col_scale=scales[1], sk_workspace=_lib.new_split_k_workspace(cuda))
    torch.cuda.synchronize()
    return got, want


@pytest.mark.parametrize("tile", [None, 0, 1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("W,m", [(2, 1), (16, 3), (4, 50), (8, 100), (3, 128), (5, 130), (2, 257), (7, 300)])
def test_bf16_rows_where_they_lie(cuda, W, m, tile):
    announce("shard rows W=%d m=%d tile=%s" % (W, m, tile))
    g = torch.Generator().manual_seed(W + m)
    shards = scattered(cuda, g, W, (m, 1000), torch.bfloat16)
    got, want = product(cuda, shards, torch.randn((264, 1000), generator=g).to(torch.bfloat16).to(cuda), tile)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype,W,m,N,K", [(torch.float8_e4m3fn, 8, 300, 1024, 2048), (torch.float8_e4m3fn, 3, 77, 520, 1040),
                                           (torch.float16, 8, 700, 2304, 512), (torch.float16, 2, 2048, 4096, 256)])
def test_other_types_and_several_rounds(cuda, dtype, W, m, N, K):
    announce("shard rows %s W=%d m=%d" % (dtype, W, m))
    g = torch.Generator().manual_seed(m)
    shards = scattered(cuda, g, W, (m, K), dtype)
    scales = (None, None)
    if dtype == torch.float8_e4m3fn:
        scales = (torch.rand(W * m, generator=g).to(cuda), torch.rand(N, generator=g).to(cuda))
    b = torch.randn((N, K), generator=g).to(torch.bfloat16).to(dtype).to(cuda)
    got, want = product(cuda, shards, b, None, scales)
    assert torch.equal(got, want)


@pytest.mark.parametrize("case", ["too many", "too far apart"])
def test_shards_out_of_reach_are_gathered(cuda, case):
    announce("shard rows %s" % case)
    g = torch.Generator().manual_seed(2)
    W = 17 if case == "too many" else 2
    shards = scattered(cuda, g, W, (40, 512), torch.bfloat16)
    if case == "too far apart":
        room = torch.empty(9 << 29, dtype=torch.uint8, device=cuda)   # 4.5 GiB with a shard at either end
        for r, at in ((0, 0), (1, room.numel() - 65536)):
            there = room[at:at + 40 * 1024].view(torch.bfloat16).view(40, 512)
            there.copy_(shards[r])
            shards[r] = there
    got, want = product(cuda, shards, torch.randn((256, 512), generator=g).to(torch.bfloat16).to(cuda), None)
    assert torch.equal(got, want)


# (tile 0: 256 x 256, 4: 128 x 256; the choice left to the call takes small ones at all of these sizes)
@pytest.mark.parametrize("tile", [None, 0, 4])
@pytest.mark.parametrize("W,m,topk,E,N,K", [(4, 7, 2, 8, 256, 512), (8, 130, 2, 4, 520, 1000), (2, 1024, 4, 8, 512, 256), (16, 33, 1, 3, 256, 264)])
def test_grouped_rows_where_they_lie(cuda, monkeypatch, W, m, topk, E, N, K, tile):
    from triton_dist import _lib
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, create_ag_group_gemm_intra_node_context
    announce("grouped shard rows W=%d m=%d E=%d tile=%s" % (W, m, E, tile))
    g = torch.Generator().manual_seed(W * m)
    shards = scattered(cuda, g, W, (m, K), torch.bfloat16)
    ids = torch.rand((W * m, E), generator=g).topk(topk, dim=1).indices.to(torch.int32).to(cuda)
    w = (torch.randn((E, N, K), generator=g) * 0.05).to(torch.bfloat16).to(cuda).transpose(1, 2)
    out = []
    for gathered in (False, True):
        ctx = create_ag_group_gemm_intra_node_context(None, shards[1], w, ids, E, max_M=W * m, rank=1, num_ranks=W)
        ctx.set_peer_shards({r: s for r, s in enumerate(shards) if r != 1})
        ctx.workspace_tensors[1].view(torch.uint8).fill_(0x7B)
        if gathered:
            monkeypatch.setattr(_lib, "shards_in_reach", lambda *_: False)
        with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, tile):
            out.append(ag_group_gemm_intra_node(shards[1], w, ctx))
        torch.cuda.synchronize()
        assert tile is None or {blocks.block_size for blocks in ctx.joined.values()} == {256 if tile == 0 else 128}
    assert torch.equal(out[0], out[1])
    token = torch.cat(shards)[:, None, :].expand(-1, topk, -1).reshape(-1, K).float()
    rows = torch.arange(0, W * m * topk, max(1, W * m * topk // 50), device=cuda)
    want = torch.stack([token[r] @ w[ids.reshape(-1)[r].long()].float() for r in rows])
    assert ((out[0][rows].float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3).all()
