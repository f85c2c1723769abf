"""MoE dispatch from expert ids where rows are shared by several waves (few tokens), and align / sort where padding outweighs
the entries: bit-exact against the oracle."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu


# one token; whole and broken workgroups; windows of 1 to 7 KB with a last one that is empty, partial or a single piece;
# rows without 16-byte pieces; the last size that is cut finer and the first that is not (1024 tokens of one window)
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("T,topk,G,W,H", [(1, 8, 256, 32, 7168), (2, 1, 8, 2, 1024), (15, 3, 16, 4, 1040), (16, 8, 64, 8, 2048), (17, 8, 64, 8, 5120),
                                          (128, 8, 256, 32, 7168), (33, 5, 8, 2, 8208), (31, 4, 8, 2, 16384), (3, 2, 4, 2, 100000),
                                          (9, 3, 4, 4, 52), (40, 2, 4, 4, 3001), (1007, 2, 32, 8, 1040), (1009, 2, 32, 8, 1040)])
def test_dispatch_from_few_ids(cuda, wide, T, topk, G, W, H):
    from triton_dist.kernels.amd import create_all_to_all_context, fast_all_to_all
    announce("dispatch from few ids T=%d topk=%d G=%d W=%d H=%d wide=%s" % (T, topk, G, W, H, wide))
    g = torch.Generator().manual_seed(T + H)
    ids = golden.random_distinct_experts(T, G, topk, g)
    x = torch.randint(0, 256, (T, H), generator=g, dtype=torch.uint8)
    scale = torch.rand(T, generator=g)
    max_m = T * topk
    ctx = create_all_to_all_context(max_m, H, 0, G, W, G // W, dtype=torch.float8_e4m3fn)
    ctx.recv_buf.view(torch.uint8).fill_(0xAB)
    dev_ids = ids.to(torch.int64 if wide else torch.int32).to(cuda)
    splits, recv, scales = fast_all_to_all(ctx, x.to(cuda).view(torch.float8_e4m3fn), None, scale.to(cuda), expert_ids=dev_ids)
    torch.cuda.synchronize()
    w_splits, w_cumsum, w_scatter, w_gather, _ = golden.moe_preprocess(ids, G)
    for got, want in zip(ctx.last_index, (w_splits, w_cumsum, w_scatter, w_gather)):
        assert torch.equal(got.cpu(), want)
    assert torch.equal(splits.cpu(), w_splits)
    recv, scales, rows = recv.view(torch.uint8).cpu(), scales.cpu(), x[w_gather.long()]
    for d in range(W):
        lo, hi = int(w_cumsum[d * (G // W)]), int(w_cumsum[(d + 1) * (G // W)])
        assert torch.equal(recv[d * max_m:d * max_m + hi - lo], rows[lo:hi])
        assert torch.equal(scales[d * max_m:d * max_m + hi - lo], scale[w_gather.long()][lo:hi])
        assert (recv[d * max_m + hi - lo:(d + 1) * max_m] == 0xAB).all()


# experts per rank that are one, odd, and as many as there can be: the rank of an expert is found by a multiplication
@pytest.mark.parametrize("T,topk,G,W", [(37, 6, 21, 7), (37, 6, 21, 21), (5, 8, 381, 3), (5, 8, 4096, 1), (9, 4, 4095, 13)])
def test_dispatch_with_any_number_of_experts_per_rank(cuda, T, topk, G, W):
    test_dispatch_from_few_ids(cuda, False, T, topk, G, W, 1024)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("R,T,topk,E,BS", [(8, 1, 8, 256, 128), (8, 125, 8, 256, 128), (1, 3, 2, 16, 256), (8, 2, 2, 64, 1024), (4, 1031, 3, 100, 64)])
def test_align_sort_with_more_padding_than_entries(cuda, dtype, R, T, topk, E, BS):
    from triton_dist.kernels.amd import sort_topk_ids_align_block_size
    announce("align R=%d T=%d topk=%d E=%d BS=%d" % (R, T, topk, E, BS))
    ids = golden.random_distinct_experts(R * T, E, topk, torch.Generator().manual_seed(T))
    want = golden.sort_topk_ids_align_block_size(ids, E, R, T, BS)
    got = sort_topk_ids_align_block_size(ids.to(dtype).to(cuda), E, R, T, BS)
    nb = want[4] // BS
    assert int(got[4].item()) == want[4]
    assert torch.equal(got[0].cpu(), want[0])   # the whole buffer, padding included
    assert torch.equal(got[1].cpu()[:nb], want[1]) and torch.equal(got[2].cpu()[:nb], want[2])
    assert torch.equal(got[3].cpu(), want[3])


# one and two passes of 64 entries per wave with many entries of one group in each (a wave's count of a group fills its byte
# up to 128), four groups to a step and a remainder, as many groups as there can be, blocks of one row and of more than 32768
@pytest.mark.parametrize("R,T,topk,E,BS", [(1, 600, 1, 1, 128), (1, 40000, 1, 2, 1), (2, 20001, 1, 1, 48), (3, 700, 2, 3, 5), (16, 130, 2, 256, 16),
                                           (5, 97, 3, 819, 3), (2, 11, 2, 7, 40000)])
def test_align_sort_counts(cuda, R, T, topk, E, BS):
    test_align_sort_with_more_padding_than_entries(cuda, torch.int32, R, T, topk, E, BS)
    test_align_sort_with_more_padding_than_entries(cuda, torch.int64, R, T, topk, E, BS)


# 64-bit ids: both block sizes of the one launch, remainders of a vector of four, ids that are not 16-byte aligned, not
# contiguous, out of range, and more of them than the one launch takes
@pytest.mark.parametrize("T,topk,G,how", [(1, 1, 1, ""), (1, 8, 256, ""), (63, 3, 7, ""), (4096, 8, 256, ""), (4097, 8, 64, ""), (8192, 8, 64, ""), (9000, 8, 64, ""),
                                          (101, 3, 40, "misaligned"), (50, 4, 16, "strided"), (77, 5, 12, "out of range"), (16, 2, 4096, "")])
def test_index_from_64_bit_ids(cuda, T, topk, G, how):
    from triton_dist.kernels.amd import create_all_to_all_context, moe_dispatch_preprocess
    announce("index from 64-bit ids T=%d topk=%d G=%d %s" % (T, topk, G, how))
    g = torch.Generator().manual_seed(T + G)
    ids = torch.randint(-1 if how == "out of range" else 0, G + (1 if how == "out of range" else 0), (T, topk), generator=g)
    if how == "misaligned":
        dev = torch.empty(T * topk + 1, dtype=torch.int64, device=cuda)[1:].view(T, topk).copy_(ids)
    elif how == "strided":
        dev = torch.empty((T, topk + 2), dtype=torch.int64, device=cuda)[:, :topk].copy_(ids)
    else:
        dev = ids.to(cuda)
    ctx = create_all_to_all_context(8, 16, 0, G, 1, G, dtype=torch.float8_e4m3fn)
    want = [t.clone() for t in moe_dispatch_preprocess(ids.int().to(cuda), G, want_topk_index=True)]
    got = moe_dispatch_preprocess(dev, G, want_topk_index=True, ctx=ctx)
    valid = int(want[1][-1])
    for name, a, b in zip(("splits", "cumsum", "scatter", "gather", "topk"), got, want):
        n = valid if name in ("gather", "topk") else a.numel()
        assert torch.equal(a.reshape(-1)[:n], b.reshape(-1)[:n]), name
    if how != "out of range":
        for a, b in zip(got, golden.moe_preprocess(ids, G)[:4]):
            assert torch.equal(a.cpu(), b)
