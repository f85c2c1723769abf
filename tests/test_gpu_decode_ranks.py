"""The streaming decode with the merge of all ranks' results in its second launch, against the stream and the merge as calls of their
own: the same bits, in this rank's place among the results as well."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


# one rank; ranks that fill the loads in flight, one more, and several times as many; sequences in one range, in few and in many;
# no keys of a sequence here, or on another rank; more sequences than ranges; results in rows that take no wide loads
@pytest.mark.parametrize("R,lens,hq,hkv,dk,dv,part,room", [
    (1, [1320], 32, 8, 128, 128, torch.float32, 0), (2, [70, 0, 3], 16, 16, 128, 128, torch.bfloat16, 0), (8, [1259], 16, 16, 128, 128, torch.bfloat16, 0),
    (9, [20000, 1, 0, 611, 64], 64, 8, 128, 128, torch.float16, 0), (17, [333, 4097], 6, 1, 256, 256, torch.float32, 0),
    (8, [16] * 40 + [900], 32, 8, 64, 64, torch.bfloat16, 0), (3, [0, 0], 32, 8, 96, 96, torch.float16, 1), (4, [50, 2000], 8, 8, 64, 64, torch.float32, 3),
    (8, [100, 2500, 0, 31], 128, 1, 576, 512, torch.bfloat16, 0), (4, [90] * 70, 64, 16, 128, 128, torch.bfloat16, 0), (2, [17] * 9, 128, 64, 64, 64, torch.float16, 2)])
def test_like_stream_and_merge(cuda, R, lens, hq, hkv, dk, dv, part, room):
    from triton_dist.kernels.amd.flash_decode import decode_stream, decode_stream_ranks, gqa_fwd_batch_decode_inter_rank_combine
    announce("decode ranks R=%d B=%d heads %d/%d dims %d/%d %s" % (R, len(lens), hq, hkv, dk, dv, part))
    g = torch.Generator(device="cuda").manual_seed(R + sum(lens) + dk)
    B, page, own = len(lens), 16, R // 2
    dtype = torch.float16 if part == torch.float16 else torch.bfloat16
    pages = [-(-n // page) for n in lens]
    k = torch.randn((sum(pages) + 1, page, hkv, dk), generator=g, device=cuda).to(dtype)
    v = k[..., :dv] if dv < dk else torch.randn((sum(pages) + 1, page, hkv, dv), generator=g, device=cuda).to(dtype)
    table, place, at = torch.zeros((B, max(pages) + 1), dtype=torch.int32, device=cuda), torch.randperm(sum(pages) + 1, generator=g, device=cuda, dtype=torch.int32), 0
    for b, n in enumerate(pages):
        table[b, :n] = place[at:at + n]
        at += n
    q = torch.randn((B, hq, dk), generator=g, device=cuda).to(dtype)
    rank_lens = torch.randint(0, 3, (R, B), generator=g, device=cuda, dtype=torch.int32)
    rank_lens[own] = torch.tensor(lens, dtype=torch.int32)
    lse = torch.randn((R, B, hq), generator=g, device=cuda)
    lse[0, 0, 0] = -float("inf")
    rows = (torch.randn((R, B, hq, dv + room), generator=g, device=cuda) * 0.1).to(part)
    got = []
    for fused in (True, False):
        all_out, all_lse = rows.clone()[..., :dv], lse.clone()
        if fused:
            out = decode_stream_ranks(q, k, v, rank_lens, table, dk ** -0.5, 0.0, own, all_out, all_lse)
        else:
            decode_stream(q, k, v, rank_lens[own], table, dk ** -0.5, 0.0, all_out[own], all_lse[own])
            out = gqa_fwd_batch_decode_inter_rank_combine(all_out, all_lse, rank_lens, out_dtype=q.dtype)
        got.append((out, all_out.contiguous(), all_lse))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_results_of_another_size_than_the_layer_is_for_are_refused(cuda):
    """This rank's result is written into the caller's rows: they have to be of the cache's width, on either route."""
    from triton_dist.kernels.amd.flash_decode import decode_stream_ranks
    from triton_dist.layers.amd.sp_flash_decode_layer import SpGQAFlashDecodeAttention
    announce("decode ranks: results of another width")
    q, cache = torch.zeros((1, 8, 128), dtype=torch.bfloat16, device=cuda), torch.zeros((4, 16, 8, 128), dtype=torch.bfloat16, device=cuda)
    table, lens = torch.zeros((1, 4), dtype=torch.int32, device=cuda), torch.full((2, 1), 16, dtype=torch.int32, device=cuda)
    for heads, width in ((8, 64), (4, 128)):
        rows, lse = torch.zeros((2, 1, heads, width), dtype=torch.bfloat16, device=cuda), torch.zeros((2, 1, heads), device=cuda)
        layer = SpGQAFlashDecodeAttention(0, 0, 2, 1, heads, heads, 128, width, page_size=16, scale=1.0)
        for peers in ((rows, lse), (rows, lse.to(torch.float64))):
            with pytest.raises(AssertionError):
                layer(q, cache, cache, lens, table, peers)
        with pytest.raises(AssertionError):
            decode_stream_ranks(q, cache, cache, lens, table, 1.0, 0.0, 0, rows, lse)
    rows, lse = torch.zeros((2, 1, 8, 128), dtype=torch.bfloat16, device=cuda), torch.zeros((2, 1, 8), device=cuda)
    for rank in (-1, 2):
        with pytest.raises(AssertionError):
            decode_stream_ranks(q, cache, cache, lens, table, 1.0, 0.0, rank, rows, lse)
