"""The decode that divides a batch's keys itself (tdist_decode_stream) against the exact closed form, at the lengths where
its ranges begin and end: blocks of 16 and 32 keys, sequences without keys, more sequences than lanes, one long sequence
among short ones (its partial results merged over many ranges), batches whose units do not fill a workgroup."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu

ATOL = 2e-3

LENS = {
    "one": [1], "block edges": [15, 16, 17, 32, 33, 64, 65], "none among some": [0, 40, 0, 0, 100, 7, 0], "no keys at all": [0, 0, 0],
    "one long": [5, 9000, 64, 1, 300], "more than lanes": [(37 * i) % 90 for i in range(150)],
}


def check(cuda, num_heads, dims, dtype, kv_lens, page, soft_cap, latent, seed):
    from triton_dist.kernels.amd.flash_decode import decode_stream
    dk, dv = dims
    Hq, Hkv = num_heads
    B = len(kv_lens)
    g = torch.Generator().manual_seed(seed)
    q = torch.randn((B, Hq, dk), generator=g).to(dtype)
    k, v, table = golden.make_paged_kv(B, max(max(kv_lens), 1), Hkv, dk, page, dtype, g, v_head_dim=dv)
    kd, td, lens = k.to(cuda), table.to(cuda), torch.tensor(kv_lens, dtype=torch.int32, device=cuda)
    if latent:
        v, vd = k[..., :dv], kd[..., :dv]
    else:
        vd = v.to(cuda)
    scale = dk**-0.5
    counters = torch.zeros(8192, dtype=torch.int32, device=cuda)
    exact, exact_lse = golden.decode_exact(q, k, v, kv_lens, table, scale, soft_cap)
    live = ~torch.isinf(exact_lse)
    first = None
    for _ in range(2):   # twice on the same counters
        out = torch.full((B, Hq, dv + 4), float("nan"), dtype=torch.float32, device=cuda)[..., :dv]
        lse = torch.full((B, Hq), float("nan"), dtype=torch.float32, device=cuda)
        decode_stream(q.to(cuda), kd, vd, lens, td, scale, soft_cap, out, lse, counters=counters)
        torch.cuda.synchronize()
        assert int(counters.abs().sum()) == 0
        assert (out.cpu().double() - exact).abs().max() <= ATOL
        assert torch.equal(torch.isinf(lse.cpu()), ~live)
        assert not live.any() or (lse.cpu().double()[live] - exact_lse[live]).abs().max() <= ATOL
        assert first is None or torch.equal(first, out)   # whoever arrives last, the sums run in order
        first = out
    out16 = torch.full((B, Hq, dv), float("nan"), dtype=dtype, device=cuda)
    decode_stream(q.to(cuda), kd, vd, lens, td, scale, soft_cap, out16)
    torch.cuda.synchronize()
    assert torch.equal(out16, first.to(dtype))


@pytest.mark.parametrize("lens", list(LENS))
@pytest.mark.parametrize("num_heads,dims,dtype,page,soft_cap", [
    ((32, 8), (128, 128), torch.bfloat16, 16, 0), ((6, 1), (128, 128), torch.float16, 1, 30), ((40, 2), (64, 64), torch.bfloat16, 16, 0),
    ((16, 16), (192, 128), torch.float16, 16, 0), ((12, 3), (256, 256), torch.bfloat16, 1, 0), ((10, 5), (96, 96), torch.bfloat16, 16, 0),
    ((8, 2), (40, 40), torch.float16, 16, 0), ((8, 8), (160, 160), torch.bfloat16, 16, 50)])
def test_ranges_against_the_exact_result(cuda, num_heads, dims, dtype, page, soft_cap, lens):
    announce("decode stream heads=%s dims=%s %s page=%d cap=%s lens: %s" % (num_heads, dims, dtype, page, soft_cap, lens))
    check(cuda, num_heads, dims, dtype, LENS[lens], page, soft_cap, False, len(lens) + dims[0])


@pytest.mark.parametrize("lens", list(LENS))
@pytest.mark.parametrize("num_heads,dtype,page,soft_cap", [((128, 1), torch.bfloat16, 16, 0), ((24, 1), torch.float16, 1, 30), ((4, 2), torch.bfloat16, 16, 0)])
def test_latent_heads_against_the_exact_result(cuda, num_heads, dtype, page, soft_cap, lens):
    """576 / 512 with the value a view of the key's first 512 columns."""
    announce("decode stream latent heads=%s %s page=%d cap=%s lens: %s" % (num_heads, dtype, page, soft_cap, lens))
    check(cuda, num_heads, (576, 512), dtype, LENS[lens], page, soft_cap, True, len(lens))


# a workgroup's 16 or 32 heads filled, overfilled by one and shared by two kv heads; lengths around its blocks of 32 keys, and
# sequences of several blocks that share a range with others
@pytest.mark.parametrize("num_heads", [(16, 1), (17, 1), (32, 1), (33, 1), (48, 1), (40, 2)])
@pytest.mark.parametrize("lens", [[31, 32, 33, 63, 64, 65, 95, 96, 97], [1, 0, 130, 0, 31, 700, 2]])
def test_latent_head_sets_and_blocks(cuda, num_heads, lens):
    announce("decode stream latent heads=%s lens: %s" % (num_heads, lens))
    check(cuda, num_heads, (576, 512), torch.bfloat16, lens, 16, 0, True, num_heads[0] + len(lens))


# sequences with few partials each (a wave merges all of them) and batches on both sides of that rule
@pytest.mark.parametrize("B,num_heads,D", [(7, (32, 8), 64), (8, (32, 8), 64), (9, (32, 8), 128), (33, (6, 1), 128), (65, (6, 1), 96)])
def test_merge_of_few_partials(cuda, B, num_heads, D):
    announce("decode stream merge B=%d heads=%s D=%d" % (B, num_heads, D))
    check(cuda, num_heads, (D, D), torch.bfloat16, [(97 * i) % 701 + 400 for i in range(B)], 16, 0, False, B + D)


def test_workspace_and_head_dimensions_are_checked(cuda):
    from triton_dist import _lib
    lib = _lib.load()
    need = lib.tdist_decode_stream_workspace_bytes(3, 32, 8, 128, 128)
    assert need > 0 and lib.tdist_decode_stream_workspace_bytes(3, 32, 5, 128, 128) == -1
    p = torch.zeros(4096, dtype=torch.uint8, device=cuda).data_ptr()

    def call(dk, dv, v, nbytes):
        return lib.tdist_decode_stream(p, p, v, 1.0, 0.0, p, p, 3, 32, 8, dk, dv, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, _lib.TDIST_BF16, p,
                                       1024, p, nbytes, p, _lib.TDIST_BF16, 0, 0, None, None)
    assert call(128, 128, p, need - 1) == _lib.TDIST_ERR_WORKSPACE
    assert call(576, 512, p + 16, 1 << 40) == _lib.TDIST_ERR_UNSUPPORTED


@pytest.mark.parametrize("B,Hq,Hkv,D,lens,dtype", [(1, 64, 8, 128, [6016], torch.bfloat16), (5, 32, 8, 96, [6001, 17, 300, 0, 2048], torch.float16),
                                                   (12, 6, 1, 128, [6100] + [33] * 11, torch.bfloat16), (8, 6, 1, 72, [1] * 8, torch.float16)])
def test_few_long_sequences_take_either_form_with_one_result(cuda, B, Hq, Hkv, D, lens, dtype):
    """A fixed number of splits and their combine on the same inputs. Both hold fp32 partial results: they differ by one
    rounding of the output. And the room a page table has beyond the sequences' pages changes nothing, not even the route:
    the same bits behind a narrow table and one four times as wide."""
    from triton_dist.kernels.amd import flash_decode as fd
    announce("few long sequences B=%d heads %d/%d D=%d" % (B, Hq, Hkv, D))
    g = torch.Generator().manual_seed(B + D)
    page, pages = 16, 400
    k = torch.randn((pages, page, Hkv, D), generator=g).to(dtype).to(cuda)
    v = torch.randn((pages, page, Hkv, D), generator=g).to(dtype).to(cuda)
    q = torch.randn((B, Hq, D), generator=g).to(dtype).to(cuda)
    need = max(1, -(-max(lens) // page))
    wide = torch.randint(0, pages, (B, 4 * max(need, 376)), generator=g, dtype=torch.int32).to(cuda)
    kv_lens = torch.tensor(lens, dtype=torch.int32, device=cuda)
    got = fd.gqa_fwd_batch_decode(q, k, v, None, [1] * B, kv_lens, wide, D ** -0.5)
    assert torch.equal(got, fd.gqa_fwd_batch_decode(q, k, v, None, [1] * B, kv_lens, wide[:, :need], D ** -0.5))
    S = fd.DEFAULT_KV_SPLITS
    part, lse, _ = fd._split_kv(q, k, v, kv_lens, wide, D ** -0.5, 0.0, S)
    want = fd.decode_combine(part, lse, S, 1, kv_lens, B, Hq, D, (part.stride(2), part.stride(0), part.stride(1)),
                             (lse.stride(2), lse.stride(0), lse.stride(1)), torch.empty_like(got))
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((got.float() - want.float()).abs() <= 2 * eps * want.float().abs() + 1e-5).all()


# one sequence over 1024, 512, 341, 256 and 128 ranges (merged by 16 waves a workgroup above 256, by four below), alone and
# beside short ones
@pytest.mark.parametrize("lens", [[21000], [3, 0, 21000, 700]])
@pytest.mark.parametrize("num_heads,D", [((6, 1), 128), ((10, 2), 64), ((24, 3), 96), ((16, 4), 128), ((16, 8), 64), ((20, 1), 256)])
def test_a_long_sequence_over_many_ranges(cuda, num_heads, D, lens):
    announce("decode stream, many ranges, heads=%s D=%d lens=%s" % (num_heads, D, lens))
    check(cuda, num_heads, (D, D), torch.bfloat16, lens, 16, 0, False, D + len(lens))


# partial results in tiles of 16 columns: one narrower tile alone, and one behind whole ones; blocks of 16 heads and of fewer
@pytest.mark.parametrize("num_heads,D", [((20, 1), 8), ((34, 2), 24), ((3, 3), 200)])
def test_narrow_tiles_of_partial_results(cuda, num_heads, D):
    announce("decode stream, narrow tiles, heads=%s D=%d" % (num_heads, D))
    check(cuda, num_heads, (D, D), torch.float16, [2500, 0, 70], 16, 0, False, D)


def test_a_long_latent_sequence(cuda):
    announce("decode stream, many ranges, latent heads")
    check(cuda, (16, 1), (576, 512), torch.bfloat16, [21000, 40], 16, 0, True, 5)


@pytest.mark.parametrize("hq", [16, 40])
def test_a_query_that_is_no_number_has_no_lse_either(cuda, hq):
    """Latent heads, a sequence in one range: the result and its LSE are no numbers, as the exact ones; other heads and sequences
    are as they were. (-inf, of a sequence without keys, would have a merge with other ranks leave the result out unseen.)"""
    from triton_dist.kernels.amd.flash_decode import decode_stream
    announce("decode stream latent, a query of NaN, %d heads" % hq)
    g = torch.Generator().manual_seed(hq)
    lens = [40, 33, 64]
    q = torch.randn((3, hq, 576), generator=g).bfloat16()
    k, _, table = golden.make_paged_kv(3, 64, 1, 576, 16, torch.bfloat16, g, v_head_dim=512)
    kd, td, ld = k.to(cuda), table.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda)

    def run(query):
        out, lse = torch.zeros((3, hq, 512), device=cuda), torch.zeros((3, hq), device=cuda)
        decode_stream(query.to(cuda), kd, kd[..., :512], ld, td, 576**-0.5, 0.0, out, lse)
        return out.cpu(), lse.cpu()

    out, lse = run(q)
    q[1, 5] = float("nan")
    bad_out, bad_lse = run(q)
    assert bad_out[1, 5].isnan().all() and bad_lse[1, 5].isnan()
    others = torch.ones((3, hq), dtype=torch.bool)
    others[1, 5] = False
    assert torch.equal(bad_out[others], out[others]) and torch.equal(bad_lse[others], lse[others])


@pytest.mark.parametrize("dtype,group", [(torch.bfloat16, 2), (torch.float16, 17)])
def test_latent_maxima_raised_within_a_range(cuda, dtype, group):
    """Scores far above those before them, in the middle of a range: the sums so far, which other waves hold, are rescaled. A quarter of
    the heads sees one such key each at a third, a half and two thirds of a sequence (it and the sequence's other keys weigh about the
    same, so that a sum left as it was, or dropped, is seen), the last quarter scores that grow with every block of 32 keys."""
    from triton_dist.kernels.amd.flash_decode import decode_stream
    announce("decode stream latent, raised maxima, %s, %d heads per kv head" % (dtype, group))
    g = torch.Generator().manual_seed(group)
    hkv, B = 8, 24
    lens = [384 - 5 * (i % 7) for i in range(B)]   # 12 blocks each over 32 ranges of 9: sequences straddle ranges, ranges hold several
    q = torch.randn((B, hkv * group, 576), generator=g) * 0.25
    k, _, table = golden.make_paged_kv(B, 384, hkv, 576, 16, torch.float32, g, v_head_dim=512)
    kind = torch.arange(hkv * group) % 4
    q[:, :, 512:516] = torch.nn.functional.one_hot(kind, 4) * 12.875
    k[..., 512:516] = 0
    for b, n in enumerate(lens):
        for key in range(n):
            k[table[b, key // 16], key % 16, :, 515] = 0.35 * key   # 6 more per block, in the scores' e-logarithm
        for j, key in enumerate((n // 3, n // 2, 2 * n // 3)):
            k[table[b, key // 16], key % 16, :, 512 + j] = 12.875     # 6.9
    q, k = q.to(dtype), k.to(dtype)
    exact, exact_lse = golden.decode_exact(q, k, k[..., :512], lens, table, 576**-0.5, 0)
    # (on the oracle's side: without its one key, a head's other scores stay more than 8 in log2 below)
    flat = q.clone()
    flat[:, :, 512:515] = 0
    most = torch.stack([(flat[b].double() @ golden._gather_kv(k, table.numpy()[b], 0, n)[:, 0].double().t()).max(1).values for b, n in enumerate(lens)])
    raised = 6.9 - 576**-0.5 * most[:, (kind < 3) & (torch.arange(hkv * group) < group)] > 8 * 0.6931
    assert raised.double().mean() > 0.8
    kd = k.to(cuda)
    out, lse = torch.empty((B, hkv * group, 512), device=cuda), torch.empty((B, hkv * group), device=cuda)
    decode_stream(q.to(cuda), kd, kd[..., :512], torch.tensor(lens, dtype=torch.int32, device=cuda), table.to(cuda), 576**-0.5, 0.0, out, lse)
    assert (out.cpu().double() - exact).abs().max() <= ATOL
    assert (lse.cpu().double() - exact_lse).abs().max() <= ATOL


@pytest.mark.parametrize("hq,hkv,ranges", [(128, 1, 32), (24, 1, 128), (40, 2, 64)])
def test_latent_heads_in_half_the_workspace(cuda, hq, hkv, ranges):
    """The room for ``ranges`` ranges, as many as one block of 16 heads per workgroup has on 256 compute units, is enough; less is
    refused."""
    from triton_dist import _lib
    lib = _lib.load()
    lens = [3000, 0, 31, 700, 64]
    announce("decode stream latent heads=%d/%d with %d ranges" % (hq, hkv, ranges))
    g = torch.Generator().manual_seed(hq)
    q = torch.randn((5, hq, 576), generator=g).bfloat16()
    k, _, table = golden.make_paged_kv(5, 3000, hkv, 576, 16, torch.bfloat16, g, v_head_dim=512)
    exact, exact_lse = golden.decode_exact(q, k, k[..., :512], lens, table, 576**-0.5, 0)
    qd, kd, td, ld = q.to(cuda), k.to(cuda), table.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda)
    per_range = 2 * hq * 513 * 4
    assert lib.tdist_num_cus() == 256 and lib.tdist_decode_stream_workspace_bytes(5, hq, hkv, 576, 512) > ranges * per_range
    memory = torch.zeros(ranges * per_range + 64, dtype=torch.uint8, device=cuda)
    memory[-64:] = 7

    def call(nbytes):
        out, lse = torch.zeros((5, hq, 512), device=cuda), torch.zeros((5, hq), device=cuda)
        rc = lib.tdist_decode_stream(qd.data_ptr(), kd.data_ptr(), kd.data_ptr(), 576**-0.5, 0.0, td.data_ptr(), ld.data_ptr(), 5, hq, hkv,
                                     576, 512, 16, *qd.stride()[:2], *kd.stride()[:3], *kd.stride()[:3], td.stride(0), _lib.TDIST_BF16, None, 0,
                                     memory.data_ptr(), nbytes, out.data_ptr(), _lib.TDIST_F32, *out.stride()[:2], lse.data_ptr(), None)
        torch.cuda.synchronize()
        return rc, out.cpu().double(), lse.cpu().double()

    assert call(ranges * per_range - 1)[0] == _lib.TDIST_ERR_WORKSPACE
    rc, out, lse = call(ranges * per_range)
    live = ~torch.isinf(exact_lse)
    assert rc == _lib.TDIST_OK and bool((memory[-64:] == 7).all())
    assert (out - exact).abs().max() <= ATOL and (lse[live] - exact_lse[live]).abs().max() <= ATOL and torch.equal(torch.isinf(lse), ~live)
