"""Experts' last rows in short blocks of a list and a launch of their own: the two lists against the plain join's one, and the grouped
GEMM over both exactly as the oracle has it (whole numbers small enough for every sum)."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


def routing(counts, g):
    """ids [n, 1] with this many entries per expert, in any order."""
    ids = torch.cat([torch.full((n, ), e, dtype=torch.int32) for e, n in enumerate(counts)])
    return ids[torch.randperm(len(ids), generator=g)].view(-1, 1)


# tails of one row, of as many as are taken and one more, none, of whole short blocks; experts without rows and with nothing else; columns for
# which no round goes away; more short tiles than compute units; experts that a thread of the scan takes several of
CASES = [([256 * 4 + t for t in (1, 128, 0, 64)], 4096, True), ([256 * 4 + t for t in (129, 1, 255, 65)], 3584, True), ([1030] * 4, 512, False),
         ([0, 256 * 8 + 3, 100, 0, 256 * 7, 256], 4096, True), ([300] * 200, 8192, False), ([260] * 16 + [0] * 600 + [7] * 40, 4096, False),
         ([512 + 5] * 32, 1024, True), ([256 * 4 + 200] * 4, 4096, False)]


@pytest.mark.parametrize("counts,n,taken", CASES)
@pytest.mark.parametrize("block", [128, 64])
def test_both_lists(cuda, counts, n, taken, block):
    from triton_dist import _lib
    from triton_dist.kernels.amd import sort_topk_ids_align_block_size
    announce("join with tails: %d experts, %d rows, %d columns, blocks of %d" % (len(counts), sum(counts), n, block))
    g = torch.Generator().manual_seed(sum(counts))
    ids, E, entries, out, most = routing(counts, g).to(cuda), len(counts), sum(counts), 256, 128
    sorted_ids, experts, _, _, padded = sort_topk_ids_align_block_size(ids, E, 1, entries, block)
    n_blocks, n_tails = entries // out + E, max(1, 256 // -(-n // 128))
    a = [torch.full((size, ), -7, dtype=torch.int32, device=cuda) for size in (n_blocks * out, n_blocks, n_blocks, 1, n_tails * 64, n_tails, n_tails, 1)]
    p = [t.data_ptr() for t in a]
    _lib.call("tdist_moe_join_blocks_tails", sorted_ids.data_ptr(), experts.data_ptr(), padded.data_ptr(),
              min(experts.numel(), sorted_ids.numel() // block), block, entries, E, out, p[0], a[0].numel(), p[1], p[2], p[3], most, 64, n, p[4],
              a[4].numel(), p[5], p[6], p[7], _lib.stream_ptr())
    torch.cuda.synchronize()
    cus, cols = _lib.load().tdist_num_cus(), -(-n // 256)
    tail = [c % out if c % out <= most else 0 for c in counts]
    rounds = [-(-sum(-(-c // out) for c in cs) * cols // cus) for cs in (counts, [c - t for c, t in zip(counts, tail)])]
    short = sum(-(-t // 64) for t in tail)
    assert (rounds[1] < rounds[0] and short <= n_tails) == taken or cus != 256
    if not (rounds[1] < rounds[0] and short <= n_tails):
        tail = [0] * E
    flat = ids.view(-1).cpu()
    lists = [[], []]
    for e in range(E):
        rows = torch.nonzero(flat == e).view(-1).tolist()
        whole = counts[e] - tail[e]
        for to, part, size in ((0, rows[:whole], out), (1, rows[whole:], 64)):
            for at in range(0, len(part), size):
                lists[to].append((e, part[at:at + size] + [entries] * (size - len(part[at:at + size]))))
    for k, size in ((0, out), (1, 64)):
        got = [t.cpu() for t in a[4 * k:4 * k + 4]]
        used = len(lists[k])
        assert int(got[3]) == used * size
        assert got[1][:used].tolist() == [e for e, _ in lists[k]] and not got[2][:used].any()
        assert got[0][:used * size].tolist() == [r for _, rows in lists[k] for r in rows]
        assert (got[0][used * size:] == -7).all() and (got[1][used:] == -7).all()


@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 320), (torch.float16, 256), (torch.float8_e4m3fn, 640)])
@pytest.mark.parametrize("counts,n,taken", [CASES[0], CASES[3], ([1200, 1030, 1024, 1025], 3840, True), ([1030, 1100, 1279, 1279], 4096, False)])
def test_products_over_both_lists(cuda, dtype, K, counts, n, taken):
    from triton_dist import _lib
    from triton_dist.kernels.amd import allgather_group_gemm as gg, sort_topk_ids_align_block_size
    announce("grouped GEMM with tails: %s, %s rows, %d x %d" % (dtype, counts, n, K))
    g = torch.Generator().manual_seed(sum(counts))
    E, entries = len(counts), sum(counts)
    ids = routing(counts, g).to(cuda)
    a = torch.randint(-2, 3, (entries, K), generator=g).float().to(dtype).to(cuda)
    w = torch.randint(-2, 3, (E, n, K), generator=g).float().to(dtype).to(cuda)
    sorted_ids, experts, _, _, padded = sort_topk_ids_align_block_size(ids, E, 1, entries, 128)
    row_bytes, ws = K * a.element_size(), _lib.new_split_k_workspace(cuda)
    out_dtype = torch.float16 if dtype == torch.float16 else torch.bfloat16
    want = torch.stack([a.float() @ w[e].float().t() for e in range(E)]).to(out_dtype)[ids.view(-1).long(), torch.arange(entries, device=cuda)]
    with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, 0):   # (256-row blocks, whatever the estimate for so short a K)
        made = {}
        for _ in range(2):
            blocks = gg.joined_row_blocks(made, sorted_ids, experts, padded, 128, entries, E, n, row_bytes, _lib.stream_ptr(), any_block=True, sk_workspace=ws)
            assert blocks.block_size == 256
            if blocks.tail is None:   # (the host's estimate goes by the mean)
                blocks.tail_most = 128
                blocks.tail = gg.RowBlocks.of(torch.empty(2 * E * 66 + 1, dtype=torch.int32, device=cuda), 0, 2 * E, 64)
                blocks = gg.joined_row_blocks(made, sorted_ids, experts, padded, 128, entries, E, n, row_bytes, _lib.stream_ptr(), any_block=True,
                                              sk_workspace=ws)
            c = torch.full((entries, n), float("nan"), dtype=out_dtype, device=cuda)
            gg.group_gemm_rows(dtype, _lib.address_table(a), 1, entries, w, c, blocks, entries, 1, None, ws, _lib.stream_ptr())
            torch.cuda.synchronize()
            tail = blocks.tail.memory[(blocks.tail.padded - blocks.tail.memory.data_ptr()) // 4]
            assert (int(tail) > 0) == taken or _lib.load().tdist_num_cus() != 256
            assert torch.equal(c, want)


def test_no_room_for_the_tails_places(cuda):
    """Blocks and experts for which the plain join's words fill the LDS: the same first list as by it, and nothing in the second."""
    from triton_dist import _lib
    from triton_dist.kernels.amd import sort_topk_ids_align_block_size
    announce("join with tails, the LDS full")
    counts, block, out, n = CASES[0][0], 64, 256, 4096
    E, entries, words = len(counts), sum(counts), (160 * 1024 - 256) // 4
    ids = routing(counts, torch.Generator().manual_seed(5)).to(cuda)
    sorted_ids, experts, _, _, padded = sort_topk_ids_align_block_size(ids, E, 1, entries, block)
    n_blocks, n_tails = entries // out + E, 8
    for num_blocks, room in ((words - 3 * E, True), (words - 3 * E + 1, False), (words - 2 * E, False)):
        ids_in = torch.full((num_blocks * block, ), entries, dtype=torch.int32, device=cuda)
        experts_in = torch.zeros(num_blocks, dtype=torch.int32, device=cuda)
        used = min(experts.numel(), sorted_ids.numel() // block)
        ids_in[:used * block], experts_in[:used] = sorted_ids[:used * block], experts[:used]

        def outputs():
            return [torch.full((size, ), -7, dtype=torch.int32, device=cuda) for size in (n_blocks * out, n_blocks, n_blocks, 1, n_tails * 64, n_tails, n_tails, 1)]

        a, b = outputs(), outputs()
        args = (ids_in.data_ptr(), experts_in.data_ptr(), padded.data_ptr(), num_blocks, block, entries, E, out)
        p, q = [t.data_ptr() for t in a], [t.data_ptr() for t in b]
        _lib.call("tdist_moe_join_blocks", *args, q[0], b[0].numel(), q[1], q[2], q[3], _lib.stream_ptr())
        _lib.call("tdist_moe_join_blocks_tails", *args, p[0], a[0].numel(), p[1], p[2], p[3], 128, 64, n, p[4], a[4].numel(), p[5], p[6], p[7],
                  _lib.stream_ptr())
        torch.cuda.synchronize()
        if room:
            assert int(a[7]) > 0 or _lib.load().tdist_num_cus() != 256
            continue
        assert int(a[7]) == 0 and all((t == -7).all() for t in a[4:7])
        assert all(torch.equal(x, y) for x, y in zip(a[:4], b[:4]))


def test_a_second_list_that_is_refused_launches_nothing(cuda):
    from triton_dist import _lib
    announce("grouped GEMM with tails: refusals")
    n, K, rows = 512, 256, 256
    a, w = torch.ones((rows, K), dtype=torch.bfloat16, device=cuda), torch.ones((1, n, K), dtype=torch.bfloat16, device=cuda)
    c = torch.full((rows, n), -3.0, dtype=torch.bfloat16, device=cuda)
    ids, zero = torch.arange(rows, dtype=torch.int32, device=cuda), torch.zeros(64, dtype=torch.int32, device=cuda)
    total = torch.full((1, ), rows, dtype=torch.int32, device=cuda)
    z = zero.data_ptr()

    def call(tail=(z, z, z, z), blocks=1, ldb=K):
        return _lib.load().tdist_group_gemm_rows_tails(_lib.TDIST_BF16, _lib.address_table(a), 1, rows, w.data_ptr(), ldb, n * K, c.data_ptr(), n, n, K,
                                                       ids.data_ptr(), z, z, total.data_ptr(), 1, 256, rows, 1, *tail, blocks, None, None, None, 0,
                                                       _lib.stream_ptr())

    for i in range(4):
        assert call(tail=tuple(None if k == i else z for k in range(4))) == _lib.TDIST_ERR_INVALID
    assert call(blocks=0) == _lib.TDIST_ERR_INVALID
    assert call(ldb=1 << 21) == _lib.TDIST_ERR_UNSUPPORTED   # (4 MiB a row: an expert's weights would be 2 GiB)
    torch.cuda.synchronize()
    assert (c == -3).all()
    assert call() == _lib.TDIST_OK
    torch.cuda.synchronize()
    assert (c == K).all()


def test_what_the_join_with_tails_refuses(cuda):
    from triton_dist import _lib
    lib = _lib.load()
    p = torch.zeros(64, dtype=torch.int32, device=cuda).data_ptr()
    call = lambda most, block, n, rows, ids=p: lib.tdist_moe_join_blocks_tails(p, p, p, 1, 128, 4, 4, 256, p, 256, p, p, p, most, block, n, ids, rows, p, p, p, None)
    assert call(0, 64, 256, 64) == call(256, 64, 256, 64) == call(128, 0, 256, 64) == call(128, 64, 0, 64) == call(128, 64, 256, 63) == call(128, 96, 256, 96) == _lib.TDIST_ERR_INVALID
    assert call(128, 64, 256, 64, None) == _lib.TDIST_ERR_INVALID
    assert lib.tdist_group_gemm_tail_rows(0, 8, 4096, 4096, 256) == lib.tdist_group_gemm_tail_rows(16384, 8, 4096, 4096, 128) == 0
