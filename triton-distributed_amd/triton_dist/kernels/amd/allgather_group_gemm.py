"""MoE tensor-parallel AG + grouped GEMM on one MI355X: the align / sort of the routing and the chunk-gated grouped
GEMM that consumes it.

Keeps the interface of the reference's kernels/nvidia/allgather_group_gemm.py: ``sort_topk_ids_align_block_size``
(:54-135; its device work is the C++ op moe_ag_scatter_align_block_size, csrc/lib/moe_utils.cu:60-186),
``MoE_AllGatherGroupGEMMTensorParallelContext`` (:494-553), ``create_ag_group_gemm_intra_node_context`` (:555-638)
and ``ag_group_gemm_intra_node`` (:641-691). As in the AG-GEMM, the other ranks' token rows are handed to the context
(``ctx.set_peer_shards``) and copy streams of this GPU deliver them into the workspace and release one flag per rank
segment (the reference's producer: cp_engine_producer_all_gather_full_mesh_push, one barrier word per rank).
"""
import dataclasses
from typing import Dict, List, Optional

import torch

from triton_dist import _lib
from triton_dist.kernels.amd.common_ops import fill_flags


_ALIGN_PLANS = {}   # (ids, experts, ranks, topk, block size) -> scratch bytes and the layout of the results


def sort_topk_ids_align_block_size(
    topk_ids: torch.Tensor,
    num_experts: int,
    num_ranks: int,
    num_tokens_per_rank: int,
    block_size: int,
    moe_stream: torch.cuda.Stream = None,
):
    """
    Sort and align the token distribution across experts to be compatible with block size for matrix multiplication.

    Parameters (reference :62-72):
    - topk_ids: [total_tokens, top_k] expert index of every (token, k), int64 (the reference's dtype) or int32.
    - num_experts, num_ranks, num_tokens_per_rank (tokens, not topk-ed, per rank), block_size.
    - moe_stream: stream for the kernels; the current stream if None.

    Returns (sorted_token_ids, expert_ids, block_barrier_ids, rank_block_num, num_tokens_post_padded), all int32,
    allocated with the reference's capacities (:100-121); padding positions of sorted_token_ids hold
    topk_ids.numel().
    """
    _lib.require_cuda(topk_ids)
    if topk_ids.dtype not in (torch.int32, torch.int64):
        raise TypeError("topk_ids must be int32 or int64, got %s" % topk_ids.dtype)
    topk_ids = topk_ids.contiguous()
    num_topk = topk_ids.shape[1]
    dev = topk_ids.device
    n_total = topk_ids.numel()
    n_per = num_tokens_per_rank * num_topk
    assert n_total == n_per * num_ranks, "topk_ids must hold num_ranks * num_tokens_per_rank tokens"
    # sizes and scratch bytes once per shape: the call itself costs less than working them out again
    key = (n_total, num_experts, num_ranks, num_topk, block_size)
    plan = _ALIGN_PLANS.get(key)
    if plan is None:
        ws_bytes = _lib.load().tdist_moe_align_workspace_bytes(n_total, num_experts, num_ranks)
        if ws_bytes == 0:
            raise _lib.TdistError(_lib.TDIST_ERR_UNSUPPORTED,
                                  "num_experts * num_ranks = %d is above what the align kernel handles" % (num_experts * num_ranks))
        # the five results are views of one allocation (sizes as in the reference, :100-121; every view 16-byte aligned)
        n_sorted = (n_per + num_experts * (block_size - 1)) * num_ranks
        n_blocks = (n_per + num_experts) * num_ranks
        sizes = (n_sorted, n_blocks, n_blocks, num_ranks, 1)
        starts, at = [], 0
        for n in sizes:
            starts.append(at)
            at += (n + 3) // 4 * 4
        plan = _ALIGN_PLANS[key] = (ws_bytes, at, tuple(starts), sizes)
    ws_bytes, n_flat, starts, sizes = plan
    if moe_stream is None:
        out = _lib.native().align(topk_ids, num_experts, num_ranks, block_size, starts, sizes, n_flat, _lib.zeroed_scratch(ws_bytes, dev), ws_bytes)
        if out is not None:
            return out
    flat = torch.empty(n_flat, dtype=torch.int32, device=dev)
    sorted_ids, expert_ids, block_barrier_ids, rank_block_num, num_tokens_post_pad = [
        flat[a:a + n] for a, n in zip(starts, sizes)]
    base = flat.data_ptr()
    ids_ptr, ids_int64 = topk_ids.data_ptr(), 1 if topk_ids.dtype == torch.int64 else 0

    def launch(stream):
        workspace = _lib.zeroed_scratch(ws_bytes, dev)   # (cached per stream: current is `stream` here)
        # (sorted_ids.fill_(numel) of the reference, :103, is done inside the call)
        _lib.call("tdist_moe_align_block_size", ids_ptr, ids_int64, n_total, num_experts, num_ranks, n_per, block_size,
                  base + 4 * starts[0], sizes[0], base + 4 * starts[1], base + 4 * starts[2], base + 4 * starts[3],
                  base + 4 * starts[4], workspace.data_ptr(), ws_bytes, stream)

    if moe_stream is None:
        launch(_lib.stream_ptr())      # no stream switch, event, Stream object or allocator bookkeeping to pay for
    else:
        with torch.cuda.stream(moe_stream):
            launch(moe_stream.cuda_stream)
        torch.cuda.current_stream().wait_stream(moe_stream)
    return (
        sorted_ids,
        expert_ids,
        block_barrier_ids,
        rank_block_num,
        num_tokens_post_pad,
    )


# Relative time of a 256 x 256 and a 128 x 256 tile (the smaller one runs at 0.8 of the larger one's rate), for the choice
# of the row block where neither the caller's is asked for nor _block_plan has one.
_BLOCK_COST = {256: 1.0, 128: 0.625}


def _row_block(entries, num_experts, n, cus):
    """Rows per block for ``entries`` (token, k) pairs spread over the experts, ``n`` output columns: every expert with rows
    pads half a block on average, and fewer tiles than compute units leave some idle whatever the tile. 256 from 192
    rows per expert on, where the chip is full (2 x 8192 entries over 8 experts, a whole layer of 4096 x 1792: 513 us against
    637 with 128; 2 x 174 rows by 6 over 64 experts, 4352 x 1024: 347 against 288)."""
    used, cols = min(num_experts, entries), -(-n // 256)
    return min(_BLOCK_COST, key=lambda b: max(1.0, (entries / b + 0.5 * used) * cols / cus) * _BLOCK_COST[b])


def _join_plan(entries, num_experts, n):
    """Rows per joined block and the most blocks they can be."""
    block = _row_block(entries, num_experts, n, _lib.load().tdist_num_cus())
    return block, (entries + num_experts * (block - 1)) // block


def _block_plan(entries, num_experts, n, row_bytes, sk_workspace):
    """Rows per joined block and the most blocks they can be for tdist_group_gemm_rows, which knows more forms than
    _row_block does and tells which one is the fastest (16 to 18731 rows over 8 to 64 experts: 39 % on average). None: it cannot."""
    block = _lib.load().tdist_group_gemm_row_block(entries, num_experts, n, row_bytes, _lib.workspace_args(sk_workspace)[1])
    return (block, (entries + min(num_experts, entries) * (block - 1)) // block) if block > 0 else None


class RowBlocks:
    """Addresses of a grouped GEMM's row blocks (sorted ids, an expert and a segment per block, the padded total), their
    number and their rows; ``memory``: the tensor they lie in."""
    __slots__ = ("sorted_ids", "experts", "segments", "padded", "num_blocks", "block_size", "memory", "tail", "tail_most")

    def __init__(self, sorted_ids, experts, segments, padded, num_blocks, block_size, memory=None):
        self.sorted_ids, self.experts, self.segments, self.padded = sorted_ids, experts, segments, padded
        self.num_blocks, self.block_size, self.memory = num_blocks, block_size, memory
        self.tail, self.tail_most = None, 0   # experts' last rows in RowBlocks of their own, and how many of them at most (0: none)

    @classmethod
    def of(cls, memory, at, num_blocks, block_size):
        """Blocks in int32 ``memory`` from element ``at`` on."""
        base, rows = memory.data_ptr() + 4 * at, num_blocks * block_size
        return cls(base, base + 4 * rows, base + 4 * (rows + num_blocks), base + 4 * (rows + 2 * num_blocks), num_blocks, block_size, memory)

    def fields(self):
        t = self.tail
        return (self.sorted_ids, self.experts, self.segments, self.padded, self.num_blocks, self.block_size, self.tail_most,
                0 if t is None else t.sorted_ids, 0 if t is None else t.num_blocks)


def joined_row_blocks(made, sorted_ids, expert_ids, num_tokens_post_padded, block_size, entries, num_experts, n, row_bytes, stream, gather=None,
                      any_block=False, sk_workspace=None):
    """The rows of ``sorted_ids`` in blocks without rank segments, for a grouped GEMM with ``n`` output columns that waits for
    nobody: RowBlocks, or None where the GEMM does not take rows of ``row_bytes`` in such blocks or the sizes are beyond
    tdist_moe_join_blocks (nothing has been launched then).

    Blocks that end with their rank segment only add padding where all rows are there (Mixtral's 8 experts x 8 ranks at
    16384 entries: 160 blocks of 128 rows for 128 that are full, and no 256-row ones), also where the chip has room for all
    of them: fewer tiles are cut along K (8 x 28 tokens by 4 over 8 experts, a layer of 5248 x 1280: 107 us joined, 198 as sorted).
    They are joined on every call, from what the tensors hold then: a caller may replace or rewrite any of them, also between
    the replays of a graph. (Kept from call to call they cost 7 to 14 us less a layer, and a rewritten routing went unseen.)
    ``made``: the context's memory for them, a RowBlocks per size (a graph may hold the address of any of them).
    ``gather``: the arguments of tdist_gather_shards but its stream; the same launch then gathers. ``any_block``: the caller's
    GEMM is tdist_group_gemm_rows with ``sk_workspace``, whatever the block."""
    if not (row_bytes % 128 == 0 or row_bytes > 128):
        return None
    _lib.require_cuda(sorted_ids, expert_ids, num_tokens_post_padded)
    key = (entries, num_experts, n, any_block and row_bytes)
    if gather is not None:
        key += ("gather", )   # (that launch makes no tails)
    out = made.get(key)
    if out is None:
        plan = _block_plan(entries, num_experts, n, row_bytes, sk_workspace) if any_block else None
        block, n_blocks = plan or _join_plan(entries, num_experts, n)
        tail_most = _lib.load().tdist_group_gemm_tail_rows(entries, num_experts, n, row_bytes, block) if any_block and gather is None else 0
        # (as many as leave two of their tiles of 128 columns to a compute unit; and with fewer places the GEMM would take K apart for them)
        tail_blocks = min(min(num_experts, entries) * (tail_most // _lib.GROUP_TAIL_BLOCK), 2 * _lib.load().tdist_num_cus() // -(-n // 128))
        size = n_blocks * (block + 2) + 1
        memory = torch.empty(size + (tail_blocks * (_lib.GROUP_TAIL_BLOCK + 2) + 1 if tail_most else 0), dtype=torch.int32, device=sorted_ids.device)
        out = made[key] = RowBlocks.of(memory, 0, n_blocks, block)
        if tail_most:
            out.tail, out.tail_most = RowBlocks.of(memory, size, tail_blocks, _lib.GROUP_TAIL_BLOCK), tail_most
    args = (sorted_ids.data_ptr(), expert_ids.data_ptr(), num_tokens_post_padded.data_ptr(),
            min(expert_ids.numel(), sorted_ids.numel() // block_size), block_size, entries, num_experts, out.block_size, out.sorted_ids,
            out.num_blocks * out.block_size, out.experts, out.segments, out.padded)
    lib, tail = _lib.load(), out.tail
    if gather is not None:
        rc = lib.tdist_moe_gather_and_join(*gather, *args, stream)
    elif tail is not None:
        rc = lib.tdist_moe_join_blocks_tails(*args, out.tail_most, _lib.GROUP_TAIL_BLOCK, n, tail.sorted_ids, tail.num_blocks * _lib.GROUP_TAIL_BLOCK, tail.experts,
                                             tail.segments, tail.padded, stream)
    else:
        rc = lib.tdist_moe_join_blocks(*args, stream)
    if rc == _lib.TDIST_ERR_UNSUPPORTED:
        return None
    _lib.check(rc)
    return out


_GROUP_GEMM_ENTRY = {
    torch.bfloat16: "tdist_group_gemm_gated_bf16",
    torch.float16: "tdist_group_gemm_gated_f16",
    torch.float8_e4m3fn: "tdist_group_gemm_gated_fp8e4m3",
}


def group_gemm_gated(a_ws, a_local, local_row_begin, b_nk, c, sorted_token_ids, expert_ids, block_barrier_ids,
                     num_tokens_post_padded, block_size, num_valid_tokens, topk, tokens_per_rank, first_block, flags, rank,
                     *, wait_value=1, spin_limit=0, status=None, max_workgroups=0, sk_workspace=None, stream=None):
    """Thin wrapper over tdist_group_gemm_gated_*. ``a_ws`` [tokens, K] gathered rows, ``a_local`` the own shard or
    None, ``b_nk`` [E, N, K] (K contiguous), ``c`` [num_valid_tokens, N]."""
    _lib.require_cuda(sorted_token_ids, expert_ids, block_barrier_ids, num_tokens_post_padded)
    blocks = RowBlocks(sorted_token_ids.data_ptr(), expert_ids.data_ptr(), block_barrier_ids.data_ptr(), num_tokens_post_padded.data_ptr(),
                       min(expert_ids.numel(), sorted_token_ids.numel() // block_size), int(block_size))
    return _group_gemm(a_ws, a_local, local_row_begin, b_nk, c, blocks, num_valid_tokens, topk, tokens_per_rank, first_block, flags, rank,
                       wait_value, spin_limit, status, max_workgroups, sk_workspace, stream)


def _group_gemm(a_ws, a_local, local_row_begin, b_nk, c, blocks, num_valid_tokens, topk, tokens_per_rank, first_block, flags, rank,
                wait_value=1, spin_limit=0, status=None, max_workgroups=0, sk_workspace=None, stream=None):
    _lib.require_cuda(a_ws, b_nk, c)
    if a_ws.dtype not in _GROUP_GEMM_ENTRY:
        raise TypeError("unsupported grouped GEMM dtype %s" % a_ws.dtype)
    if a_ws.stride(1) != 1 or b_nk.stride(2) != 1 or c.stride(1) != 1:
        raise ValueError("A, B ([E, N, K]) and C need a contiguous last dimension")
    E, N, K = b_nk.shape
    assert a_ws.shape[1] == K and c.shape[1] == N
    _lib.call(_GROUP_GEMM_ENTRY[a_ws.dtype], a_ws.data_ptr(), a_ws.stride(0), _lib.ptr(a_local),
              a_local.stride(0) if a_local is not None else 0, int(local_row_begin),
              a_local.shape[0] if a_local is not None else 0, b_nk.data_ptr(), b_nk.stride(1), b_nk.stride(0), c.data_ptr(),
              c.stride(0), a_ws.shape[0], N, K, blocks.sorted_ids, blocks.experts, blocks.segments, blocks.padded, blocks.num_blocks,
              blocks.block_size,
              int(num_valid_tokens), int(topk), int(tokens_per_rank), int(first_block), _lib.ptr(flags), int(wait_value),
              int(rank), int(spin_limit), _lib.ptr(status), int(max_workgroups), *_lib.workspace_args(sk_workspace),
              _lib.stream_ptr(stream))
    return c


def any_block_fits(a_rows, row_bytes, b_nk, elem_size):
    """Whether tdist_group_gemm_rows takes such operands in blocks of any size (its offsets are of 32 bits)."""
    return a_rows * row_bytes < 1 << 32 and b_nk.shape[1] * b_nk.stride(1) * elem_size < 1 << 31


def group_gemm_rows(dtype, shards, num_shards, rows_per_shard, b_nk, c, blocks, num_valid_tokens, topk, status=None, sk_workspace=None, stream=None):
    """Thin wrapper over tdist_group_gemm_rows. ``shards``: addresses of the shards, or of all rows in one piece."""
    if b_nk.stride(2) != 1 or c.stride(1) != 1:
        raise ValueError("A, B ([E, N, K]) and C need a contiguous last dimension")
    _, N, K = b_nk.shape
    assert c.shape[1] == N
    args = (_lib.dtype_code(dtype), shards, num_shards, rows_per_shard, b_nk.data_ptr(), b_nk.stride(1), b_nk.stride(0), c.data_ptr(), c.stride(0),
            N, K, blocks.sorted_ids, blocks.experts, blocks.segments, blocks.padded, blocks.num_blocks, blocks.block_size, int(num_valid_tokens),
            int(topk))
    rest = (status, None if status is None else status + 8, *_lib.workspace_args(sk_workspace), stream)
    tail = blocks.tail
    if tail is None:
        _lib.call("tdist_group_gemm_rows", *args, *rest)
    else:
        _lib.call("tdist_group_gemm_rows_tails", *args, tail.sorted_ids, tail.experts, tail.segments, tail.padded, tail.num_blocks, *rest)
    return c


@dataclasses.dataclass
class MoE_AllGatherGroupGEMMTensorParallelContext:
    rank: int
    num_ranks: int
    num_experts: int
    topk: int
    full_num_tokens: int
    sorted_topk_ids: torch.Tensor
    aligned_expert_ids: torch.Tensor
    aligned_barrier_ids: torch.Tensor
    aligned_num_tokens: torch.Tensor
    workspace_tensors: List[Optional[torch.Tensor]]
    barrier_tensors: List[Optional[torch.Tensor]]
    internode_ag_stream: Optional[torch.cuda.streams.Stream] = None
    ag_stream: Optional[torch.cuda.streams.Stream] = None
    group_gemm_stream: Optional[torch.cuda.streams.Stream] = None
    local_world_size: int = 8
    BLOCK_M: int = 128
    BLOCK_N: int = 256
    BLOCK_K: int = 64
    GROUP_SIZE_M: int = 8
    stages: int = 3
    warps: int = 8
    # ---- one-GPU additions -------------------------------------------------------------------
    rank_block_num: Optional[torch.Tensor] = None
    first_block: int = 0                 # first row block of the own rank's segment (consumed first)
    peer_shards: Dict[int, torch.Tensor] = dataclasses.field(default_factory=dict)
    one: Optional[torch.Tensor] = None
    status: Optional[torch.Tensor] = None
    spin_limit: int = 0
    held_ranks: tuple = ()               # test hook: segments that are never delivered
    producer_cus: int = 32               # compute units left to the copies (see the AG-GEMM context)
    weight_nk: Optional[torch.Tensor] = None   # [E, N, K] copy of a [E, K, N] weight, made once per weight tensor
    weight_key: Optional[tuple] = None
    sk_workspace: Optional[torch.Tensor] = None   # the context's GEMM workspace (split of a last round along K); None = off
    # False: the other ranks' rows come by copies beside a GEMM that waits for their flags also where they are at hand and
    # one launch could gather them in front of it
    gather_rows: bool = True
    joined: dict = dataclasses.field(default_factory=dict)   # memory for the row blocks of a call, see joined_row_blocks

    def set_peer_shards(self, shards):
        """``shards``: dict rank -> [M_per_rank, K] tensor (or a list; the own entry is ignored): the token rows that
        live on the other ranks."""
        if not isinstance(shards, dict):
            shards = {r: t for r, t in enumerate(shards) if t is not None}
        for r, t in shards.items():
            if r != self.rank:
                _lib.require_cuda(t)
                if not t.is_contiguous():
                    raise ValueError("peer shard of rank %d must be contiguous" % r)
        self.peer_shards = {r: t for r, t in shards.items() if r != self.rank}

    def check_status(self):
        """Synchronises and raises TdistError if a bounded flag wait expired in an earlier call (the earliest one
        since the last check; status[0:2] is the current call's, [2:4] the first of the calls before it)."""
        torch.cuda.synchronize()
        code, segment, first_code, first_segment = self.status.tolist()
        if first_code != 0:
            code, segment = first_code, first_segment
        if code != 0:
            self.status.zero_()
            raise _lib.TdistError(code, "flag wait expired for rank segment %d" % segment)


def create_ag_group_gemm_intra_node_context(tp_pg, tensor_A, tensor_B, full_topk_ids, num_experts, max_M=2**14, BLOCK_M=128,
                                            BLOCK_N=256, BLOCK_K=64, GROUP_SIZE_M=8, stages=3, warps=8, ag_stream=None,
                                            group_gemm_stream=None, rank=None, num_ranks=None, split_k=True):
    """create context for allgather group gemm intra-node (reference :555-638).

    tensor_A [M_per_rank, K] local tokens, tensor_B [E, K, N_per_rank] local expert weights, full_topk_ids
    [M_per_rank * num_ranks, topk]. ``tp_pg`` may be None on one GPU: pass ``rank`` / ``num_ranks``. BLOCK_M is the
    row block of the align / sort and of the GEMM tile (128 or 256); the other tiling arguments are accepted for
    signature compatibility. ``split_k``: give the context a GEMM workspace (64 MiB): the number of row blocks
    in use is seldom a multiple of the grid, and with the workspace the grouped GEMM cuts the tiles of a last round that
    fills at most half of the grid along K."""
    if not torch.cuda.is_available():
        raise RuntimeError("create_ag_group_gemm_intra_node_context needs a GPU")
    _lib.check(_lib.load().tdist_init())
    M_per_rank, K = tensor_A.shape
    _, topk = full_topk_ids.shape
    assert tensor_B.shape[1] == K, "tensor_B should have shape [E, %d, N_per_rank], got %s" % (K, tuple(tensor_B.shape))
    assert tensor_A.dtype == tensor_B.dtype
    if tp_pg is not None:
        rank, num_ranks = tp_pg.rank(), tp_pg.size()
    assert rank is not None and num_ranks is not None
    assert full_topk_ids.shape[0] == M_per_rank * num_ranks and M_per_rank * num_ranks <= max_M
    device = tensor_A.device
    workspaces: List[Optional[torch.Tensor]] = [None] * num_ranks
    barriers: List[Optional[torch.Tensor]] = [None] * num_ranks
    workspaces[rank] = torch.empty([max_M, K], dtype=tensor_A.dtype, device=device)
    barriers[rank] = torch.zeros([num_ranks], dtype=torch.int32, device=device)
    sorted_ids, expert_ids, barrier_ids, rank_block_num, post_pad = sort_topk_ids_align_block_size(
        full_topk_ids, num_experts, num_ranks, M_per_rank, BLOCK_M)
    torch.cuda.synchronize()
    first_block = int(rank_block_num[:rank].sum().item()) if rank > 0 else 0
    return MoE_AllGatherGroupGEMMTensorParallelContext(
        rank=rank, num_ranks=num_ranks, num_experts=num_experts, topk=topk, full_num_tokens=full_topk_ids.numel(),
        sorted_topk_ids=sorted_ids, aligned_expert_ids=expert_ids, aligned_barrier_ids=barrier_ids,
        aligned_num_tokens=post_pad, workspace_tensors=workspaces, barrier_tensors=barriers,
        ag_stream=torch.cuda.Stream() if ag_stream is None else ag_stream,
        group_gemm_stream=group_gemm_stream, BLOCK_M=BLOCK_M, BLOCK_N=BLOCK_N, BLOCK_K=BLOCK_K,
        GROUP_SIZE_M=GROUP_SIZE_M, stages=stages, warps=warps, rank_block_num=rank_block_num, first_block=first_block,
        one=torch.ones((16, ), dtype=torch.int32, device=device), status=torch.zeros((4, ), dtype=torch.int32, device=device),
        sk_workspace=_lib.new_split_k_workspace(device) if split_k else None)


def _gather_and_multiply(a, b_nk, c, ctx, shards):
    """With every rank's rows at hand: one launch joins the row blocks across the rank segments (and brings the rows into the
    workspace where they lie too far apart to be read where they are), the next multiplies them, on one stream. Against
    copies beside a flag-gated GEMM on 32 compute units less, in blocks that end with their segment (8 x 1024 tokens by 4096,
    top 2 of 8 experts, 1792 columns): 339 -> 219 us with the gather. False where the blocks cannot be joined (nothing has been
    launched then). The workspace is scratch here."""
    M_per_rank, K = a.shape
    workspace = ctx.workspace_tensors[ctx.rank]
    M = M_per_rank * ctx.num_ranks
    current = _lib.stream_ptr()
    stream = current if ctx.group_gemm_stream is None else ctx.group_gemm_stream.cuda_stream
    if stream != current:
        ctx.group_gemm_stream.wait_stream(torch.cuda.current_stream())
    row_bytes = K * a.element_size()
    known = a.dtype in _GROUP_GEMM_ENTRY
    in_place = known and _lib.shards_in_reach(shards, M_per_rank, row_bytes)
    any_block = known and any_block_fits(M, row_bytes, b_nk, a.element_size())
    status = ctx.status.data_ptr()
    blocks = joined_row_blocks(ctx.joined, ctx.sorted_topk_ids, ctx.aligned_expert_ids, ctx.aligned_num_tokens, ctx.BLOCK_M, ctx.full_num_tokens,
                               b_nk.shape[0], b_nk.shape[1], row_bytes, stream,
                               gather=None if in_place else (workspace.data_ptr(), shards, ctx.num_ranks, M_per_rank * row_bytes, status, status + 8),
                               any_block=any_block, sk_workspace=ctx.sk_workspace)
    if blocks is None:
        return False
    assert b_nk.shape[2] == K
    if in_place:
        group_gemm_rows(a.dtype, shards, ctx.num_ranks, M_per_rank, b_nk, c, blocks, ctx.full_num_tokens, ctx.topk, status, ctx.sk_workspace, stream)
    elif any_block:
        group_gemm_rows(a.dtype, _lib.address_table(workspace), 1, M, b_nk, c, blocks, ctx.full_num_tokens, ctx.topk, None, ctx.sk_workspace, stream)
    else:
        _group_gemm(workspace[:M], None, 0, b_nk, c, blocks, ctx.full_num_tokens, ctx.topk, M, 0, None, ctx.rank,
                    sk_workspace=ctx.sk_workspace, stream=ctx.group_gemm_stream)
    if stream != current:
        torch.cuda.current_stream().wait_stream(ctx.group_gemm_stream)
    return True


def _weight_nk(ctx, b):
    """[E, K, N] weights as an [E, N, K] K-contiguous tensor: a view when the caller's tensor already is one
    (stride of K == 1), else a transposed copy made once per weight tensor and kept in the context."""
    if b.stride(1) == 1:
        return b.transpose(1, 2)
    key = (b.data_ptr(), tuple(b.shape), b._version)
    if ctx.weight_key != key:
        ctx.weight_nk = b.transpose(1, 2).contiguous()
        ctx.weight_key = key
    return ctx.weight_nk


def ag_group_gemm_intra_node(a, b, ctx=None, full_topk_ids=None, num_experts=None):
    """intra-node allgather group gemm (reference :641-691)

    a [M_per_rank, K] local tokens, b [E, K, N_per_rank] local expert weights. Returns C [M * topk, N_per_rank]:
    row t*topk + k is token t of the gathered A times the weights of its k-th expert."""
    if ctx is None:
        raise RuntimeError("one GPU holds a single rank: create the context first and hand it the peers' rows")
    M_per_rank, K = a.shape
    E, _, N_per_rank = b.shape
    W, rank = ctx.num_ranks, ctx.rank
    if W > 1 and ctx.gather_rows and not ctx.held_ranks and ctx.group_gemm_stream is None:
        blocks = ctx.joined.get((ctx.full_num_tokens, E, N_per_rank, K * a.element_size()))   # (what _gather_and_multiply has made)
        if blocks is not None:
            C = _lib.native().ag_group_gemm(a, b, ctx.peer_shards, rank, W, ctx.topk, ctx.workspace_tensors[rank], ctx.status, ctx.sk_workspace,
                                            ctx.sorted_topk_ids, ctx.aligned_expert_ids, ctx.aligned_num_tokens, ctx.BLOCK_M, ctx.full_num_tokens,
                                            *blocks.fields())
            if C is not None:
                return C
    _lib.require_cuda(a, b)
    missing = [r for r in range(W) if r != rank and r not in ctx.peer_shards]
    if missing:
        raise RuntimeError("hand the other ranks' token rows to the context first (ctx.set_peer_shards); missing %s" % missing)
    out_dtype = a.dtype if a.dtype in (torch.bfloat16, torch.float16) else torch.bfloat16
    # the routing names rows of C, the gather and the copies write what ``a`` is sized, and the GEMM reads b as a's type
    if ctx.full_num_tokens > ctx.topk * M_per_rank * W:
        raise ValueError("the context's routing is of %d rows, the call of %d" % (ctx.full_num_tokens, ctx.topk * M_per_rank * W))
    if b.shape[1] != K or a.element_size() != b.element_size():
        raise ValueError("Incompatible operands: %s %s and %s %s" % (tuple(a.shape), a.dtype, tuple(b.shape), b.dtype))
    if ctx.workspace_tensors[rank].nbytes < W * a.nbytes:
        raise ValueError("the context's workspace has no room for %d shards of %d x %d %s" % (W, M_per_rank, K, a.dtype))
    C = torch.empty([ctx.topk * M_per_rank * W, N_per_rank], dtype=out_dtype, device=a.device)
    b_nk = _weight_nk(ctx, b)
    if W > 1 and ctx.gather_rows and not ctx.held_ranks and a.is_contiguous() and (M_per_rank * K * a.element_size()) % 16 == 0:
        shards = _lib.shard_table(a, ctx.peer_shards, rank, W)
        if shards is not None and _gather_and_multiply(a, b_nk, C, ctx, shards):
            return C
    workspace, barrier = ctx.workspace_tensors[rank], ctx.barrier_tensors[rank]
    if workspace.element_size() != a.element_size():   # (the GEMM takes rows and type from it)
        raise ValueError("the workspace holds %s, not %s" % (workspace.dtype, a.dtype))
    current = torch.cuda.current_stream()
    gemm_stream = current if ctx.group_gemm_stream is None else ctx.group_gemm_stream
    fork = current.record_event()   # one event for both streams; a GEMM on the caller's own stream needs none
    ctx.ag_stream.wait_event(fork)
    if gemm_stream is not current:
        gemm_stream.wait_event(fork)
    # producer: one copy and one flag per peer rank (reference :354-361)
    nbytes = M_per_rank * K * a.element_size()
    for idx in range(1, W):
        r = (rank + idx) % W
        if r in ctx.held_ranks:
            continue
        _lib.call("tdist_producer_push_chunk", workspace.data_ptr() + r * nbytes, ctx.peer_shards[r].data_ptr(), nbytes,
                  barrier.data_ptr() + 4 * r, ctx.one.data_ptr(), 0, ctx.ag_stream.cuda_stream)
    max_wgs = max(1, _lib.load().tdist_num_cus() - ctx.producer_cus) if (W > 1 and ctx.producer_cus > 0) else 0
    # the launch before may have given up on a flag: keep what it reported, start this one clean
    _lib.call("tdist_status_retire", ctx.status.data_ptr(), ctx.status.data_ptr() + 8, gemm_stream.cuda_stream)
    # (the launch names its stream; nothing here runs on torch's current stream)
    group_gemm_gated(workspace[:M_per_rank * W], a, rank * M_per_rank, b_nk, C, ctx.sorted_topk_ids,
                     ctx.aligned_expert_ids, ctx.aligned_barrier_ids, ctx.aligned_num_tokens, ctx.BLOCK_M,
                     ctx.full_num_tokens, ctx.topk, M_per_rank, ctx.first_block, barrier, rank,
                     spin_limit=ctx.spin_limit, status=ctx.status, max_workgroups=max_wgs, sk_workspace=ctx.sk_workspace,
                     stream=gemm_stream)
    current.wait_stream(ctx.ag_stream)
    if gemm_stream is not current:
        current.wait_stream(gemm_stream)
    fill_flags(barrier, 0)   # the reference's block_barriers[rank].zero_() (:399)
    return C
