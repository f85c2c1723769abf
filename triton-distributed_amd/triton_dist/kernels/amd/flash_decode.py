"""Split-KV GQA flash decode on one MI355X and the LSE-weighted merges.

Keeps the launcher signatures of the reference's kernels/nvidia/flash_decode.py:
``gqa_fwd_batch_decode`` (:763-844), ``gqa_fwd_batch_decode_intra_rank`` (:847-928) and
``gqa_fwd_batch_decode_persistent`` (:931-1004). The per-split partial results are kept as an fp32
``[B, Hq, S, Dv]`` tensor plus an fp32 ``[B, Hq, S]`` LSE tensor (the reference packs the LSE into column
Dv of a ``[.., Dv+1]`` buffer of the query dtype, :235-239).
"""
from typing import Optional

import torch

from triton_dist import _lib

DEFAULT_KV_SPLITS = 32  # reference :777, :861


# (q/k head dim, v head dim) with compiled shapes of their own; beside them every equal pair that is a multiple of 8
# up to 256 runs on the shape of the next power of two (the reference splits a head into BLOCK_DMODEL + BLOCK_DPE and
# masks, kernels/nvidia/flash_decode.py:771-772)
SUPPORTED_HEAD_DIMS = ((64, 64), (128, 128), (256, 256), (192, 128), (576, 512))


def head_dims_supported(dk, dv):
    return (dk, dv) in SUPPORTED_HEAD_DIMS or (dk == dv and 0 < dk <= 256 and dk % 8 == 0)


def _check_kv_split(kv_split):
    """A number of splits, or -1 for the library's choice; refused otherwise, also where the number changes nothing."""
    if kv_split != -1 and not 1 <= kv_split <= 65535:
        raise _lib.TdistError(_lib.TDIST_ERR_INVALID if kv_split < 1 else _lib.TDIST_ERR_UNSUPPORTED, "kv_split %d" % kv_split)


def _check_inputs(q, k_cache, v_cache, kv_lens, block_table):
    _lib.require_cuda(q, k_cache, v_cache, kv_lens, block_table)
    batch, q_heads, q_head_dim = q.shape
    _, page_size, kv_heads, k_head_dim = k_cache.shape
    assert page_size == v_cache.shape[1] and kv_heads == v_cache.shape[2] and k_head_dim == q_head_dim
    v_head_dim = v_cache.shape[-1]
    assert q_heads % kv_heads == 0
    if not head_dims_supported(q_head_dim, v_head_dim):
        raise NotImplementedError("head dims (%d, %d); supported: equal ones that are a multiple of 8 up to 256 and %s" %
                                  (q_head_dim, v_head_dim, SUPPORTED_HEAD_DIMS[3:]))
    if q.dtype != k_cache.dtype or q.dtype != v_cache.dtype:
        raise TypeError("q, k_cache and v_cache must share one dtype")
    if q.stride(-1) != 1 or k_cache.stride(-1) != 1 or v_cache.stride(-1) != 1:
        raise ValueError("the head dimension must be contiguous")
    if kv_lens.dtype != torch.int32:
        kv_lens = kv_lens.to(torch.int32)
    if block_table.dtype != torch.int32:
        block_table = block_table.to(torch.int32)
    assert block_table.stride(-1) == 1
    return kv_lens, block_table


def _decode_args(q, k_cache, v_cache, out_split, lse_split, scale, soft_cap, block_table, kv_lens, num_splits):
    batch, q_heads, q_head_dim = q.shape
    _, page_size, kv_heads, _ = k_cache.shape
    return [q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), out_split.data_ptr(), lse_split.data_ptr(),
            float(scale), float(soft_cap), block_table.data_ptr(), kv_lens.data_ptr(), batch, q_heads, kv_heads,
            q_head_dim, v_cache.shape[-1], page_size, num_splits, q.stride(0), q.stride(1), k_cache.stride(0),
            k_cache.stride(1), k_cache.stride(2), v_cache.stride(0), v_cache.stride(1), v_cache.stride(2),
            block_table.stride(0), _lib.dtype_code(q.dtype)]


def _split_buffers(q, v_cache, num_splits, out_split, lse_split):
    batch, q_heads, _ = q.shape
    if out_split is None:
        out_split = torch.empty((batch, q_heads, num_splits, v_cache.shape[-1]), dtype=torch.float32, device=q.device)
    if lse_split is None:
        lse_split = torch.empty((batch, q_heads, num_splits), dtype=torch.float32, device=q.device)
    return out_split, lse_split


def _split_kv(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, num_splits, out_split=None, lse_split=None):
    kv_lens, block_table = _check_inputs(q, k_cache, v_cache, kv_lens, block_table)
    out_split, lse_split = _split_buffers(q, v_cache, num_splits, out_split, lse_split)
    _lib.call("tdist_decode_split_kv",
              *_decode_args(q, k_cache, v_cache, out_split, lse_split, scale, soft_cap, block_table, kv_lens, num_splits),
              _lib.stream_ptr())
    return out_split, lse_split, kv_lens


_fused_counters = {}   # (device index, stream handle) -> zero-initialised int32 counters (the kernel leaves them zero)


def _check_counters(q, kv_heads, counters):
    """``counters``: a contiguous int32 device tensor of at least tdist_decode_fused_counters(...) entries; that many."""
    need = _lib.load().tdist_decode_fused_counters(q.shape[0], q.shape[1], kv_heads)
    if counters is not None and not (isinstance(counters, torch.Tensor) and counters.is_cuda and counters.dtype == torch.int32
                                     and counters.is_contiguous() and counters.numel() >= need):
        raise ValueError("counters: a contiguous int32 device tensor of at least %d zeroed entries" % need)
    return need


def _counters_for(q, kv_heads, counters):
    """Arrival counters of the fused launch. ``counters`` (an explicit opt-in of decode_fused's callers): see _check_counters;
    ALL ZERO and shared with no launch that may overlap this one; the kernel leaves it zero. None: the library's own, a
    zeroed buffer per device and stream (_lib.zeros_per_stream)."""
    need = _check_counters(q, kv_heads, counters)
    if counters is None:
        counters = _lib.zeros_per_stream(_fused_counters, need, 4096, torch.int32, q.device)
    return counters, counters.numel()


def decode_fused(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, num_splits, out, lse_out=None,
                 workspace=None, out_split=None, lse_split=None):
    """tdist_decode_fused: split-KV decode and the merge of the splits in one launch. ``out`` [B,Hq,Dv]
    (bf16 / f16 / fp32), ``lse_out`` fp32 [B,Hq] or None. ``workspace``: None, or zeroed arrival counters of the
    caller's own (see _counters_for; anything else is an error). Returns (out, out_split, lse_split)."""
    kv_lens, block_table = _check_inputs(q, k_cache, v_cache, kv_lens, block_table)
    out_split, lse_split = _split_buffers(q, v_cache, num_splits, out_split, lse_split)
    assert out.stride(-1) == 1 and (lse_out is None or (lse_out.dtype == torch.float32 and lse_out.is_contiguous()))
    counters, n_counters = _counters_for(q, k_cache.shape[2], workspace)
    _lib.call("tdist_decode_fused",
              *_decode_args(q, k_cache, v_cache, out_split, lse_split, scale, soft_cap, block_table, kv_lens, num_splits),
              counters.data_ptr(), n_counters, out.data_ptr(), _lib.dtype_code(out.dtype), out.stride(0), out.stride(1),
              _lib.ptr(lse_out), _lib.stream_ptr())
    return out, out_split, lse_split


_STREAM_PLANS = {}   # (batch, q heads, kv heads, head dims, device) -> workspace bytes


def decode_stream(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, out, lse_out=None, counters=None):
    """tdist_decode_stream: a launch that divides the batch's keys itself and one that merges the sequences it spread over
    several places. ``out`` [B,Hq,Dv] (bf16 / f16 / fp32), ``lse_out`` contiguous fp32 [B,Hq] or None. No state outlives the
    call (``counters`` is checked and not used). The 576 / 512 heads take
    this form where the value is a view of the key's first columns; with a value cache of its own the call runs as a fixed
    number of splits and their combine. Returns ``out``."""
    kv_lens, block_table = _check_inputs(q, k_cache, v_cache, kv_lens, block_table)
    batch, q_heads, dk = q.shape
    _, page_size, kv_heads, dv = v_cache.shape
    assert out.stride(-1) == 1 and (lse_out is None or (lse_out.dtype == torch.float32 and lse_out.is_contiguous()))
    qs, ks, vs, os = q.stride(), k_cache.stride(), v_cache.stride(), out.stride()
    if dk > 256 and (k_cache.data_ptr() != v_cache.data_ptr() or ks != vs):
        S = DEFAULT_KV_SPLITS
        part, lse, kv_lens = _split_kv(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, S)
        return decode_combine(part, lse, S, 1, kv_lens, batch, q_heads, dv, (part.stride(2), part.stride(0), part.stride(1)),
                              (lse.stride(2), lse.stride(0), lse.stride(1)), out, lse_out)
    key = (batch, q_heads, kv_heads, dk, dv, q.device.index)
    need = _STREAM_PLANS.get(key) or _stream_workspace_bytes(key)
    if counters is not None:
        _check_counters(q, kv_heads, counters)
    workspace = torch.empty(need, dtype=torch.uint8, device=q.device)
    _lib.call("tdist_decode_stream", q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), scale, soft_cap,
              block_table.data_ptr(), kv_lens.data_ptr(), batch, q_heads, kv_heads, dk, dv, page_size, qs[0], qs[1], ks[0],
              ks[1], ks[2], vs[0], vs[1], vs[2], block_table.stride(0), _lib.dtype_code(q.dtype), None, 0,
              workspace.data_ptr(), need, out.data_ptr(), _lib.dtype_code(out.dtype), os[0], os[1],
              _lib.ptr(lse_out), _lib.stream_ptr())
    return out


def _stream_workspace_bytes(key):
    if len(_STREAM_PLANS) >= 1024:
        _STREAM_PLANS.clear()
    need = _STREAM_PLANS[key] = _lib.load().tdist_decode_stream_workspace_bytes(*key[:5])
    return need


def decode_stream_ranks(q, k_cache, v_cache, global_kv_lens, block_table, scale, soft_cap, rank, all_out, all_lse):
    """tdist_decode_stream_ranks: decode_stream over rank ``rank``'s keys into its place in ``all_out`` [R,B,Hq,Dv] and ``all_lse``
    (fp32 [R,B,Hq], contiguous per rank), and gqa_fwd_batch_decode_inter_rank_combine of all of them, a launch less. Returns
    [B,Hq,Dv] in q's dtype, or None where the head dimensions have no streaming form (nothing has been launched then)."""
    if global_kv_lens.dtype != torch.int32:
        global_kv_lens = global_kv_lens.to(torch.int32)
    global_kv_lens = global_kv_lens.contiguous()
    _, block_table = _check_inputs(q, k_cache, v_cache, global_kv_lens, block_table)
    batch, q_heads, dk = q.shape
    _, page_size, kv_heads, dv = v_cache.shape
    ks, vs = k_cache.stride(), v_cache.stride()
    if dk > 256 and (k_cache.data_ptr() != v_cache.data_ptr() or ks != vs):
        return None
    R = all_out.shape[0]
    _lib.require_cuda(all_out, all_lse)
    assert all_out.shape == (R, batch, q_heads, dv) and all_lse.shape == (R, batch, q_heads) and all_out.stride(-1) == 1
    assert global_kv_lens.shape == (R, batch) and 0 <= rank < R
    qs, os = q.stride(), all_out.stride()
    key = (batch, q_heads, kv_heads, dk, dv, q.device.index)
    need = _STREAM_PLANS.get(key) or _stream_workspace_bytes(key)
    workspace = torch.empty(need, dtype=torch.uint8, device=q.device)
    out = torch.empty((batch, q_heads, dv), dtype=q.dtype, device=q.device)
    dtype = _lib.dtype_code(q.dtype)
    _lib.call("tdist_decode_stream_ranks", q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), scale, soft_cap, block_table.data_ptr(),
              global_kv_lens.data_ptr(), rank, R, batch, q_heads, kv_heads, dk, dv, page_size, qs[0], qs[1], ks[0], ks[1], ks[2], vs[0], vs[1], vs[2],
              block_table.stride(0), dtype, workspace.data_ptr(), need, all_out.data_ptr(), _lib.dtype_code(all_out.dtype), os[0], os[1], os[2],
              all_lse.data_ptr(), all_lse.stride(0), out.data_ptr(), dtype, _lib.stream_ptr())
    return out


def decode_combine(part, lse, num_partials, mode, lens, batch, q_heads, dv, part_strides, lse_strides, out,
                   lse_out=None):
    """tdist_decode_combine with explicit element strides (p, b, h) for ``part`` and ``lse``."""
    _lib.call("tdist_decode_combine", part.data_ptr(), _lib.dtype_code(part.dtype), lse.data_ptr(), num_partials, mode,
              _lib.ptr(lens), batch, q_heads, dv, part_strides[0], part_strides[1], part_strides[2], lse_strides[0],
              lse_strides[1], lse_strides[2], out.data_ptr(), _lib.dtype_code(out.dtype), out.stride(0), out.stride(1),
              _lib.ptr(lse_out), _lib.stream_ptr())
    return out


def gqa_fwd_batch_decode(q, k_cache, v_cache, workspace, q_lens, kv_lens, block_table, scale, soft_cap=0.0,
                         output_split=None, output_combine=None, kv_split=-1):
    """Decode attention of one query token per sequence over a paged KV cache (reference :763-844).

    q [B,Hq,D]; k_cache / v_cache [num_pages, page_size, Hkv, D]; kv_lens int32[B]; block_table int32
    [B, max_pages]. ``workspace`` and ``q_lens`` are accepted and unused, as in the reference.
    ``output_split`` is ignored: the keys of the whole batch are divided evenly over the chip, whatever the
    lengths (``kv_split``, the reference's fixed number of splits per sequence, is accepted for its signature and
    changes nothing in the result). Returns ``output_combine`` [B,Hq,Dv] (default dtype: q's; the reference hard-codes
    float16, :784)."""
    if output_combine is None and kv_split == -1:
        out = _lib.native().decode(q, k_cache, v_cache, block_table, scale, soft_cap, kv_lens)
        if out is not None:
            return out
    _check_kv_split(kv_split)
    if output_combine is None:
        output_combine = torch.empty((q.shape[0], q.shape[1], v_cache.shape[-1]), dtype=q.dtype, device=q.device)
    return decode_stream(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, output_combine)


def gqa_fwd_batch_decode_persistent(q, k_cache, v_cache, workspace, q_lens, kv_lens, block_table, scale, soft_cap=0.0,
                                    output_split=None, output_combine=None, kv_split=-1):
    """Same result as gqa_fwd_batch_decode (reference :931-1004: split-KV, a grid barrier on ``workspace``, then the
    combine). ``kv_split`` = -1: as gqa_fwd_batch_decode. Otherwise every sequence is cut into that many splits in one
    launch, in which the last workgroup to finish a (sequence, head block) merges its splits. ``workspace`` (the
    reference's barrier buffer) and ``q_lens`` are accepted and unused: nothing says what a caller's buffer holds or who
    else uses it, and a counter that does not start at zero makes a merge fire early or never, so the arrival counters
    are the library's own (_lib.zeros_per_stream). ``output_split`` is ignored
    (partials are fp32 internally)."""
    _check_kv_split(kv_split)
    batch, q_heads, _ = q.shape
    if output_combine is None:
        output_combine = torch.empty((batch, q_heads, v_cache.shape[-1]), dtype=q.dtype, device=q.device)
    if kv_split == -1:
        return decode_stream(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, output_combine)
    decode_fused(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, kv_split, output_combine)
    return output_combine


def gqa_fwd_batch_decode_intra_rank(q, k_cache, v_cache, workspace, q_lens, kv_lens, block_table, scale, soft_cap=0.0,
                                    output_split=None, output_combine=None, kv_split=-1, return_lse=False, counters=None):
    """One rank's KV shard: split-KV decode, then the merge of its splits keeping the LSE (reference
    :847-928). Returns ``output_combine`` [B,Hq,Dv+1] with the LSE in column Dv, fp32 unless the caller
    passes a buffer of another dtype (the reference uses q's dtype). With ``return_lse`` also returns the
    fp32 (out [B,Hq,Dv], lse [B,Hq]) pair the merge produced. ``workspace`` and ``q_lens`` are accepted and unused, as
    in the reference; ``counters`` (keyword only in spirit: an addition) likewise, if it is what _check_counters asks for."""
    _check_kv_split(kv_split)
    batch, q_heads, _ = q.shape
    dv = v_cache.shape[-1]
    if output_combine is None:
        output_combine = torch.empty((batch, q_heads, dv + 1), dtype=torch.float32, device=q.device)
    out32 = torch.empty((batch, q_heads, dv), dtype=torch.float32, device=q.device)
    lse32 = torch.empty((batch, q_heads), dtype=torch.float32, device=q.device)
    # the keys divided and merged, keeping the LSE
    decode_stream(q, k_cache, v_cache, kv_lens, block_table, scale, soft_cap, out32, lse32, counters=counters)
    output_combine[..., :dv].copy_(out32)
    output_combine[..., dv].copy_(lse32)
    if return_lse:
        return output_combine, out32, lse32
    return output_combine


def gqa_fwd_batch_decode_inter_rank_combine(all_ranks_out, all_ranks_lse, global_kv_lens, final_output=None,
                                            out_dtype=None):
    """Merge of the ranks' partial results by LSE (reference kernel :481-532, call shape
    layers/nvidia/sp_flash_decode_layer.py:172-182): all_ranks_out [R,B,Hq,Dv] (fp32 / bf16 / f16),
    all_ranks_lse fp32 [R,B,Hq], global_kv_lens int32 [R,B] (a rank whose length is 0 is skipped,
    :513-515). Returns [B,Hq,Dv]."""
    _lib.require_cuda(all_ranks_out, all_ranks_lse, global_kv_lens)
    R, B, Hq, dv = all_ranks_out.shape
    assert all_ranks_lse.shape == (R, B, Hq) and all_ranks_lse.dtype == torch.float32
    assert all_ranks_out.stride(-1) == 1
    if global_kv_lens.dtype != torch.int32:
        global_kv_lens = global_kv_lens.to(torch.int32)
    global_kv_lens = global_kv_lens.contiguous()
    assert global_kv_lens.shape == (R, B)
    if final_output is None:
        final_output = torch.empty((B, Hq, dv), dtype=out_dtype or all_ranks_out.dtype, device=all_ranks_out.device)
    decode_combine(all_ranks_out, all_ranks_lse, R, 2, global_kv_lens, B, Hq, dv,
                   (all_ranks_out.stride(0), all_ranks_out.stride(1), all_ranks_out.stride(2)),
                   (all_ranks_lse.stride(0), all_ranks_lse.stride(1), all_ranks_lse.stride(2)), final_output)
    return final_output
