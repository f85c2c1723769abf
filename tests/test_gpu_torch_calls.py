"""The calls of tdist_torch (csrc/torch_calls.cpp) against the Python code that takes every call they leave alone: the same bits in the
ordinary form, and any other form, one changed argument at a time, is left alone with nothing done. Without a GPU: everything is."""
import functools

import pytest
import torch

from tests.conftest import announce
from triton_dist import _lib

NAMES = ("decode", "decode_ranks", "ag_gemm", "gemm_rs", "ag_group_gemm", "reduce_rs", "preprocess", "dispatch_ids", "dispatch_quant", "combine", "align")


class Recorder:
    """Stands for the module: notes whether each call was taken, or takes none."""

    def __init__(self, module, take=True):
        self.taken = []
        for name in NAMES:
            setattr(self, name, functools.partial(self._call, name, getattr(module, name), take))

    def _call(self, name, fn, take, *args):
        out = fn(*args) if take else None
        self.taken.append((name, out is not None))
        return out


@pytest.fixture
def route(monkeypatch):
    """route(f) -> (results of f by the module, of f without it, names that the module took in the first)."""
    module = _lib.native()

    def run(f):
        first, second = Recorder(module), Recorder(module, take=False)
        monkeypatch.setattr(_lib, "native", lambda: first)
        a = f()
        monkeypatch.setattr(_lib, "native", lambda: second)
        b = f()
        monkeypatch.setattr(_lib, "native", lambda: module)
        assert [n for n, _ in second.taken] and not any(t for _, t in second.taken)
        return a, b, [n for n, t in first.taken if t]

    return run


def same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
    elif isinstance(a, (list, tuple)):
        assert type(a) is type(b) and len(a) == len(b)
        for x, y in zip(a, b):
            same(x, y)
    else:
        assert a == b


def test_nothing_is_taken_without_a_gpu():
    module, cpu = _lib.native(), torch.zeros(4, 4)
    counts = dict(decode=7, decode_ranks=14, ag_gemm=11, gemm_rs=9, ag_group_gemm=23, reduce_rs=22, preprocess=3, dispatch_ids=4, dispatch_quant=4,
                  combine=6, align=9)
    for name in NAMES:
        fn = getattr(module, name)
        assert fn(*[None] * counts[name]) is None and fn(*[cpu] * counts[name]) is None
        with pytest.raises(TypeError):
            fn(cpu)


def test_a_module_built_for_another_torch_is_refused(monkeypatch):
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    with pytest.raises(RuntimeError, match="0.0.0"):
        _lib.native()


class Subclass(torch.Tensor):
    pass


def decode_inputs(cuda, dims, dtype, batch=3):
    hq, hkv, dk, dv = dims
    g = torch.Generator(device=cuda).manual_seed(dk + hq)
    pages = 24
    k = torch.randn((pages, 16, hkv, dk), generator=g, device=cuda).to(dtype)
    v = k[..., :dv] if dv < dk else torch.randn((pages, 16, hkv, dv), generator=g, device=cuda).to(dtype)
    table = torch.randperm(pages, generator=g, device=cuda, dtype=torch.int32).view(batch, pages // batch)
    return dict(q=torch.randn((batch, hq, dk), generator=g, device=cuda).to(dtype), k=k, v=v, lens=torch.tensor([1, 100, 128], dtype=torch.int32, device=cuda),
                table=table, scale=dk ** -0.5, soft_cap=0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,dtype", [((32, 8, 128, 128), torch.bfloat16), ((6, 1, 96, 96), torch.float16), ((16, 1, 576, 512), torch.bfloat16)])
def test_decode(cuda, route, dims, dtype):
    from triton_dist.kernels.amd import gqa_fwd_batch_decode
    from triton_dist.layers.amd.sp_flash_decode_layer import SpGQAFlashDecodeAttention
    announce("torch calls, decode %s" % (dims, ))
    x = decode_inputs(cuda, dims, dtype)

    def call(**kw):
        y = {**x, **kw}
        return lambda: gqa_fwd_batch_decode(y["q"], y["k"], y["v"], None, [1] * 3, y["lens"], y["table"], y["scale"], y["soft_cap"])

    a, b, taken = route(call())
    same(a, b)
    assert taken == ["decode"]
    q = x["q"]
    strided = torch.stack([q, q], dim=1)[:, 1]                      # rows of another stride: ordinary
    wide = torch.cat([x["table"], x["table"]], dim=1)[:, :x["table"].shape[1]]
    a, c, taken = route(call(q=strided, table=wide, soft_cap=0))
    same(a, c)
    same(a, b)
    assert taken == ["decode"]
    for kw in (dict(lens=x["lens"].long()), dict(table=x["table"].long()), dict(scale=torch.tensor(x["scale"])), dict(q=q.as_subclass(Subclass))):
        a, c, taken = route(call(**kw))
        same(a, c)
        same(a, b)
        assert not taken
    R, B, Hq = 3, 3, dims[0]
    peers = torch.randn((R, B, Hq, dims[3]), device=cuda).to(dtype), torch.randn((R, B, Hq), device=cuda)
    layer = SpGQAFlashDecodeAttention(1, 0, R, 1, Hq, dims[1], dims[2], dims[3], page_size=16, scale=x["scale"], max_allowed_batch=B)
    lens = x["lens"].repeat(R, 1).contiguous()

    def forward(all_out=peers[0], all_lse=peers[1]):
        def f():
            out, lse = all_out.clone(memory_format=torch.preserve_format), all_lse.clone(memory_format=torch.preserve_format)
            return layer(q, x["k"], x["v"], lens, x["table"], (out, lse)), out, lse
        return f

    a, b, taken = route(forward())
    same(a, b)
    assert taken == ["decode_ranks"]
    a, b, taken = route(forward(all_lse=peers[1].transpose(1, 2).contiguous().transpose(1, 2)))
    same(a, b)
    assert not taken
    with pytest.raises(AssertionError):
        layer(q, x["k"], x["v"], lens[:2], x["table"], peers)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
def test_gemms(cuda, route, dtype):
    from triton_dist.kernels.amd import (ag_gemm_intra_node, create_ag_gemm_intra_node_context, create_gemm_rs_intra_node_context, gemm_rs_intra_node)
    announce("torch calls, GEMMs %s" % dtype)
    g = torch.Generator(device=cuda).manual_seed(3)

    def rand(*shape):
        return torch.randn(shape, generator=g, device=cuda).to(dtype)

    out = torch.bfloat16 if dtype == torch.float8_e4m3fn else dtype
    W, mpr, K, N = 4, 37, 272, 200
    ctx = create_ag_gemm_intra_node_context(W * mpr, N, K, dtype, out, 2, W, None, M_PER_CHUNK=mpr, ragged_chunks=True)
    shards = [rand(mpr, K) for _ in range(W)]
    ctx.set_peer_shards({r: s for r, s in enumerate(shards) if r != 2})
    b, scales = rand(N, K), {}
    if dtype == torch.float8_e4m3fn:
        scales = dict(row_scale=torch.rand(W * mpr, generator=g, device=cuda), col_scale=torch.rand(N, generator=g, device=cuda))
    strided = torch.cat([b, b], dim=1)[:, :K]
    for weight in (b, strided):
        x, y, taken = route(lambda: ag_gemm_intra_node(shards[2], weight, False, ctx, **scales))
        same(x, y)
        assert taken == ["ag_gemm"]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):     # (the context's stream is another one than the caller's)
        stream.wait_stream(torch.cuda.default_stream())
        z, y, taken = route(lambda: ag_gemm_intra_node(shards[2], b, False, ctx, **scales))
        stream.synchronize()
        same(z, x)
        same(z, y)
        assert not taken
    for wrong in (rand(N, K + 16), b.float()):
        with pytest.raises((AssertionError, TypeError)):
            ag_gemm_intra_node(shards[2], wrong, False, ctx)
    W, M, K, N = 2, 256, 256, 512
    rs = create_gemm_rs_intra_node_context(M, N, out, 1, W, None)
    rs.set_peer_partials({0: torch.randn((M // W, N), generator=g, device=cuda).to(out)})
    a, b = rand(M, K), rand(N, K)
    if scales:
        scales = dict(row_scale=torch.rand(M, generator=g, device=cuda), col_scale=torch.rand(N, generator=g, device=cuda))
    x, y, taken = route(lambda: [gemm_rs_intra_node(a, b, rs, **scales)] + [t.clone() for t in rs.scatter_bufs])
    same(x, y)
    assert taken == ["gemm_rs"]
    for wrong in (a[:, :128].contiguous(), a.t()):
        with pytest.raises(AssertionError):
            gemm_rs_intra_node(wrong, b[:, :wrong.shape[1]].contiguous(), rs)


@pytest.mark.gpu
@pytest.mark.parametrize("ids_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype,quant", [(torch.bfloat16, False), (torch.float8_e4m3fn, False), (torch.float8_e4m3fn, True)])
def test_moe_dispatch(cuda, route, dtype, quant, ids_dtype):
    from triton_dist.kernels.amd import (create_all_to_all_context, fast_all_to_all, moe_dispatch_preprocess, moe_weighted_combine,
                                         sort_topk_ids_align_block_size)
    announce("torch calls, dispatch %s %s" % (dtype, quant))
    T, topk, G, W, H = 48, 3, 16, 4, 1024
    g = torch.Generator(device=cuda).manual_seed(5)
    ids = torch.rand((T, G), generator=g, device=cuda).topk(topk, dim=1).indices.to(ids_dtype)
    x = torch.randn((T, H), generator=g, device=cuda).to(torch.bfloat16 if quant else dtype)
    scale = torch.rand(T, generator=g, device=cuda) if dtype == torch.float8_e4m3fn and not quant else None
    w = torch.rand((T, topk), generator=g, device=cuda)

    def context():
        ctx = create_all_to_all_context(T * topk, H, 0, G, W, G // W, dtype=dtype, fp8_group_size=128 if quant else 0)
        ctx.recv_buf.view(torch.uint8).zero_()
        ctx.scale_recv_buf.zero_()
        return ctx

    made = []

    def run(ids=ids, x=x):
        def f():
            ctx = context()
            made.append(ctx)
            out = []
            for _ in range(3):   # (the first call makes the context's index tensors; both halves and sets)
                if quant:
                    _, cumsum, scatter, gather = moe_dispatch_preprocess(ids, G, ctx=ctx)
                    r = fast_all_to_all(ctx, x, cumsum, None, scatter_index=scatter, online_quant_fp8=True)
                else:
                    r = fast_all_to_all(ctx, x, None, scale, expert_ids=ids)
                    _, cumsum, scatter, gather = ctx.last_index
                y = moe_weighted_combine(ctx, r[1], r[2], scatter, w, cumsum)
                out.append([t.clone() for t in (r[0], r[1], cumsum, scatter, gather, y)] + [None if r[2] is None else r[2].clone()])
                assert r[1].data_ptr() != out[0][1].data_ptr()
            out.append((ctx.call_count, ctx.index_calls))
            rows, _, _, blocks, padded = sort_topk_ids_align_block_size(ids, G, W, T // W, 64)   # (the others are not written whole)
            out.append((rows, blocks, padded))
            return out
        return f

    a, b, taken = route(run())
    same(a, b)
    assert taken == (["dispatch_quant", "combine"] + ["preprocess", "dispatch_quant", "combine"] * 2 if quant else ["dispatch_ids", "combine"] * 3) + ["align"]
    # a result is the call's own: a caller's change of its shape is not seen by a later call
    if not quant:
        ctx = made[0]
        first = fast_all_to_all(ctx, x, None, scale, expert_ids=ids)[1]
        shape = first.shape
        first.resize_(1, shape[1])
        fast_all_to_all(ctx, x, None, scale, expert_ids=ids)
        assert fast_all_to_all(ctx, x, None, scale, expert_ids=ids)[1].shape == shape
    # other forms: ids that are not contiguous, tokens that are not
    a, c, taken = route(run(ids=ids.t().contiguous().t(), x=torch.cat([x, x], dim=1)[:, :H]))
    same(a, c)
    same(a, b)
    assert "dispatch_ids" not in taken and "dispatch_quant" not in taken and "preprocess" not in taken


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
def test_moe_layer(cuda, route, dtype):
    from triton_dist.kernels.amd import (ag_group_gemm_intra_node, create_ag_group_gemm_intra_node_context, create_moe_rs_context, moe_reduce_rs,
                                         select_experts)
    announce("torch calls, MoE layer %s" % dtype)
    W, mpr, E, H, I, topk, rank = 2, 24, 4, 256, 192, 2, 1
    g = torch.Generator(device=cuda).manual_seed(7)

    def rand(*shape):
        return (torch.randn(shape, generator=g, device=cuda) * 0.1).to(dtype)

    shards, logits = [rand(mpr, H) for _ in range(W)], [torch.randn((mpr, E), generator=g, device=cuda) for _ in range(W)]
    up, down = rand(E, I, H).transpose(1, 2), rand(E, H, I).transpose(1, 2)
    peers = {r: t for r, t in enumerate(logits) if r != rank}
    ids, _ = select_experts(None, W, topk, torch.bfloat16, cuda, logits[rank], peers, rank)
    partial = torch.randn((mpr, H), generator=g, device=cuda).bfloat16()

    def run(up=up, down=down):
        def f():
            ag = create_ag_group_gemm_intra_node_context(None, shards[rank], up, ids, E, max_M=W * mpr, rank=rank, num_ranks=W)
            ag.set_peer_shards({0: shards[0]})
            rs = create_moe_rs_context(None, rank, W, W, W * mpr, H, E, topk, torch.bfloat16, torch.bfloat16, cuda, 128, logits[rank], peers)
            rs.set_peer_partials({0: partial})
            out = []
            for _ in range(3):
                h = ag_group_gemm_intra_node(shards[rank], up, ag)
                if dtype == torch.float16:   # (the reduction is of bf16 rows)
                    with pytest.raises(TypeError):
                        moe_reduce_rs(rank, W, W, h, down, rs)
                    out += [h]
                    continue
                out += [h, moe_reduce_rs(rank, W, W, h.to(dtype), down, rs), rs.rs_buffers[rank].clone(), rs.final_output_buffer.clone()]
            ag.check_status()
            return out
        return f

    a, b, taken = route(run())
    same(a, b)
    second = ["ag_group_gemm"] if dtype == torch.float16 else ["ag_group_gemm", "reduce_rs"]
    assert taken == ["align"] * 2 + second * 2   # (the contexts' own; the first calls make the memory of the row blocks)
    a, c, taken = route(run(up=up.contiguous(), down=down.contiguous()))   # weights that are transposed first
    same(a, c)
    same(a, b)
    assert taken == ["align"] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_moe_layer_with_two_lists(cuda, route, dtype):
    """Experts' last rows in a list of their own, by the module and by the Python code, whole numbers exactly: 512 rows per expert on average
    and 4096 columns are two rounds of 256-row blocks with the last rows, one without."""
    from triton_dist.kernels.amd import (ag_group_gemm_intra_node, create_ag_group_gemm_intra_node_context, create_moe_rs_context, moe_reduce_rs)
    announce("torch calls, MoE layer with two lists %s" % dtype)
    W, mpr, E, N, K, topk, rank = 4, 512, 8, 4096, 192, 2, 1
    g = torch.Generator(device=cuda).manual_seed(11)

    def whole(*shape):
        return torch.randint(-1, 2, shape, generator=g, device=cuda).float().to(dtype)

    shards, logits = [whole(mpr, K) for _ in range(W)], [torch.randn((mpr, E), generator=g, device=cuda) for _ in range(W)]
    up, down, states = whole(E, N, K).transpose(1, 2), whole(E, N, K).transpose(1, 2), whole(W * mpr * topk, K)
    peers = {r: t for r, t in enumerate(logits) if r != rank}
    weight = torch.randint(1, 3, (W * mpr, topk), generator=g, device=cuda).float()
    partials = [torch.randint(-8, 9, (mpr, N), generator=g, device=cuda).bfloat16() for _ in range(W)]
    ids = torch.cat(logits).softmax(-1).topk(topk).indices.int()
    made = []

    def f():
        ag = create_ag_group_gemm_intra_node_context(None, shards[rank], up, ids, E, max_M=W * mpr, rank=rank, num_ranks=W)
        ag.set_peer_shards({r: s for r, s in enumerate(shards) if r != rank})
        rs = create_moe_rs_context(None, rank, W, W, W * mpr, N, E, topk, torch.bfloat16, torch.bfloat16, cuda, 128, logits[rank], peers)
        rs.topk_weight_f32 = weight
        rs.set_peer_partials({r: t for r, t in enumerate(partials) if r != rank})
        made.append((ag, rs))
        out = []
        for _ in range(3):
            out += [ag_group_gemm_intra_node(shards[rank], up, ag), moe_reduce_rs(rank, W, W, states, down, rs)]
        ag.check_status()
        return out

    with _lib.debug_switch(_lib.TDIST_DEBUG_GEMM_TILE, 0):   # (256-row blocks, whatever the estimate for so short a K)
        a, b, taken = route(f)
    same(a, b)
    assert taken == ["align"] * 2 + ["ag_group_gemm", "reduce_rs"] * 2
    for ctx in (c for pair in made for c in pair):
        blocks, = ctx.joined.values()
        assert blocks.block_size == 256 and blocks.tail_most > 0
        at = (blocks.tail.padded - blocks.memory.data_ptr()) // 4
        assert int(blocks.memory[at]) > 0 or _lib.load().tdist_num_cus() != 256
    entry = torch.arange(W * mpr * topk, device=cuda)

    def products(rows, w):
        out = torch.empty((rows.shape[0], N), device=cuda)
        for e in range(E):
            of = entry[ids.view(-1) == e]
            out[of] = rows[of].float() @ w[e].float()
        return out

    h = products(torch.cat([s.float() for s in shards]).repeat_interleave(topk, 0), up)
    sums = (products(states, down).view(W * mpr, topk, N) * weight[:, :, None]).sum(1)[rank * mpr:(rank + 1) * mpr]
    y = sum(t.float() for r, t in enumerate(partials) if r != rank) + sums
    assert max(t.abs().max() for t in (h, sums, y)) <= 256   # every value is an integer that bf16 holds
    for i in range(0, 6, 2):
        assert torch.equal(a[i].float(), h) and torch.equal(a[i + 1].float(), y)


@pytest.mark.gpu
def test_modes(cuda, route):
    """A mode that sees the calls of torch sees those of the Python code; states that change nothing for the call leave it to the module."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from triton_dist.kernels.amd import gqa_fwd_batch_decode
    announce("torch calls, modes")

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x = decode_inputs(cuda, (32, 8, 128, 128), torch.bfloat16)
    want = gqa_fwd_batch_decode(x["q"], x["k"], x["v"], None, [1] * 3, x["lens"], x["table"], x["scale"], x["soft_cap"])

    def f(mode):
        def g():
            with mode():
                return gqa_fwd_batch_decode(x["q"], x["k"], x["v"], None, [1] * 3, x["lens"], x["table"], x["scale"], x["soft_cap"])
        return g

    for mode, by_module in ((Function, False), (Dispatch, False), (torch.inference_mode, True), (torch.no_grad, True), (torch.enable_grad, True),
                            (lambda: torch.autocast("cuda"), True)):
        a, b, taken = route(f(mode))
        assert bool(taken) == by_module
        assert a.is_inference() == b.is_inference()
        with torch.inference_mode():
            same(a, b)
            same(a, want)


@pytest.mark.gpu
def test_captured(cuda, monkeypatch):
    """Calls that the module takes while a graph is captured: every replay, on inputs that have changed, with eager calls between, against the
    eager result."""
    from triton_dist.kernels.amd import (ag_group_gemm_intra_node, create_ag_group_gemm_intra_node_context, create_all_to_all_context,
                                         create_gemm_rs_intra_node_context, create_moe_rs_context, fast_all_to_all, gemm_rs_intra_node,
                                         gqa_fwd_batch_decode, moe_reduce_rs, moe_weighted_combine, sort_topk_ids_align_block_size)
    announce("torch calls, captured")
    g, module = torch.Generator(device=cuda).manual_seed(13), _lib.native()
    d = decode_inputs(cuda, (32, 8, 128, 128), torch.bfloat16)
    T, topk, G, W, H = 48, 3, 16, 4, 1024
    x, w = torch.randn((T, H), generator=g, device=cuda).bfloat16(), torch.rand((T, topk), generator=g, device=cuda)
    ids = torch.rand((T, G), generator=g, device=cuda).topk(topk, dim=1).indices
    contexts = [create_all_to_all_context(T * topk, H, 0, G, W, G // W) for _ in range(2)]
    R, mpr, E, I, rank = 2, 24, 4, 192, 1
    shards, logits = [torch.randn((mpr, 256), generator=g, device=cuda).bfloat16() for _ in range(R)], [torch.randn((mpr, E), generator=g, device=cuda) for _ in range(R)]
    up, down = (torch.randn((E, *s), generator=g, device=cuda).bfloat16().transpose(1, 2) for s in ((I, 256), (256, I)))
    rs = create_moe_rs_context(None, rank, R, R, R * mpr, 256, E, 2, torch.bfloat16, torch.bfloat16, cuda, 128, logits[rank], {0: logits[0]})
    rs.set_peer_partials({0: torch.randn((mpr, 256), generator=g, device=cuda)})
    ag = create_ag_group_gemm_intra_node_context(None, shards[rank], up, rs.precompute_ctx.full_topk_ids, E, max_M=R * mpr, rank=rank, num_ranks=R)
    ag.set_peer_shards({0: shards[0]})
    gemm = create_gemm_rs_intra_node_context(256, 512, torch.bfloat16, 1, 2, None)
    gemm.set_peer_partials({0: torch.randn((128, 512), generator=g, device=cuda)})
    a, b = (torch.randn(s, generator=g, device=cuda).bfloat16() for s in ((256, 256), (512, 256)))

    def calls(ctx):
        out = [gqa_fwd_batch_decode(d["q"], d["k"], d["v"], None, [1] * 3, d["lens"], d["table"], d["scale"], d["soft_cap"])]
        splits, recv, _ = fast_all_to_all(ctx, x, None, None, expert_ids=ids)
        _, cumsum, scatter, gather = ctx.last_index
        out += [splits, cumsum, scatter, gather, moe_weighted_combine(ctx, recv, None, scatter, w, cumsum)]
        rows, _, _, blocks, padded = sort_topk_ids_align_block_size(ids, G, W, T // W, 64)
        h = ag_group_gemm_intra_node(shards[rank], up, ag)
        return out + [rows, blocks, padded, h, moe_reduce_rs(rank, R, R, h, down, rs), gemm_rs_intra_node(a, b, gemm)]

    for ctx in contexts:
        calls(ctx)   # (what a context makes at its first call)
    recorder = Recorder(module)
    monkeypatch.setattr(_lib, "native", lambda: recorder)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = calls(contexts[0])
    monkeypatch.setattr(_lib, "native", lambda: module)
    assert recorder.taken == [(n, True) for n in ("decode", "dispatch_ids", "combine", "align", "ag_group_gemm", "reduce_rs", "gemm_rs")]
    for turn in range(4):
        for t in (d["q"], x, shards[rank], shards[0], a):
            t.copy_(torch.randn(t.shape, generator=g, device=cuda))
        ids.copy_(torch.rand((T, G), generator=g, device=cuda).topk(topk, dim=1).indices)
        d["lens"].copy_(torch.tensor([turn, 128 - turn, 17 * turn], dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        same(got, calls(contexts[1]))
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_threads(cuda):
    """Threads with contexts and streams of their own, their calls in flight together: the results of one thread alone."""
    import threading

    from triton_dist.kernels.amd import (create_all_to_all_context, fast_all_to_all, gqa_fwd_batch_decode, moe_weighted_combine,
                                         sort_topk_ids_align_block_size)
    announce("torch calls, threads")
    T, topk, G, W, H = 64, 4, 16, 4, 512

    def job(seed):
        g = torch.Generator(device=cuda).manual_seed(seed)
        d = decode_inputs(cuda, (32, 8, 128, 128), torch.bfloat16)
        q = torch.randn(d["q"].shape, generator=g, device=cuda).bfloat16()
        x, w = torch.randn((T, H), generator=g, device=cuda).bfloat16(), torch.rand((T, topk), generator=g, device=cuda)
        ids = torch.rand((T, G), generator=g, device=cuda).topk(topk, dim=1).indices
        ctx = create_all_to_all_context(T * topk, H, 0, G, W, G // W)

        def calls():
            out = [gqa_fwd_batch_decode(q, d["k"], d["v"], None, [1] * 3, d["lens"], d["table"], d["scale"], 0.0)]
            splits, recv, _ = fast_all_to_all(ctx, x, None, None, expert_ids=ids)
            _, cumsum, scatter, gather = ctx.last_index
            out += [splits, cumsum, scatter, gather, moe_weighted_combine(ctx, recv, None, scatter, w, cumsum)]
            rows, _, _, blocks, padded = sort_topk_ids_align_block_size(ids, G, W, T // W, 64)
            return [t.clone() for t in out + [rows, blocks, padded]]
        return calls

    jobs = [job(seed) for seed in range(4)]
    want = [calls() for calls in jobs]
    torch.cuda.synchronize()
    got, failed = [None] * len(jobs), []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                got[i] = [jobs[i]() for _ in range(20)]
            stream.synchronize()
        except Exception as e:   # (a thread's own exception would be lost)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i, )) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for i, results in enumerate(got):
        for r in results:
            same(r, want[i])
