"""What fast_all_to_all returns are the call's own tensors over the context's buffers, whatever becomes of either."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu
T, TOPK, G, W, H, MAX_M = 40, 2, 16, 4, 128, 48


def _context(cuda):
    from triton_dist.kernels.amd import create_all_to_all_context
    g = torch.Generator().manual_seed(1)
    ctx = create_all_to_all_context(MAX_M, H, 0, G, W, G // W, dtype=torch.bfloat16)
    ids = golden.random_distinct_experts(T, G, TOPK, g).to(cuda)
    x, scale = torch.randn((T, H), generator=g).bfloat16().to(cuda), torch.rand(T, generator=g).to(cuda)
    return ctx, ids, x, scale


def _slots(ctx, ids, x, rows):
    """The rows that every slot holds, in order."""
    from triton_dist.kernels.amd import moe_dispatch_preprocess
    _, cumsum, _, gather = moe_dispatch_preprocess(ids, G)
    per = G // W
    for d in range(W):
        lo, hi = int(cumsum[d * per]), int(cumsum[(d + 1) * per])
        assert torch.equal(rows[d * MAX_M:d * MAX_M + hi - lo], x[gather[lo:hi].long()])


def _run(form, ctx, ids, x, scale):
    from triton_dist.kernels.amd import fast_all_to_all, moe_dispatch_preprocess
    if form == "ids":
        return fast_all_to_all(ctx, x, None, scale, expert_ids=ids)
    _, cumsum, scatter, gather = moe_dispatch_preprocess(ids, G)
    return fast_all_to_all(ctx, x, cumsum, scale, **({"scatter_index": scatter} if form == "scatter" else {"gather_index": gather}))


@pytest.mark.parametrize("form", ["ids", "scatter", "gather"])
def test_a_returned_tensor_changed_in_place_is_seen_by_no_other_call(cuda, form):
    announce("a2a %s: returned tensors changed in place" % form)
    ctx, ids, x, scale = _context(cuda)
    for _ in range(2):   # either half
        splits, recv, scales = _run(form, ctx, ids, x, scale)
        recv.unsqueeze_(0)
        recv.mine = True
        scales.requires_grad_()
        splits.resize_(3)
    for _ in range(2):
        splits, recv, scales = _run(form, ctx, ids, x, scale)
        assert recv.shape == (W * MAX_M, H) and not hasattr(recv, "mine") and not scales.requires_grad and splits.shape == (G, )
        _slots(ctx, ids, x, recv)


@pytest.mark.parametrize("form", ["ids", "scatter", "gather"])
@pytest.mark.parametrize("how", ["another tensor", "the tensor's memory"])
def test_replaced_buffers_are_the_ones_that_are_filled(cuda, form, how):
    announce("a2a %s: %s replaced" % (form, how))
    ctx, ids, x, scale = _context(cuda)
    for _ in range(2):
        _run(form, ctx, ids, x, scale)
    old = ctx.recv_buf.clone()
    new = {n: torch.zeros_like(getattr(ctx, n)) for n in ("recv_buf", "scale_recv_buf", "split_recv_buf")}
    for n, t in new.items():
        if how == "another tensor":
            setattr(ctx, n, t)
        else:
            getattr(ctx, n).data = t
    for half in (0, 1):
        splits, recv, scales = _run(form, ctx, ids, 2 * x, scale)
        at = ctx.WORLD_SIZE * MAX_M * ((ctx.call_count - 1) % 2)
        assert recv.data_ptr() == new["recv_buf"][at:].data_ptr()
        assert scales.data_ptr() == new["scale_recv_buf"][at:].data_ptr()
        assert splits.data_ptr() == new["split_recv_buf"][G * ((ctx.call_count - 1) % 2):].data_ptr()
        _slots(ctx, ids, 2 * x, recv)
    assert old.shape == new["recv_buf"].shape
