"""Calls whose rows the context has no room for are refused, on every route."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


def _ag_gemm(cuda, made_for, dtype, m_per_rank, K, flags):
    from triton_dist.kernels.amd import ag_gemm_intra_node, create_ag_gemm_intra_node_context
    W, N = 2, 256
    ctx = create_ag_gemm_intra_node_context(W * 128, N, 256, made_for, torch.bfloat16, 0, W, None, M_PER_CHUNK=128)
    ctx.preset_flags = flags
    shards = [torch.ones((m_per_rank, K), device=cuda).to(dtype) for _ in range(W)]
    ctx.set_peer_shards({1: shards[1]})
    return ag_gemm_intra_node(shards[0], torch.ones((N, K), device=cuda).to(dtype), False, ctx)


@pytest.mark.parametrize("flags", [False, True])
@pytest.mark.parametrize("made_for,dtype,m_per_rank,K", [
    (torch.float8_e4m3fn, torch.bfloat16, 128, 256), (torch.bfloat16, torch.bfloat16, 256, 256), (torch.bfloat16, torch.bfloat16, 128, 264)])
def test_ag_gemm_refuses_rows_beyond_the_workspace(cuda, flags, made_for, dtype, m_per_rank, K):
    announce("ag_gemm: a workspace for less than %s %d x %d" % (dtype, m_per_rank, K))
    with pytest.raises(ValueError):
        _ag_gemm(cuda, made_for, dtype, m_per_rank, K, flags)
    # what fits is taken: another type of the same size, (rows at hand) more columns of a narrower one, and bytes
    if not flags:
        assert float(_ag_gemm(cuda, torch.bfloat16, torch.float16, 128, 256, flags)[0, 0]) == 256
        assert float(_ag_gemm(cuda, torch.bfloat16, torch.float8_e4m3fn, 128, 512, flags)[0, 0]) == 512
    as_bytes = _ag_gemm(cuda, torch.float8_e4m3fn, torch.uint8, 128, 256, flags)   # e4m3 bits: 1 is 2 ** -9
    assert float(as_bytes[0, 0]) == 256 * 2.0**-18


def _group_gemm(cuda, made_for, dtype, b_dtype, made_rows, rows, K, flags):
    from triton_dist.kernels.amd import ag_group_gemm_intra_node, create_ag_group_gemm_intra_node_context
    W, E, topk, N = 2, 4, 2, 256
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(i))[:topk] for i in range(W * made_rows)]).to(cuda)
    made = torch.zeros((made_rows, 256), device=cuda).to(made_for)
    ctx = create_ag_group_gemm_intra_node_context(None, made, torch.zeros((E, 256, N), device=cuda).to(made_for), ids, E, max_M=W * made_rows,
                                                  rank=0, num_ranks=W)
    ctx.gather_rows = not flags
    shards = [torch.ones((rows, K), device=cuda).to(dtype) for _ in range(W)]
    ctx.set_peer_shards({1: shards[1]})
    return ag_group_gemm_intra_node(shards[0], torch.ones((E, K, N), device=cuda).to(b_dtype), ctx)


# a workspace for half the bytes; more rows than there is room for; fewer rows than the routing names; weights of a narrower type
@pytest.mark.parametrize("flags", [False, True])
@pytest.mark.parametrize("made_for,dtype,b_dtype,made_rows,rows", [
    (torch.float8_e4m3fn, torch.bfloat16, torch.bfloat16, 64, 64), (torch.bfloat16, torch.bfloat16, torch.bfloat16, 64, 80),
    (torch.bfloat16, torch.bfloat16, torch.bfloat16, 64, 48), (torch.bfloat16, torch.bfloat16, torch.float8_e4m3fn, 64, 64)])
def test_group_gemm_refuses_what_the_context_is_not_made_for(cuda, flags, made_for, dtype, b_dtype, made_rows, rows):
    announce("ag_group_gemm: a context of %s x %d for %s x %d, weights %s" % (made_for, made_rows, dtype, rows, b_dtype))
    with pytest.raises(ValueError):
        _group_gemm(cuda, made_for, dtype, b_dtype, made_rows, rows, 256, flags)
    c = _group_gemm(cuda, torch.bfloat16, torch.bfloat16, torch.bfloat16, 64, 64, 256, flags)
    assert c.shape == (256, 256) and float(c.min()) == float(c.max()) == 256
