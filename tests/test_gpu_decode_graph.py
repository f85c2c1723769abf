"""Decode under HIP graphs, as it is served: one graph per batch size, captured one after the other on torch's capture
stream, replayed in any order and from several streams, on lengths that change between the replays. A captured call keeps nothing
that outlives it, so no graph depends on another's having run, or on eager calls. Likewise the align / sort in the form that
goes through scratch memory."""
import pytest
import torch

from oracle import golden
from tests.conftest import announce

pytestmark = pytest.mark.gpu

ATOL = 2e-3   # the parity bar of an fp32 result


class Served:
    """Static inputs of one batch size, the graph of a call on them and its output."""

    def __init__(self, cuda, heads, dims, lens_max, seed, latent=False):
        Hq, Hkv = heads
        dk, dv = dims
        B, g = len(lens_max), torch.Generator().manual_seed(seed)
        dtype = torch.bfloat16
        self.q = torch.randn((B, Hq, dk), generator=g).to(dtype)
        self.k, self.v, self.table = golden.make_paged_kv(B, max(lens_max), Hkv, dk, 16, dtype, g, v_head_dim=dv)
        kd = self.k.to(cuda)
        if latent:
            self.v = self.k[..., :dv]
        self.lens = torch.tensor(lens_max, dtype=torch.int32, device=cuda)
        self.out = torch.full((B, Hq, dv), float("nan"), dtype=torch.float32, device=cuda)
        self.scale = dk ** -0.5
        self.args = (self.q.to(cuda), kd, kd[..., :dv] if latent else self.v.to(cuda), None, [1] * B, self.lens, self.table.to(cuda), self.scale)

    def capture(self, call):
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            call(*self.args, output_combine=self.out)
        return self

    def check(self, lens):
        exact, _ = golden.decode_exact(self.q, self.k, self.v, lens, self.table, self.scale, 0)
        assert (self.out.cpu().double() - exact).abs().max() <= ATOL


@pytest.mark.parametrize("entry,split", [("gqa_fwd_batch_decode", -1), ("gqa_fwd_batch_decode_persistent", -1),
                                         ("gqa_fwd_batch_decode_persistent", 16)])
@pytest.mark.parametrize("heads,dims,latent", [((32, 8), (128, 128), False), ((128, 1), (576, 512), True)])
def test_graphs_of_two_batch_sizes_in_reverse_order_and_on_two_streams(cuda, entry, split, heads, dims, latent):
    from triton_dist.kernels.amd import flash_decode
    announce("decode graphs %s split=%d heads=%s dims=%s" % (entry, split, heads, dims))
    call = lambda *a, **kw: getattr(flash_decode, entry)(*a, kv_split=split, **kw)
    call(*Served(cuda, heads, dims, [300, 5], 1, latent).args)   # (an eager call first, as a server's warm-up)
    small, large = (Served(cuda, heads, dims, lens, 2 + i, latent).capture(call) for i, lens in enumerate(([700, 333], [1500, 40, 900, 64, 1, 1111])))
    # the graph captured last first; poisoned outputs and new lengths before every replay
    for lens_small, lens_large in (([700, 333], [1500, 40, 900, 64, 1, 1111]), ([17, 0], [64, 1400, 0, 800, 1200, 3])):
        for s, lens in ((large, lens_large), (small, lens_small)):
            s.out.fill_(float("nan"))
            s.lens.copy_(torch.tensor(lens, dtype=torch.int32))
            s.graph.replay()
            torch.cuda.synchronize()
            s.check(lens)
        # both at once, each on a stream of its own, several times
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        small.out.fill_(float("nan"))
        large.out.fill_(float("nan"))
        torch.cuda.synchronize()
        for _ in range(5):
            for s, stream in zip((small, large), streams):
                with torch.cuda.stream(stream):
                    s.graph.replay()
        torch.cuda.synchronize()
        small.check(lens_small)
        large.check(lens_large)


def test_layer_captured_twice(cuda):
    """The sequence-parallel layer under two graphs that nothing ran before."""
    from triton_dist.layers.amd.sp_flash_decode_layer import SpGQAFlashDecodeAttention
    announce("decode layer graphs")
    Hq, Hkv, D, B = 16, 4, 128, 3
    layer = SpGQAFlashDecodeAttention(0, 0, 1, 1, Hq, Hkv, D, D, page_size=16, scale=D ** -0.5, max_allowed_batch=8)

    def call(q, k, v, _w, _ones, lens, table, _scale, output_combine):
        output_combine.copy_(layer(q, k, v, lens.view(1, -1), table))
    first, second = (Served(cuda, (Hq, Hkv), (D, D), lens, 9 + i).capture(call) for i, lens in enumerate(([900, 40, 1300], [2000, 1])))
    for s, lens in ((second, [2000, 1]), (first, [900, 40, 1300])):
        s.graph.replay()
        torch.cuda.synchronize()
        exact, _ = golden.decode_exact(s.q, s.k, s.v, lens, s.table, s.scale, 0)
        # the layer's result is bf16: its rounding step beside the bar
        assert ((s.out.cpu().double() - exact).abs() <= ATOL + 2.0 ** -8 * exact.abs()).all()


def test_sort_in_two_graphs_at_once(cuda):
    """More entries than the one-launch form takes: three launches through a scratch tensor, which eager calls share per
    stream and captured ones must not."""
    from triton_dist import _lib
    from triton_dist.kernels.amd import sort_topk_ids_align_block_size
    announce("align / sort graphs")
    E, block = 16, 128
    made = []
    for tokens, seed in ((9000, 1), (20000, 2)):
        ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(seed * 100000 + t))[:8] for t in range(64)])
        ids = ids.repeat(-(-tokens // 64), 1)[:tokens].contiguous()
        ids_d = ids.to(cuda)
        sort_topk_ids_align_block_size(ids_d, E, 1, tokens, block)
        graph = torch.cuda.CUDAGraph()
        before = dict(_lib._zero_scratch)
        with torch.cuda.graph(graph):
            out = sort_topk_ids_align_block_size(ids_d, E, 1, tokens, block)
        assert {k: v.data_ptr() for k, v in _lib._zero_scratch.items()} == {k: v.data_ptr() for k, v in before.items()}
        want = golden.sort_topk_ids_align_block_size(ids, E, 1, tokens, block)
        made.append((graph, ids_d, out, want))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(3):
        for _, _, out, _ in made:
            for t in out:
                t.fill_(-5)
        torch.cuda.synchronize()
        for (graph, *_), stream in zip(reversed(made), streams):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        for _, _, out, want in made:
            total = int(out[4].item())
            assert total == int(want[4])
            assert torch.equal(out[0][:total].cpu(), want[0][:total].to(torch.int32))
            assert torch.equal(out[1][:total // block].cpu(), want[1][:total // block].to(torch.int32))
