"""Chunks in a HIP graph: what a captured launch holds of the context's scratch stays, whatever eager calls on the same stream
ask for afterwards. Every replay against the eager result of the same launches, bit for bit, with eager work that outgrows the
stream's scratch in between."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import saragossa_amd as skv

pytestmark = pytest.mark.gpu

# every chunk of 64 slots and more by the chunk kernels; a captured chunk makes no terms, so the eager one must not either
WAYS = {"bf16": {"SKV_PREFILL_TILES": "2"}, "f32": {"SKV_PREFILL_TILES": "2", "SKV_F32_TERMS": "0"}}


class under:
    def __init__(self, env):
        self.env = env

    def __enter__(self):
        self.saved = {k: os.environ.get(k) for k in self.env}
        os.environ.update(self.env)
        skv.flags.reload()

    def __exit__(self, *exc):
        for k, v in self.saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
        skv.flags.reload()


def make(ctx, element, dims, capacity, window=0):
    return ctx.full_attention_with_element(capacity, *dims, skv.DTYPE_F32 if element == "f32" else skv.DTYPE_BF16, window)


class Chunk:
    """A layer of `base` rows and one chunk over it, on the device."""

    def __init__(self, ctx, element, dims, window, base, rows, gen):
        q_heads, kv_heads, head_dim = dims
        self.kv, self.base, self.rows, self.window = make(ctx, element, dims, base + rows, window), base, rows, window
        r = lambda n, heads: torch.randn(n, heads * head_dim, device="cuda", generator=gen)
        self.old = r(base, kv_heads), r(base, kv_heads)
        self.q, self.k, self.v = r(rows, q_heads), r(rows, kv_heads), r(rows, kv_heads)
        self.out = torch.zeros(rows, q_heads * head_dim, device="cuda")

    def refill(self, stream):
        self.kv.truncate(0)
        self.kv.encode_append_batch(stream.cuda_stream, self.old[0].data_ptr(), self.old[1].data_ptr(), self.base)

    def run(self, stream):
        self.kv.encode_prefill_rows(stream.cuda_stream, self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.rows,
                                    self.out.data_ptr())


@pytest.mark.parametrize("element,dims,window,base,rows", [
    ("bf16", (16, 2, 256), 0, 2000, 6),    # few rows, split over the context
    ("bf16", (8, 2, 64), 0, 900, 130),     # a tile chunk with splits
    ("bf16", (8, 2, 64), 100, 300, 130),   # a ring chunk, its rows' pages in the scratch too
    ("f32", (16, 2, 64), 0, 900, 130),
    ("f32", (8, 2, 64), 100, 300, 130),
])
def test_captured_chunks_keep_their_scratch(element, dims, window, base, rows):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(base + rows)
    ctx = skv.DecodeResidentState(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), under(WAYS[element]):
        c = Chunk(ctx, element, dims, window, base, rows, gen)
        c.refill(side)
        c.run(side)                          # outside the capture: the stream's scratch, lazy kernel attributes
        side.synchronize()
        want = c.out.clone()
        c.refill(side)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            c.run(side)
        for replay, more in enumerate((40, 300, 600)):
            # more partials than the stream has scratch for, and the terms of f32 pages
            for other, env in (("bf16", {}), ("f32", {"SKV_F32_TERMS": "2"})):
                with under({**WAYS[other], **env}):
                    big = Chunk(ctx, other, (32, 4, 128), 0, 3000 + more, more, gen)
                    big.refill(side)
                    big.run(side)
                    side.synchronize()
                    assert torch.isfinite(big.out).all()
            c.refill(side)
            c.kv.truncate(base)
            c.out.fill_(float("nan"))
            side.synchronize()
            graph.replay()
            side.synchronize()
            assert torch.equal(c.out, want), f"replay {replay}"
        del graph
    torch.cuda.synchronize()


def test_scratch_is_not_replaced_during_a_capture():
    """A chunk that needs more than the captured stream's scratch is refused, and its layer counts no row of it; the capture goes on."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    ctx = skv.DecodeResidentState(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        small = Chunk(ctx, "bf16", (16, 2, 256), 0, 2000, 3, gen)
        large = Chunk(ctx, "bf16", (16, 2, 256), 0, 9000, 6, gen)
        for c in (small, large):
            c.refill(side)
        small.run(side)
        side.synchronize()
        want = small.out.clone()
        small.refill(side)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            with pytest.raises(skv.DeviceError):
                large.run(side)
            small.run(side)
        assert large.kv.len() == 9000
        for replay in range(3):
            small.refill(side)
            small.out.zero_()
            side.synchronize()
            graph.replay()
            side.synchronize()
            assert torch.equal(small.out, want), f"replay {replay}"
        large.run(side)                      # outside a capture it gets what it needs
        side.synchronize()
        assert torch.isfinite(large.out).all() and large.kv.len() == 9006
        del graph
    torch.cuda.synchronize()
