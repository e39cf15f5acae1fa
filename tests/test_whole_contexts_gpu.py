"""Decode steps and chunks over few pages are attended without a split: on both sides of the lines against the oracle, and with a
context that lies over what the launch reads, where the split stays."""
import os

import numpy as np
import pytest
import torch

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu


def _layer(state, dims, element, rows, extra, seed):
    q_heads, kv_heads, head_dim = dims
    rng = np.random.default_rng(seed)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(rows + extra, q_heads, kv_heads, head_dim)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    k, v = (rng.standard_normal((rows + extra, kv_heads * head_dim), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((extra, q_heads * head_dim), dtype=np.float32)
    kv.seed(k[:rows], v[:rows], rows)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache.append_batch(k[:rows], v[:rows], lay)
    want = np.stack([oracle.decode_step(cache, k[rows + i], v[rows + i], q[i], lay) for i in range(extra)])
    return kv, q, k[rows:], v[rows:], want


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("dims,pages", [((8, 2, 64), 24), ((8, 8, 80), 24), ((16, 4, 128), 16), ((24, 1, 128), 16), ((8, 2, 256), 10)])
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_steps_around_the_line(state, dims, pages, past):
    rows = pages * 16 - 1 + past
    kv, q, k, v, want = _layer(state, dims, "bf16", rows, 1, rows)
    qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v))
    out = torch.full((1, q.shape[1]), float("nan"), device="cuda")
    kv.encode_decode_step(_stream(), kd.data_ptr(), 0, vd.data_ptr(), 0, qd.data_ptr(), out.data_ptr())
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-4


def _chunk(state, dims, element, chunk, pages, env):
    """A chunk over a context of so many pages with itself: within the element's tolerance of the oracle"""
    saved = {name: os.environ.get(name) for name in env}
    os.environ.update(env)
    skv.flags.reload()
    try:
        rows = pages * 16 - chunk - 1
        kv, q, k, v, want = _layer(state, dims, element, rows, chunk, rows)
        qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v))
        out = torch.full(q.shape, float("nan"), device="cuda")
        kv.encode_prefill_rows(_stream(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), chunk, out.data_ptr())
        got = out.cpu().numpy()
        assert np.abs(got - want).max() <= (2e-5 if element == "f32" else 1e-4)
        return got
    finally:
        for name, was in saved.items():
            os.environ.pop(name) if was is None else os.environ.__setitem__(name, was)
        skv.flags.reload()


@pytest.mark.parametrize("dims,element,chunk,pages,whole", [
    ((8, 2, 64), "bf16", 5, 28, True), ((8, 2, 64), "bf16", 5, 29, False),          # two tiles a kv head, appended
    ((8, 2, 64), "bf16", 16, 26, True), ((8, 2, 64), "bf16", 16, 27, False),        # four, on four XCDs
    ((8, 2, 32), "bf16", 16, 28, True), ((8, 2, 32), "bf16", 16, 29, False),
    ((16, 1, 96), "bf16", 12, 25, True), ((16, 1, 96), "bf16", 12, 26, False),
    ((16, 16, 96), "bf16", 3, 32, True), ((16, 16, 96), "bf16", 3, 33, False),      # more than eight kv heads
    ((32, 8, 128), "bf16", 3, 27, True), ((32, 8, 128), "bf16", 3, 28, False),      # one tile a kv head
    ((32, 8, 128), "bf16", 16, 39, True), ((32, 8, 128), "bf16", 16, 40, False),    # four, on one XCD
    ((32, 8, 128), "bf16", 30, 58, True), ((32, 8, 128), "bf16", 30, 59, False),    # eight, rows appended in front
    ((24, 1, 128), "bf16", 6, 22, True), ((24, 1, 128), "bf16", 6, 23, False),      # nine, on eight XCDs
    ((36, 3, 128), "bf16", 6, 21, True), ((36, 3, 128), "bf16", 6, 22, False),
    ((32, 16, 128), "bf16", 10, 32, True), ((32, 16, 128), "bf16", 10, 33, False),
    ((16, 2, 256), "bf16", 6, 16, True), ((16, 2, 256), "bf16", 6, 17, False),
    ((16, 8, 256), "bf16", 16, 18, True), ((16, 8, 256), "bf16", 16, 19, False),
    ((16, 2, 256), "bf16", 40, 29, True), ((16, 2, 256), "bf16", 40, 30, False),
    ((8, 2, 64), "f32", 48, 10, True), ((8, 2, 64), "f32", 48, 11, False),
    ((32, 8, 64), "f32", 30, 14, True), ((32, 8, 128), "f32", 30, 12, True), ((32, 8, 128), "f32", 30, 13, False),
    ((32, 8, 128), "f32", 30, 16, False), ((32, 8, 128), "f32", 30, 17, True), ((32, 8, 128), "f32", 30, 20, True), ((32, 8, 128), "f32", 30, 21, False),
    ((32, 8, 64), "f32", 60, 28, True), ((32, 8, 64), "f32", 60, 29, False), ((32, 8, 96), "f32", 66, 36, True), ((32, 8, 96), "f32", 66, 37, False),
    ((16, 2, 256), "f32", 24, 9, False),
])
def test_chunks_around_the_line(state, dims, element, chunk, pages, whole):
    """Whole up to the line, and behind it bit for bit what the chunk is where a knob of the splits is set."""
    split = _chunk(state, dims, element, chunk, pages, {"RETI_RUST_SDPA_2PASS_MIN_LEN": "128"})
    assert np.array_equal(_chunk(state, dims, element, chunk, pages, {}), split) != whole


@pytest.mark.parametrize("over", ["q", "k", "v"])
def test_a_step_over_its_own_rows(state, over):
    """The context lies over the step's query or new row, one head further: what the launch still reads stays whole until it is done."""
    dims, rows = (32, 8, 128), 200
    kv, q, k, v, want = _layer(state, dims, "bf16", rows, 1, 7)
    buf = {n: torch.zeros(6000, device="cuda") for n in "qkv"}
    for n, a in zip("qkv", (q, k, v)):
        buf[n][128:128 + a.size] = torch.from_numpy(a.reshape(-1)).cuda()
    at = {n: b.data_ptr() + 128 * 4 for n, b in buf.items()}
    kv.encode_decode_step(_stream(), at["k"], 0, at["v"], 0, at["q"], buf[over].data_ptr())
    assert np.abs(buf[over][:q.size].cpu().numpy() - want[0]).max() <= 1e-4


def test_a_batch_over_another_sequences_rows(state):
    dims, rows = (8, 2, 64), 150
    seqs = [_layer(state, dims, "bf16", rows + 9 * i, 1, i) for i in range(3)]
    kd = torch.from_numpy(np.concatenate([s[2] for s in seqs])).cuda()
    vd = torch.from_numpy(np.concatenate([s[3] for s in seqs])).cuda()
    qd = torch.from_numpy(np.concatenate([s[1] for s in seqs])).cuda()
    q_dim, kv_dim = qd.shape[1], kd.shape[1]
    rest = torch.zeros(2, q_dim, device="cuda")
    # the first sequence's context over the last ones' queries
    outs = [qd.data_ptr() + q_dim * 4, rest[0].data_ptr(), rest[1].data_ptr()]
    skv.encode_decode_step_batch([s[0] for s in seqs], _stream(), [kd.data_ptr() + i * kv_dim * 4 for i in range(3)],
                                 [vd.data_ptr() + i * kv_dim * 4 for i in range(3)], [qd.data_ptr() + i * q_dim * 4 for i in range(3)], outs)
    got = np.stack([qd[1].cpu().numpy(), rest[0].cpu().numpy(), rest[1].cpu().numpy()])
    assert np.abs(got - np.concatenate([s[4] for s in seqs])).max() <= 1e-4


@pytest.mark.parametrize("knob", ["SKV_DECODE_WGS", "SKV_PREFILL_WGS"])
@pytest.mark.parametrize("chunk", [1, 16])
def test_a_given_number_of_workgroups_splits(state, knob, chunk):
    """Where a knob of the splits is set, to its default here, short contexts are split as they are with any other such knob: bit for bit."""
    def run(env):
        saved = {name: os.environ.get(name) for name in env}
        os.environ.update(env)
        skv.flags.reload()
        try:
            kv, q, k, v, want = _layer(state, (32, 8, 128), "bf16", 220, chunk, 3)
            qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v))
            out = torch.full(q.shape, float("nan"), device="cuda")
            kv.encode_prefill_rows(_stream(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), chunk, out.data_ptr())
            got = out.cpu().numpy()
            assert np.abs(got - want).max() <= 1e-4
            return got
        finally:
            for name, was in saved.items():
                os.environ.pop(name) if was is None else os.environ.__setitem__(name, was)
            skv.flags.reload()
    split = run({"RETI_RUST_SDPA_2PASS_MIN_LEN": "128"})
    assert np.array_equal(run({knob: "256"}), split)
    assert not np.array_equal(run({}), split)


def _batch(state, dims, lens, env, apart=False):
    saved = {name: os.environ.get(name) for name in env}
    os.environ.update(env)
    skv.flags.reload()
    try:
        seqs = [_layer(state, dims, "bf16", n, 1, i) for i, n in enumerate(lens)]
        q, k, v = (torch.from_numpy(np.concatenate([s[i] for s in seqs])).cuda() for i in (1, 2, 3))
        out = torch.full(q.shape, float("nan"), device="cuda")
        if apart: # every sequence's q, k, v and context side by side, as where each has buffers of its own
            rows = torch.cat([q, k, v, out], dim=1)
            q, k, v, out = rows.split([q.shape[1], k.shape[1], v.shape[1], out.shape[1]], dim=1)
        at = lambda t: [row.data_ptr() for row in t]
        skv.encode_decode_step_batch([s[0] for s in seqs], _stream(), at(k), at(v), at(q), at(out))
        got = out.cpu().numpy()
        assert np.abs(got - np.concatenate([s[4] for s in seqs])).max() <= 1e-4
        return got
    finally:
        for name, was in saved.items():
            os.environ.pop(name) if was is None else os.environ.__setitem__(name, was)
        skv.flags.reload()


@pytest.mark.parametrize("dims,lens", [((8, 2, 64), [300, 900]), ((8, 2, 64), [900, 300, 90]), ((16, 2, 256), [140, 400])])
def test_a_batch_stays_whole_together(state, dims, lens):
    """One context past the line splits the others as well: bit for bit what they are where a knob of the splits is set."""
    assert np.array_equal(_batch(state, dims, lens, {}), _batch(state, dims, lens, {"RETI_RUST_SDPA_2PASS_MIN_LEN": "128"}))


@pytest.mark.parametrize("dims,lens", [((8, 2, 64), [300, 200]), ((16, 2, 256), [140, 90, 60])])
def test_a_batch_of_buffers_apart_stays_whole(state, dims, lens):
    """Rows between the contexts but under none of them: bit for bit what the batch is with one tensor of each kind."""
    assert np.array_equal(_batch(state, dims, lens, {}, apart=True), _batch(state, dims, lens, {}))


@pytest.mark.parametrize("dims,n_seq,pages", [((8, 2, 64), 3, 25), ((8, 8, 80), 16, 49), ((16, 4, 128), 16, 28), ((8, 2, 256), 16, 10), ((16, 8, 256), 8, 15)])
def test_batches_around_the_line(state, dims, n_seq, pages):
    lens = [pages * 16 - 1 - 3 * i for i in range(n_seq)]
    split = {"RETI_RUST_SDPA_2PASS_MIN_LEN": "128"}
    below = _batch(state, dims, lens, {})       # all whole
    lens[-1] = pages * 16
    above = _batch(state, dims, lens, {})       # one page too many
    assert np.array_equal(above, _batch(state, dims, lens, split))
    assert not np.array_equal(below[:-1], above[:-1])


@pytest.mark.parametrize("rows,merged", [(150, False), (1000, True)])
def test_the_probe_of_the_merge_is_the_steps_own(state, rows, merged):
    """Nothing is launched where the step stays whole."""
    kv, q, k, v, want = _layer(state, (16, 4, 128), "bf16", rows, 1, rows)
    qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v))
    out = torch.full((1, q.shape[1]), float("nan"), device="cuda")
    kv.encode_decode_step(_stream(), kd.data_ptr(), 0, vd.data_ptr(), 0, qd.data_ptr(), out.data_ptr())
    again = torch.full_like(out, 7.0)
    kv.encode_probe_merge(_stream(), again.data_ptr())
    assert torch.equal(again, out) if merged else bool((again == 7.0).all())


@pytest.mark.parametrize("dims,element,rows,chunk,env", [
    ((32, 8, 128), "bf16", 200, 1, {}),                                      # whole step
    ((32, 8, 128), "bf16", 2000, 1, {}),                                     # split, merged
    ((32, 8, 128), "bf16", 200, 16, {}),                                     # whole chunk
    ((8, 2, 64), "bf16", 2400, 100, {"SKV_PREFILL_TILES": "2"}),             # chunk of splits, merged row by row
    ((8, 2, 64), "f32", 2400, 100, {"SKV_PREFILL_TILES": "2"}),
    ((8, 2, 64), "f32", 2400, 1, {}),
])
def test_a_context_at_any_floats_address(state, dims, element, rows, chunk, env):
    """The one at an address of whole 16 bytes, up to the order in which a merge adds its splits: up to 32 of them, 32 roundings of
    2^-24 of values of about 1."""
    saved = {name: os.environ.get(name) for name in env}
    os.environ.update(env)
    skv.flags.reload()
    try:
        got = []
        for lead in (0, 1, 2, 3):
            kv, q, k, v, _ = _layer(state, dims, element, rows, chunk, 5)
            qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v))
            buf = torch.full((q.size + 8,), 7.0, device="cuda")
            kv.encode_prefill_rows(_stream(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), chunk, buf.data_ptr() + lead * 4)
            assert bool((buf[:lead] == 7.0).all() and (buf[lead + q.size:] == 7.0).all())
            got.append(buf[lead:lead + q.size])
        assert all((g - got[0]).abs().max().item() <= 2e-6 for g in got)
    finally:
        for name, was in saved.items():
            os.environ.pop(name) if was is None else os.environ.__setitem__(name, was)
        skv.flags.reload()


class _Step:
    """One step of a kind over a context of so many pages with itself, as often as it is asked for"""

    def __init__(self, state, kind, dims, pages):
        q_heads, kv_heads, head_dim = dims
        self.kind, self.rows, self.head_dim = kind, pages * 16 - 1, head_dim
        self.kv, q, k, v, _ = _layer(state, dims, "bf16", self.rows, 1, pages)
        rng = np.random.default_rng(pages)
        if kind == "gated":
            q = rng.standard_normal((1, 2 * q.size), dtype=np.float32)
        w = (0.7 + rng.random((2, head_dim))).astype(np.float32)
        self.q, self.k, self.v, self.w = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v, w))
        self.rope = state.rope_table(self.rows + 1, head_dim, 10000.0)
        self.out = torch.full((q_heads * head_dim,), float("nan"), device="cuda")

    def __call__(self, stream):
        self.kv.truncate(self.rows)
        q, k, v, out = (t.data_ptr() for t in (self.q, self.k, self.v, self.out))
        if self.kind in ("prekv", "gated"):
            step = self.kv.encode_decode_step_prekv if self.kind == "prekv" else self.kv.encode_decode_step_gated
            step(stream, self.rope, self.rows, q, 0, k, 0, v, 0, self.w[0].data_ptr(), self.w[1].data_ptr(), 1e-6, float(self.head_dim), out)
        else:
            step = self.kv.encode_decode_step_static if self.kind == "static" else self.kv.encode_decode_step
            step(stream, k, 0, v, 0, q, out)
        return self.out


LINES = [((8, 2, 32), 24), ((16, 2, 64), 24), ((8, 8, 80), 24), ((32, 8, 128), 16), ((16, 1, 128), 16), ((16, 2, 256), 10)]


@pytest.mark.parametrize("kind", ["plain", "static", "prekv", "gated"])
@pytest.mark.parametrize("dims,pages", LINES)
@pytest.mark.parametrize("past", [0, 1])
def test_steps_of_all_kinds_around_the_line(state, kind, dims, pages, past):
    """Whole up to the line, and behind it bit for bit what the step is where a knob of the splits is set."""
    step = _Step(state, kind, dims, pages + past)
    got = step(_stream()).cpu().numpy().copy()
    os.environ["RETI_RUST_SDPA_2PASS_MIN_LEN"] = "128"
    skv.flags.reload()
    try:
        split = step(_stream()).cpu().numpy()
    finally:
        del os.environ["RETI_RUST_SDPA_2PASS_MIN_LEN"]
        skv.flags.reload()
    assert np.array_equal(got, split) == bool(past)
    # (some 24 pages in another order: 24 roundings of 2^-24 of values up to 4)
    assert np.abs(got - split).max() <= 6e-6


@pytest.mark.parametrize("kind", ["plain", "static", "prekv", "gated"])
@pytest.mark.parametrize("past", [0, 1])
def test_captured_steps_around_the_line(state, kind, past):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step = _Step(state, kind, (32, 8, 128), 16 + past)
        want = step(side.cuda_stream).clone()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step(side.cuda_stream)
        other = _Step(state, kind, (32, 8, 128), 9)
        for replay in range(3):
            other(side.cuda_stream)
            step.out.fill_(float("nan"))
            side.synchronize()
            graph.replay()
            side.synchronize()
            assert torch.equal(step.out, want), f"replay {replay}"
        del graph
    torch.cuda.synchronize()
