"""The work this framework is used for, as measurable cases over its public entry points.

A case is one pass of the KV path of a model step: decode steps of one or several sequences,
chunks of new rows over a cache (a prompt, a long context, a speculative verify), and the prefix
hot cache (a cached session picked up again, a conversation turn). The head geometries are
those of the benchmark's configurations: 32 query / 8 kv heads of 128, 16 / 2 of 256 (hybrid
model at 32k context), 16 / 8 of 256 (sliding-window model, window 1024); drawn cases add
narrower, odd and wider heads of the tests.

Every pass first takes the caches back to the length the case starts from (`truncate`, host
bookkeeping only, what a rollback does), so passes repeat; the rows a pass appends are attended
by its later steps, so its contexts carry the updated caches too.
"""
import numpy as np
import torch

import saragossa_amd as skv

EPS = 1.0e-6
THETA = 1.0e6
_CTX = []


def _context():
    # one context per process, as a serving program has
    if not _CTX:
        _CTX.append(skv.DecodeResidentState(0))
    return _CTX[0]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def listed():
    qwen = {"q_heads": 32, "kv_heads": 8, "head_dim": 128}
    hybrid = {"q_heads": 16, "kv_heads": 2, "head_dim": 256}
    sliding = {"q_heads": 16, "kv_heads": 8, "head_dim": 256}
    return [
        # one step of one attention layer at 1024 cached rows: the smallest call a host makes
        {"name": "decode_one_layer_1k", "kind": "decode", **qwen, "element": "bf16", "layers": 1, "window": 0,
         "rows": 1024, "tokens": 1, "seqs": 1, "step": "plain"},
        # a chat answer after a 2048-token prompt: two tokens through all 36 layers, norms and
        # rotation fused into the step
        {"name": "decode_36_layers_2k", "kind": "decode", **qwen, "element": "bf16", "layers": 36, "window": 0,
         "rows": 2048, "tokens": 2, "seqs": 1, "step": "prekv"},
        # long-context decode of the hybrid model's 10 full-attention layers, with its output gate
        {"name": "decode_gated_32k", "kind": "decode", **hybrid, "element": "bf16", "layers": 10, "window": 0,
         "rows": 32768, "tokens": 2, "seqs": 1, "step": "gated"},
        # greedy decoding keeps f32 rows (the default policy): mid-length context, ragged length
        {"name": "decode_f32_greedy", "kind": "decode", **qwen, "element": "f32", "layers": 36, "window": 0,
         "rows": 5003, "tokens": 1, "seqs": 1, "step": "prekv"},
        # four users of the sliding-window model at 65536 context, one period of its layers
        # (five local, one global)
        {"name": "batch4_sliding_64k", "kind": "sliding", **sliding, "element": "bf16", "window": 1024,
         "rows": 65536, "tokens": 2, "seqs": 4, "periods": 1},
        # speculative decoding: a draft of six tokens verified over 8k rows, then rolled back
        {"name": "verify_6_rows_8k", "kind": "chunk", **hybrid, "element": "bf16", "layers": 10, "window": 0,
         "rows": 8192, "chunk": 6, "norm": True},
        # a prompt of 2000 tokens (not a multiple of the chunk) prefilled in chunks of 512
        {"name": "prompt_2000", "kind": "prompt", **qwen, "element": "bf16", "layers": 4, "window": 0,
         "rows": 2000, "chunk": 512},
        # one more chunk of a long document
        {"name": "chunk_512_over_32k", "kind": "chunk", **hybrid, "element": "bf16", "layers": 2, "window": 0,
         "rows": 32768, "chunk": 512, "norm": True},
        # a prompt through the sliding-window model's local layers (ring caches)
        {"name": "prompt_ring_3000", "kind": "prompt", **sliding, "element": "bf16", "layers": 5, "window": 1024,
         "rows": 3000, "chunk": 512},
        # the prompt of a greedy request: f32 rows
        {"name": "prompt_f32_1500", "kind": "prompt", **qwen, "element": "f32", "layers": 4, "window": 0,
         "rows": 1500, "chunk": 512},
        # a session whose prompt is in the hot cache is picked up: blocks restored, first token
        {"name": "resume_4864", "kind": "resume", **qwen, "element": "bf16", "layers": 36, "window": 0,
         "rows": 4864},
        # the next turn of a conversation over a full block pool: restore of the cached prefix,
        # prefill of 512 new tokens, their blocks remembered, older ones evicted
        {"name": "turn_512_over_4700", "kind": "turn", **qwen, "element": "bf16", "layers": 36, "window": 0,
         "rows": 4700, "chunk": 512, "blocks_per_chunk": 32},
    ]


GEOMETRIES = [(32, 8, 128), (16, 2, 256), (16, 8, 256), (8, 2, 64), (12, 4, 96), (8, 8, 80), (28, 4, 128),
              (8, 2, 512), (24, 8, 128)]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _cost(case):
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / (1e14 if case["element"] == "f32" else 4e14)


def draw(rng):
    q, kv, hd = rng.choice(GEOMETRIES)
    case = {"kind": rng.choice(["decode", "decode", "decode", "sliding", "chunk", "chunk", "prompt", "prompt", "resume", "turn"]),
            "q_heads": q, "kv_heads": kv, "head_dim": hd, "element": rng.choice(["bf16", "bf16", "f32"])}
    kind = case["kind"]
    if kind == "decode":
        case.update(layers=rng.randint(1, 24), window=rng.choice([0, 0, 0, 512, 1024]), rows=_log_int(rng, 17, 32768),
                    tokens=rng.randint(1, 2), seqs=rng.choice([1, 1, 1, 2, 4, 7]), step=rng.choice(["plain", "prekv", "gated"]))
        if case["seqs"] > 1:
            case.update(step="plain", layers=rng.randint(1, 6))
    elif kind == "sliding":
        case.update(q_heads=16, kv_heads=8, head_dim=256, window=rng.choice([512, 1024]), rows=_log_int(rng, 1500, 40000),
                    tokens=rng.randint(1, 2), seqs=rng.randint(1, 4), periods=1)
    elif kind == "chunk":
        case.update(layers=rng.randint(1, 2), window=0, rows=_log_int(rng, 64, 24000), chunk=_log_int(rng, 2, 512),
                    norm=rng.random() < 0.5)
    elif kind == "prompt":
        case.update(layers=rng.randint(1, 3), window=rng.choice([0, 0, 512, 1024]), rows=_log_int(rng, 33, 2500),
                    chunk=rng.choice([256, 512, 512, 1024]))
    elif kind == "resume":
        case.update(element="bf16", layers=rng.randint(4, 36), window=0, rows=_log_int(rng, 64, 4800))
    else:
        case.update(element="bf16", layers=rng.randint(2, 12), window=0, rows=_log_int(rng, 200, 4000),
                    chunk=rng.randint(40, 512), blocks_per_chunk=rng.choice([4, 32]))
    # no drawn case costs more than the largest listed one
    limit = max(_cost(c) for c in listed())
    while _cost(case) > limit and case.get("layers", 1) > 1:
        case["layers"] = (case["layers"] + 1) // 2
    while _cost(case) > limit:
        case["rows"] = case["rows"] * 2 // 3
    return case


# ---- inputs ------------------------------------------------------------------------------

class _Inputs:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.host = np.random.default_rng(seed)

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", dtype=torch.float32, generator=self.gen)


def _layer(case, inputs, capacity, window=0):
    element = skv.DTYPE_F32 if case["element"] == "f32" else skv.DTYPE_BF16
    kv = _context().full_attention_with_element(capacity, case["q_heads"], case["kv_heads"], case["head_dim"], element, window)
    kv.set_block_table(inputs.host.permutation(kv.pages()).astype(np.int32))
    return kv


def _fill(kv, inputs, rows):
    """rows cached rows of N(0, 1), as after a prompt."""
    step = 16384
    for first in range(0, rows, step):
        n = min(step, rows - first)
        k, v = inputs.normal(n, kv.kv_dim()), inputs.normal(n, kv.kv_dim())
        kv.encode_append_batch(_stream(), k.data_ptr(), v.data_ptr(), n)


def _rope(case, positions):
    return _context().rope_table(positions, case["head_dim"], THETA)


def _norm_weights(case, inputs, layers):
    return 1.0 + 0.1 * inputs.normal(layers, 2, case["head_dim"])


def prepare(case, seed):
    x = _Inputs(seed)
    q_dim, kv_dim = case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    s = {"case": case, "q_dim": q_dim, "kv_dim": kv_dim}
    kind = case["kind"]
    if kind in ("decode", "sliding"):
        tokens, rows, seqs = case["tokens"], case["rows"], case["seqs"]
        if kind == "sliding":
            windows = ([case["window"]] * 5 + [0]) * case["periods"]
        else:
            windows = [case["window"]] * case["layers"]
        s["layers"] = []
        for w in windows:
            group = []
            for i in range(seqs):
                n = rows - 37 * i if rows > 400 else rows  # independent sequences, lengths of their own
                kv = _layer(case, x, n + tokens, w)
                _fill(kv, x, n)
                group.append((kv, n))
            s["layers"].append(group)
        gated = kind == "decode" and case["step"] == "gated"
        n_layers = len(windows)
        s["q"] = x.normal(tokens, n_layers, seqs, (2 if gated else 1) * q_dim)
        s["k"] = x.normal(tokens, n_layers, seqs, kv_dim)
        s["v"] = x.normal(tokens, n_layers, seqs, kv_dim)
        s["out"] = torch.empty(tokens, n_layers, seqs, q_dim, device="cuda")
        if kind == "decode" and case["step"] != "plain":
            s["rope"] = _rope(case, rows + tokens)
            s["w"] = _norm_weights(case, x, n_layers)
    elif kind in ("chunk", "prompt"):
        rows = case["rows"]
        base, new = (rows, case["chunk"]) if kind == "chunk" else (0, rows)
        s["layers"] = []
        for _ in range(case["layers"]):
            kv = _layer(case, x, base + new, case["window"])
            _fill(kv, x, base)
            s["layers"].append(kv)
        _new_rows(s, case, x, new)
        s["rope"] = _rope(case, base + new)
    elif kind == "resume":
        rows, layers = case["rows"], case["layers"]
        bt = 16
        blocks = rows // bt
        s["layers"] = [_layer(case, x, rows + 2) for _ in range(layers)]
        for kv in s["layers"]:
            _fill(kv, x, rows)
        s["tokens"] = x.host.integers(0, 151936, size=rows).astype(np.uint64)
        s["hot"] = skv.HotCache(_context(), bt, blocks, blocks, s["layers"])
        s["root"] = h = skv.BlockHash.for_session("session")
        hashes = []
        for b in range(blocks):
            h = skv.BlockHash.chain(h, s["tokens"][b * bt:(b + 1) * bt])
            hashes.append(h)
        s["hot"].remember_prefix_blocks(s["root"], hashes, bt, s["layers"], stream=_stream())
        s["q"], s["k"], s["v"] = x.normal(layers, q_dim), x.normal(layers, kv_dim), x.normal(layers, kv_dim)
        s["out"] = torch.empty(layers, q_dim, device="cuda")
        s["rope"] = _rope(case, rows + 2)
        s["w"] = _norm_weights(case, x, layers)
    else:  # turn
        rows, layers, bt = case["rows"], case["layers"], 16
        new = case["chunk"] + bt  # the cached prefix ends at a block boundary: up to 15 rows more
        s["layers"] = [_layer(case, x, rows + new) for _ in range(layers)]
        for kv in s["layers"]:
            _fill(kv, x, rows)
        s["history"] = x.host.integers(0, 151936, size=rows).astype(np.uint64)
        s["turn_rng"] = x.host
        # room for the history and one and a half turns: the second turn evicts blocks of the first
        pool = rows // bt + (case["chunk"] + 15) // bt * 3 // 2 + 1
        s["hot"] = skv.HotCache(_context(), bt, pool, pool, s["layers"])
        h = root = skv.BlockHash.for_session("session")
        hashes = []
        for b in range(rows // bt):
            h = skv.BlockHash.chain(h, s["history"][b * bt:(b + 1) * bt])
            hashes.append(h)
        s["hot"].remember_prefix_blocks(root, hashes, bt, s["layers"], stream=_stream())
        s["model"] = skv.LoadedModelKv(s["hot"], enabled=True)
        _new_rows(s, case, x, new)
        s["first"] = rows // bt * bt
        s["rope"] = _rope(case, rows + new)
    return s


def _new_rows(s, case, x, new):
    """The raw projections of the new rows of every layer, and where their finished q and k and
    their contexts go."""
    n = case["layers"]
    s["q"], s["k"], s["v"] = x.normal(n, new, s["q_dim"]), x.normal(n, new, s["kv_dim"]), x.normal(n, new, s["kv_dim"])
    s["w"] = _norm_weights(case, x, n)
    s["out"] = torch.zeros(n, new, s["q_dim"], device="cuda")
    # scratch of the finished rows, one layer's worth, as a decoder keeps it
    s["q_fin"] = torch.empty(new, s["q_dim"], device="cuda")
    s["k_fin"] = torch.empty(new, s["kv_dim"], device="cuda")


# ---- passes ------------------------------------------------------------------------------

def run(s):
    return {"decode": _run_decode, "sliding": _run_decode, "chunk": _run_chunk, "prompt": _run_prompt,
            "resume": _run_resume, "turn": _run_turn}[s["case"]["kind"]](s)


def _run_decode(s):
    case, stream = s["case"], _stream()
    q, k, v, out = s["q"], s["k"], s["v"], s["out"]
    tokens, n_layers, seqs = k.shape[:3]
    for group in s["layers"]:
        for kv, n in group:
            kv.truncate(n)
    qs, ks, os_ = q.shape[3] * 4, k.shape[3] * 4, out.shape[3] * 4
    q0, k0, v0, o0 = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    step = case.get("step", "plain")
    for t in range(tokens):
        for li, group in enumerate(s["layers"]):
            at = (t * n_layers + li) * seqs
            if seqs > 1:
                skv.encode_decode_step_batch([g[0] for g in group], stream, [k0 + (at + i) * ks for i in range(seqs)],
                                             [v0 + (at + i) * ks for i in range(seqs)], [q0 + (at + i) * qs for i in range(seqs)],
                                             [o0 + (at + i) * os_ for i in range(seqs)])
            elif step == "plain":
                group[0][0].encode_decode_step(stream, k0 + at * ks, 0, v0 + at * ks, 0, q0 + at * qs, o0 + at * os_)
            else:
                kv, n = group[0]
                fn = kv.encode_decode_step_gated if step == "gated" else kv.encode_decode_step_prekv
                w = s["w"][li]
                fn(stream, s["rope"], n + t, q0, at * qs, k0, at * ks, v0, at * ks, w[0].data_ptr(), w[1].data_ptr(),
                   EPS, float(case["head_dim"]), o0 + at * os_)
    return out


def _prefill(s, li, first, last, base, norm=True):
    """Rows [first, last) of the new ones through layer li: norms and rotation, then the chunk."""
    case, stream, n = s["case"], _stream(), last - first
    q, k, v, out = s["q"][li, first:last], s["k"][li, first:last], s["v"][li, first:last], s["out"][li, first:last]
    qp, kp = q.data_ptr(), k.data_ptr()
    if norm:
        w = s["w"][li]
        _context().encode_rms_norm_rope_rows(stream, s["rope"], base + first, qp, w[0].data_ptr(), n, case["q_heads"],
                                             case["head_dim"], EPS, s["q_fin"].data_ptr())
        _context().encode_rms_norm_rope_rows(stream, s["rope"], base + first, kp, w[1].data_ptr(), n, case["kv_heads"],
                                             case["head_dim"], EPS, s["k_fin"].data_ptr())
        qp, kp = s["q_fin"].data_ptr(), s["k_fin"].data_ptr()
    s["layers"][li].encode_prefill_rows(stream, qp, kp, v.data_ptr(), n, out.data_ptr())


def _run_chunk(s):
    case = s["case"]
    for li, kv in enumerate(s["layers"]):
        kv.truncate(case["rows"])
        _prefill(s, li, 0, case["chunk"], case["rows"], case["norm"])
    return s["out"]


def _run_prompt(s):
    case = s["case"]
    rows, chunk = case["rows"], case["chunk"]
    for kv in s["layers"]:
        kv.truncate(0)
    for first in range(0, rows, chunk):
        for li in range(len(s["layers"])):
            _prefill(s, li, first, min(first + chunk, rows), 0)
    return s["out"]


def _run_resume(s):
    case, stream = s["case"], _stream()
    reused, digest = s["hot"].match_restore(s["root"], s["tokens"], s["layers"], stream=stream)
    q0, k0, v0, o0 = (s[n].data_ptr() for n in ("q", "k", "v", "out"))
    for li, kv in enumerate(s["layers"]):
        w = s["w"][li]
        kv.encode_decode_step_prekv(stream, s["rope"], reused, q0, li * s["q_dim"] * 4, k0, li * s["kv_dim"] * 4, v0,
                                    li * s["kv_dim"] * 4, w[0].data_ptr(), w[1].data_ptr(), EPS, float(case["head_dim"]),
                                    o0 + li * s["q_dim"] * 4)
    return [s["out"], reused, np.frombuffer(digest, dtype=np.uint8)]


def _run_turn(s):
    case, first = s["case"], s["first"]
    # the user's new message: other tokens every turn
    tokens = np.concatenate([s["history"], s["turn_rng"].integers(0, 151936, size=case["chunk"]).astype(np.uint64)])

    def prefill_rows(lo, hi):
        # a decoder runs the model over [lo, hi) layer by layer
        for li in range(len(s["layers"])):
            _prefill(s, li, lo - first, hi - first, first)

    reused = s["model"].prefill_prompt_state(tokens, "session", s["layers"], prefill_rows, stream=_stream(),
                                             blocks_per_chunk=case["blocks_per_chunk"])
    return [s["out"][:, :len(tokens) - first], reused, len(s["hot"])]


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    q_dim, kv_dim = case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    elem = 4 if case["element"] == "f32" else 2
    kind, window, rows = case["kind"], case["window"], case["rows"]
    gate = 1 if case.get("step") == "gated" else 0

    def attended(n, w):  # rows the query at position n - 1 sees
        return min(n, w) if w else n

    if kind in ("decode", "sliding"):
        windows = ([window] * 5 + [0]) * case["periods"] if kind == "sliding" else [window] * case["layers"]
        nbytes = flops = 0
        for w in windows:
            for i in range(case["seqs"]):
                n = rows - 37 * i if rows > 400 else rows
                for t in range(case["tokens"]):
                    seen = attended(n + t + 1, w)
                    # cached rows read, the new row in (f32) and out, q (and gate) in, context out
                    nbytes += 2 * (seen - 1) * kv_dim * elem + 2 * kv_dim * (4 + elem) + (2 + gate) * q_dim * 4
                    flops += 4 * seen * q_dim
        return {"bytes": nbytes, "flops": flops}
    if kind in ("chunk", "prompt", "turn"):
        if kind == "prompt":
            base, new, chunk = 0, rows, case["chunk"]
        elif kind == "chunk":
            base, new, chunk = rows, case["chunk"], case["chunk"]
        else:
            base = rows // 16 * 16
            new = rows + case["chunk"] - base
            chunk = case["blocks_per_chunk"] * 16
        nbytes = flops = 0
        for first in range(0, new, chunk):
            n = min(chunk, new - first)
            old = base + first
            kept = min(old, window) if window else old
            # cached rows read once per chunk, the new rows in and out, q in and context out
            nbytes += 2 * kept * kv_dim * elem + n * (2 * kv_dim * (4 + elem) + 2 * q_dim * 4)
            pairs = sum(attended(old + i + 1, window) for i in range(n))
            flops += 4 * pairs * q_dim
        if kind == "turn":
            nbytes += 2 * 2 * (base + (rows + case["chunk"]) // 16 * 16 - base) * kv_dim * elem  # restored, remembered
        return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}
    # resume: blocks read from the pool and written to the caches, then attended once
    n = rows // 16 * 16
    one = 3 * 2 * n * kv_dim * elem + 2 * kv_dim * (4 + elem) + 2 * q_dim * 4
    return {"bytes": one * case["layers"], "flops": 4 * (n + 1) * q_dim * case["layers"]}


def tolerance(case):
    # About four times the distance of the contexts from attention in 64 bits over the same cached
    # rows, over these cases and drawn ones: bf16 caches multiply 16-bit queries and probabilities
    # (relative 3e-6 to 1e-5, largest 3e-4 of the root mean square), f32 caches sum in 32 bits
    # (relative 2e-7 to 1e-6, largest 1.2e-5, whichever order the sums are taken in).
    if case["element"] == "f32":
        return {"rel": 4.0e-6, "max": 5.0e-5}
    return {"rel": 4.0e-5, "max": 1.2e-3}
