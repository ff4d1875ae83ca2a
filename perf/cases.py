"""The attention path's workloads, as a program that serves a model with this library runs them.

A case is one of two kinds of pass:

  "step"     one decode or verify step of `layers` full-attention layers: per layer attn_prep (q | gate split, norm, rope,
             quantizing write of the new K / V rows) and attn_decode / attn_decode_dev / attn_decode_rows with the fused
             output gate. `slots` sequences of `rows` new tokens each; their lengths, the new tokens included, are spread
             log-uniformly over [ctx_min, ctx].
  "prefill"  one chunk of `tokens` new tokens behind `past` cached ones, one layer: attn_prep (or kv_append, where the
             caller norms and ropes by itself) and attn_prefill.

`graph` steps are recorded once and replayed, the way a serving loop runs its decode step (positions and page tables
are device data, so one recording serves every depth); the others are plain calls. Values are N(0, 1), keys and queries
RMS-normed per head; pages of a pool are handed out in random order.
"""
import importlib
import math

import torch

p1a = importlib.import_module("p100e-engine_amd")

KV_TYPES = {"f16": p1a.KV_F16, "q8_0": p1a.KV_Q8_0, "q4_0": p1a.KV_Q4_0}
FREQ_BASE, EPS = 1.0e6, 1e-6


def _step(name, kv, heads, kv_heads, dim, page, ctx, ctx_min=None, slots=1, rows=1, layers=1, graph=False, a16=False, gate=True,
          position="host"):
    return {"name": name, "kind": "step", "kv": kv, "heads": heads, "kv_heads": kv_heads, "dim": dim, "page": page, "ctx": ctx,
            "ctx_min": ctx if ctx_min is None else ctx_min, "slots": slots, "rows": rows, "layers": layers, "graph": graph, "a16": a16,
            "gate": gate, "position": position}


def _prefill(name, kv, heads, kv_heads, dim, page, tokens, past, gate=True, scratch=False, prep=True):
    return {"name": name, "kind": "prefill", "kv": kv, "heads": heads, "kv_heads": kv_heads, "dim": dim, "page": page, "tokens": tokens,
            "past": past, "gate": gate, "scratch": scratch, "prep": prep}


def listed():
    return [
        # the smallest model the tests run, called plainly: what a call costs when there is next to nothing to compute
        _step("tiny_f16_512", "f16", 4, 1, 64, 16, 512, gate=False),
        # a single user in a long chat with the 27B shape: eight of its full-attention layers, a16 output for the next matvec
        _step("one_27b_q8_32k", "q8_0", 24, 4, 256, 256, 32768, layers=8, graph=True, a16=True, position="device"),
        # eight users of different history on one server
        _step("slots8_27b_q8", "q8_0", 24, 4, 256, 256, 32768, ctx_min=1024, slots=8, layers=4, graph=True),
        # many users early in their chats: a full call of 32 rows
        _step("slots32_27b_q8", "q8_0", 24, 4, 256, 256, 5000, ctx_min=300, slots=32, layers=4, graph=True),
        # speculative decoding: four users, one accepted token and three drafts each, a compact cache
        _step("verify_27b_q4_64k", "q4_0", 24, 4, 256, 256, 65536, slots=4, rows=4, layers=2, graph=True),
        # the same for one user, at a depth where the cache is kept unquantized
        _step("verify_27b_f16_48k", "f16", 24, 4, 256, 256, 49153, rows=4, layers=2, graph=True, position="device"),
        # heads of 128 (the common size of dense models) behind small pages, plain calls
        _step("slots4_d128_f16", "f16", 32, 8, 128, 16, 9001, ctx_min=2000, slots=4, layers=4),
        # a head size that is no power of two
        _step("one_d96_q8_8k", "q8_0", 24, 4, 96, 256, 8190, layers=2),
        # a chunk of a long document, all of its context behind it: the largest call
        _prefill("chunk_27b_q8_32k", "q8_0", 24, 4, 256, 256, 4096, 28672, scratch=True),
        # the first prompt of a chat, heads of 128
        _prefill("prompt_d128_f16_2k", "f16", 32, 8, 128, 16, 2003, 0),
        # a user's next message: a few dozen tokens behind a long history
        _prefill("turn_27b_q8_16k", "q8_0", 24, 4, 256, 256, 77, 16000),
        # a middling chunk over a compact cache; the caller has its own norm and rope and its own gate
        _prefill("chunk_27b_q4_4k", "q4_0", 24, 4, 256, 256, 512, 3500, gate=False, prep=False),
    ]


HEADS = [(4, 1), (24, 4), (16, 2), (32, 8), (8, 8), (16, 4)]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    heads, kv_heads = rng.choice(HEADS)
    kv = rng.choice(["f16", "q8_0", "q8_0", "q4_0"])
    page = rng.choice([16, 64, 256])
    if rng.random() < 0.6:
        dim = rng.choice([64, 128, 128, 256, 256, 256, 96, 192])
        rows = rng.choice([1, 1, 1, 2, 4])
        slots = rng.choice([1, 1, 2, 4, 8, 16, 32])
        slots = min(slots, 32 // rows)
        # at most 384 MB of cache a layer (24 MB for head sizes that are no power of two)
        most = (24 if dim in (96, 192) else 384) * 1_000_000 // (slots * 2 * p1a.kv_row_bytes(KV_TYPES[kv], kv_heads, dim))
        ctx = _log_uniform(rng, 64, min(131072, most))
        c = _step("", kv, heads, kv_heads, dim, page, ctx, ctx_min=max(rows, ctx // rng.choice([1, 4, 16])), slots=slots, rows=rows,
                  layers=rng.choice([1, 2, 4]), graph=rng.random() < 0.6, a16=rng.random() < 0.3, gate=rng.random() < 0.8,
                  position=rng.choice(["host", "device"]))
    else:
        dim = rng.choice([64, 128, 256, 256])
        past = rng.choice([0, _log_uniform(rng, 100, 28672)])
        tokens = _log_uniform(rng, 17, 4096)
        c = _prefill("", kv, heads, kv_heads, dim, page, tokens, past, gate=rng.random() < 0.8, scratch=rng.random() < 0.5, prep=rng.random() < 0.7)
        while work(c)["flops"] > 2.9e12:                       # (32 heads of 256 over the longest context)
            c["tokens"] = c["tokens"] * 3 // 4
    del c["name"]
    return c


def _lengths(case):
    """the sequences' lengths, the new tokens included: evenly spread over the logarithm, in an order that is not sorted"""
    n, lo, hi = case["slots"], case["ctx_min"], case["ctx"]
    if n == 1:
        return [hi]
    at = [(i * 5) % n for i in range(n)]                       # (n is a power of two: a permutation)
    return [max(case["rows"], int(round(lo * (hi / lo) ** (a / (n - 1))))) for a in at]


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _normed(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _fill(g, cache, n, kv_heads, dim):
    """positions 0 .. n - 1 of one sequence, through the library's own append"""
    for a in range(0, n, 8192):
        t = min(8192, n - a)
        p1a.kv_append(cache, _normed(_randn(g, t, kv_heads, dim)), _randn(g, t, kv_heads, dim), a, t)


def _pool(g, case, lengths, layers):
    """a pool of `layers` layers with the sequences' pages in random order, and each layer's cache"""
    kv, hkv, dim, page = KV_TYPES[case["kv"]], case["kv_heads"], case["dim"], case["page"]
    psh = page.bit_length() - 1
    need = [-(-n // page) for n in lengths]
    per_seq = max(need)
    order = torch.randperm(sum(need), generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(lengths) * per_seq, dtype=torch.int32, device="cuda")
    at = 0
    for s, n in enumerate(need):
        table[s * per_seq:s * per_seq + n] = order[at:at + n]
        at += n
    pool = torch.zeros(sum(need) * layers * 2 * page * p1a.kv_row_bytes(kv, hkv, dim), dtype=torch.uint8, device="cuda")
    caches = [p1a.KVCache.paged(kv, hkv, dim, psh, sum(need), table, per_seq, n_layers=layers, layer=i, pool=pool) for i in range(layers)]
    for c in caches:
        for s, n in enumerate(lengths):
            _fill(g, c.slot(s, per_seq), n, hkv, dim)
    return pool, caches, per_seq


def _rotary(dim):
    return 64 if dim == 256 else dim


def _prepare_step(case, g):
    hq, hkv, dim, slots, rows, layers = (case[k] for k in ("heads", "kv_heads", "dim", "slots", "rows", "layers"))
    lengths = _lengths(case)
    t = slots * rows
    pool, caches, per_seq = _pool(g, case, lengths, layers)
    pos = [n - rows + r for n in lengths for r in range(rows)]
    s = {"case": case, "pool": pool, "p0": pos[0], "pos": torch.tensor(pos, dtype=torch.int32, device="cuda")}
    if slots == 1:
        s["caches"] = [c.slot(0, per_seq) for c in caches]
    else:
        rtab = torch.tensor([q * per_seq for q in range(slots) for _ in range(rows)], dtype=torch.int32, device="cuda")
        s["caches"] = [c.with_rows(rtab) for c in caches]
    # what the layers' projections hand over
    s["qg"], s["k"], s["v"] = _randn(g, layers, t, hq * 2 * dim), _randn(g, layers, t, hkv, dim), _randn(g, layers, t, hkv, dim)
    s["q_norm"], s["k_norm"] = 1 + 0.1 * _randn(g, dim), 1 + 0.1 * _randn(g, dim)
    s["q"], s["gate"], s["out"] = (torch.empty((layers, t, hq, dim), device="cuda") for _ in range(3))
    s["a16"] = torch.zeros((layers, p1a.a16_bytes(t, hq * dim) // 2), dtype=torch.float16, device="cuda") if case["a16"] else None
    return s


def _run_step(s):
    case = s["case"]
    hq, dim, slots, rows = case["heads"], case["dim"], case["slots"], case["rows"]
    t, scale = slots * rows, case["dim"] ** -0.5
    for i, c in enumerate(s["caches"]):
        q, gate, out = s["q"][i], s["gate"][i], s["out"][i]
        by_pos = slots > 1 or case["position"] == "device"
        p1a.attn_prep(s["qg"][i], s["k"][i], s["v"][i], s["q_norm"], s["k_norm"], s["pos"], q, gate, c, -1 if by_pos else s["p0"], t, hq,
                      _rotary(dim), FREQ_BASE, EPS)
        g = gate if case["gate"] else None
        if s["a16"] is not None or slots > 1:
            p1a.attn_decode_rows(q, c, out, t, s["pos"], hq, scale, gate=g, rows_per_seq=rows, qbuf=None if s["a16"] is None else s["a16"][i])
        elif by_pos:
            p1a.attn_decode_dev(q, c, out, t, s["pos"], case["ctx"], hq, scale, gate=g)
        else:
            p1a.attn_decode(q, c, out, t, s["p0"], hq, scale, gate=g)


_recording = None   # the stream that steps are recorded on: one for the program, as a serving loop has


def _record(s):
    global _recording
    if _recording is None:
        _recording = torch.cuda.Stream()
    case = s["case"]
    _recording.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(_recording):
        p1a.warmup(case["slots"] * case["rows"], case["heads"], case["kv_heads"], case["dim"])
        with torch.cuda.graph(graph, stream=_recording):
            _run_step(s)
    torch.cuda.current_stream().wait_stream(_recording)
    return graph


def _prepare_prefill(case, g):
    hq, hkv, dim, t, past = (case[k] for k in ("heads", "kv_heads", "dim", "tokens", "past"))
    pool, caches, per_seq = _pool(g, case, [past + t], 1)
    s = {"case": case, "pool": pool, "cache": caches[0].slot(0, per_seq), "out": torch.empty((t, hq, dim), device="cuda"), "scratch": None}
    if case["prep"]:
        s["pos"] = torch.arange(past, past + t, dtype=torch.int32, device="cuda")
        s["qg"], s["k"], s["v"] = _randn(g, t, hq * 2 * dim), _randn(g, t, hkv, dim), _randn(g, t, hkv, dim)
        s["q_norm"], s["k_norm"] = 1 + 0.1 * _randn(g, dim), 1 + 0.1 * _randn(g, dim)
        s["q"], s["gate"] = torch.empty((t, hq, dim), device="cuda"), torch.empty((t, hq, dim), device="cuda")
    else:
        s["q"], s["k"], s["v"] = _normed(_randn(g, t, hq, dim)), _normed(_randn(g, t, hkv, dim)), _randn(g, t, hkv, dim)
        s["gate"] = _randn(g, t, hq, dim)
    if case["scratch"]:
        s["scratch"] = torch.empty(p1a.prefill_scratch_bytes(t, past, hq, hkv, dim), dtype=torch.uint8, device="cuda")
    return s


def _run_prefill(s):
    case = s["case"]
    t, past, hq, dim = case["tokens"], case["past"], case["heads"], case["dim"]
    if case["prep"]:
        p1a.attn_prep(s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["pos"], s["q"], s["gate"], s["cache"], past, t, hq, _rotary(dim),
                      FREQ_BASE, EPS)
    else:
        p1a.kv_append(s["cache"], s["k"], s["v"], past, t)
    p1a.attn_prefill(s["q"], s["cache"], s["out"], t, past, hq, dim ** -0.5, gate=s["gate"] if case["gate"] else None, scratch=s["scratch"])


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["kind"] == "prefill":
        return _prepare_prefill(case, g)
    s = _prepare_step(case, g)
    s["graph"] = _record(s) if case["graph"] else None
    return s


def run(state):
    case = state["case"]
    if case["kind"] == "prefill":
        _run_prefill(state)
    elif state["graph"] is not None:
        state["graph"].replay()
    else:
        _run_step(state)
    got = {"out": state["out"], "cache": state["pool"]}
    if case["kind"] == "step" or case["prep"]:
        got["q"], got["gate"] = state["q"], state["gate"]
    if case["kind"] == "step" and case["a16"]:
        got["a16"] = state["a16"]
    return got


def work(case):
    hq, hkv, dim = case["heads"], case["kv_heads"], case["dim"]
    row = 2 * p1a.kv_row_bytes(KV_TYPES[case["kv"]], hkv, dim)           # K and V of one position
    if case["kind"] == "step":
        t, layers, rows, lengths = case["slots"] * case["rows"], case["layers"], case["rows"], _lengths(case)
        keys = sum(sum(n - r for r in range(rows)) for n in lengths)       # (query, key) pairs of one head
        read = sum(lengths) * row
    else:
        t, layers, prep = case["tokens"], 1, case["prep"]
        keys = case["past"] * t + t * (t + 1) // 2
        read = (case["past"] + t) * row
    qh = t * hq * dim * 4
    new = t * 2 * hkv * dim * 4 + t * row                                  # new K / V rows: fp32 in, cache rows out
    if case["kind"] == "step" or prep:
        new += 2 * qh + 2 * qh                                             # q | gate in, q and gate out
    moved = read + new + (3 if case["gate"] else 2) * qh                   # q (and the gate) in, the result out
    if case.get("a16"):
        moved += p1a.a16_bytes(t, hq * dim)
    return {"bytes": layers * moved, "flops": layers * 4 * dim * hq * keys}


def tolerance(case):
    # The products take f16 operands (2^-11 each) and sum in fp32: against the same pass in float64 the results of the listed
    # and of drawn cases are 0.2e-4 .. 4.3e-4 off (2-norm), and a16 values are rounded to f16 once more. Four times that;
    # cache bytes are whole numbers and stay the same.
    return {"rel": 1.6e-3}
