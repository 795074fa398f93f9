"""The workloads this package is timed on, through its public entry points.

Each case is one attention call of one layer, as a serving program makes it:
decode over a slot pool or over a runtime cache, prompt chunks over cached
pages, and decode with part of the cache in host memory.  Shapes are those of
the package's own workloads (``helm_amd/workloads.py``, ``bench.py``) and of
the architectures its patched forwards cover: head dimensions 64, 128 and 256,
grouped and plain heads, soft-capped and windowed attention.

Query and key values are N(0, 1) with the query scaled by ``Q_STD`` (logits of
standard deviation ~1.5, a moderately peaked softmax), values N(0, 1).
"""
import math

import torch

from helm_amd.paged import prepare_paged_decode
from helm_amd.runtime.kv_allocator import KVAllocator
from helm_amd.runtime.kv_cache import KVCacheManager, perform_streaming_attention
from helm_amd.runtime.kv_offload import _decode_batched, _stream_prefill_batched

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
Q_STD = 1.5
NO_EVICTION = 10 ** 15
LARGEST_KV_BYTES = 2 * 131072 * 40 * 128 * 2      # decode-128k-mha
LARGEST_PREFILL_FLOPS = 4 * 512 * 32768 * 32 * 128  # prefill-512-over-32k


# kind "pool": prepare_paged_decode(...).run() over a slot pool, `lens` tokens
#   per sequence (the serving loop that keeps its own page table);
# kind "step": _decode_batched over the contiguous all-GPU cache under the
#   decode mask of a left-padded batch: the token written, then attention;
# kind "stream": perform_streaming_attention over a cache manager's pages.
#   mask "none" (with q_len > 1: HELM's top-left causal), "zeros" (the decode
#   mask), "window" (Gemma-2's sliding window of `window` tokens);
#   host = the oldest fraction of the pages evicted to pinned host memory;
# kind "chunk": _stream_prefill_batched, a later prompt chunk of q_len tokens
#   under the chunk-causal mask the pipeline builds, T tokens cached with it.
def _pool(name, dt, Hq, Hkv, D, page, lens):
    return dict(name=name, kind="pool", dtype=dt, Hq=Hq, Hkv=Hkv, D=D, page=page,
                lens=",".join(str(x) for x in lens))


def _step(name, dt, Hq, Hkv, D, B, T):
    return dict(name=name, kind="step", dtype=dt, Hq=Hq, Hkv=Hkv, D=D, B=B, T=T)


def _stream(name, dt, Hq, Hkv, D, page, q_len, T, mask="none", window=0, cap=0.0, host=0.0):
    return dict(name=name, kind="stream", dtype=dt, Hq=Hq, Hkv=Hkv, D=D, page=page, q_len=q_len,
                T=T, mask=mask, window=window, cap=cap, host=host)


def _chunk(name, dt, Hq, Hkv, D, page, q_len, T):
    return dict(name=name, kind="chunk", dtype=dt, Hq=Hq, Hkv=Hkv, D=D, page=page, q_len=q_len,
                T=T)


def listed():
    return [
        # a small model answering a short chat: launch and latency bound
        _pool("decode-2k", "f16", 16, 8, 128, 16, [2048]),
        # the headline: one long conversation, grouped heads, everything resident
        _pool("decode-32k", "bf16", 32, 8, 128, 16, [32768]),
        # a serving batch of unrelated requests, lengths as they come
        _pool("decode-ragged-b8", "bf16", 40, 8, 128, 16,
              [4101, 30177, 12553, 23016, 8190, 27811, 17408, 5999]),
        # plain (ungrouped) heads at the longest context: the most KV one call reads
        _pool("decode-128k-mha", "f16", 40, 40, 128, 16, [131072]),
        # small head dimension, a batch of four
        _pool("decode-d64-b4", "f16", 32, 8, 64, 64, [8192, 12001, 3333, 16000]),
        # the production decode step: append + decode mask over a padded batch
        _step("decode-step-b4", "bf16", 40, 8, 128, 4, 8200),
        # soft-capped, windowed decode at head dimension 256
        _stream("decode-d256-softcap", "bf16", 16, 8, 256, 64, 1, 8000, "window", 4096, 50.0),
        # half of the context in pinned host memory, streamed over the host link
        _stream("decode-32k-offload50", "bf16", 32, 8, 128, 16, 1, 32768, "zeros", host=0.5),
        # a later prompt chunk over a long context: the matrix-core-bound call
        _chunk("prefill-512-over-32k", "bf16", 32, 8, 128, 16, 512, 32768),
        # a whole prompt at once, causal
        _stream("prefill-first-2k", "bf16", 40, 8, 128, 16, 2048, 2048),
        # a later prompt chunk of a small model, sizes as they come
        _chunk("prefill-d64", "f16", 14, 2, 64, 64, 777, 2777),
        # a soft-capped, windowed prompt chunk at head dimension 256
        _stream("prefill-d256-window", "bf16", 16, 8, 256, 64, 512, 4700, "window", 4096, 50.0),
    ]


def _size(rng, lo, hi):
    """A size in [lo, hi], spread over its logarithm, usually odd."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, D):
    """(Hq, Hkv) of the architectures the patched forwards cover."""
    return rng.choice({64: [(32, 8), (14, 2), (12, 12), (16, 16)],
                       128: [(16, 8), (32, 8), (40, 8), (40, 40), (28, 4), (32, 32)],
                       256: [(16, 8), (8, 4), (8, 8)]}[D])


def draw(rng):
    kind = rng.choice(["pool", "pool", "step", "stream", "chunk", "chunk", "first", "host"])
    D = rng.choice([64, 128, 128, 128, 256])
    Hq, Hkv = _heads(rng, D)
    dt = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f16", "f32"])
    page = rng.choice([16, 16, 64])
    tok = 2 * Hkv * D * (4 if dt == "f32" else 2)        # K+V bytes of a token
    cap = rng.choice([0.0, 0.0, 0.0, 50.0])
    if kind == "pool":
        B = rng.choice([1, 1, 2, 4, 8, 13])
        hi = min(65536, LARGEST_KV_BYTES // (2 * tok * B))
        c = _pool("", dt, Hq, Hkv, D, page, [_size(rng, 17, hi) for _ in range(B)])
    elif kind == "step":
        B = rng.choice([1, 2, 4, 8])
        c = _step("", dt, Hq, Hkv, D, B, _size(rng, 100, min(32768, LARGEST_KV_BYTES // (2 * tok * B))))
    elif kind == "stream":
        T = _size(rng, 100, 16384)
        mask = rng.choice(["zeros", "window"])
        c = _stream("", dt, Hq, Hkv, D, page, 1, T, mask, max(1, T // 2), cap)
    elif kind == "host":
        T = _size(rng, 1000, 32768)
        c = _stream("", dt, Hq, Hkv, D, page, 1, T, "zeros", host=rng.choice([0.25, 0.5]))
    else:
        S = _size(rng, 17, 2048)
        room = LARGEST_PREFILL_FLOPS // (4 * S * Hq * D) // (8 if dt == "f32" else 1)
        T = S + (0 if kind == "first" else _size(rng, 16, 16384))
        T = max(S, min(T, room))
        if kind == "chunk" and T > S and cap == 0.0:
            c = _chunk("", dt, Hq, Hkv, D, page, S, T)
        elif kind == "chunk" and T > S:
            c = _stream("", dt, Hq, Hkv, D, page, S, T, "window", max(1, T // 2), cap)
        else:
            c = _stream("", dt, Hq, Hkv, D, page, S, S)
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, shape, dtype, std=1.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    return x.mul_(std) if std != 1.0 else x


def _lens(c):
    return [int(x) for x in c["lens"].split(",")]


def _inputs(c, seed):
    """The case's tensors from the seed: query, keys / values (a pool and its
    table, or one [1, Hkv, T, D] pair per sequence), mask."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    Hq, Hkv, D = c["Hq"], c["Hkv"], c["D"]
    x = {}
    if c["kind"] == "pool":
        lens, P = _lens(c), c["page"]
        pages = [-(-t // P) for t in lens]
        x["q"] = _randn(g, (len(lens), Hq, 1, D), dt, Q_STD)
        x["pool"] = _randn(g, (sum(pages), 2, Hkv, P, D), dt)
        slots = torch.randperm(sum(pages), generator=g, device="cuda").to(torch.int32)
        x["table"] = torch.zeros((len(lens), max(pages)), dtype=torch.int32, device="cuda")
        at = 0
        for b, n in enumerate(pages):
            x["table"][b, :n] = slots[at:at + n]
            at += n
        return x
    B, T, S = c.get("B", 1), c["T"], c.get("q_len", 1)
    x["q"] = _randn(g, (B, Hq, S, D), dt, Q_STD)
    x["kv"] = [(_randn(g, (1, Hkv, T, D), dt), _randn(g, (1, Hkv, T, D), dt)) for _ in range(B)]
    low = torch.finfo(dt).min
    if c["kind"] == "step":
        x["k_new"], x["v_new"] = _randn(g, (B, Hkv, 1, D), dt), _randn(g, (B, Hkv, 1, D), dt)
        # a left-padded batch: item b's first pads are masked for every step
        x["mask"] = torch.zeros((B, 1, 1, T + 1), dtype=dt, device="cuda")
        for b in range(B):
            x["mask"][b, :, :, :b * T // (4 * B)] = low
    elif c["kind"] == "chunk" or c["mask"] != "none":
        pos = torch.arange(T - S, T, device="cuda")[:, None]
        key = torch.arange(T, device="cuda")[None, :]
        seen = key <= pos
        if c.get("window"):
            seen &= key > pos - c["window"]
        x["mask"] = torch.zeros((S, T), dtype=dt, device="cuda").masked_fill_(~seen, low)[None, None]
    return x


def prepare(case, seed):
    c, x = case, _inputs(case, seed)
    Hkv, D, dt = c["Hkv"], c["D"], DTYPES[c["dtype"]]
    s = {"c": c, "q": x["q"], "mask": x.get("mask")}
    if c["kind"] == "pool":
        lens = _lens(c)
        pages = [-(-t // c["page"]) for t in lens]
        s["call"] = prepare_paged_decode(
            x["q"], x["pool"][:, 0], x["pool"][:, 1], x["table"],
            torch.tensor(lens, dtype=torch.int32, device="cuda"), max_pages=max(pages),
            total_pages=sum(pages), host_lens=lens)
        return s
    if c["kind"] == "step":
        s["k_new"], s["v_new"] = x["k_new"], x["v_new"]
        s["mgrs"] = []
        for k, v in x["kv"]:
            # two layers, of which the first is stepped: the step's token is
            # committed after the last layer, so a pass can be repeated
            m = KVCacheManager(KVAllocator(2, Hkv, D, page_size=16, dtype=dt), NO_EVICTION)
            if not m.build_contiguous(2, Hkv, D, c["T"] + 64, torch.device("cuda", 0), dt):
                raise MemoryError("out of memory: contiguous cache")
            m.prefill_contiguous(0, k, v)
            s["mgrs"].append(m)
        return s
    m = KVCacheManager(KVAllocator(1, Hkv, D, page_size=c["page"], dtype=dt), NO_EVICTION)
    k, v = x["kv"][0]
    m.append_prefill(0, k, v)
    if c.get("host"):
        m.evict_pages(int(c["host"] * c["T"] * 2 * Hkv * D * k.element_size()))
    s["mgr"] = m
    return s


def run(state):
    s, c = state, state["c"]
    scale = 1.0 / math.sqrt(c["D"])
    if c["kind"] == "pool":
        return s["call"].run()
    if c["kind"] == "step":
        return _decode_batched(s["mgrs"], s["q"], s["k_new"], s["v_new"], 0, scale,
                               attention_mask=s["mask"])
    if c["kind"] == "chunk":
        return _stream_prefill_batched([s["mgr"]], s["q"], 0, scale, attention_mask=s["mask"])
    return perform_streaming_attention(s["q"], s["mgr"].iterate_layer_pages(0), scale=scale,
                                       attention_mask=s["mask"], softcap=c["cap"] or None)


# ---- what a pass cannot do without -----------------------------------------------
def work(case):
    c = case
    es = 4 if c["dtype"] == "f32" else 2
    Hq, Hkv, D = c["Hq"], c["Hkv"], c["D"]
    if c["kind"] == "pool":
        lens, S = _lens(c), 1
        seen = keys = sum(lens)
        extra = 4 * sum(-(-t // c["page"]) for t in lens)
        B = len(lens)
    else:
        B, S, T = c.get("B", 1), c.get("q_len", 1), c["T"]
        T += 1 if c["kind"] == "step" else 0
        first = c["kind"] == "stream" and c["mask"] == "none" and S > 1
        past = 0 if first else T - S
        w = c.get("window") or T
        # (query, key) pairs visible under the mask, and keys seen by any query
        seen = B * sum(min(past + i + 1, w) for i in range(S))
        keys = B * min(T, w + S - 1)
        masked = c["kind"] == "step" or (c["kind"] == "stream" and c["mask"] != "none")
        extra = B * S * T * es if masked else 0
    return {"bytes": keys * 2 * Hkv * D * es + 2 * B * S * Hq * D * es + extra,
            "flops": 4 * seen * Hq * D}


# Largest relative errors, about four times what the calls show against the
# float64 result (bf16 1.6e-3 .. 2.3e-3, f16 2.1e-4, f32 3e-7 .. 6e-7): the
# output's own rounding dominates, in a prompt chunk the weights' joins it.
def tolerance(case):
    return {"bf16": {"rel": 8e-3, "max": 3e-2}, "f16": {"rel": 1e-3, "max": 4e-3},
            "f32": {"rel": 3e-6, "max": 3e-5}}[case["dtype"]]


# ---- the same results in 64 bits ----------------------------------------------------
def _attend64(q, K, V, scale, mask=None, cap=0.0, causal=False):
    """softmax(cap(q K^T scale) + mask) V in float64: q [Hq, S, D], K and V
    [Hkv, T, D], mask [S, T]; causal: top-left.  Laid out [Hq, S, D]."""
    Hq, S, _ = q.shape
    Hkv, T, _ = K.shape
    G = Hq // Hkv
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for h in range(Hkv):
        k, v = K[h].double(), V[h].double()
        for r in range(0, S, 256):
            x = torch.matmul(q[h * G:(h + 1) * G, r:r + 256].double(), k.t().contiguous()) * scale
            if cap:
                x = torch.tanh(x / cap) * cap
            if mask is not None:
                x = x + mask[r:r + 256].double()
            if causal:
                pos = torch.arange(r, min(r + 256, S), device=q.device)[:, None]
                x = x.masked_fill(torch.arange(T, device=q.device)[None, :] > pos, -math.inf)
            out[h * G:(h + 1) * G, r:r + 256] = torch.matmul(torch.softmax(x, -1), v)
    return out


def exact(case, seed):
    c, x = case, _inputs(case, seed)
    scale = 1.0 / math.sqrt(c["D"])
    outs = []
    if c["kind"] == "pool":
        for b, t in enumerate(_lens(c)):
            n = -(-t // c["page"])
            rows = x["pool"][x["table"][b, :n].long()]            # [n, 2, Hkv, P, D]
            kv = rows.permute(1, 2, 0, 3, 4).reshape(2, c["Hkv"], -1, c["D"])[:, :, :t]
            outs.append(_attend64(x["q"][b], kv[0], kv[1], scale))
    elif c["kind"] == "step":
        for b, (k, v) in enumerate(x["kv"]):
            k, v = torch.cat([k[0], x["k_new"][b]], 1), torch.cat([v[0], x["v_new"][b]], 1)
            outs.append(_attend64(x["q"][b], k, v, scale, x["mask"][b, 0]))
    else:
        k, v = x["kv"][0]
        m = x["mask"][0, 0] if x.get("mask") is not None else None
        outs.append(_attend64(x["q"][0], k[0], v[0], scale, m, c.get("cap", 0.0),
                              causal=m is None and c["q_len"] > 1))
    return torch.stack(outs)
