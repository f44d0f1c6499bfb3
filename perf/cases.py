"""The work that a user of this library has it do, as timed cases.

Each case is one pass through public entry points of gkv.py on inputs of the
gpt-oss shapes (64 query heads, 8 kv heads, head_dim 64, hidden 2880, a window
of 128 on every other layer; also the head counts that a tensor-parallel rank
of 2, 4 or 8 keeps). Kinds:

  decode   one decode layer of a batch: append of the new tokens, attention
  step     the layers of one decode step, each kind's plan kept by its first
           layer and reused by the others
  qkv      the QKV projection with the append in its epilogue
  prompt   one layer of whole prompts: append, then causal attention on the
           packed rows
  chunk    one layer of prompt chunks that continue a cached history
  exact    the fp32 path that repeats the CPU forward bit for bit

Lengths are spread evenly over [lo, hi] (the same for every seed, so that a
case's work is known) and dealt to the sequences in the seed's order; block
tables are random permutations of the pool's blocks.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = 64    # head dim
BT = 16   # tokens per paged block
HIDDEN = 2880
BF16, INT8, FP8 = 0, 1, 2  # cache formats (gkv.V_BF16, V_INT8, KV_FP8)

_gkv = None


def gkv():
    global _gkv
    if _gkv is None:
        path = os.path.join(ROOT, "optimize_inference_gpt-oss_amd", "gkv.py")
        spec = importlib.util.spec_from_file_location("gkv", path)
        _gkv = importlib.util.module_from_spec(spec)
        sys.modules["gkv"] = _gkv
        spec.loader.exec_module(_gkv)
        _gkv.lib()
    return _gkv


# ---- cases ------------------------------------------------------------------


def listed():
    return [
        # The headline workload: one full-attention decode layer of gpt-oss-20b
        # at a serving batch, bf16 cache.
        dict(name="decode_full_b512", kind="decode", B=512, lo=129, hi=2049, window=0, fmt=BF16,
             Hq=64, Hkv=8),
        # Its sliding-window layer: a ring of 128 slots, short streams.
        dict(name="decode_window_b512", kind="decode", B=512, lo=1, hi=4096, window=128, fmt=BF16,
             Hq=64, Hkv=8),
        # A handful of chats on one GPU: launches and round trips count.
        dict(name="decode_full_b4", kind="decode", B=4, lo=129, hi=2049, window=0, fmt=BF16,
             Hq=64, Hkv=8),
        # The e4m3 K/V cache at an odd batch.
        dict(name="decode_fp8_b333", kind="decode", B=333, lo=129, hi=2049, window=0, fmt=FP8,
             Hq=64, Hkv=8),
        # Four layers (window, full, window, full) of the decode step of a large
        # batch with long contexts, on the int8-V cache.
        dict(name="step_int8_b640", kind="step", B=640, lo=1025, hi=3073, window=128, fmt=INT8,
             Hq=64, Hkv=8, layers=4),
        # The projection of a small decode batch: the weights' bytes count.
        dict(name="qkv_rows24", kind="qkv", rows=24, prompts=0, fmt=BF16, Hq=64, Hkv=8),
        # ... of a serving batch.
        dict(name="qkv_rows512", kind="qkv", rows=512, prompts=0, fmt=BF16, Hq=64, Hkv=8),
        # ... of a batch of prompts: the matrix cores count.
        dict(name="qkv_rows9507", kind="qkv", rows=9507, prompts=32, fmt=BF16, Hq=64, Hkv=8),
        # A full layer of 64 prompts: append (cache and packed rows), attention.
        dict(name="prompt_full_b64", kind="prompt", B=64, lo=64, hi=512, window=0, fmt=BF16,
             Hq=64, Hkv=8),
        # The window layer of the same prompts.
        dict(name="prompt_window_b64", kind="prompt", B=64, lo=64, hi=512, window=128, fmt=BF16,
             Hq=64, Hkv=8),
        # Chunks of long prompts after a cached history, int8-V cache.
        dict(name="chunk_int8_b8", kind="chunk", B=8, lo=100, hi=700, hist=1536, window=0,
             fmt=INT8, Hq=64, Hkv=8),
        # The exact engine build's decode attention, fp32 caches.
        dict(name="exact_b32", kind="exact", B=32, lo=128, hi=2048, window=0, Hq=64, Hkv=8),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "step", "qkv", "qkv", "prompt", "prompt",
                       "chunk", "exact"])
    Hq, Hkv = rng.choice([(64, 8)] * 5 + [(32, 4), (16, 2), (8, 1)])
    window = rng.choice([0, 128])
    fmt = rng.choice([BF16, BF16, INT8, FP8])
    if kind == "decode":
        B = _log(rng, 1, 512)
        hi = _log(rng, 64, 4096 if B <= 256 else 2049)
        return dict(kind=kind, B=B, lo=rng.randint(1, hi), hi=hi, window=window, fmt=fmt, Hq=Hq,
                    Hkv=Hkv)
    if kind == "step":
        hi = _log(rng, 256, 3073)
        return dict(kind=kind, B=_log(rng, 4, 640), lo=rng.randint(1, hi // 3), hi=hi, window=128,
                    fmt=rng.choice([BF16, INT8, FP8]) if hi < 1500 else INT8, Hq=64, Hkv=8,
                    layers=rng.randint(2, 4))
    if kind == "qkv":
        rows = _log(rng, 1, 9507)
        return dict(kind=kind, rows=rows, prompts=0 if rows <= 1024 else rng.randint(1, 32),
                    fmt=fmt, Hq=Hq, Hkv=Hkv)
    if kind == "prompt":
        hi = _log(rng, 32, 900)
        return dict(kind=kind, B=_log(rng, 1, min(64, 19024 // hi)), lo=rng.randint(1, hi), hi=hi,
                    window=window, fmt=fmt, Hq=Hq, Hkv=Hkv)
    if kind == "chunk":
        hi = _log(rng, 32, 700)
        return dict(kind=kind, B=rng.randint(1, 8), lo=rng.randint(1, hi), hi=hi,
                    hist=16 * rng.randint(0, 96), window=window, fmt=fmt, Hq=Hq, Hkv=Hkv)
    hi = _log(rng, 64, 2048)
    return dict(kind=kind, B=rng.randint(1, 32), lo=rng.randint(1, hi), hi=hi, window=window, Hq=Hq,
                Hkv=Hkv)


def _spread(n, lo, hi):
    """n lengths spread evenly over [lo, hi]."""
    return [lo + int((i + 0.5) / n * (hi - lo + 1)) for i in range(n)]


def _prompt_lens(case):
    """Lengths of the prompts whose rows a qkv case projects."""
    q, r = divmod(case["rows"], case["prompts"])
    return [q + (1 if i < r else 0) for i in range(case["prompts"])]


# ---- inputs -----------------------------------------------------------------


class Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.np = np.random.default_rng(seed)

    def normal(self, shape, std, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=self.g)

    def lens(self, lens):
        return self.np.permutation(np.asarray(lens, np.int32)).astype(np.int32)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _cache(rnd, fmt, n_blocks, Hkv, std=0.5):
    """A pool's arrays {k, v, vs} with a history of N(0, std) values."""
    n = (n_blocks, Hkv, BT * D)
    if fmt == BF16:
        return dict(k=rnd.normal(n, std, torch.bfloat16), v=rnd.normal(n, std, torch.bfloat16),
                    vs=None)
    if fmt == INT8:
        v = rnd.normal(n, 45.0, torch.bfloat16).round_().clamp_(-127, 127).to(torch.int8)
        vs = torch.empty((n_blocks, Hkv, BT), device="cuda").uniform_(
            0.8 * std / 45, 1.2 * std / 45, generator=rnd.g)
        return dict(k=rnd.normal(n, std, torch.bfloat16), v=v, vs=vs)
    code = lambda: rnd.normal(n, 150.0, torch.bfloat16).clamp_(-448, 448).to(  # noqa: E731
        torch.float8_e4m3fn).view(torch.uint8)
    vs = torch.empty((n_blocks, Hkv, 2 * BT), device="cuda").uniform_(
        0.8 * std / 150, 1.2 * std / 150, generator=rnd.g)
    return dict(k=code(), v=code(), vs=vs)


def _table(rnd, per_seq, spare=5):
    """(block table [B, max blocks], blocks in the pool): a random permutation."""
    per_seq = np.asarray(per_seq)
    n_blocks = int(per_seq.sum()) + spare
    ids = rnd.np.permutation(n_blocks).astype(np.int32)
    tab = np.zeros((len(per_seq), max(1, int(per_seq.max()))), np.int32)
    at = 0
    for b, n in enumerate(per_seq):
        tab[b, :n] = ids[at:at + n]
        at += n
    return tab, n_blocks


def _layer(rnd, seq_lens, window, fmt, Hkv, tab=None):
    """One layer's cache, block table and view for sequences of these lengths."""
    if tab is None:
        per = np.full(len(seq_lens), window // BT) if window else (np.asarray(seq_lens) + 15) // BT
        tab = _table(rnd, per)
    t, n_blocks = tab
    c = _cache(rnd, fmt, n_blocks, Hkv)
    c["table"] = _dev(t)
    c["view"] = gkv().cache_view(c["k"], c["v"], c["table"], Hkv, ring=window, v_scale=c["vs"],
                                 v_format=fmt)
    c["window"] = window
    return c


def _written(c, exact=True):
    """The cache arrays of a layer as outputs: bits where they have to be the
    same, bf16 values where the rows come from 32-bit sums."""
    if c["k"].dtype == torch.bfloat16 and exact:
        k = c["k"].view(torch.int16)
        v = c["v"].view(torch.int16) if c["v"].dtype == torch.bfloat16 else c["v"]
    else:
        k, v = c["k"], c["v"]
    return {"k": k, "v": v} if c["vs"] is None else {"k": k, "v": v, "vs": c["vs"]}


def _width(case):
    return (case["Hq"] + 2 * case["Hkv"]) * D


def prepare(case, seed):
    G, rnd, kind = gkv(), Rand(seed), case["kind"]
    Hq, Hkv = case["Hq"], case["Hkv"]
    s = dict(case=case, err=torch.zeros(1, dtype=torch.int32, device="cuda"))
    s["sinks"] = rnd.normal((Hq,), 1.0)

    def tables(n):
        c, sn = G.rope_table(n)
        s["cos"], s["sin"] = _dev(c), _dev(sn)

    if kind in ("decode", "step"):
        B, window = case["B"], case["window"]
        lens = rnd.lens(_spread(B, case["lo"], case["hi"]))
        s["lens_h"], s["lens"], s["max_len"] = lens, _dev(lens), int(lens.max())
        tables(s["max_len"])
        n = case.get("layers", 1)
        windows = [window if kind == "decode" or i % 2 == 0 else 0 for i in range(n)]
        tabs = {w: _table(rnd, np.full(B, w // BT) if w else (lens + 15) // BT)
                for w in sorted(set(windows))}
        s["layers"] = [_layer(rnd, lens, w, case["fmt"], Hkv, tabs[w]) for w in windows]
        for c in s["layers"]:
            c["qkv"] = rnd.normal((B, _width(case)), 0.5)
            c["out"] = torch.empty((B, Hq * D), dtype=torch.bfloat16, device="cuda")
        s["ws"] = {w: torch.empty(G.workspace_bytes(B, Hkv, s["max_len"], w), dtype=torch.uint8,
                                  device="cuda") for w in set(windows)}
    elif kind == "qkv":
        rows = case["rows"]
        s["x"] = rnd.normal((rows, HIDDEN), 1.0, torch.bfloat16)
        s["w"] = rnd.normal((_width(case), HIDDEN), HIDDEN ** -0.5, torch.bfloat16)
        s["bias"] = rnd.normal((_width(case),), 0.1)
        s["qkv"] = torch.empty((rows, _width(case)), device="cuda")
        if case["prompts"]:
            pl = rnd.lens(_prompt_lens(case))
            s["pos"] = _dev(np.concatenate([np.arange(n) for n in pl]).astype(np.int32))
            s["seq"] = _dev(np.repeat(np.arange(len(pl)), pl).astype(np.int32))
            lens = pl
        else:  # a decode step: row b is the new token of sequence b
            s["pos"] = s["seq"] = None
            lens = rnd.lens(_spread(rows, 17, 64))
        s["lens_h"], s["lens"] = lens, _dev(lens)
        tables(int(lens.max()))
        s["layers"] = [_layer(rnd, lens, 0, case["fmt"], Hkv)]
    elif kind in ("prompt", "chunk"):
        B, window = case["B"], case["window"]
        pl = rnd.lens(_spread(B, case["lo"], case["hi"]))
        rows, hist = int(pl.sum()), case.get("hist", 0)
        s["pl"], s["rows"], s["max_len"] = pl, rows, int(pl.max())
        s["cu"] = _dev(np.concatenate([[0], np.cumsum(pl)]).astype(np.int32))
        s["pos"] = _dev(np.concatenate([hist + np.arange(n) for n in pl]).astype(np.int32))
        s["seq"] = _dev(np.repeat(np.arange(B), pl).astype(np.int32))
        s["start"] = _dev(np.full(B, hist, np.int32))
        s["lens"] = _dev((pl + hist).astype(np.int32))
        tables(hist + s["max_len"])
        c = _layer(rnd, pl + hist, window, case["fmt"], Hkv)
        s["layers"] = [c]
        c["qkv"] = rnd.normal((rows, _width(case)), 0.5)
        c["out"] = torch.empty((rows, Hq * D), dtype=torch.bfloat16, device="cuda")
        s["kp"] = torch.empty((rows, Hkv * D), dtype=torch.bfloat16, device="cuda")
        s["vp"] = torch.empty((rows, Hkv * D), dtype=torch.bfloat16, device="cuda")
        if kind == "chunk" and window:
            # a ring is attended before its chunk is appended, so the packed
            # rows come without the cache write
            G.kv_append(c["qkv"], Hq, s["cos"], s["sin"], s["pos"],
                        G.CacheView(n_kv_heads=Hkv), row_seq=s["seq"], k_pack=s["kp"],
                        v_pack=s["vp"])
    else:
        B, window = case["B"], case["window"]
        lens = rnd.lens(_spread(B, case["lo"], case["hi"]))
        s["lens_h"], s["max_len"] = lens, int(lens.max())
        slots = max(window, 1) if window else s["max_len"]
        s["pos"] = _dev((lens - 1).astype(np.int32))
        s["qkv"] = rnd.normal((B, _width(case)), 0.5)
        s["kc"] = rnd.normal((B, slots, Hkv * D), 0.5)
        s["vc"] = rnd.normal((B, slots, Hkv * D), 0.5)
        s["out"] = torch.empty((B, Hq * D), device="cuda")
    return s


# ---- one pass ---------------------------------------------------------------


def run(s):
    G, case = gkv(), s["case"]
    kind, Hq, Hkv = case["kind"], case["Hq"], case["Hkv"]
    if kind == "decode":
        c = s["layers"][0]
        G.decode_layer(c["qkv"], s["lens"], s["max_len"], c["view"], s["sinks"], c["out"],
                       s["cos"], s["sin"], window=c["window"], workspace=s["ws"][c["window"]],
                       dev_err=s["err"])
        return {"out": c["out"], "cache": _written(c)}
    if kind == "step":
        kept, outs = set(), []
        for c in s["layers"]:
            w = c["window"]
            G.decode_layer_planned(c["qkv"], s["lens"], s["max_len"], c["view"], s["sinks"],
                                   c["out"], s["cos"], s["sin"],
                                   G.PLAN_REUSE if w in kept else G.PLAN_KEEP, window=w,
                                   workspace=s["ws"][w], dev_err=s["err"])
            kept.add(w)
            outs.append({"out": c["out"], "cache": _written(c)})
        return outs
    if kind == "qkv":
        c = s["layers"][0]
        G.qkv_append(s["x"], s["w"], s["bias"], Hq, s["cos"], s["sin"], c["view"],
                     row_pos=s["pos"], row_seq=s["seq"], seq_lens=s["lens"], qkv_out=s["qkv"],
                     dev_err=s["err"])
        return {"qkv": s["qkv"], "cache": _written(c, exact=False)}
    if kind == "exact":
        w = case["window"]
        G.kv_write_exact(s["qkv"], Hq * D, (Hq + Hkv) * D, s["kc"], s["vc"], Hkv * D,
                         positions=s["pos"], window=w, dev_err=s["err"])
        G.attention_exact(s["qkv"], Hq, Hkv, s["kc"], s["vc"], s["sinks"], s["out"],
                          positions=s["pos"], max_pos=s["max_len"] - 1, window=w,
                          dev_err=s["err"])
        return {"out": s["out"], "kc": s["kc"], "vc": s["vc"]}
    c = s["layers"][0]
    w = c["window"]
    if kind == "chunk" and w:
        # the ring still holds the history: attend on the packed rows
        G.prefill_paged(s["cu"], s["max_len"], c["qkv"], c["view"], s["sinks"], c["out"],
                        start_pos=s["start"], k=s["kp"], v=s["vp"], window=w, cos_tab=s["cos"],
                        sin_tab=s["sin"], dev_err=s["err"])
        return {"out": c["out"]}
    G.kv_append(c["qkv"], Hq, s["cos"], s["sin"], s["pos"], c["view"], row_seq=s["seq"],
                seq_lens=s["lens"], k_pack=s["kp"], v_pack=s["vp"], dev_err=s["err"])
    if kind == "prompt":
        G.prefill_attention(s["cu"], s["max_len"], c["qkv"], s["kp"], s["vp"], s["sinks"],
                            c["out"], Hkv, window=w, cos_tab=s["cos"], sin_tab=s["sin"])
    else:
        G.prefill_paged(s["cu"], s["max_len"], c["qkv"], c["view"], s["sinks"], c["out"],
                        start_pos=s["start"], k=s["kp"], v=s["vp"], window=w, cos_tab=s["cos"],
                        sin_tab=s["sin"], dev_err=s["err"])
    return {"out": c["out"], "cache": _written(c), "kp": s["kp"].view(torch.int16),
            "vp": s["vp"].view(torch.int16)}


# ---- what a pass cannot do without ------------------------------------------


def _token_bytes(fmt, Hkv):
    """Cache bytes of one token: K and V of every kv head, with its scales."""
    return Hkv * {BF16: 256, INT8: 128 + 64 + 4, FP8: 128 + 8}[fmt]


def work(case):
    kind, Hq, Hkv = case["kind"], case["Hq"], case["Hkv"]
    width = (Hq + 2 * Hkv) * D
    if kind in ("decode", "step"):
        by = fl = 0
        lens = _spread(case["B"], case["lo"], case["hi"])
        for i in range(case.get("layers", 1)):
            w = case["window"] if kind == "decode" or i % 2 == 0 else 0
            n = sum(min(x, w) if w else x for x in lens)
            by += (n + case["B"]) * _token_bytes(case["fmt"], Hkv)  # read, and the new written
            by += case["B"] * (4 * width + 2 * Hq * D)              # qkv rows in, outputs out
            fl += 4 * n * Hq * D
        return {"bytes": by, "flops": fl}
    if kind == "qkv":
        r = case["rows"]
        by = 2 * r * HIDDEN + 2 * width * HIDDEN + 4 * width + 4 * r * width
        return {"bytes": by + r * _token_bytes(case["fmt"], Hkv), "flops": 2 * r * width * HIDDEN}
    if kind == "exact":
        lens = _spread(case["B"], case["lo"], case["hi"])
        n = sum(min(x, case["window"]) if case["window"] else x for x in lens)
        return {"bytes": n * Hkv * D * 8 + case["B"] * (width + 2 * Hkv * D + Hq * D) * 4,
                "flops": 4 * n * Hq * D}
    pl, hist, w = _spread(case["B"], case["lo"], case["hi"]), case.get("hist", 0), case["window"]
    pairs = read = 0
    for n in pl:
        pairs += sum(min(hist + t + 1, w) if w else hist + t + 1 for t in range(n))
        read += min(hist, w - 1) if w else hist
    rows = sum(pl)
    by = rows * (4 * width + 2 * Hq * D) + read * _token_bytes(case["fmt"], Hkv)
    if kind == "chunk" and w:
        by += rows * 4 * Hkv * D                          # the packed rows read
    else:
        kept = sum(min(n, w) if w else n for n in pl)     # cache and packed rows written
        by += kept * _token_bytes(case["fmt"], Hkv) + rows * 4 * Hkv * D
    return {"bytes": by, "flops": 4 * pairs * Hq * D}


def tolerance(case):
    kind = case["kind"]
    if kind == "exact":
        return "exact"  # the path's contract: the CPU forward's bits
    if kind == "qkv":
        # 32-bit sums of 2880 products in another order (3e-7 off the exact
        # rows as measured); in the cache a few in ten thousand of them round
        # to the neighbouring bf16 value or code (at most 2^-7 of the value)
        return {"rel": 2e-4, "max": 0.01, "differ": 1e-3}
    # bf16 outputs (2^-9 each, 1.7e-3 off the exact ones as measured); every
    # stored K/V byte is bit-exact by contract
    return {"rel": 5e-3, "max": 0.03, "differ": 0.0}


# ---- the same in 64 bits ----------------------------------------------------


def _k_rows(c, blocks, fmt):
    """K of pool blocks, fp64 [n, 16 tokens, Hkv, 64] from the block layout."""
    k = c["k"][blocks]
    n, Hkv = k.shape[:2]
    if fmt == FP8:
        k = k.view(torch.float8_e4m3fn).double().view(n, Hkv, 4, BT, 2, 8)
        k = k.permute(0, 3, 1, 4, 2, 5).reshape(n, BT, Hkv, D)
        return k * c["vs"][blocks][:, :, :BT].double().permute(0, 2, 1)[..., None]
    return k.double().view(n, Hkv, 2, 4, BT, 8).permute(0, 4, 1, 2, 3, 5).reshape(n, BT, Hkv, D)


def _v_rows(c, blocks, fmt):
    v = c["v"][blocks]
    n, Hkv = v.shape[:2]
    if fmt == BF16:
        v = v.double().view(n, Hkv, 2, 4, 16, 2, 4)
        return v.permute(0, 3, 6, 1, 2, 5, 4).reshape(n, BT, Hkv, D)
    v = (v.double() if fmt == INT8 else v.view(torch.float8_e4m3fn).double()).view(
        n, Hkv, 16, 4, 4, 4)
    v = v.permute(0, 3, 5, 1, 4, 2).reshape(n, BT, Hkv, D)
    vs = c["vs"][blocks] if fmt == INT8 else c["vs"][blocks][:, :, BT:]
    return v * vs.double().permute(0, 2, 1)[..., None]


def _rotate(x, cos, sin):
    """RoPE of [rows, heads, 64] fp64 at per-row angles [rows, 32]."""
    a, b = x[..., :32], x[..., 32:]
    c, s = cos.double()[:, None], sin.double()[:, None]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _stored(k, v, fmt):
    """New fp64 K and V rows [.., Hkv, 64] as the cache stands for them."""
    if fmt == FP8:
        def q(x):
            sc = x.abs().amax(-1, keepdim=True) / 448
            sc = torch.where(sc > 0, sc, torch.ones_like(sc))
            return (x / sc).clamp(-448, 448).float().to(torch.float8_e4m3fn).double() * sc
        return q(k), q(v)
    k = k.float().bfloat16().double()
    if fmt == INT8:
        sc = v.abs().amax(-1, keepdim=True) / 127
        sc = torch.where(sc > 0, sc, torch.ones_like(sc))
        return k, (v / sc).round().clamp(-127, 127) * sc
    return k, v.float().bfloat16().double()


def _attend(q, k, v, sinks, mask=None):
    """fp64 attention of q [rows, Hq, 64] over k, v [n, Hkv, 64], with sinks."""
    Hq, Hkv = q.shape[1], k.shape[1]
    rows = q.shape[0]
    g = Hq // Hkv
    qg = q.permute(1, 0, 2).reshape(Hkv, g * rows, D)
    sc = (qg @ k.permute(1, 2, 0).contiguous()).view(Hq, rows, -1) / 8.0
    if mask is not None:
        sc = sc.masked_fill(~mask, -math.inf)
    sk = sinks.double().view(Hq, 1, 1).expand(Hq, rows, 1)
    p = torch.softmax(torch.cat([sc, sk], -1), -1)[..., :-1]
    o = p.reshape(Hkv, g * rows, -1) @ v.permute(1, 0, 2).contiguous()
    return o.view(Hq, rows, D).permute(1, 0, 2).reshape(rows, Hq * D)


def _nothing(c):
    return {k: None for k in _written(c)}


def exact(case, seed):
    s = prepare(case, seed)
    kind, Hq, Hkv = case["kind"], case["Hq"], case["Hkv"]
    if kind in ("decode", "step"):
        if kind == "step" and case["B"] * case["hi"] * case["layers"] > 2e6:
            return None  # gathered in 64 bits it takes too long
        res = []
        for c in s["layers"]:
            x = c["qkv"].double().view(-1, Hq + 2 * Hkv, D)
            at = (s["lens"] - 1).long()
            rot = _rotate(x[:, :Hq + Hkv], s["cos"][at], s["sin"][at])
            kn, vn = _stored(rot[:, Hq:], x[:, Hq + Hkv:], case["fmt"])
            out = torch.empty((case["B"], Hq * D), dtype=torch.float64, device="cuda")
            for b, L in enumerate(s["lens_h"].tolist()):
                n = min(L, c["window"]) if c["window"] else L
                slot = (L - 1) % c["window"] if c["window"] else L - 1
                blocks = c["table"][b, :(n + 15) // BT].long()
                k = _k_rows(c, blocks, case["fmt"]).reshape(-1, Hkv, D)[:n]
                v = _v_rows(c, blocks, case["fmt"]).reshape(-1, Hkv, D)[:n]
                k[slot], v[slot] = kn[b], vn[b]
                out[b] = _attend(rot[b:b + 1, :Hq], k, v, s["sinks"])[0]
            res.append({"out": out, "cache": _nothing(c)})
        return res if kind == "step" else res[0]
    if kind == "qkv":
        out = s["x"].double() @ s["w"].double().t() + s["bias"].double()
        return {"qkv": out, "cache": _nothing(s["layers"][0])}
    if kind == "exact":
        x = s["qkv"].double().view(-1, Hq + 2 * Hkv, D)
        out = torch.empty((case["B"], Hq * D), dtype=torch.float64, device="cuda")
        for b, L in enumerate(s["lens_h"].tolist()):
            w = case["window"]
            n = min(L, w) if w else L
            slot = (L - 1) % w if w else L - 1
            k = s["kc"][b, :n].double().view(n, Hkv, D)
            v = s["vc"][b, :n].double().view(n, Hkv, D)
            k[slot], v[slot] = x[b, Hq:Hq + Hkv], x[b, Hq + Hkv:]
            out[b] = _attend(x[b:b + 1, :Hq], k, v, s["sinks"])[0]
        return {"out": out, "kc": None, "vc": None}
    c, hist, w = s["layers"][0], case.get("hist", 0), case["window"]
    x = c["qkv"].double().view(-1, Hq + 2 * Hkv, D)
    at = s["pos"].long()
    rot = _rotate(x[:, :Hq + Hkv], s["cos"][at], s["sin"][at])
    kn = rot[:, Hq:].float().bfloat16().double()  # the chunk's keys: packed bf16 rows
    vn = x[:, Hq + Hkv:].float().bfloat16().double()
    out = torch.empty((s["rows"], Hq * D), dtype=torch.float64, device="cuda")
    row = 0
    for b, n in enumerate(s["pl"].tolist()):
        k, v, k0 = kn[row:row + n], vn[row:row + n], hist
        if hist:
            k0 = max(0, hist - w) if w else 0
            slots = torch.arange(k0, hist, device="cuda")
            slots = slots % w if w else slots
            blocks = c["table"][b].long()
            kh = _k_rows(c, blocks, case["fmt"]).reshape(-1, Hkv, D)[slots]
            vh = _v_rows(c, blocks, case["fmt"]).reshape(-1, Hkv, D)[slots]
            k, v = torch.cat([kh, k]), torch.cat([vh, v])
        qp = hist + torch.arange(n, device="cuda")[:, None]
        kp = k0 + torch.arange(k.shape[0], device="cuda")[None]
        mask = (kp <= qp) & (kp > qp - w if w else kp >= 0)
        out[row:row + n] = _attend(rot[row:row + n, :Hq], k, v, s["sinks"], mask)
        row += n
    if kind == "chunk" and w:
        return {"out": out}
    return {"out": out, "cache": _nothing(c), "kp": None, "vp": None}
