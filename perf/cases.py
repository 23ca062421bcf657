"""Performance cases of the block-sparse causal attention forward.

Each case is one call of a public entry point (block_sparse_attn_fwd, block_sparse_attn_fwd_window
or block_sparse_attn_fwd_generic) on inputs resident on the GPU, over the range the package is used
for: T from one block to 32768, few and many heads, the scored families (sliding window, global
prefix, retrieval), short rows, full causal rows, mixed heads, fp16 and bf16, with and without
ragged seq_lens.

A case:
    entry    "default", "window" (no CSR) or "generic" (rows in any order, diagonal optional)
    B, H, T  batch, heads, tokens (a multiple of 128)
    dtype    "fp16" or "bf16"
    pattern  "rows": every query block attends the first `g` blocks, the last `w` blocks up to its
                     own and `r` more, drawn from the ones between (w >= T/128: full causal rows)
             "mixed": of 16 heads 6 are sliding (16), 5 global (8 + 8) and 5 retrieval (2 + 24)
             "random": every key block with probability `density`, in any order, above the
                     diagonal too, the diagonal present in most rows (generic walk only)
    lens     "none" (seq_lens=None), "first" (the first sequence full, the others cut) or "ragged"
             (every sequence cut)
    fresh    the CSR tensors are new ones in every call
"""

from __future__ import annotations

import math

import numpy as np
import torch

import usagi_amd

BLOCK = 128
D = 128
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
MAX_ITEMS = 2048        # query blocks of the largest listed calls
MAX_ACTIVE = 36000      # key blocks the largest listed call visits


def _case(name, entry, B, H, T, dtype, pattern="rows", w=0, g=0, r=0, density=0.0, lens="none",
          fresh=False):
    c = dict(entry=entry, B=B, H=H, T=T, dtype=dtype, pattern=pattern, w=w, g=g, r=r,
             density=density, lens=lens, fresh=fresh)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call: four heads over a short context (launch and host cost count).
        _case("sliding_1k", "default", 1, 4, 1024, "fp16", w=4),
        # A batch of short prompts of unequal length with full causal attention, an odd number of
        # blocks.
        _case("prompts_ragged", "default", 4, 8, 896, "bf16", w=7, lens="ragged"),
        # One sequence of a layer with few heads, analytic rows without a CSR.
        _case("window_2k", "window", 1, 8, 2048, "bf16", w=8, g=2),
        # Block lists in any order, some without their diagonal, over ragged sequences.
        _case("generic_ragged", "generic", 2, 6, 1920, "fp16", pattern="random", density=0.5,
              lens="ragged"),
        # Blocks chosen anew for every call (query-dependent retrieval).
        _case("retrieval_4k_fresh", "default", 1, 8, 4096, "fp16", w=2, r=14, fresh=True),
        # Dense causal prefill through the block-sparse entry point.
        _case("full_causal_4k", "default", 1, 16, 4096, "bf16", w=32),
        # Short rows: a 256-token window over a long context.
        _case("sliding_w2_8k", "default", 2, 16, 8192, "fp16", w=2),
        # The scored families at their scored size; the global one as the reference runs it (bf16,
        # the second sequence cut).
        _case("sliding_8k", "default", 2, 16, 8192, "fp16", w=8),
        _case("global_8k_lens", "default", 2, 16, 8192, "bf16", w=4, g=4, lens="first"),
        _case("retrieval_8k", "default", 2, 16, 8192, "fp16", w=2, r=14),
        # A layer whose heads use different patterns, so their rows differ in length.
        _case("mixed_16k", "default", 1, 16, 16384, "fp16", pattern="mixed"),
        # A long context on a shard with two heads, rows of up to 80 blocks.
        _case("long_32k", "default", 1, 2, 32768, "bf16", w=8, g=4, r=68),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        entry = rng.choice(["default", "default", "default", "window", "generic"])
        nqb = _log_int(rng, 1, 256)
        B = rng.choice([1, 1, 1, 2, 2, 3, 4])
        H = rng.choice([1, 2, 3, 4, 5, 6, 8, 12, 16, 16, 24, 32])
        if B * H * nqb > MAX_ITEMS:
            continue
        c = _case(None, entry, B, H, nqb * BLOCK, rng.choice(["fp16", "bf16"]),
                  lens=rng.choice(["none", "none", "first", "ragged"]),
                  fresh=entry == "default" and rng.random() < 0.15)
        if entry == "generic":
            c["pattern"] = "random"
            c["density"] = round(rng.uniform(0.05, 0.7), 2)
        else:
            kind = rng.choice(["sliding", "global", "retrieval", "full", "mixed"])
            if entry == "window" and kind in ("retrieval", "mixed"):
                kind = "global"
            if kind == "mixed":
                c["pattern"] = "mixed"
            elif kind == "full":
                c["w"] = nqb
            else:
                c["w"] = _log_int(rng, 1, 32)
                if kind == "global":
                    c["g"] = _log_int(rng, 1, 8)
                elif kind == "retrieval":
                    c["r"] = _log_int(rng, 2, 68)
        if int(_counts(c, 0).sum()) <= MAX_ACTIVE:
            return c


# ------------------------------------------------------------------------------ patterns


def _rows(nqb, heads, w, g, r, rs):
    """bool [heads, nqb, nqb]: the first g blocks, the last w, and r more from those between."""
    i = np.arange(nqb)[:, None]
    j = np.arange(nqb)[None, :]
    base = (j <= i) & ((j > i - w) | (j < g))
    m = np.broadcast_to(base, (heads, nqb, nqb)).copy()
    if r:
        free = (j <= i) & ~base
        key = np.where(free, rs.random_sample((heads, nqb, nqb)), 2.0)
        order = np.argsort(key, axis=-1)[..., :r]
        picked = np.zeros_like(m)
        np.put_along_axis(picked, order, True, axis=-1)
        m |= picked & free
    return m


def _mask(case, seed):
    """bool [B*H, nqb, nqb]: the key blocks each query block lists."""
    nqb, H = case["T"] // BLOCK, case["H"]
    bh = case["B"] * H
    rs = np.random.RandomState(seed % (1 << 31))
    if case["pattern"] == "mixed":
        m = np.empty((bh, nqb, nqb), dtype=bool)
        h = (np.arange(bh) % H) * 16 // H
        for sel, (w, g, r) in ((h <= 5, (16, 0, 0)), ((h > 5) & (h <= 10), (8, 8, 0)),
                               (h > 10, (2, 0, 24))):
            m[sel] = _rows(nqb, int(sel.sum()), w, g, r, rs)
        return m
    if case["pattern"] == "random":
        m = rs.random_sample((bh, nqb, nqb)) < case["density"]
        diag = np.arange(nqb)
        m[:, diag, diag] = rs.random_sample((bh, nqb)) < 0.9
        return m
    return _rows(nqb, bh, case["w"], case["g"], case["r"], rs)


def _lens(case):
    """Sequence lengths (the same for every seed: they set how much work the case is)."""
    B, T = case["B"], case["T"]
    if case["lens"] == "none":
        return [T] * B
    cut = [max(1, int(T * f)) for f in (0.611, 0.97, 0.34, 0.83)]
    if case["lens"] == "first":
        return [T if b == 0 else cut[(b - 1) % 4] for b in range(B)]
    return [cut[(b + 1) % 4] for b in range(B)]


def _counts(case, seed):
    return _mask(case, seed).sum(axis=-1)


def _csr(case, seed):
    """(row_ptr [B, H, nqb+1], col_idx [B, H, max_nnz]) int32; rows ascending, or in any order
    for the generic walk."""
    B, H, nqb = case["B"], case["H"], case["T"] // BLOCK
    m = _mask(case, seed)
    counts = m.sum(axis=-1)
    rp = np.zeros((B * H, nqb + 1), dtype=np.int32)
    rp[:, 1:] = np.cumsum(counts, axis=-1)
    ci = np.zeros((B * H, max(1, int(rp[:, -1].max()))), dtype=np.int32)
    bh, row, col = np.nonzero(m)
    if case["entry"] == "generic":
        rs = np.random.RandomState((seed + 1) % (1 << 31))
        order = np.lexsort((rs.random_sample(len(col)), row, bh))
        bh, row, col = bh[order], row[order], col[order]
    start = np.concatenate(([0], np.cumsum(rp[:, -1])[:-1]))
    ci[bh, np.arange(len(col)) - start[bh]] = col
    return rp.reshape(B, H, nqb + 1), ci.reshape(B, H, -1)


# ------------------------------------------------------------------------------ the calls


def _qkv(case, seed):
    """q, k, v ~ N(0, 1), as the benchmark's."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["B"], case["H"], case["T"], D)
    return [torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
            .to(DTYPES[case["dtype"]]) for _ in range(3)]


def prepare(case, seed):
    q, k, v = _qkv(case, seed)
    s = {"entry": case["entry"], "q": q, "k": k, "v": v, "w": case["w"], "g": case["g"],
         "fresh": case["fresh"], "sl": None}
    if case["entry"] != "window":
        rp, ci = _csr(case, seed)
        s["rp"] = torch.from_numpy(rp).cuda()
        s["ci"] = torch.from_numpy(ci).cuda()
    if case["lens"] != "none":
        s["sl"] = torch.tensor(_lens(case), dtype=torch.int32, device="cuda")
    return s


def run(s):
    if s["entry"] == "window":
        return usagi_amd.block_sparse_attn_fwd_window(s["q"], s["k"], s["v"], s["w"], s["g"], s["sl"])
    rp, ci = s["rp"], s["ci"]
    if s["fresh"]:  # what a block selector hands over: tensors that no earlier call has seen
        rp, ci = rp.clone(), ci.clone()
    fn = (usagi_amd.block_sparse_attn_fwd_generic if s["entry"] == "generic"
          else usagi_amd.block_sparse_attn_fwd)
    return fn(s["q"], s["k"], s["v"], rp, ci, s["sl"])


# ------------------------------------------------------------------------------ floors and checks


def work(case):
    """Visible (query, key) pairs x 4 x 128 operations; q, k, v and the CSR read once, O and LSE
    written once."""
    B, H, T = case["B"], case["H"], case["T"]
    nqb = T // BLOCK
    lens = np.repeat(np.array(_lens(case)), H)                      # [B*H]
    valid = np.clip(lens[:, None] - BLOCK * np.arange(nqb), 0, BLOCK)   # rows / keys of a block
    m = _mask(case, 0)
    diag = np.arange(nqb)
    on = m[:, diag, diag]
    m[:, diag, diag] = False
    pairs = float((valid * (m * valid[:, None, :]).sum(axis=-1)).sum())
    pairs += float((on * valid * (valid + 1) / 2).sum())
    tokens = float(lens.sum())
    csr = 0.0 if case["entry"] == "window" else 4.0 * (B * H * (nqb + 1) + m.sum() + on.sum())
    return {"bytes": 3 * tokens * D * 2 + B * H * T * (D * 2 + 4) + csr, "flops": 4.0 * D * pairs}


def tolerance(case):
    """O is rounded to its type and P to fp16: against 64 bits O is off by 2.6e-4 (fp16) and 1.6e-3
    (bf16) over these cases, LSE by less than 1e-5. `max` is larger because the first rows, which
    average few keys, hold values far above the whole output's root mean square."""
    return {"rel": 6e-3, "max": 1e-1} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 4e-2}


def exact(case, seed):
    """Dense masked attention in float64, slabs of query blocks at a time."""
    B, H, T = case["B"], case["H"], case["T"]
    nqb = T // BLOCK
    q, k, v = _qkv(case, seed)
    m = _mask(case, seed)
    lens = _lens(case)
    O = torch.zeros((B, H, T, D), dtype=torch.float64, device="cuda")
    L = torch.full((B, H, T), -math.inf, dtype=torch.float64, device="cuda")
    tri = torch.ones((BLOCK, BLOCK), dtype=torch.bool, device="cuda").tril()
    slab = 16
    for b in range(B):
        n = lens[b]
        for h in range(H):
            kd = k[b, h, :n].double()
            vd = v[b, h, :n].double()
            mh = torch.from_numpy(m[b * H + h]).cuda()
            for i0 in range(0, min(nqb, -(-n // BLOCK)), slab):
                rows = range(i0, min(nqb, i0 + slab))
                r0, r1 = i0 * BLOCK, min(n, (i0 + len(rows)) * BLOCK)
                allow = mh[i0:i0 + len(rows)].repeat_interleave(BLOCK, 0).repeat_interleave(BLOCK, 1)
                for x, i in enumerate(rows):
                    allow[x * BLOCK:(x + 1) * BLOCK, i * BLOCK:(i + 1) * BLOCK] &= tri
                s = q[b, h, r0:r1].double() @ kd.t() / math.sqrt(D)
                s.masked_fill_(~allow[:r1 - r0, :n], -math.inf)
                lse = torch.logsumexp(s, dim=-1)
                L[b, h, r0:r1] = lse
                p = torch.exp(s - torch.where(torch.isinf(lse), torch.zeros_like(lse), lse)[:, None])
                O[b, h, r0:r1] = p @ vd
    return O, L
