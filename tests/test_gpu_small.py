"""The kernels for few query blocks (bsa_ksplit.hip) at the sizes where their choice or their tiling
changes: 64 / 128 / 256 / 512 query blocks, counts that are no multiple of 8, rows of 1, 2, 3 and more
than 64 blocks, rows without their diagonal, and sequences cut inside and between the 32- and 64-row
parts of a query block, NaN and infinities past seq_len. Against the fp32 walk; atol = rtol = 2e-3, half a bf16 ulp more for bf16 O."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import c_ref
from tests._helpers import assert_close
from usagi_amd import (block_sparse_attn_fwd, block_sparse_attn_fwd_generic,
                       block_sparse_attn_fwd_window)
from usagi_amd import patterns as P

pytestmark = pytest.mark.gpu

DEV = "cuda"


def check(fn, rp, ci, q, k, v, sl=None):
    dsl = None if sl is None else torch.tensor(sl, dtype=torch.int32, device=DEV)
    o, lse = fn(q.to(DEV), k.to(DEV), v.to(DEV), torch.from_numpy(rp).to(DEV),
                torch.from_numpy(ci).to(DEV), dsl)
    torch.cuda.synchronize()
    oo, ol = c_ref.fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), rp, ci,
                       None if sl is None else np.asarray(sl, np.int32), round_p_fp16=False,
                       generic=fn is block_sparse_attn_fwd_generic)
    rtol = 2e-3 + (2.0 ** -9 if q.dtype == torch.bfloat16 else 0.0)
    assert_close(o.float().cpu().numpy(), oo, rtol=rtol)
    assert_close(lse.cpu().numpy(), ol, what="LSE")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T,w", [
    (1, 1, 128, 1), (1, 3, 384, 3), (1, 7, 1152, 9),      # n = 1, 9, 63: 32 query rows
    (1, 8, 1024, 8),                                      # n = 64
    (1, 5, 1664, 5), (1, 8, 2048, 16),                    # n = 65, 128: 64 query rows
    (1, 3, 5504, 8), (1, 16, 2048, 7),                    # n = 129, 256: 128 query rows
    (1, 3, 5504, 43),                                     # n = 129, full causal rows: 64
    (1, 10, 4096, 32), (1, 16, 4096, 32),                 # n = 320, 512, full causal rows: 128
])
def test_window_rows(B, H, T, w, dtype):
    rp, ci = P.sliding_csr(B, H, T, w)
    q, k, v = P.make_qkv(B, H, T, seed=B * H * w, dtype=dtype)
    print(f"case small window B{B} H{H} T{T} w{w} {dtype}", flush=True)
    check(block_sparse_attn_fwd, rp, ci, q, k, v)


@pytest.mark.parametrize("H", [1, 9, 17, 27])  # n = 10 .. 270 query blocks in two sequences
@pytest.mark.parametrize("cuts", [(640, 33), (31, 97), (609, 512), (0, 128)])
def test_ragged_generic_rows(H, cuts):
    """Rows of 0-9 entries in any order, with repeats, above the diagonal and without it."""
    T = 640
    rng = np.random.default_rng(H)

    def row(b, h, i):
        r = [int(x) for x in rng.integers(0, T // 128, size=int(rng.integers(0, 9)))]
        if rng.random() < 0.7:
            r.insert(int(rng.integers(0, len(r) + 1)), i)
        return r

    rp, ci = P.make_csr(2, H, T, row)
    q, k, v = P.make_qkv(2, H, T, seed=H)
    print(f"case small generic H{H} seq_lens={cuts}", flush=True)
    check(block_sparse_attn_fwd_generic, rp, ci, q, k, v, list(cuts))


@pytest.mark.parametrize("H,T", [(1, 16384), (2, 16384)])  # n = 128 and 256, rows of up to 90 blocks
def test_rows_longer_than_a_column_chunk(H, T):
    rng = np.random.default_rng(H)

    def row(b, h, i):
        n = min(i, int(rng.choice([0, 1, 2, 62, 63, 64, 65, 89])))
        return sorted(int(x) for x in rng.choice(i, size=n, replace=False)) + [i]

    rp, ci = P.make_csr(1, H, T, row)
    q, k, v = P.make_qkv(1, H, T, seed=3 + H)
    print(f"case small long rows H{H} T{T}", flush=True)
    check(block_sparse_attn_fwd, rp, ci, q, k, v, [T - 45])


@pytest.mark.parametrize("H", [2, 4, 8])  # n = 32, 64, 128 (32 and 64 rows), 200 by T below
@pytest.mark.parametrize("T", [2048, 3200])
def test_scores_that_outgrow_the_running_max(H, T):
    """Key block 0's scores far above the diagonal's: every key group has to move its row max."""
    rp, ci = P.global_csr(1, H, T, 1, 6)
    q, k, v = P.make_qkv(1, H, T, seed=H)
    k = k.clone()
    k[:, :, 37:128] *= 6.0
    print(f"case small growth H{H} T{T}", flush=True)
    check(block_sparse_attn_fwd, rp, ci, q, k, v)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H", [2, 8, 40])  # n = 32, 128 and 640: bsa_ksplit.hip and bsa_fwd_dma_kernel
def test_rows_past_seq_len_hold_anything(H, dtype):
    """q, k and v past seq_len are NaN: the rows before it (seq_len a multiple of 32, the keys of a
    P·V step) are those of clean inputs, the rows past it O = 0 and LSE = -inf."""
    B, T, sl = 2, 1024, [608, 96]
    rp, ci = P.sliding_csr(B, H, T, 3)
    q, k, v = P.make_qkv(B, H, T, seed=H, dtype=dtype)
    dirty = [x.clone() for x in (q, k, v)]
    for x in dirty:
        for b in range(B):
            x[b, :, sl[b]:] = float("nan")
    print(f"case dirty tail H{H} {dtype}", flush=True)
    o, lse = block_sparse_attn_fwd(*(x.to(DEV) for x in dirty), torch.from_numpy(rp).to(DEV),
                                   torch.from_numpy(ci).to(DEV),
                                   torch.tensor(sl, dtype=torch.int32, device=DEV))
    torch.cuda.synchronize()
    oo, ol = c_ref.fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), rp, ci,
                       np.asarray(sl, np.int32), round_p_fp16=False)
    rtol = 2e-3 + (2.0 ** -9 if dtype == torch.bfloat16 else 0.0)
    assert_close(o.float().cpu().numpy(), oo, rtol=rtol)
    assert_close(lse.cpu().numpy(), ol, what="LSE")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
# n = 32, 128, 256 and 640: 32, 64 and 128 query rows per workgroup, and bsa_fwd_dma_kernel
@pytest.mark.parametrize("H", [2, 8, 16, 40])
@pytest.mark.parametrize("entry", ["csr", "window", "generic"])
@pytest.mark.parametrize("sl", [(609, 33), (1, 895)])
def test_tail_inside_a_step_of_32_keys(sl, entry, H, dtype):
    """q, k and v past seq_len are NaN or infinite and seq_len lies inside the 32 keys of a P·V step:
    the rows before it are those of clean inputs. Generic rows list blocks that seq_len cuts above
    the diagonal too."""
    B, T, w = 2, 1024, 7
    nqb = T // 128
    if entry == "generic":
        rng = np.random.default_rng(H)
        rp, ci = P.make_csr(B, H, T, lambda b, h, i: [int(x) for x in rng.permutation(nqb)[:w]])
    else:
        rp, ci = P.sliding_csr(B, H, T, w)
    q, k, v = P.make_qkv(B, H, T, seed=H, dtype=dtype)
    dirty = [x.clone() for x in (q, k, v)]
    for x, bad in zip(dirty, (float("nan"), float("nan"), float("inf"))):
        for b in range(B):
            x[b, :, sl[b]:] = bad
            x[b, :, sl[b] + 1::2] = float("nan")
    dirty = [x.to(DEV) for x in dirty]
    drp, dci = torch.from_numpy(rp).to(DEV), torch.from_numpy(ci).to(DEV)
    dsl = torch.tensor(sl, dtype=torch.int32, device=DEV)
    print(f"case tail in a step {entry} H{H} {dtype} seq_lens={sl}", flush=True)
    if entry == "window":
        o, lse = block_sparse_attn_fwd_window(*dirty, w, 0, dsl)
    elif entry == "generic":
        o, lse = block_sparse_attn_fwd_generic(*dirty, drp, dci, dsl)
    else:  # not routed to the analytic rows: two entries of one row in the other order
        ci2 = ci.copy()
        ci2[0, 0, rp[0, 0, 4]:rp[0, 0, 4] + 2] = ci[0, 0, rp[0, 0, 4]:rp[0, 0, 4] + 2][::-1]
        o, lse = block_sparse_attn_fwd(*dirty, drp, torch.from_numpy(ci2).to(DEV), dsl)
    torch.cuda.synchronize()
    oo, ol = c_ref.fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), rp, ci,
                       np.asarray(sl, np.int32), round_p_fp16=False, generic=entry == "generic")
    rtol = 2e-3 + (2.0 ** -9 if dtype == torch.bfloat16 else 0.0)
    assert_close(o.float().cpu().numpy(), oo, rtol=rtol)
    assert_close(lse.cpu().numpy(), ol, what="LSE")
