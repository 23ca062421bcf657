"""Submission-module entry points, same names and contract as the reference
(kernels/v7_blockptr_warpspec.py:15-24, 201-252):

    VARIANT_MANIFEST
    setup(suite_specs, device, variants)
    block_sparse_attn_fwd(q, k, v, row_ptr, col_idx, seq_lens) -> (O, LSE)

plus block_sparse_attn_fwd_generic (the order-free CSR walk of kernels/v1_baseline.py:331-406)
and block_sparse_attn_fwd_window (analytic window rows, kernels/v1_baseline.py:141-322).

Differences from the reference, all deliberate:
  * fp16 q/k/v/O is the primary dtype; bf16 is also accepted (O in bf16, P·V in fp16 as in
    kernels/v7_blockptr_warpspec.py:107).
  * The launch goes through the C ABI of libusagi_bsa.so (compiled ahead of time for gfx950)
    instead of a Triton JIT launch.
  * The first call with a given pair of CSR tensors checks every row on the GPU, ahead of the
    forward kernel, and waits for the result while that one runs (CSR tensors on the host, and a
    CSR that the GPU check rejects, are checked on the host). block_sparse_attn_fwd raises
    ValueError on a row that is empty, repeats a block, lists a block outside [0, qb) before its
    last entry, or does not end with its diagonal (the reference's walk,
    kernels/v7_blockptr_warpspec.py:83-111, would silently attend future tokens or count a block
    twice there; the entries before the diagonal
    may come in any order; rows of query blocks at or past seq_len, which the walk never reads
    (v7:63-67), may hold anything). The same call plans the work order of more than 256 query
    blocks. Later calls with the same tensor objects, unmodified, reuse that (the reference memoises converted metadata on
    data_ptr() alone, kernels/v7_blockptr_warpspec.py:167-176; here the key also holds the
    shapes, dtypes, torch's in-place version counters and the tensor objects themselves, and,
    for a CSR that is only valid before seq_len, the seq_lens it was checked with). A CSR
    changed outside torch (e.g. through a NumPy view of its memory), or an inference-mode CSR
    changed in place (inference tensors have no version counter), needs clear_csr_cache().
    USAGI_BSA_VALIDATE=0 (read at import) skips the check and with it the synchronisation: the
    first call runs the CSR walk in the built-in order while a copy of the CSR goes to pinned
    host memory behind it, and a later call, finding that copy done, plans the work order and
    looks for a window pattern (like the reference, a malformed CSR then goes unreported).
  * A CSR whose rows are exactly the analytic rows of a window or window + global-prefix
    pattern (found by that same first-call check) runs the analytic-row kernel, which reads no
    CSR and gives the same bits; USAGI_BSA_ROUTE_WINDOW=0 (read at import) turns that off.
  * Like the reference, `setup` returns None without doing anything for a non-GPU device or
    no specs (kernels/v7_blockptr_warpspec.py:202-203); on a GPU it loads the ahead-of-time
    library first, so a missing build fails at setup time. The entry points reject CPU tensors
    (there is no CPU path).
"""

from __future__ import annotations

import contextlib
import math
import os
import weakref
from collections import OrderedDict

import torch

from . import _native

BLOCK_SIZE = 128
HEAD_DIM = 128

VARIANT_MANIFEST = [{"name": "default"}]

VALIDATE_CSR = os.environ.get("USAGI_BSA_VALIDATE", "1") not in ("", "0")
# A CSR whose rows are exactly an analytic window / window + global-prefix pattern runs the
# analytic-row kernel (no CSR reads, same result bit for bit); USAGI_BSA_ROUTE_WINDOW=0 (read
# at import) keeps every call on the CSR walk.
ROUTE_WINDOW = os.environ.get("USAGI_BSA_ROUTE_WINDOW", "1") not in ("", "0")

_DTYPE_CODES = {torch.float16: _native.FP16, torch.bfloat16: _native.BF16}

_CSR_CACHE_SIZE = 64

# Handle of the current stream of a device (by index), as torch.cuda.current_stream().cuda_stream; torch's
# own short cut to it (no Stream object: 0.05 us a call instead of 2.1) where it is there.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream",
                      lambda index: torch.cuda.current_stream(index).cuda_stream)

_NOTHING = contextlib.nullcontext()

# Query blocks up to which no work plan is made. All workgroups then run at once, but for the kernel with two
# per query block at 129 .. 256 query blocks (long growing rows), whose second half waits for a CU: there a
# plan can help (one full causal head of 8, T 4096: 35 us against 46) or hurt as much (two full causal heads,
# T 16384: 239 against 157), and mostly does neither (heads of mixed patterns, T 4096: 45.7 against 45.6).
_PLAN_ITEMS = 256


class _CsrEntry:
    """What the first call learnt about one (row_ptr, col_idx) pair: the tensors it was made
    for (weak references), the device copy of its work plan (None: built-in order) and the
    stream that copy was made on, the analytic (window, n_global) pattern the rows spell out
    (None: not one), and, when the rows are only valid before seq_len, the seq_lens they were
    checked with (seq_key; None: every row is valid)."""

    __slots__ = ("row_ptr", "col_idx", "sched", "n_slots", "stream", "window", "seq_key",
                 "seq_ref", "pending", "sched_ready", "unchecked", "entries")

    def __init__(self, row_ptr, col_idx, sched, n_slots, stream, window, seq_key, seq_ref):
        self.row_ptr = weakref.ref(row_ptr)
        self.col_idx = weakref.ref(col_idx)
        self.sched = sched
        self.n_slots = n_slots
        self.stream = stream
        self.window = window
        self.seq_key = seq_key
        self.seq_ref = seq_ref
        # Unchecked CSRs (USAGI_BSA_VALIDATE=0): (event, pinned row_ptr, pinned col_idx, B, H,
        # nqb) of the host copy still in flight, or None.
        self.pending = None
        # Event after an asynchronous copy of the plan to the device (or None: the copy was
        # synchronous); a launch on another stream waits for it.
        self.sched_ready = None
        # Entries of the head that holds most of them, or -1 (not known): the width of the column list
        # may be far above.
        self.entries = -1
        # The key of an entry that is not in the cache yet (else None): the call that made it checks
        # the CSR on the GPU (_start_check, _finish_check) around its launch.
        self.unchecked = None

    def valid_before(self, seq_lens) -> None:
        """Rows past seq_len may hold anything: the entry stands for calls with these seq_lens."""
        self.seq_key, ref = _seq_key(seq_lens)
        self.seq_ref = None if ref is None else weakref.ref(ref)


_csr_cache: "OrderedDict[tuple, _CsrEntry]" = OrderedDict()


def clear_csr_cache() -> None:
    """Forget every checked and planned CSR (the next call with any CSR checks it again)."""
    _csr_cache.clear()


def _tensor_key(t: torch.Tensor) -> tuple:
    # Inference tensors have no version counter: an in-place change to one made in inference
    # mode is not seen (like a change made outside torch, it needs clear_csr_cache()).
    version = None if t.is_inference() else t._version
    return (t.device, t.data_ptr(), t.shape, t.stride(), t.dtype, version)


def _seq_key(seq_lens):
    """Cache key of a seq_lens argument and the tensor to hold a weak reference to (or None)."""
    if seq_lens is None:
        return None, None
    if isinstance(seq_lens, torch.Tensor):
        return ("tensor",) + _tensor_key(seq_lens), seq_lens
    return ("values", tuple(int(x) for x in seq_lens)), None


def window_pattern(rp, ci, nqb: int):
    """(window, n_global) when every (b, h) row of the host CSR (rp [BH, nqb+1], ci [BH,
    max_nnz]) is exactly the analytic row of that pattern: query block i attends blocks
    0 .. n_global-1 and max(0, i-window+1) .. i, deduplicated and ascending (the rows of the
    reference's _fwd_window / _fwd_window_global, kernels/v1_baseline.py:141-322); else None.
    The pattern is read off the last row (a run of consecutive blocks ending at the diagonal,
    after a prefix 0 .. g-1), then every row of every head is compared with it."""
    import numpy as np

    rp = np.asarray(rp).reshape(-1, nqb + 1)
    ci = np.asarray(ci).reshape(rp.shape[0], -1)
    last = nqb - 1
    rs, re = int(rp[0, last]), int(rp[0, nqb])
    if not (0 <= rs < re <= ci.shape[1]):
        return None
    row = ci[0, rs:re]
    n = len(row)
    if row[-1] != last:
        return None
    run = 1
    while run < n and row[n - 1 - run] == last - run:
        run += 1
    g = n - run
    if g and not np.array_equal(row[:g], np.arange(g)):
        return None
    window, n_global = run, g
    q = np.arange(nqb)
    lo = np.maximum(q - window + 1, 0)
    ng = np.minimum(n_global, lo)
    counts = ng + (q - lo + 1)
    exp_rp = np.concatenate(([0], np.cumsum(counts)))
    nnz = int(exp_rp[-1])
    if nnz > ci.shape[1] or not np.array_equal(rp, np.broadcast_to(exp_rp, rp.shape)):
        return None
    # Entry p of row i: p itself in the global prefix (p < ng[i]), else lo[i] + (p - ng[i]).
    row_of = np.repeat(q, counts)
    p = np.arange(nnz) - np.repeat(exp_rp[:-1], counts)
    ng_r = ng[row_of]
    exp_ci = np.where(p < ng_r, p, lo[row_of] + (p - ng_r))
    if not np.array_equal(ci[:, :nnz], np.broadcast_to(exp_ci, (ci.shape[0], nnz))):
        return None
    return window, n_global


def _csr_entry(row_ptr, col_idx, B, H, nqb, dev, generic: bool, seq_lens=None) -> _CsrEntry:
    key = (generic, dev, _tensor_key(row_ptr), _tensor_key(col_idx))
    e = _csr_cache.get(key)
    if e is not None and e.row_ptr() is row_ptr and e.col_idx() is col_idx:
        if e.seq_key is None or (_seq_key(seq_lens)[0] == e.seq_key and
                                 (e.seq_ref is None or e.seq_ref() is seq_lens)):
            _csr_cache.move_to_end(key)
            if e.pending is not None and e.pending[0].query():
                _finish_pending(e, dev, generic)
            return e
    max_nnz = col_idx.shape[-1] if col_idx.dim() else 0
    stream = torch.cuda.current_stream(dev) if dev.type == "cuda" else None
    if not VALIDATE_CSR and dev.type == "cuda":
        # No check, so nothing has to be known before this launch: it runs the CSR walk in the
        # built-in order while a copy of the CSR goes to pinned host memory behind it on the
        # stream; a later call finds the copy done (an event query, no synchronisation) and
        # plans the work order and looks for a window pattern then.
        rp_h = torch.empty((B, H, nqb + 1), dtype=torch.int32, pin_memory=True)
        ci_h = torch.empty((B, H, max_nnz), dtype=torch.int32, pin_memory=True)
        rp_h.copy_(_as_int32_device(row_ptr, dev, (B, H, nqb + 1)), non_blocking=True)
        ci_h.copy_(_as_int32_device(col_idx, dev, (B, H, max_nnz)), non_blocking=True)
        done = torch.cuda.Event()
        done.record(stream)
        e = _CsrEntry(row_ptr, col_idx, None, 0, stream, None, None, None)
        e.pending = (done, rp_h, ci_h, B, H, nqb)
    elif _on_gpu(row_ptr, col_idx, dev, nqb, max_nnz):
        e = _CsrEntry(row_ptr, col_idx, None, 0, stream, None, None, None)
        if not generic or B * H * nqb > _PLAN_ITEMS:
            e.unchecked = key
            return e
    else:
        e = _CsrEntry(row_ptr, col_idx, None, 0, stream, None, None, None)
        _check_on_host(e, row_ptr, col_idx, B, H, nqb, dev, generic, seq_lens)
    _remember(e, key)
    return e


def _remember(e: _CsrEntry, key: tuple) -> None:
    _csr_cache[key] = e
    while len(_csr_cache) > _CSR_CACHE_SIZE:
        _csr_cache.popitem(last=False)


def _on_gpu(row_ptr, col_idx, dev, nqb: int, max_nnz: int) -> bool:
    """Whether the CSR can be checked on the GPU: there already, with any rows, and not under stream
    capture (the result is waited for)."""
    return (dev.type == "cuda" and row_ptr.device == dev and col_idx.device == dev
            and max_nnz > 0 and row_ptr.numel() > 0
            and nqb <= _native.CHECK_MAX_BLOCKS and not torch.cuda.is_current_stream_capturing())


def _check_on_host(e: _CsrEntry, row_ptr, col_idx, B, H, nqb, dev, generic: bool, seq_lens) -> None:
    """Check, window pattern and plan over host copies of the CSR; raises ValueError on a row that
    the walk would misread."""
    max_nnz = col_idx.shape[-1] if col_idx.dim() else 0
    rp = row_ptr.detach().reshape(B, H, nqb + 1).to("cpu", torch.int32).contiguous().numpy()
    ci = col_idx.detach().reshape(B, H, max_nnz).to("cpu", torch.int32).contiguous().numpy()
    if not generic and VALIDATE_CSR:
        try:
            _native.check_csr_host(rp, ci, B, H, nqb, max_nnz)
        except ValueError:
            # Rows past seq_len are never read, so they may hold anything: check the rest.
            if seq_lens is None:
                raise
            sl = torch.as_tensor(seq_lens).detach().to("cpu", torch.int32).reshape(-1).numpy()
            _native.check_csr_host(rp, ci, B, H, nqb, max_nnz, seq_lens=sl)
            e.valid_before(seq_lens)
    _plan_entry(e, rp, ci, B, H, nqb, dev, generic)


def _start_check(result, rp, ci, sl, B, H, nqb, max_nnz, stream) -> tuple:
    """Launch the GPU check of int32 device tensors; the forward launch follows it on the stream.
    result: pinned memory that the caller keeps until the check has run."""
    n_flags = _native.check_csr_gpu(rp.data_ptr(), ci.data_ptr(), B, H, nqb, max_nnz,
                                    result.data_ptr(), result.numel(), stream,
                                    sl.data_ptr() if sl is not None else None)
    done = torch.cuda.Event()
    done.record()
    return done, result, n_flags


def _finish_check(e: _CsrEntry, check: tuple, row_ptr, col_idx, B, H, nqb, dev, generic: bool,
                  seq_lens) -> None:
    """Wait for the check (the forward kernel is queued behind it or running), keep what it found in
    the entry and the entry in the cache; a CSR that it rejects is looked at again on the host, which
    raises with the row's position."""
    import numpy as np

    done, result, n_flags = check
    done.synchronize()
    r = result.numpy()
    flags = int(np.bitwise_or.reduce(r[:n_flags]))
    key, e.unchecked = e.unchecked, None
    if flags & 1 and not generic:
        _check_on_host(e, row_ptr, col_idx, B, H, nqb, dev, generic, seq_lens)
    else:
        if flags & 4 and not generic:
            e.valid_before(seq_lens)
        rows = B * H * nqb
        e.entries = int(r[:n_flags].max()) >> _native.CHECK_FLAG_BITS
        if rows > _PLAN_ITEMS:
            rp = np.zeros((B * H, nqb + 1), dtype=np.int32)
            np.cumsum(r[n_flags + 2:n_flags + 2 + rows].reshape(B * H, nqb), axis=1, out=rp[:, 1:])
            _plan_rows(e, rp, B, H, nqb, dev, generic, pinned=True)
        if not generic and ROUTE_WINDOW and not flags & 2 and e.sched is None:
            e.window = (int(r[n_flags]), int(r[n_flags + 1]))
    _remember(e, key)


def _plan_rows(e: _CsrEntry, rp, B, H, nqb, dev, generic: bool, pinned=False) -> None:
    """Work plan of a host row_ptr, into the entry. With at most _PLAN_ITEMS query blocks every
    workgroup runs at once and the order does not matter."""
    if B * H * nqb <= _PLAN_ITEMS:
        return
    sched = _native.plan_host(rp, B, H, nqb, generic)
    if sched is None:
        return
    src = torch.from_numpy(sched)
    if pinned:  # copied behind the stream's queued work, no synchronisation; torch keeps the pinned
        src = src.pin_memory()  # memory from being reused until the copy has run
    e.sched = src.to(dev, non_blocking=pinned)
    e.n_slots = len(sched)
    e.stream = torch.cuda.current_stream(dev) if dev.type == "cuda" else None
    if pinned:
        e.sched_ready = torch.cuda.Event()
        e.sched_ready.record(e.stream)


def _plan_entry(e: _CsrEntry, rp, ci, B, H, nqb, dev, generic: bool, pinned=False) -> None:
    """Entries, work plan and window pattern of a host copy of the CSR, into the entry."""
    e.entries = max(int(rp.max(initial=0)), 0)
    _plan_rows(e, rp, B, H, nqb, dev, generic, pinned)
    if e.sched is None and not generic and ROUTE_WINDOW and ci.shape[-1]:
        e.window = window_pattern(rp, ci, nqb)


def _finish_pending(e: _CsrEntry, dev, generic: bool) -> None:
    _, rp_h, ci_h, B, H, nqb = e.pending
    e.pending = None
    _plan_entry(e, rp_h.numpy(), ci_h.numpy(), B, H, nqb, dev, generic, pinned=True)


def _as_int32_device(t: torch.Tensor, device: torch.device, shape: tuple) -> torch.Tensor:
    """t's values as contiguous int32 on the device (in `shape`'s order; its own shape where it
    already is that: only the memory is used)."""
    if (t.dtype == torch.int32 and t.device == device and t.is_contiguous()
            and t.numel() == math.prod(shape)):
        return t
    t = t.reshape(shape)
    if t.device != device or t.dtype != torch.int32 or not t.is_contiguous():
        t = t.to(device=device, dtype=torch.int32).contiguous()
    return t


def _on_device(dev: torch.device):
    """Context in which dev is the current device (nothing to switch where it already is)."""
    if dev.index == torch.cuda.current_device():
        return _NOTHING
    return torch.cuda.device(dev)


def _check_inputs(q, k, v):
    # What every good call passes first, in few attribute reads; anything else is named below.
    if isinstance(q, torch.Tensor) and isinstance(k, torch.Tensor) and isinstance(v, torch.Tensor):
        shape, dtype, dev = q.shape, q.dtype, q.device
        if (dev.type == "cuda" and dtype in _DTYPE_CODES and len(shape) == 4
                and k.shape == shape and v.shape == shape and k.dtype == dtype
                and v.dtype == dtype and k.device == dev and v.device == dev):
            B, H, T, D = shape
            if D == HEAD_DIM and T > 0 and T % BLOCK_SIZE == 0:
                return B, H, T, D
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor")
        if t.device.type != "cuda":
            raise ValueError(f"{name} must be on a ROCm GPU device, got {t.device}")
        if t.dtype not in _DTYPE_CODES:
            raise TypeError(f"{name} must be float16 or bfloat16, got {t.dtype}")
        if t.dim() != 4:
            raise ValueError(f"{name} must be [B, H, T, D], got shape {tuple(t.shape)}")
    if not (q.shape == k.shape == v.shape):
        raise ValueError(f"q/k/v shapes differ: {tuple(q.shape)} {tuple(k.shape)} {tuple(v.shape)}")
    if not (q.dtype == k.dtype == v.dtype):
        raise TypeError("q/k/v dtypes differ")
    if not (q.device == k.device == v.device):
        raise ValueError("q/k/v are on different devices")
    B, H, T, D = q.shape
    if D != HEAD_DIM:
        raise ValueError(f"head dim must be {HEAD_DIM}, got {D}")
    if T <= 0 or T % BLOCK_SIZE:
        raise ValueError(f"T must be a positive multiple of {BLOCK_SIZE}, got {T}")
    return B, H, T, D


def _run_csr(q, k, v, row_ptr, col_idx, seq_lens, generic: bool):
    B, H, T, D = _check_inputs(q, k, v)
    dev = q.device
    nqb = T // BLOCK_SIZE
    if not isinstance(row_ptr, torch.Tensor) or not isinstance(col_idx, torch.Tensor):
        raise TypeError("row_ptr and col_idx must be torch.Tensors")
    if row_ptr.numel() != B * H * (nqb + 1):
        raise ValueError(f"row_ptr must hold [B, H, T/128 + 1] = [{B}, {H}, {nqb + 1}] values, "
                         f"got shape {tuple(row_ptr.shape)}")
    max_nnz = col_idx.shape[-1] if col_idx.dim() else 0
    if col_idx.numel() != B * H * max_nnz:
        raise ValueError(f"col_idx must be [B, H, max_nnz], got shape {tuple(col_idx.shape)}")
    plan = _csr_entry(row_ptr, col_idx, B, H, nqb, dev, generic, seq_lens)
    q = q.contiguous()
    k = k.contiguous()
    v = v.contiguous()
    sl = None
    if seq_lens is not None:
        sl = _as_int32_device(torch.as_tensor(seq_lens), dev, (B,))
    out = torch.empty((B, H, T, D), device=dev, dtype=q.dtype)
    lse = torch.empty((B, H, T), device=dev, dtype=torch.float32)
    with _on_device(dev):
        stream = _raw_stream(dev.index)  # of torch's current stream; no Stream object per call

        def launch_window():
            _native.fwd_window(q.data_ptr(), k.data_ptr(), v.data_ptr(), plan.window[0],
                               plan.window[1], sl.data_ptr() if sl is not None else None,
                               out.data_ptr(), lse.data_ptr(), B, H, T, D,
                               _DTYPE_CODES[q.dtype], stream)

        if plan.window is not None:
            launch_window()
            return out, lse
        rp = _as_int32_device(row_ptr, dev, (B, H, nqb + 1))
        ci = _as_int32_device(col_idx, dev, (B, H, max_nnz))
        if plan.sched is not None and stream != plan.stream.cuda_stream:
            # The plan's memory belongs to the stream it was copied on; a launch on another
            # stream waits for an asynchronous copy to land and keeps the memory from being
            # reused while the kernel reads it.
            current = torch.cuda.current_stream(dev)
            if plan.sched_ready is not None:
                current.wait_event(plan.sched_ready)
            plan.sched.record_stream(current)

        def launch(entries):
            _native.fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), rp.data_ptr(),
                        ci.data_ptr() if max_nnz else None, sl.data_ptr() if sl is not None else None,
                        out.data_ptr(), lse.data_ptr(), B, H, T, D, max_nnz, _DTYPE_CODES[q.dtype],
                        plan.sched.data_ptr() if plan.sched is not None else None, plan.n_slots,
                        stream, generic=generic, entries=entries)

        if plan.unchecked is None:
            launch(plan.entries)
            return out, lse
        result = torch.empty(_native.check_cap(B * H * nqb), dtype=torch.int32, pin_memory=True)
        try:
            check = _start_check(result, rp, ci, sl, B, H, nqb, max_nnz, stream)
            launch(-1)
            _finish_check(plan, check, row_ptr, col_idx, B, H, nqb, dev, generic, seq_lens)
        except BaseException:
            # The check may be queued still, and torch does not know that it writes to the result:
            # the memory must not go back before it has run.
            torch.cuda.current_stream(dev).synchronize()
            raise
        if 0 <= plan.entries < max_nnz:
            # A column list wider than its rows need may have led to another kernel than the later
            # calls', whose results differ in the last bits: this call gives theirs.
            lens = sl is not None
            later = plan.entries if plan.window is not None else max_nnz
            if (_native.kernel_of(B, H, T, lens, max_nnz, generic)
                    != _native.kernel_of(B, H, T, lens, later, generic, plan.entries)):
                if plan.window is not None:
                    launch_window()
                else:
                    launch(plan.entries)
    return out, lse


def block_sparse_attn_fwd(q, k, v, row_ptr, col_idx, seq_lens):
    """Block-sparse causal attention forward (kernels/v7_blockptr_warpspec.py:251-252).

    q, k, v: [B, H, T, 128] fp16 (or bf16) on the GPU.
    row_ptr: [B, H, T/128 + 1] integer, offsets local to each (b, h) row of col_idx.
    col_idx: [B, H, max_nnz] integer; each row lists distinct key blocks below its query block,
        in any order, then the diagonal (the reference's rows are ascending, which qualifies).
    seq_lens: [B] integer (or None = all T).
    Returns (O [B, H, T, 128] in q.dtype, LSE [B, H, T] float32), as
    kernels/v7_blockptr_warpspec.py:191.
    """
    return _run_csr(q, k, v, row_ptr, col_idx, seq_lens, generic=False)


def block_sparse_attn_fwd_generic(q, k, v, row_ptr, col_idx, seq_lens):
    """The generic CSR walk of kernels/v1_baseline.py:331-406: every entry of a row in any
    order, no implicit diagonal (an entry equal to the query block is causally masked, an empty
    row gives O = 0 and LSE = -inf), keys at or past seq_len masked. Same tensors and returns
    as block_sparse_attn_fwd; rows are not checked (any content is defined)."""
    return _run_csr(q, k, v, row_ptr, col_idx, seq_lens, generic=True)


def block_sparse_attn_fwd_window(q, k, v, window, n_global=0, seq_lens=None):
    """Forward pass over an analytic pattern: query block i attends the global prefix
    0 .. n_global-1 and the window max(0, i-window+1) .. i (the rows of the reference's unused
    analytic kernels _fwd_window / _fwd_window_global, kernels/v1_baseline.py:141-322), with no
    CSR. Equal to block_sparse_attn_fwd on the CSR of that pattern; same tensors and returns.
    """
    B, H, T, D = _check_inputs(q, k, v)
    window, n_global = int(window), int(n_global)
    if window < 1 or n_global < 0:
        raise ValueError(f"need window >= 1 and n_global >= 0, got {window}, {n_global}")
    dev = q.device
    q = q.contiguous()
    k = k.contiguous()
    v = v.contiguous()
    sl = None
    if seq_lens is not None:
        sl = _as_int32_device(torch.as_tensor(seq_lens), dev, (B,))
    out = torch.empty((B, H, T, D), device=dev, dtype=q.dtype)
    lse = torch.empty((B, H, T), device=dev, dtype=torch.float32)
    with _on_device(dev):
        stream = _raw_stream(dev.index)
        _native.fwd_window(q.data_ptr(), k.data_ptr(), v.data_ptr(), window, n_global,
                           sl.data_ptr() if sl is not None else None, out.data_ptr(),
                           lse.data_ptr(), B, H, T, D, _DTYPE_CODES[q.dtype], stream)
    return out, lse


def setup(suite_specs, device, variants):
    """Load the ahead-of-time library and run one tiny launch per distinct T.

    Mirrors kernels/v7_blockptr_warpspec.py:201-247: None without doing anything for a non-GPU
    device or no specs (v7:202-203), else a diagonal-only CSR launch per spec, then a
    synchronise. Specs only need a `t_max` attribute.
    """
    if str(device) != "cuda" and not str(device).startswith("cuda:"):
        return None
    if not suite_specs:
        return None
    _native.load()
    dev = torch.device(device)
    seen = set()
    for spec in suite_specs:
        T = int(spec.t_max)
        if T in seen:
            continue
        seen.add(T)
        nqb = T // BLOCK_SIZE
        x = torch.zeros((1, 1, T, HEAD_DIM), device=dev, dtype=torch.float16)
        rp = torch.arange(nqb + 1, device=dev, dtype=torch.int32).view(1, 1, nqb + 1)
        ci = torch.arange(nqb, device=dev, dtype=torch.int32).view(1, 1, nqb)
        sl = torch.tensor([T], device=dev, dtype=torch.int32)
        block_sparse_attn_fwd(x, x, x, rp, ci, sl)
    torch.cuda.synchronize(dev)
    return None
