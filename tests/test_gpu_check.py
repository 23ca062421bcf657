"""The CSR check on the GPU against the host check, window_pattern and the CSR itself: valid rows,
rows broken in each way the host check names, window and near-window patterns, rows longer than a
wave, few and many rows per wave, rows past seq_len; the first call of the shim around it (padded lists,
rows that end at seq_len) and captured calls after it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests._helpers import assert_close
from oracle import c_ref
from usagi_amd import (_native, block_sparse_attn_fwd, block_sparse_attn_fwd_generic,
                       submission)
from usagi_amd import patterns as P

pytestmark = pytest.mark.gpu


def gpu_check(rp, ci):
    B, H, n1 = rp.shape
    rows = B * H * (n1 - 1)
    drp, dci = torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda()
    result = torch.empty(_native.check_cap(rows), dtype=torch.int32, pin_memory=True)
    n = _native.check_csr_gpu(drp.data_ptr(), dci.data_ptr(), B, H, n1 - 1, ci.shape[-1],
                              result.data_ptr(), result.numel(),
                              torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    r = result.numpy()
    flags = int(np.bitwise_or.reduce(r[:n]))
    window = None if flags & 2 else (int(r[n]), int(r[n + 1]))
    return bool(flags & 1), window, r[n + 2:n + 2 + rows].reshape(B, H, n1 - 1).copy()


def host_check(rp, ci):
    B, H, n1 = rp.shape
    try:
        _native.check_csr_host(rp, ci, B, H, n1 - 1, ci.shape[-1])
    except ValueError:
        return True
    return False


@pytest.mark.parametrize("B,H,T,w,g", [(1, 1, 128, 1, 0), (1, 3, 384, 2, 0), (2, 4, 1024, 3, 2),
                                       (1, 2, 12800, 70, 5), (1, 1, 8192, 100, 0), (3, 40, 2560, 4, 0),
                                       (1, 2, 1024, 2, 9)])
def test_window_patterns(B, H, T, w, g):
    rp, ci = P.global_csr(B, H, T, g, w) if g else P.sliding_csr(B, H, T, w)
    print(f"case check window B{B} H{H} T{T} w{w} g{g}", flush=True)
    bad, window, counts = gpu_check(rp, ci)
    assert not bad and window == submission.window_pattern(rp, ci, T // 128)
    assert np.array_equal(counts, np.diff(rp, axis=-1))
    # one entry changed in the last head: a valid row or not, never the pattern
    if T > 256:
        rp2, ci2 = rp.copy(), ci.copy()
        at = rp2[-1, -1, T // 128 - 1]
        ci2[-1, -1, at] = (ci2[-1, -1, at] + 1) % (T // 128)
        bad, window, _ = gpu_check(rp2, ci2)
        assert bad == host_check(rp2, ci2)
        assert window == submission.window_pattern(rp2, ci2, T // 128)


def broken(rp, ci, how, rng):
    b, h = rng.integers(0, rp.shape[0]), rng.integers(0, rp.shape[1])
    qb = int(rng.integers(2, rp.shape[2] - 1))
    rs, re = rp[b, h, qb], rp[b, h, qb + 1]
    if how == "not diagonal":
        ci[b, h, re - 1] = qb - 1
    elif how == "above":
        ci[b, h, rs] = qb
    elif how == "negative":
        ci[b, h, rs] = -3
    elif how == "twice":
        ci[b, h, re - 2] = ci[b, h, rs]
    elif how == "empty":
        rp[b, h, qb + 1] = rs
    elif how == "past the list":
        rp[b, h, -1] = ci.shape[-1] + 1
    elif how == "start":
        rp[b, h, 0] = 1


@pytest.mark.parametrize("how", ["none", "not diagonal", "above", "negative", "twice", "empty",
                                 "past the list", "start"])
@pytest.mark.parametrize("B,H,T", [(1, 2, 2048), (2, 3, 12800), (1, 64, 4096)])
def test_rows_against_the_host_check(B, H, T, how):
    nqb = T // 128
    rng = np.random.default_rng(nqb)

    def row(b, h, i):  # entries before the diagonal in any order, at least two where there are two
        n = min(i, int(rng.integers(2, 80)))
        return [int(x) for x in rng.permutation(i)[:n]] + [i]

    rp, ci = P.make_csr(B, H, T, row)
    if how != "none":
        broken(rp, ci, how, rng)
    print(f"case check rows B{B} H{H} T{T} {how}", flush=True)
    bad, window, counts = gpu_check(rp, ci)
    assert bad == host_check(rp, ci) == (how != "none")
    assert window == submission.window_pattern(rp, ci, nqb)
    assert np.array_equal(counts, np.maximum(np.diff(rp, axis=-1), 0))


@pytest.mark.parametrize("pad", [0, 700])
def test_first_call_equals_later_calls(pad):
    """The first call launches before the check's result is known; a window-shaped CSR (also one
    with a padded column list) gives the same bits in every call, and a broken one raises."""
    submission.clear_csr_cache()
    B, H, T = 1, 8, 4096
    rp, ci = P.sliding_csr(B, H, T, 4)
    ci = np.concatenate([ci, np.zeros((B, H, pad), np.int32)], axis=-1)
    q, k, v = P.make_qkv(B, H, T, seed=5)
    dev = [x.cuda() for x in (q, k, v)] + [torch.from_numpy(x).cuda() for x in (rp, ci)]
    print(f"case first call pad {pad}", flush=True)
    o1, l1 = block_sparse_attn_fwd(*dev, None)
    (entry,) = submission._csr_cache.values()
    assert entry.window == (4, 0)
    o2, l2 = block_sparse_attn_fwd(*dev, None)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(l1, l2)
    oo, _ = c_ref.fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), rp, ci, None,
                      round_p_fp16=False)
    assert_close(o1.float().cpu().numpy(), oo)
    dev[4][0, 3, 9] = 31
    with pytest.raises(ValueError, match="h=3"):
        block_sparse_attn_fwd(*dev, None)
    submission.clear_csr_cache()


@pytest.mark.parametrize("H,T,width", [(8, 4096, 528), (16, 4096, 528), (4, 8192, 2080), (3, 5504, 946),
                                       (8, 8320, 4225)])
def test_padded_list_equals_the_list_of_its_rows(H, T, width, monkeypatch):
    """A column list allocated for full causal rows or more: every call, the first one too, gives the
    bits of the list that just holds the rows (so runs the same kernel), and only a first call whose
    width led to another kernel launches twice."""
    submission.clear_csr_cache()
    rp, ci = P.retrieval_csr(1, H, T, 6, 3)
    wide = np.concatenate([ci, np.zeros((1, H, width - ci.shape[-1]), np.int32)], axis=-1)
    qkv = [x.cuda() for x in P.make_qkv(1, H, T, seed=H)]
    drp, dci, dwide = (torch.from_numpy(x).cuda() for x in (rp, ci, wide))
    launches = []
    fwd = _native.fwd
    monkeypatch.setattr(_native, "fwd", lambda *a, **kw: (launches.append(1), fwd(*a, **kw)))
    print(f"case padded list H{H} T{T} width {width}", flush=True)
    o, l = block_sparse_attn_fwd(*qkv, drp, dci, None)
    for call in range(2):
        launches.clear()
        ow, lw = block_sparse_attn_fwd(*qkv, drp, dwide, None)
        torch.cuda.synchronize()
        assert torch.equal(o, ow) and torch.equal(l, lw)
        twice = _native.kernel_of(1, H, T, False, width) != _native.kernel_of(1, H, T, False, ci.shape[-1])
        assert len(launches) == (2 if twice and call == 0 else 1)
    submission.clear_csr_cache()


def test_padded_window_of_the_same_kernel_launches_once(monkeypatch):
    submission.clear_csr_cache()
    B, H, T = 1, 8, 8320
    rp, ci = P.sliding_csr(B, H, T, 8)
    ci = np.concatenate([ci, np.zeros((B, H, 900), np.int32)], axis=-1)
    dev = [x.cuda() for x in P.make_qkv(B, H, T, seed=5)] + [torch.from_numpy(x).cuda() for x in (rp, ci)]
    launches = []
    for name in ("fwd", "fwd_window"):
        f = getattr(_native, name)
        monkeypatch.setattr(_native, name, lambda *a, f=f, **kw: (launches.append(1), f(*a, **kw)))
    print("case padded window, one launch", flush=True)
    o1, l1 = block_sparse_attn_fwd(*dev, None)
    assert len(launches) == 1
    o2, l2 = block_sparse_attn_fwd(*dev, None)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(l1, l2)
    submission.clear_csr_cache()


@pytest.mark.parametrize("how", ["none", "not diagonal", "above", "twice", "empty", "past the list"])
@pytest.mark.parametrize("lens", [(2048, 2048), (2000, 1), (640, 641), (0, 129)])
def test_rows_past_seq_len_against_the_host_check(lens, how):
    """One broken row, before and past seq_len, in each of the sequences: the flags are the host
    check's with and without seq_lens."""
    B, H, T = 2, 3, 2048
    nqb = T // 128
    rng = np.random.default_rng(7)
    sl = np.asarray(lens, np.int32)
    dsl = torch.from_numpy(sl).cuda()
    print(f"case check lens {lens} {how}", flush=True)
    for _ in range(6):
        rp, ci = P.retrieval_csr(B, H, T, 5, int(rng.integers(1 << 20)))
        if how != "none":
            broken(rp, ci, how, rng)

        def rejected(seq_lens):
            try:
                _native.check_csr_host(rp, ci, B, H, nqb, ci.shape[-1], seq_lens=seq_lens)
            except ValueError:
                return True
            return False

        result = torch.empty(_native.check_cap(B * H * nqb), dtype=torch.int32, pin_memory=True)
        drp, dci = torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda()
        n = _native.check_csr_gpu(drp.data_ptr(), dci.data_ptr(), B, H, nqb, ci.shape[-1],
                                  result.data_ptr(), result.numel(),
                                  torch.cuda.current_stream().cuda_stream, dsl.data_ptr())
        torch.cuda.synchronize()
        flags = int(np.bitwise_or.reduce(result.numpy()[:n]))
        if how in ("none", "not diagonal", "above", "twice"):
            assert int(result.numpy()[:n].max()) >> _native.CHECK_FLAG_BITS == rp[..., -1].max()
        assert bool(flags & 1) == rejected(sl)
        assert bool(flags & 5) == rejected(None)


@pytest.mark.parametrize("on_host", [False, True])
def test_rows_that_end_at_seq_len_are_checked_on_the_gpu(on_host, monkeypatch):
    """A CSR without rows past seq_len, as a selector over ragged sequences makes it: no copy to the
    host, one check for these seq_lens, another for other ones, a broken row before seq_len raises."""
    submission.clear_csr_cache()
    B, H, T, lens = 2, 3, 1024, [700, 1024]
    rp, ci = P.make_csr(B, H, T, lambda b, h, i: [] if i * 128 >= lens[b]
                        else sorted({0, i // 2, i}))
    q, k, v = P.make_qkv(B, H, T, seed=11)
    dev = [x.cuda() for x in (q, k, v)] + [torch.from_numpy(x).cuda() for x in (rp, ci)]
    sl = torch.tensor(lens, dtype=torch.int32, device="cpu" if on_host else "cuda")
    calls = []
    host = submission._check_on_host
    monkeypatch.setattr(submission, "_check_on_host", lambda *a: (calls.append(1), host(*a)))
    print(f"case rows end at seq_len, seq_lens on the host {on_host}", flush=True)
    for _ in range(2):
        o, l = block_sparse_attn_fwd(*dev, sl)
        torch.cuda.synchronize()
        oo, ol = c_ref.fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), rp, ci,
                           np.asarray(lens, np.int32), round_p_fp16=False)
        assert_close(o.float().cpu().numpy(), oo)
        assert_close(l.cpu().numpy(), ol, what="LSE")
    assert not calls and len(submission._csr_cache) == 1
    with pytest.raises(ValueError, match="empty"):  # the same CSR does not do without seq_lens
        block_sparse_attn_fwd(*dev, None)
    with pytest.raises(ValueError, match="b=0,h=0,qb=6"):
        block_sparse_attn_fwd(*dev, torch.tensor([800, 1024], dtype=torch.int32))
    dev[4][1, 2, 5] = 7
    with pytest.raises(ValueError, match="b=1,h=2"):
        block_sparse_attn_fwd(*dev, sl)
    submission.clear_csr_cache()


@pytest.mark.parametrize("case", ["plan", "few query blocks", "padded", "rows end at seq_len"])
def test_calls_captured_after_a_first_call(case):
    """A CSR seen before is launched from its cache entry under stream capture; every replay, with eager
    work between them, gives the eager result."""
    submission.clear_csr_cache()
    sl = None
    if case == "plan":
        rp, ci = P.mixed_csr(1, 16, 4096, 3)
    elif case == "few query blocks":
        rp, ci = P.retrieval_csr(1, 4, 2048, 6, 1)
    elif case == "padded":
        rp, ci = P.retrieval_csr(1, 8, 4096, 6, 1)
        ci = np.concatenate([ci, np.zeros((1, 8, 400), np.int32)], axis=-1)
    else:
        rp, ci = P.make_csr(2, 3, 1024, lambda b, h, i: [] if i * 128 >= 700 else sorted({0, i // 2, i}))
        sl = torch.tensor([700, 650], dtype=torch.int32, device="cuda")
    B, H, n1 = rp.shape
    dev = [x.cuda() for x in P.make_qkv(B, H, (n1 - 1) * 128, seed=2)]
    dev += [torch.from_numpy(x).cuda() for x in (rp, ci)] + [sl]
    print(f"case captured {case}", flush=True)
    want, want_lse = block_sparse_attn_fwd(*dev)
    torch.cuda.synchronize()
    assert (next(iter(submission._csr_cache.values())).sched is not None) == (case == "plan")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o, lse = block_sparse_attn_fwd(*dev)
    for _ in range(4):
        o.zero_()
        lse.zero_()
        block_sparse_attn_fwd(*dev)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(lse, want_lse)
    submission.clear_csr_cache()


@pytest.mark.parametrize("on_host", [False, True])
def test_an_empty_batch_is_rejected_as_before_the_gpu_check(on_host):
    q = torch.empty((0, 3, 1024, 128), dtype=torch.float16, device="cuda")
    dev = "cpu" if on_host else "cuda"
    rp, ci = (torch.empty((0, 3, n), dtype=torch.int32, device=dev) for n in (9, 20))
    with pytest.raises(ValueError):
        block_sparse_attn_fwd(q, q, q, rp, ci, None)
    with pytest.raises(_native.NativeError):
        block_sparse_attn_fwd_generic(q, q, q, rp, ci, None)
