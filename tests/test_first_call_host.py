"""The first call with a CSR, without a GPU: the memory that the queued check writes to outlives it,
whatever raises before the result is read. The device calls are stand-ins that note what is queued."""

from __future__ import annotations

import contextlib
import os
import subprocess
import sys
import weakref

import pytest
import torch

from usagi_amd import _native, submission
from usagi_amd import patterns as P

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class FakeGpu:
    """One stream: the check is queued until an event or the stream is waited for."""

    def __init__(self, monkeypatch, fail):
        self.fail = fail
        self.queued = False       # the check may still write to the result
        self.released_while = []  # was it, when the result's memory was given back
        gpu, empty = self, torch.empty

        def pinned_empty(*a, pin_memory=False, **kw):
            t = empty(*a, **kw)
            if pin_memory:
                weakref.finalize(t, lambda: gpu.released_while.append(gpu.queued))
            return t

        def check(*a):
            gpu.queued = True
            return 1

        class Event:
            def record(self, stream=None):
                if gpu.fail == "record":
                    raise RuntimeError("record")

            def synchronize(self):
                if gpu.fail == "wait":
                    raise KeyboardInterrupt
                gpu.queued = False

        class Stream:
            cuda_stream = 0

            def synchronize(self):
                gpu.queued = False

        def fwd(*a, **kw):
            if gpu.fail == "launch":
                raise _native.NativeError(-1, "problem too large")

        monkeypatch.setattr(torch, "empty", pinned_empty)
        monkeypatch.setattr(torch.cuda, "Event", Event)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: Stream())
        monkeypatch.setattr(_native, "check_csr_gpu", check)
        monkeypatch.setattr(_native, "fwd", fwd)
        monkeypatch.setattr(submission, "_check_inputs", lambda q, k, v: tuple(q.shape))
        monkeypatch.setattr(submission, "_on_gpu", lambda *a: True)
        monkeypatch.setattr(submission, "_on_device", lambda dev: contextlib.nullcontext())
        monkeypatch.setattr(submission, "_raw_stream", lambda index: 0)


@pytest.mark.parametrize("fail,error", [("record", RuntimeError), ("launch", _native.NativeError),
                                        ("wait", KeyboardInterrupt)])
def test_a_queued_check_outlives_no_error(monkeypatch, fail, error):
    submission.clear_csr_cache()
    rp, ci = P.sliding_csr(1, 2, 512, 2)
    q = torch.zeros((1, 2, 512, 128), dtype=torch.float16)
    rp, ci = torch.from_numpy(rp), torch.from_numpy(ci)
    gpu = FakeGpu(monkeypatch, fail)
    with pytest.raises(error) as caught:
        submission.block_sparse_attn_fwd(q, q, q, rp, ci, None)
    del caught
    assert gpu.released_while == [False] and not gpu.queued
    assert not submission._csr_cache  # nothing is kept of a CSR that was not checked


def test_import_needs_no_private_torch_name():
    """A torch without its ROCm parts lacks _cuda_getCurrentRawStream; the planner, the patterns and the
    host check are there all the same."""
    code = ("import torch\n"
            "del torch._C._cuda_getCurrentRawStream\n"
            "import usagi_amd\n"
            "from usagi_amd import _native, patterns as P\n"
            "rp, ci = P.sliding_csr(1, 2, 512, 2)\n"
            "_native.check_csr_host(rp, ci, 1, 2, 4, ci.shape[-1])\n")
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=REPO)
    assert res.returncode == 0, res.stderr[-2000:]
