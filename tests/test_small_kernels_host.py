"""CPU checks of the choice among the kernels and of bsa_ksplit.hip and bsa_check.hip: the gfx950 assembly spills nothing, emits no
packed-FP32 instruction and writes M0 only right before an LDS DMA; the GPU check's entry point rejects
bad arguments before any launch."""

from __future__ import annotations

import re
import subprocess

import pytest

from usagi_amd import _native
from usagi_amd import build as B


@pytest.fixture(scope="module", params=["bsa_ksplit.hip", "bsa_check.hip"])
def asm(request, tmp_path_factory) -> str:
    try:
        B.hipcc_path()
    except RuntimeError:
        pytest.skip("hipcc not available")
    src = next(s for s in B.SRCS if s.endswith(request.param))
    out = str(tmp_path_factory.mktemp("isa") / "out.s")
    cmd = [c for c in B.hipcc_command(srcs=[src], out=out) if c not in ("-shared", "-fPIC")]
    cmd[1:1] = ["--offload-device-only", "-S"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    with open(out) as f:
        return f.read()


def test_no_spills_no_packed_fp32(asm):
    for key in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"):
        vals = [int(v) for v in re.findall(rf"\.{key}:\s+(\d+)", asm)]
        assert vals and all(v == 0 for v in vals), (key, vals)
    assert not re.search(r"v_pk_(add|mul|fma|mov)_f32", asm)


def test_m0_only_feeds_the_dma(asm):
    ins = [ln.split(";")[0].strip() for ln in asm.splitlines()]
    ins = [ln for ln in ins if ln and not ln.startswith(".") and not ln.endswith(":")]
    for i, ln in enumerate(ins):
        if ln.startswith("global_load_lds_dwordx4"):
            assert ins[i - 2].startswith("s_mov_b32 m0, s") and ins[i - 1] == "s_nop 0", ins[i - 2:i + 1]
        elif re.search(r"\bm0\b", ln):
            assert re.fullmatch(r"s_mov_b32 m0, s\d+", ln), ln
            assert ins[i + 2].startswith("global_load_lds_dwordx4"), ins[i:i + 3]


@pytest.mark.parametrize("over", [dict(rp=None), dict(ci=None), dict(B=0), dict(H=-1), dict(nqb=0),
                                  dict(nnz=-1), dict(result=None), dict(cap=100),
                                  dict(nqb=_native.CHECK_MAX_BLOCKS + 1, cap=1 << 30)])
def test_gpu_check_rejects_bad_arguments(over):
    a = dict(rp=1, ci=1, B=1, H=1, nqb=128, nnz=9, result=1, cap=_native.check_cap(128), stream=None)
    a.update(over)
    code = _native.load().usagi_bsa_check_csr_gpu(a["rp"], a["ci"], a["B"], a["H"], a["nqb"], a["nnz"],
                                                  a["result"], a["cap"], a["stream"])
    assert code < 0 and _native.last_error()


@pytest.mark.parametrize("with_seq_lens", [False, True])
@pytest.mark.parametrize("H,nqb", [(3, 43), (8, 32), (10, 32), (16, 32), (4, 64), (8, 64), (33, 16)])
@pytest.mark.parametrize("w", [5, 8, 16])
def test_a_padded_column_list_runs_the_kernel_of_its_rows(w, H, nqb, with_seq_lens):
    """Once the entries are known, the width of col_idx does not decide between the kernels for few
    query blocks and bsa_fwd_dma_kernel."""
    nnz = sum(min(i + 1, w) for i in range(nqb))
    want = _native.kernel_of(1, H, nqb * 128, with_seq_lens, nnz)
    for width in (nnz + 1, nqb * (nqb + 1) // 2, nqb * nqb):
        assert _native.kernel_of(1, H, nqb * 128, with_seq_lens, max(width, nnz), False, nnz) == want
    # more entries than the list is wide count as its width
    assert _native.kernel_of(1, H, nqb * 128, with_seq_lens, nnz, False, nqb * nqb) == want


def test_kernel_of_and_fwd_entries_reject_what_the_forward_rejects():
    lib = _native.load()
    for B, H, T, nnz in ((0, 1, 128, 1), (1, 0, 128, 1), (1, 1, 100, 1), (1, 1, 128, -1), (64, 64, 1 << 20, 1)):
        assert lib.usagi_bsa_kernel_of(B, H, T, 0, nnz, 0, -1) < 0 and _native.last_error()
        assert lib.usagi_bsa_fwd_entries(1, 1, 1, 1, 1, None, 1, None, B, H, T, 128, nnz, 0, None, 0, None,
                                         0, 1) < 0


def test_generic_rows_of_one_block_take_the_small_kernels_up_to_64_query_blocks():
    for H, nqb, want in ((4, 8, 32), (8, 8, 32), (9, 8, 0), (16, 8, 0)):
        T = nqb * 128
        assert _native.kernel_of(1, H, T, False, nqb, True) == want
        assert _native.kernel_of(1, H, T, False, 2 * nqb, True) == (want or 64)
        assert _native.kernel_of(1, H, T, True, nqb, False) == (want or 64)
