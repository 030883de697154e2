"""Build-time limits of the kernels (CPU: hipcc only, nothing runs).

The mixed kernel plans a batch in LDS (plan tables of up to kMaxSeqs
sequences beside its static arrays).  A build whose LDS could exceed what one
gfx950 workgroup may have (160 KiB) must not compile: an 8-wave build of the
mixed kernel once asked for 170,004 bytes at 1,024 sequences and its dispatch
was rejected on the GPU.  The shipped build's static LDS must match the
kernel's own account of it (MixedLds), so the bound covers what the compiler
allocates.
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from custom_inference_engine_amd import _build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
SRC = os.path.join(_build.CSRC, "mixed_attention.hip")
DECODE = os.path.join(_build.CSRC, "paged_decode.hip")


def _compile(tmp_path, *defines, src=SRC):
    flags = [f for f in _build.HIPCC_FLAGS if f != "-fPIC"]
    cmd = [HIPCC, *flags, *(f"-D{d}" for d in defines), "-I", _build.INCLUDE, "-I", _build.CSRC,
           "--offload-device-only", "-c", src, "-o", str(tmp_path / "kernels.o"),
           "-Rpass-analysis=kernel-resource-usage"]
    return subprocess.run(cmd, capture_output=True, text=True)


def test_mixed_build_past_the_lds_budget_does_not_compile(tmp_path):
    res = _compile(tmp_path, "CIE_MIXED_WAVES=8")
    assert res.returncode != 0
    assert "exceed a workgroup's LDS" in res.stderr


@pytest.fixture(scope="module")
def shipped(tmp_path_factory):
    """The compiler's remarks on the shipped mixed kernels."""
    res = _compile(tmp_path_factory.mktemp("shipped"))
    assert res.returncode == 0, res.stderr[-3000:]
    return res.stderr


def _wide_kernels(stderr, d):
    """Names of the D = d kernels that run wide items (the last template argument)."""
    return set(re.findall(rf"mixed_attention_kernelILi{d}ELb[01]ELb[01]ELb1EE", stderr))


@pytest.mark.parametrize("waves", [2, 8])
def test_mixed_build_of_other_wave_counts_has_no_wide_launch(tmp_path, waves):
    """Wide items are laid out for four waves: with two, half of each K/V stage would stay
    unwritten, with eight the stages would be written past their end."""
    res = _compile(tmp_path, f"CIE_MIXED_WAVES={waves}", "CIE_MIXED_CG=2")
    assert res.returncode == 0, res.stderr[-3000:]
    assert not _wide_kernels(res.stderr, 64)
    assert _wide_kernels(res.stderr, 128)  # always four waves


def test_shipped_mixed_build_plans_its_largest_batch_within_lds(shipped):
    assert len(_wide_kernels(shipped, 64)) == len(_wide_kernels(shipped, 128)) == 4
    sizes = [int(m) for m in re.findall(r"mixed_attention_kernel\w*.*?\n.*?LDS Size \[bytes/block\]: (\d+)",
                                        shipped, flags=re.S)]
    if not sizes:  # remarks printed in another order: take every LDS size line of the file
        sizes = [int(m) for m in re.findall(r"LDS Size \[bytes/block\]: (\d+)", shipped)]
    assert sizes
    k_max_seqs = 1024  # kMaxSeqs: the ABI's batch limit for cie_mixed_attention
    plan = k_max_seqs * 8 + (4 * k_max_seqs + k_max_seqs + 1) * 4
    # three wide workgroups a CU at D = 64, two at D = 128 (LDS goes in 1,280 bytes; the
    # plan tables of a wide launch lie in its stages)
    wide = re.findall(r"mixed_attention_kernelILi(\d+)ELb[01]ELb[01]ELb1EE.*?LDS Size \[bytes/block\]: (\d+)",
                      shipped, flags=re.S)
    assert len(wide) == 8
    for d, static in wide:
        assert 160 * 1024 // (-(-int(static) // 1280) * 1280) >= (3 if d == "64" else 2), (d, static)
    for static in sizes:
        assert static + plan <= 160 * 1024, (static, plan)


def test_launches_of_16_row_tiles_keep_their_scalars(shipped):
    """The 16-row kernels' scalars are spilled to vector lanes, a few cycles an item each: no
    more of them than these kernels had before some launches became wide."""
    spills = re.findall(r"mixed_attention_kernelILi(\d+)ELb1ELb([01])ELb0EE.*?SGPRs Spill: (\d+)", shipped,
                        flags=re.S)
    most = {("64", "0"): 47, ("64", "1"): 40, ("128", "0"): 33, ("128", "1"): 27}
    assert {(d, planned) for d, planned, _ in spills} == set(most)
    for d, planned, n in spills:
        assert int(n) <= most[d, planned], (d, planned, n)
    # their plan kernels know at build time that no tile is wide
    plans = re.findall(r"mixed_plan_kernelILi(\d+)ELb0EE.*?TotalSGPRs: (\d+)", shipped, flags=re.S)
    assert len(plans) == 2 and all(int(n) <= {"64": 79, "128": 75}[d] for d, n in plans)


@pytest.mark.parametrize("waves", [1, 4])
def test_decode_merge_of_many_splits_fits_its_lds(tmp_path, waves):
    """The merge keeps a float for each of 16 heads x 64 splits and 16 bytes a thread in the
    fold's LDS, which a one-wave build's fold alone does not fill."""
    res = _compile(tmp_path, f"CIE_DECODE_WAVES={waves}", src=DECODE)
    assert res.returncode == 0, res.stderr[-3000:]
    many = re.findall(r"decode_kernelILi(\d+)ELi(\d+)ELb[01]ELb[01]ELb[01]ELb1EE.*?LDS Size \[bytes/block\]: (\d+)",
                      res.stderr, flags=re.S)
    assert any(int(w) == waves for _, w, _ in many)
    for d, w, lds in many:
        rest = 2 * int(w) * 16 * 4 + 4  # the waves' maxima and sums, the arrival flag
        assert int(lds) - rest >= 16 * 64 * 4 + int(w) * 64 * 16, (d, w, lds)
