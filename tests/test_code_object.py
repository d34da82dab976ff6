"""What the host's plans assume of the compiled kernels (the registers and LDS
in the code object's metadata), on the CPU: csrc/matmat.c counts on four waves
per SIMD of every exact GEMM kernel on the matrix cores; and the sizes that a
kernel and the host code launching it both state.
"""
from __future__ import annotations

import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJECT = os.path.join(ROOT, "mynah-slm_amd", "_build", "kernels.hsaco")
READELF = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
LDS_PER_CU, VGPRS_PER_SIMD = 160 * 1024, 512


@pytest.fixture(scope="module")
def kernels():
    if not (os.path.exists(OBJECT) and os.path.exists(READELF)):
        pytest.skip("no code object or no llvm-readelf beside the library")
    notes = subprocess.run([READELF, "--notes", OBJECT], check=True, capture_output=True,
                           text=True).stdout
    out = {}
    for k in re.split(r"\n  - \.agpr_count", notes)[1:]:
        def field(f):
            return re.search(rf"\.{f}:\s+(\S+)", k).group(1)
        out[field("name")] = {f: int(field(f)) for f in (
            "vgpr_count", "group_segment_fixed_size", "max_flat_workgroup_size",
            "vgpr_spill_count")}
    return out


def workgroups_per_cu(k):
    waves = k["max_flat_workgroup_size"] // 64
    by_vgpr = 4 * min(8, VGPRS_PER_SIMD // (-(-k["vgpr_count"] // 8) * 8)) // waves
    lds = k["group_segment_fixed_size"]
    return min(by_vgpr, LDS_PER_CU // lds if lds else by_vgpr)


def test_exact_gemm_kernels_hold_four_waves_per_simd(kernels):
    names = [n for n in kernels if re.search(r"gemm_\w*(mfma[124]|few(16|32))$", n)]
    assert len(names) == 33
    for n in names:
        k = kernels[n]
        assert workgroups_per_cu(k) * (k["max_flat_workgroup_size"] // 64) >= 16, (n, k)
        assert k["vgpr_spill_count"] <= 1, (n, k)


@pytest.mark.parametrize("host,source,kernel", [
    ("MYNAH_DQ_STEP", "dequant.hip", "DQ_STEP"), ("MYNAH_PV_SW", "decode.hip", "DPV_SW"),
    ("MYNAH_ATTN_SHORT_N", "decode.hip", "ASH_N"), ("MYNAH_AS_CH", "common.hip.h", "AS_CH")])
def test_sizes_stated_twice_agree(host, source, kernel):
    def value(path, name):
        with open(os.path.join(ROOT, "mynah-slm_amd", "csrc", path)) as f:
            text = f.read()
        expr = re.search(rf"#define {name} ([^\n/]+)", text).group(1).strip()
        while re.search(r"[A-Z_]{3,}", expr):
            expr = re.sub(r"[A-Z_]{3,}", lambda m: str(value(path, m.group(0))), expr)
        return eval(re.sub(r"(\d)u\b", r"\1", expr))      # noqa: S307 (the source's own constant)
    assert value("runtime_internal.h", host) == value(source, kernel)
