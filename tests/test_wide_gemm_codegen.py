"""What the dense product's wide tiles rely on, checked in the generated code: the compiler keeps nothing of its own in m0, which the
transfers into LDS write, no vector load of its own is under way where theirs are counted by hand, and nothing is kept in memory."""

import re
import shutil
import subprocess

import pytest

from neuropress_amd import build


def test_wide_tiles(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not build.Path(hipcc).exists():
        pytest.skip("needs hipcc")
    out = tmp_path / "wide_gemm.s"
    res = subprocess.run([hipcc, *build.CXXFLAGS, *build.DEVICE_FLAGS, "-S", "--cuda-device-only",
                          str(build.CSRC / "wide_gemm.hip"), "-o", str(out)], capture_output=True, text=True)  # fmt: skip
    assert res.returncode == 0, res.stderr[-2000:]
    lines = out.read_text().split("\n")
    starts = [i for i, ln in enumerate(lines) if re.match(r"^_ZN5npamd\S*wide_gemm_kernel\S*:", ln)]
    assert len(starts) == 26  # two activation types, thirteen tiles
    for i in starts:
        body = lines[i : next(j for j in range(i, len(lines)) if lines[j].startswith(".Lfunc_end"))]
        code = [ln.split(";")[0] for ln in body]
        assert not [ln for ln in code if re.search(r"\bm0\b", ln) and not re.match(r"\s+s_mov_b32 m0, s\d+", ln)]
        assert not [ln for ln in code if "scratch_" in ln]
        first = next(k for k, ln in enumerate(code) if "global_load_lds" in ln)
        last = max(k for k, ln in enumerate(code) if "v_mfma" in ln)
        loop = code[first : last + 1]
        assert not [ln for ln in loop if re.search(r"v_accvgpr_(mov|read|write)", ln)]
        assert not [ln for ln in loop if re.search(r"global_load_(?!lds)|flat_load|buffer_load", ln)]
