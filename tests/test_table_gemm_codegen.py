"""What the table GEMM's transfers into LDS rely on, checked in the generated code: the compiler keeps nothing of its own in m0, which
their asm statements cannot declare as written, no vector load of its own is under way in the loop, where they are counted by
hand, and the loop moves no accumulators."""

import re
import shutil
import subprocess

import pytest

from neuropress_amd import build


def test_transfers_and_accumulators(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not build.Path(hipcc).exists():
        pytest.skip("needs hipcc")
    out = tmp_path / "table_gemm.s"
    res = subprocess.run([hipcc, *build.CXXFLAGS, *build.DEVICE_FLAGS, "-S", "--cuda-device-only",
                          str(build.CSRC / "table_gemm.hip"), "-o", str(out)], capture_output=True, text=True)  # fmt: skip
    assert res.returncode == 0, res.stderr[-2000:]
    lines = out.read_text().split("\n")
    starts = [i for i, ln in enumerate(lines) if re.match(r"^_ZN5npamd\S*table_gemm_kernel\S*:", ln)]
    assert len(starts) == 30  # two activation types, three index widths, five tiles
    for i in starts:
        body = lines[i : next(j for j in range(i, len(lines)) if lines[j].startswith(".Lfunc_end"))]
        code = [ln.split(";")[0] for ln in body]
        assert not [ln for ln in code if re.search(r"\bm0\b", ln) and not re.match(r"\s+s_mov_b32 m0, s\d+", ln)]
        assert not [ln for ln in code if "scratch_" in ln]
        first = next(k for k, ln in enumerate(code) if "v_mfma" in ln)
        last = max(k for k, ln in enumerate(code) if "v_mfma" in ln)
        # the loop: from the wait for a step's activations on
        top = max(k for k in range(first) if "s_waitcnt vmcnt(0)" in code[k])
        loop = code[top : last + 1]
        assert not [ln for ln in loop if re.search(r"v_accvgpr_(mov|read|write)", ln)]
        assert not [ln for ln in loop if re.search(r"global_load_(?!lds)|flat_load|buffer_load", ln)]
