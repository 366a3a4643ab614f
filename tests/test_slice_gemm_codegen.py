"""What the slice GEMM's relaxed barriers rely on, checked in the generated code.

``slice_gemm_kernel`` passes its two barriers of a super-step with the youngest codebook lookups still under way
(``s_waitcnt lgkmcnt(N); s_barrier``): LDS operations of a wave complete in order, so whatever is older is done.  The
barrier in front of the stores of the next activations needs every read of the last ones to be older, the one behind them
the stores.  No scalar or flat operation, whose return is counted out of order, may be under way with them.
"""

import re
import shutil
import subprocess

import pytest

from neuropress_amd import build


def test_relaxed_barriers_leave_only_lookups_under_way(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not build.Path(hipcc).exists():
        pytest.skip("needs hipcc")
    out = tmp_path / "slice_gemm.s"
    res = subprocess.run([hipcc, *build.CXXFLAGS, *build.DEVICE_FLAGS, "-S", "--cuda-device-only",
                          str(build.CSRC / "slice_gemm.hip"), "-o", str(out)], capture_output=True, text=True)  # fmt: skip
    assert res.returncode == 0, res.stderr[-2000:]
    lines = out.read_text().split("\n")
    starts = [i for i, ln in enumerate(lines) if re.match(r"^_ZN5npamd17slice_gemm_kernel\S*: ;", ln)]
    assert len(starts) == 24  # two activation types, two token tiles, three row tiles, indices clamped or not
    for i in starts:
        body = lines[i : next(j for j in range(i, len(lines)) if lines[j].startswith(".Lfunc_end"))]
        m0 = [ln for ln in body if re.search(r"\bm0\b", ln) and not re.match(r"\s+s_mov_b32 m0, s\d+", ln)]
        assert not m0, m0  # nothing but the transfers into LDS keeps anything there
        relaxed = 0
        for k, ln in enumerate(body[:-1]):
            m = re.search(r"s_waitcnt lgkmcnt\((\d+)\)", ln)
            if not (m and int(m.group(1)) > 0 and "s_barrier" in body[k + 1]):
                continue
            relaxed += 1
            ops, fenced, j = [], None, k - 1
            while j >= 0 and "s_barrier" not in body[j]:
                op = re.match(r"\s+(ds_\w+|s_load\w+|s_buffer_load\w+|flat_\w+)", body[j])
                if op:
                    ops.append(op.group(1))
                if fenced is None and "; sched_barrier" in body[j]:
                    fenced = len(ops)  # operations since the last stage ended
                j -= 1
            keep = int(m.group(1))
            assert all(o.startswith("ds_") for o in ops), ops
            assert len(ops) >= keep and all(o == "ds_read_b128" for o in ops[:keep]), ops
            # Either the stores of the next activations are behind this barrier, and the lookups since the last stage
            # are all that may be under way, or they are in front of it among the older operations.
            stores_after = any("ds_write" in x for x in body[k + 2 : k + 40])
            assert (fenced is None or fenced >= keep) if stores_after else "ds_write_b128" in ops[keep:], (ops, fenced)
        assert relaxed >= 2
