"""What the dense product's plan chooses, host arithmetic."""

import re
import time

import pytest

from neuropress_amd import _lib, build
from tests import cases


@pytest.mark.parametrize("m,n,k,parts", [(548, 320, 9728, 7), (444, 352, 9856, 7), (529, 312, 9728, 7), (601, 432, 9344, 5), (512, 512, 8192, 5)])
def test_long_k_over_few_tiles(m, n, k, parts):
    """Parts of K that make about one round of 64 x 128 tiles, the tile in two groups.  With wide tiles alone 5, 6, 5, 3 and 4 parts, 3 to 13 % slower."""
    assert _lib.load().npamd_dense_gemm_workspace_bytes(m, n, k) == parts * m * n * 4


def test_tests_know_every_tile():
    source = (build.CSRC / "dense_gemm.hip").read_text()
    rows = re.search(r"kDenseCost\[\] = \{\n(.*?)\n\};", source, re.S).group(1)
    assert [tuple(map(int, m)) for m in re.findall(r"^\s+\{(\d+), (\d+),", rows, re.M)] == [cases.DENSE_TILES[i] for i in sorted(cases.DENSE_TILES)]


# Products (tokens, rows, columns) that one of the two serves faster, by 3 % and more on both types; the last is one that no wide tile takes.
LIBRARY = [(4095, 4096, 4096), (4096, 4096, 4096), (4000, 8192, 8192), (3500, 4096, 14336), (8000, 4096, 14336), (2842, 64000, 4992), (14422, 16128, 5760), (32461, 37751, 640),
           (5000, 128256, 2048), (3500, 32000, 4096), (6144, 14336, 8192), (3000, 28672, 8192), (64, 1 << 22, 64)]  # fmt: skip
PACKAGE = [(1646, 13120, 11136), (2048, 4096, 4096), (4096, 11008, 4096), (4000, 11008, 4096), (3072, 9728, 12288), (2687, 10983, 7232), (4096, 11008, 1280), (2789, 11008, 1664),
           (2048, 13824, 13824), (384, 4096, 4096), (777, 1280, 8192)]  # fmt: skip


def test_line_to_the_library():
    preferred = _lib.load().npamd_dense_gemm_preferred
    assert [p for p in LIBRARY if preferred(*p)] == []
    assert [p for p in PACKAGE if not preferred(*p)] == []


def test_a_plan_costs_a_call_little():
    """Every decode + product call is planned at its launch.  With all tiles and parts estimated in turn 0.6 and 0.8 us, now 0.17 and 0.16."""
    plan = _lib.load().npamd_dense_gemm_workspace_bytes

    def least(*shape):
        best = 1.0
        for _ in range(60):
            t0 = time.perf_counter()
            for _ in range(300):
                plan(*shape)
            best = min(best, (time.perf_counter() - t0) / 300)
        return best

    for shape in ((384, 4096, 4096), (77, 3003, 2176)):
        # Without the call itself.  On a machine that is busy with something else for a while, once more.
        assert any(least(*shape) - least(0, 0, 0) < 0.4e-6 for _ in range(20)), shape
