"""The line between the blocks entries and decode + product, host arithmetic: calls on both sides of it that were measured."""

import pytest

# kind, rows of the codebook, then tokens, rows and columns of layers where one of the two is ahead by 8 % or more
PRODUCT = [
    (8, 0, ((358, 1102, 6656), (614, 691, 6272), (1084, 466, 4864), (1611, 280, 11520), (426, 1095, 4480))),
    (4, 0, ((362, 1276, 6400), (408, 1128, 4608), (174, 3945, 5376), (914, 544, 5248))),
    (0, 65536, ((100, 491, 6272), (62, 373, 7296), (42, 319, 7680), (56, 299, 4992))),
    (1, 65536, ((53, 679, 7168), (46, 285, 5504), (42, 506, 4864), (106, 373, 5120))),
]
BLOCKS = [
    (8, 0, ((500, 377, 8064), (262, 820, 7936), (177, 625, 13056), (101, 1163, 6784), (106, 3825, 2048))),
    (4, 0, ((441, 404, 7296), (383, 373, 6144), (169, 1658, 5120), (60, 586, 13952), (64, 512, 512))),
    (0, 65536, ((81, 1308, 4096), (75, 901, 5120), (54, 883, 5120), (64, 1024, 4096))),
    (1, 65536, ((35, 1871, 3968), (33, 1705, 4224))),
    (1, 4096, ((56, 2015, 3840), (60, 1600, 4480), (58, 777, 7296))),
]


@pytest.mark.parametrize("kind,rows,calls,blocks", [(*c, 0) for c in PRODUCT] + [(*c, 1) for c in BLOCKS])
def test_calls_that_were_measured(kind, rows, calls, blocks):
    from neuropress_amd import _lib

    asked = [_lib.load().npamd_gemv_blocks_preferred(m, n, k, kind, rows, 0, 0) for m, n, k in calls]
    assert asked == [blocks] * len(calls)
