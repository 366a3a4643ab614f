"""The GEMV of the group-affine formats that brings codes, scales and activations through LDS in whole lines: every token-count
class, one and two row tiles per block, one to many 256-k steps and their remainders, group sizes from one to four
chunks, against the decoded weight in float64; and the calls its dispatch leaves to the other kernel."""

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture
def row_tiles(monkeypatch):
    from neuropress_amd import _lib

    def force(tiles):
        monkeypatch.setenv("NPAMD_GEMV_R", str(tiles))
        monkeypatch.setenv("NPAMD_Q4_ROWWISE", "0")
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.undo()
    _lib.load().npamd_diag_reload_tuning()


def _layer(n, k, bits, group, zero_point, gpu):
    g = cases.gen(n + k + bits)
    codes = torch.randint(0, 256, (n, k * bits // 8), generator=g, dtype=torch.uint8).to(gpu)
    scale = (torch.randn(n * (k // group), generator=g) * 0.02).half().to(gpu)
    zp = torch.randint(0, 1 << bits, (n * (k // group),), generator=g).half().to(gpu) if zero_point else None
    return codes, scale, zp


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits,zero_point", [(4, False), (4, True), (8, False), (8, True)])
@pytest.mark.parametrize("tiles", [1, 2])
def test_q_gemv(gpu, row_tiles, tiles, bits, zero_point, act):
    from neuropress_amd import kernels

    row_tiles(tiles)
    # tokens at the ends of each class; rows around the tiles; K of one chunk, a ragged last step, more steps than waves; a few
    # rows past half of 256 compute units' tiles, or more tokens than K in parts is taken for
    for m, n, k, group in ((9, 16, 64, 32), (16, 33, 64, 64), (17, 1, 320, 32), (32, 50, 2176, 128), (31, 47, 576, 64), (1, 2050, 320, 64),
                           (2, 2081, 1024, 256), (3, 2064, 2240, 32), (8, 2100, 4160, 64), (16, 2049, 192, 32), (24, 130, 8448, 256)):  # fmt: skip
        codes, scale, zp = _layer(n, k, bits, group, zero_point, gpu)
        x = torch.randn(m, k, generator=cases.gen(m)).to(act).to(gpu)
        bias = torch.randn(n, generator=cases.gen(n)).to(gpu)
        w = kernels.q_dequant(codes, scale, bits, group, zp, act).double()
        y = kernels.q_linear(x, codes, scale, bits, group, zp, bias).double()
        ref = x.double() @ w.T + bias.double()
        tol = 2.0 ** (-10 if act == torch.float16 else -7)  # the rounding of the output; f32 sums of k products
        slack = 2.0 ** -22 * (x.double().abs() @ w.abs().T)
        assert bool(((y - ref).abs() <= tol * ref.abs() + slack + 1e-6).all()), (m, n, k, group, float((y - ref).abs().max()))


def test_q_gemv_past_k_counts_as_zero(gpu, row_tiles):
    """K = 320: three of the last step's four chunks lie past K and read the last chunk again.  An infinite activation or scale
    in it makes an infinite result, as its own product does, not a NaN, as zero times infinity would."""
    from neuropress_amd import kernels

    row_tiles(1)
    m, n, k = 9, 40, 320
    codes = torch.full((n, k // 2), 0x99, dtype=torch.uint8, device=gpu)  # q - 8 = 1
    scale = torch.full((n, k // 32), 0.5, dtype=torch.half, device=gpu)
    x = torch.ones(m, k, dtype=torch.half, device=gpu)
    x[3, -1] = float("inf")
    y = kernels.q_linear(x, codes, scale.view(-1), 4, 32)
    assert bool((y[3] == float("inf")).all()) and bool((y[[0, 1, 2, 4, 5, 6, 7, 8]] == k * 0.5).all())
    scale[7, -1] = float("inf")
    y = kernels.q_linear(torch.ones_like(x), codes, scale.view(-1), 4, 32)
    assert bool((y[:, 7] == float("inf")).all()) and bool((y[:, :7] == k * 0.5).all()) and bool((y[:, 8:] == k * 0.5).all())


@pytest.mark.parametrize("bits", [4, 8])
def test_calls_the_q_gemv_does_not_take(gpu, row_tiles, bits):
    """An odd count of scales, scales that start between two dwords: the same numbers as the calls it takes, up to the order of
    f32 sums."""
    from neuropress_amd import kernels

    row_tiles(1)
    n, k, m = 2065, 192, 9
    codes, scale, _ = _layer(n, k, bits, 64, False, gpu)  # 3 x 2065 scales: odd
    x = torch.randn(m, k, generator=cases.gen(5)).half().to(gpu)
    whole = kernels.q_linear(x, codes[:-1], scale[:-3], bits, 64)
    odd = kernels.q_linear(x, codes, scale, bits, 64)
    shifted = torch.cat([scale[:1], scale[:-3]])[1:]
    assert shifted.data_ptr() % 4 == 2
    for y in (odd[:, :-1], kernels.q_linear(x, codes[:-1], shifted, bits, 64)):
        assert torch.allclose(y.float(), whole.float(), rtol=2.0 ** -10, atol=1e-3)
