"""The dense product of the decode + GEMM band: its tiles at shapes around their edges, ragged rows and columns, one to
many 64-k steps (fewer than a ring is deep, and counts its groups of waves do not divide)."""

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture
def dense_tile(monkeypatch):
    from neuropress_amd import _lib

    def force(tile):
        monkeypatch.setenv("NPAMD_DENSE_TILE", str(tile))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.delenv("NPAMD_DENSE_TILE", raising=False)
    _lib.load().npamd_diag_reload_tuning()


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", sorted(cases.DENSE_TILES))
def test_dense_gemm_tiles(gpu, dense_tile, tile, act):
    from neuropress_amd import kernels

    dense_tile(tile)
    for m, n, k in ((1, 1, 64), (31, 63, 128), (33, 65, 192), (64, 128, 256), (65, 129, 320), (127, 200, 448), (129, 257, 704),
                    (256, 130, 576), (300, 500, 1088), (520, 40, 64), (193, 129, 320)):  # fmt: skip
        g = cases.gen(m + n + k)
        x = torch.randn(m, k, generator=g).to(act)
        w = (torch.randn(n, k, generator=g) * 0.05).to(act)
        bias = torch.randn(n, generator=g)
        y = kernels.dense_linear(x.to(gpu), w.to(gpu), bias.to(gpu)).float().cpu()
        ref = x.double() @ w.double().T + bias.double()
        tol = 2.0 ** (-10 if act == torch.float16 else -7)  # the rounding of the output, and f32 sums
        assert bool(((y - ref).abs() <= tol * ref.abs() + 1e-4).all()), (tile, m, n, k, float((y - ref).abs().max()))
    wide = torch.zeros(70, 200, dtype=act)  # rows of x at a stride; the same bits as dense rows
    wide[:, :192] = torch.randn(70, 192, generator=cases.gen(1)).to(act)
    w = (torch.randn(90, 192, generator=cases.gen(2)) * 0.05).to(act).to(gpu)
    xs = wide.to(gpu)[:, :192]
    assert torch.equal(kernels.dense_linear(xs, w), kernels.dense_linear(xs.contiguous(), w))


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile,splits", [(1, 2), (1, 16), (2, 9), (3, 3), (4, 8), (5, 7), (6, 2), (7, 3), (15, 2), (15, 8)])
def test_dense_gemm_parts_of_k(gpu, dense_tile, monkeypatch, tile, splits, act):
    """K in parts over blocks: parts of unequal length, of fewer steps than a ring is deep or a block has groups of
    waves, columns the reduction reads four at a time and not."""
    from neuropress_amd import _lib, kernels

    monkeypatch.setenv("NPAMD_DENSE_SPLITS", str(splits))
    dense_tile(tile)
    for m, n, k in ((1, 1, 128), (33, 65, 576), (65, 130, 1088), (129, 260, 1600), (70, 257, 2112)):
        assert _lib.load().npamd_dense_gemm_workspace_bytes(m, n, k) == min(splits, k // 64) * m * n * 4
        g = cases.gen(m + n + k)
        x = torch.randn(m, k, generator=g).to(act)
        w = (torch.randn(n, k, generator=g) * 0.05).to(act)
        bias = torch.randn(n, generator=g)
        y = kernels.dense_linear(x.to(gpu), w.to(gpu), bias.to(gpu)).float().cpu()
        ref = x.double() @ w.double().T + bias.double()
        tol = 2.0 ** (-10 if act == torch.float16 else -7)  # the rounding of the output, and f32 sums
        assert bool(((y - ref).abs() <= tol * ref.abs() + 1e-4).all()), (tile, splits, m, n, k, float((y - ref).abs().max()))


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("splits", [0, 3])
def test_dense_gemm_96_rows(gpu, dense_tile, monkeypatch, splits, act):
    """Tiles of 96 x 64, of four waves of 48 x 32: the same sums in the same order as 64 x 128's, whole and in parts, around the edges
    of both; and what the plan takes by itself."""
    from neuropress_amd import kernels

    monkeypatch.setenv("NPAMD_DENSE_SPLITS", str(splits))
    for m, n, k in ((1, 1, 64), (95, 63, 192), (96, 64, 448), (97, 65, 512), (193, 129, 576), (384, 200, 1088), (300, 2560, 2048)):
        g = cases.gen(m + n + k)
        x = torch.randn(m, k, generator=g).to(act).to(gpu)
        w = (torch.randn(n, k, generator=g) * 0.05).to(act).to(gpu)
        bias = torch.randn(n, generator=g).to(gpu)
        out = []
        for tile in (3, 13, 0):
            dense_tile(tile)
            out.append(kernels.dense_linear(x, w, bias))
        ref = x.double() @ w.double().T + bias.double()
        tol = 2.0 ** (-10 if act == torch.float16 else -7)  # the rounding of the output, and f32 sums
        assert torch.equal(out[0], out[1]), (m, n, k)
        for y in out[1:]:
            assert bool(((y.double() - ref).abs() <= tol * ref.abs() + 1e-4).all()), (m, n, k)


def test_dense_linear_copies_rows_the_kernel_does_not_take(gpu):
    """Dense rows at an odd address, one row at an odd distance, rows far apart: each equals the product of the copy."""
    from neuropress_amd import kernels

    m, n, k = 40, 96, 128
    w = (torch.randn(n, k, generator=cases.gen(3)) * 0.05).half().to(gpu)
    flat = torch.randn(m * (k + 1) + 1, generator=cases.gen(4)).half().to(gpu)
    far = torch.zeros(2, (1 << 22) + 8, dtype=torch.half, device=gpu)
    far[:, :k] = flat[: 2 * k].view(2, k)
    for x in (flat[1 : 1 + m * k].view(m, k), flat[: m * (k + 1)].view(m, k + 1)[:1, :k], far[:, :k]):
        assert torch.equal(kernels.dense_linear(x, w), kernels.dense_linear(x.clone(memory_format=torch.contiguous_format), w))
    assert not kernels.dense_preferred(1, 1, 1 << 22)


def test_dense_gemm_refuses_what_it_does_not_take(gpu):
    from neuropress_amd import kernels

    x, w = torch.zeros(4, 96, dtype=torch.half, device=gpu), torch.zeros(8, 96, dtype=torch.half, device=gpu)
    with pytest.raises(RuntimeError, match="multiple of 64"):
        kernels.dense_linear(x, w)
    assert not kernels.dense_preferred(4, 8, 96) and not kernels.dense_preferred(4096, 14336, 4096)
    assert kernels.dense_preferred(171, 256, 640)
