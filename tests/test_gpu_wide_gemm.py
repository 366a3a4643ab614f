"""The wide tiles of the dense product around their edges: rows and columns one off a tile, fewer steps of K than a ring is deep, rows that
end inside a step, columns that leave as whole pieces and one by one, K in parts whose sums are stored either way."""

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

TILES = {number: tile for number, tile in cases.DENSE_TILES.items() if number not in (1, 15)}  # those are the other kernel's


@pytest.fixture
def tuned(monkeypatch):
    from neuropress_amd import _lib

    def force(tile, splits):
        monkeypatch.setenv("NPAMD_DENSE_TILE", str(tile))
        monkeypatch.setenv("NPAMD_DENSE_SPLITS", str(splits))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    for name in ("NPAMD_DENSE_TILE", "NPAMD_DENSE_SPLITS"):
        monkeypatch.delenv(name, raising=False)
    _lib.load().npamd_diag_reload_tuning()


def check(gpu, m, n, k, act, what):
    from neuropress_amd import kernels

    g = cases.gen(m + n + k)
    x = torch.randn(m, k, generator=g).to(act)
    w = (torch.randn(n, k, generator=g) * 0.05).to(act)
    bias = torch.randn(n, generator=g)
    y = kernels.dense_linear(x.to(gpu), w.to(gpu), bias.to(gpu), ragged=k % 64 != 0).double().cpu()
    ref, size = x.double() @ w.double().T + bias.double(), x.double().abs() @ w.double().abs().T + bias.double().abs()
    tol = ref.abs() * 2.0 ** (-10 if act == torch.float16 else -7) + size * k * 2.0**-24  # the rounding of the output, and f32 sums
    assert bool(((y - ref).abs() <= tol).all()), (what, m, n, k, float((y - ref).abs().max()))


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", sorted(TILES))
def test_edges(gpu, tuned, tile, act):
    bm, bn = TILES[tile]
    tuned(tile, 1)
    for m, n, k in ((1, 8, 64), (bm - 1, bn, 128), (bm, bn - 8, 192), (bm + 1, bn + 1, 256), (2 * bm + 15, bn + 8, 320), (bm, 2 * bn + 3, 384),
                    (33, bn - 1, 448), (4 * bm + 1, 24, 512)):  # fmt: skip
        check(gpu, m, n, k, act, tile)
    for k in (8, 56, 72, 136, 200, 264, 328, 392, 456, 520):  # rows that end inside the first to the ninth step
        check(gpu, bm + 3, bn // 2 + 8, k, act, tile)


@pytest.mark.parametrize("tile", sorted(TILES))
def test_parts_of_k(gpu, tuned, tile):
    tuned(tile, 3)
    for m, n, k in ((70, 132, 192), (70, 133, 704), (TILES[tile][0] + 1, 40, 1160), (5, 9, 584)):
        check(gpu, m, n, k, torch.bfloat16, tile)


def test_rows_past_a_product(gpu, tuned):
    """Only the result is written: what lies around it stays, also where its tiles reach past it on both sides."""
    from neuropress_amd import _lib

    lib = _lib.load()
    for tile, (bm, bn) in TILES.items():
        tuned(tile, 1)
        for n, ldy in ((bn - 8, bn + 16), (bn - 3, bn + 5)):
            m, k = bm - 5, 128
            x = torch.randn(m, k, generator=cases.gen(1)).half().to(gpu)
            w = (torch.randn(n, k, generator=cases.gen(2)) * 0.05).half().to(gpu)
            y = torch.full((m + 40, ldy), 7.0, device=gpu, dtype=torch.half)
            assert lib.npamd_dense_gemm(x.data_ptr(), k, w.data_ptr(), k, None, y.data_ptr(), ldy, m, n, k, 0, None, 0,
                                        torch.cuda.current_stream().cuda_stream) == 0  # fmt: skip
            assert torch.allclose(y[:m, :n].float(), x.float() @ w.float().T, rtol=2e-3, atol=2e-3)
            assert bool((y[m:] == 7).all()) and bool((y[:, n:] == 7).all()), (tile, n)


def large(gpu, m, n, k, act, what):
    """As `check`, on the GPU in float64."""
    from neuropress_amd import kernels

    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=gpu).to(act)
    w = (torch.randn(n, k, generator=g, device=gpu) * 0.05).to(act)
    y = kernels.dense_linear(x, w).double()
    ref, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    tol = ref.abs() * 2.0 ** (-10 if act == torch.float16 else -7) + size * k * 2.0**-24
    assert bool(((y - ref).abs() <= tol).all()), (what, m, n, k)


@pytest.mark.parametrize("tile", sorted(TILES))
def test_groups_of_row_tiles(gpu, tuned, tile):
    """Units are counted down the columns of groups of row tiles: several groups, the last of them not full, of several columns, whole and in
    parts of K.  Groups of 2048 rows (y not much longer than wide) and of four tiles (longer)."""
    bm, bn = TILES[tile]
    for splits in (1, 2, 3):
        tuned(tile, splits)
        large(gpu, 2048 // bm * bm * 2 + bm + 7, 3800, 256, torch.bfloat16, (tile, splits))
        large(gpu, 4 * bm * 2 + bm + 9, 2 * bn + 5, 256, torch.float16, (tile, splits))
