"""The table GEMM, in which the blocks entry ends past a few dozen tokens: every tile at its edges -- token counts around whole tiles, rows of
8, 12 and 16 bits, tables from one row to 4096, K of one step up to several turns per wave, an odd number of them, rows of x
that end inside the last -- against the decoded weight in float64."""

import pytest
import torch

from neuropress_amd.transforms.vq_packing import IndexPacking
from tests import cases

TILES = ((32, 8), (64, 8), (64, 4), (96, 4), (128, 4))  # rows, waves


def test_every_tile_is_the_best_somewhere():
    from neuropress_amd import _lib

    plan = _lib.load().npamd_diag_table_tile
    found = {plan(m, n, k, rows) for m in (32, 64, 256, 384, 512) for n in (512, 4096, 8192) for k in (256, 4096) for rows in (256, 4096)}
    assert found == set(range(len(TILES)))
    for m, n, k, rows in ((16, 512, 512, 256), (64, 512, 500, 256), (64, 512, 512, 4097), (64, 0, 512, 256), (64, 512, 0, 256)):
        assert plan(m, n, k, rows) == -1


def test_switched_off_it_is_not_what_the_band_line_counts_on(monkeypatch):
    """The line that sends calls to the blocks entry and the entry itself ask the same plan."""
    from neuropress_amd import _lib

    lib = _lib.load()
    large = ((384, 14336, 14336, 4096), (256, 9856, 12544, 256), (1024, 4096, 4096, 1000))
    assert all(lib.npamd_gemv_blocks_preferred(m, n, k, 0, rows, 0, 1) == 1 for m, n, k, rows in large)
    with monkeypatch.context() as mp:
        mp.setenv("NPAMD_TABLE_TILE", "-1")
        lib.npamd_diag_reload_tuning()
        off = [(lib.npamd_gemv_blocks_preferred(m, n, k, 0, rows, 0, 1), lib.npamd_diag_table_tile(m, n, k, rows)) for m, n, k, rows in large]
    lib.npamd_diag_reload_tuning()
    assert off == [(0, -1)] * len(large)


def test_staging_and_the_band_are_two_questions(monkeypatch):
    """Past 16 tokens layers whose table LDS holds stage their activations, and do not stay ahead of the tile GEMM at any K for it."""
    from neuropress_amd import _lib, kernels

    lib = _lib.load()
    for m, n, k, nc, stages, ahead in ((24, 4096, 4096, 4096, 1, 0), (32, 2048, 8192, 256, 1, 0), (24, 4096, 4096, 65536, 1, 1), (2, 14336, 4096, 65536, 0, 0),
                                       (16, 4096, 4096, 4096, 1, 1), (24, 4096, 4096, 0, 1, 1)):
        asked = lib.npamd_gemv_stages_activations(m, n, k, nc), lib.npamd_gemv_ahead_of_tile(m, n, k, nc)
        assert asked == (stages, ahead), (m, n, k, nc, asked)
        assert kernels.gemv_stages_activations(m, n, k, nc) == bool(ahead)
    with monkeypatch.context() as mp:
        mp.setenv("NPAMD_GEMV_XSTAGE", "0")
        lib.npamd_diag_reload_tuning()
        assert lib.npamd_gemv_stages_activations(24, 4096, 4096, 4096) == 0


@pytest.fixture(params=range(1, len(TILES) + 1))
def forced(request, monkeypatch):
    from neuropress_amd import _lib

    lib = _lib.load()
    with monkeypatch.context() as mp:
        mp.setenv("NPAMD_TABLE_TILE", str(request.param))
        lib.npamd_diag_reload_tuning()
        yield TILES[request.param - 1][0]
    lib.npamd_diag_reload_tuning()


@pytest.mark.gpu
def test_tiles(gpu, forced):
    from neuropress_amd import _lib, kernels

    rows = forced
    shapes = ((259, 64, 0), (64, 128, 56), (300, 192, 0), (256, 2112, 8), (65, 1088, 40), (130, 4096 + 64, 24))
    for act in (torch.float16, torch.bfloat16):
        for nc, bits in ((1, 8), (200, 8), (1000, 16), (4096, 12), (4096, 16)):
            g = cases.gen(nc + bits)
            cb = (torch.randn(nc, 8, generator=g) * 0.05).to(act).to(gpu)
            for n, k, short in shapes:
                idx = torch.randint(0, nc, (n, k // 8), generator=g)
                packed = IndexPacking.pack(idx.reshape(-1), bits).to(gpu)
                w = cb[idx.to(gpu)].reshape(n, k)[:, : k - short].double()
                bias = torch.randn(n, generator=g).to(gpu) if n % 2 else None
                for m in (17, rows - 1, rows, rows + 1, 2 * rows + 33):
                    x = torch.full((m, k + 16), float("nan"), dtype=act)
                    x[:, : k - short] = torch.randn(m, k - short, generator=g).to(act)  # what lies behind a row counts for nothing
                    x = x.to(gpu)[:, : k - short]
                    y = kernels.vq_linear_blocks(x, packed, cb, bits, n, bias, width=k).double()
                    assert TILES[_lib.load().npamd_diag_last_table_tile()][0] == rows  # not the GEMV, which would be as right
                    xd = x.double()
                    ref, size = xd @ w.T, xd.abs() @ w.abs().T
                    if bias is not None:
                        ref, size = ref + bias.double(), size + bias.double().abs()
                    # one rounding of the output, and f32 sums of K products in some order
                    bound = ref.abs() * (2.0**-10 if act == torch.float16 else 2.0**-7) + size * k * 2.0**-24 + 2.0**-24
                    assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,nc", [(4096, 12544, 256), (1100, 2040, 4096)])
def test_17_to_32_tokens_run_one_kernel_on_every_way(gpu, n, k, nc):
    """Long or ragged rows, where the blocks entry serves as few tokens as the GEMV: planned, first, with rows at odd addresses and captured calls give the
    same bits, those of the entry itself."""
    from neuropress_amd import kernels
    from neuropress_amd.nn import NPVQLinear, VQProxy

    L = cases.vq_layer(n, n, k, nc)
    layer = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, 8, "cuda_wmma").to(gpu)
    for m in (24, 32):
        base = torch.randn(m, k + 3, generator=cases.gen(m)).half().to(gpu)
        x = base[:, :k].contiguous()
        stream, bits = layer._kernel_stream()
        expect = kernels.vq_linear_blocks(x, stream, layer.proxy.centroids, bits, n, width=layer._kernel_k())
        for given in (x, x, base[:, :k], base[:, :k]):
            assert torch.equal(layer(given), expect)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = layer(x)
        for _ in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, expect)
