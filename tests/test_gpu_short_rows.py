"""Rows that end inside the last 64 columns, read where they lie: the dense product on every tile and with K split over blocks, and
residual layers of such a K in every band; against float64."""

import pytest
import torch

import neuropress_amd.nn.np_vq_linear as vqmod
from neuropress_amd.nn import NPVQLinear, VQProxy
from neuropress_amd.transforms.vq_packing import IndexPacking
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture
def dense(monkeypatch):
    from neuropress_amd import _lib

    def force(tile, splits):
        monkeypatch.setenv("NPAMD_DENSE_TILE", str(tile))
        monkeypatch.setenv("NPAMD_DENSE_SPLITS", str(splits))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.undo()
    _lib.load().npamd_diag_reload_tuning()


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [0, *cases.DENSE_TILES])
def test_dense_product(gpu, dense, tile, act):
    from neuropress_amd import kernels

    for splits in (0, 1, 3) if tile else (0,):
        dense(tile, splits)
        for m, n, k in ((1, 3, 8), (33, 70, 56), (130, 257, 72), (300, 130, 584), (77, 301, 2184), (65, 65, 320), (260, 390, 1336)):
            g = cases.gen(m + k)
            x = torch.randn(m, k + 40, generator=g).to(act).to(gpu)[:, :k]
            w = (torch.randn(n, k, generator=g) * 0.05).to(act).to(gpu)
            w[:, -1] = w[:, -1].abs() + 0.01
            x[m // 2, -1] = float("inf")  # past the end of K the last pieces come again: they must not count
            bias = torch.randn(n, generator=g).to(gpu)
            y = kernels.dense_linear(x, w, bias, ragged=True).double()
            ref, size = x.double() @ w.double().T + bias.double(), x.double().abs() @ w.double().abs().T + bias.double().abs()
            assert bool((y[m // 2] == float("inf")).all())
            rows = torch.arange(m, device=gpu) != m // 2
            bound = ref.abs() * (2.0**-10 if act == torch.float16 else 2.0**-7) + size * k * 2.0**-24 + 2.0**-24  # a rounding and f32 sums
            assert bool(((y - ref).abs() <= bound)[rows].all()), (tile, splits, m, n, k)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k,nc,ncr,perm", [(70, 8, 256, 256, False), (384, 672, 4096, 256, False), (611, 464, 65536, 256, True),
                                             (1157, 272, 4096, 3000, False), (300, 2184, 1000, 16, True)])  # fmt: skip
def test_residual_layers(gpu, n, k, nc, ncr, perm, act):
    L = cases.rvq_layer(n + k, n, k, nc, ncr, zipf=False)
    cp = torch.randperm(k, generator=cases.gen(k)) if perm else None
    bias = torch.randn(n, generator=cases.gen(n))
    layer = NPVQLinear(VQProxy(L["cbm"]).to(gpu), L["pm"], L["bm"], n, k, 8, "cuda_wmma", bias=bias, column_perm=cp,
                       residual_proxy=VQProxy(L["cbr"]).to(gpu), packed_residual=L["pr"], residual_bits=L["br"],
                       row_scale=L["scale"], row_bias=L["wbias"]).to(gpu)  # fmt: skip
    w = (((L["cbm"][L["im"]] + L["cbr"][L["ir"]]).reshape(n, k) * L["scale"][:, None]) + L["wbias"][:, None]).to(act).float()
    for m in (1, 3, 17, 40, 100, 400, 1100):
        base = torch.randn(m, k + 3, generator=cases.gen(m)).to(act)
        x = base[:, :k].contiguous()
        ref = torch.nn.functional.linear((x if cp is None else x[:, cp]).float(), w, bias)
        for given in (x.to(gpu), x.to(gpu), base.to(gpu)[:, :k]):  # the first call, the planned one, rows at odd addresses
            err = (layer(given).float().cpu() - ref).abs()
            assert bool((err <= 1e-2 + 1e-2 * ref.abs()).all()), (m, float(err.max()))
        lead = layer(x.to(gpu).reshape(1, m, k))
        assert lead.shape == (1, m, n)
        xg = x.to(gpu).requires_grad_()
        layer(xg).sum().backward()  # followed by torch: the library's product
        assert torch.isfinite(xg.grad).all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("perm", [False, True])
def test_unused_rows_of_a_residual_codebook_count_for_nothing(gpu, perm, bad, monkeypatch):
    """Row 0 of the residual codebook is not finite and no index names it (what a cluster without members leaves behind): rows of x read where
    they lie, copied for a permutation or from odd addresses, and past 32 tokens with the GEMV's band raised."""
    monkeypatch.setattr(vqmod, "_FUSED_MAX_TOKENS", 64)
    n, k, bias = 96, 200, torch.randn(96, generator=cases.gen(1))
    L = cases.rvq_layer(5, n, k, 4096, 256, zipf=False)
    ir = L["ir"].clamp(min=1)
    L["cbr"][0] = bad
    cp = torch.randperm(k, generator=cases.gen(k)) if perm else None
    layer = NPVQLinear(VQProxy(L["cbm"]).to(gpu), L["pm"], L["bm"], n, k, 8, "cuda_wmma", bias=bias, column_perm=cp,
                       residual_proxy=VQProxy(L["cbr"]).to(gpu), packed_residual=IndexPacking.pack(ir, L["br"]), residual_bits=L["br"],
                       row_scale=L["scale"], row_bias=L["wbias"]).to(gpu)  # fmt: skip
    w = ((L["cbm"][L["im"]] + L["cbr"][ir]).reshape(n, k) * L["scale"][:, None] + L["wbias"][:, None]).float()
    for m in (1, 5, 20, 40):
        base = torch.randn(m, k + 3, generator=cases.gen(m)).half()
        x = base[:, :k].contiguous()
        ref = torch.nn.functional.linear((x if cp is None else x[:, cp]).float(), w, bias)
        for given in (x.to(gpu), x.to(gpu), base.to(gpu)[:, :k], base.to(gpu)[:, :k]):  # the first call, the planned one, rows at odd addresses
            err = (layer(given).float().cpu() - ref).abs()
            assert bool((err <= 1e-2 + 1e-2 * ref.abs()).all()), (m, float(err.max()))


@pytest.mark.parametrize("k,nc,ncr,tokens", [(200, 65536, 0, (3, 24)), (200, 4096, 256, (3, 24)), (204, 1000, 0, (3, 24)), (2184, 65536, 0, (40,))])
def test_a_planned_call_keeps_the_gradient_of_the_bias(gpu, k, nc, ncr, tokens, monkeypatch):
    """A layer planned where no gradient was asked for, and called again where the bias asks for one: as without a plan, the library's
    product, which carries it.  Vector length 8 and 4, residual layers, the GEMV's band and the tile GEMM's."""
    monkeypatch.setattr(vqmod, "_TILE_MIN_GRID_FRACTION", 0.0)
    n, vl = 96, 4 if k % 8 else 8
    L = cases.rvq_layer(5, n, k, nc, ncr, zipf=False) if ncr else cases.vq_layer(n, n, k, nc, vl=vl)
    more = dict(residual_proxy=VQProxy(L["cbr"]).to(gpu), packed_residual=L["pr"], residual_bits=L["br"], row_scale=L["scale"],
                row_bias=L["wbias"]) if ncr else {}  # fmt: skip
    cb, packed, bits = (L["cbm"], L["pm"], L["bm"]) if ncr else (L["cb"], L["packed"], L["bits"])
    layer = NPVQLinear(VQProxy(cb).to(gpu), packed, bits, n, k, vl, "cuda_wmma", bias=torch.zeros(n), **more).to(gpu)
    layer.bias.requires_grad_()
    for m in tokens:
        x = torch.randn(m, k, generator=cases.gen(3)).half().to(gpu)
        with torch.no_grad():
            y = layer(x)
            assert torch.equal(layer(x), y) and not y.requires_grad
        y = layer(x)
        assert y.requires_grad
        y.float().sum().backward()
        assert torch.equal(layer.bias.grad, torch.full_like(layer.bias, m))
        layer.bias.grad = None


@pytest.mark.parametrize("rows", [1, 2, 4])
def test_row_tiles_asked_for(gpu, monkeypatch, rows):
    """NPAMD_GEMV_R asks for more row tiles per block than the kernels that look where a row ends have: such layers run with what those have."""
    from neuropress_amd import _lib, kernels

    monkeypatch.setenv("NPAMD_GEMV_R", str(rows))
    _lib.load().npamd_diag_reload_tuning()
    n, k, width = 200, 552, 576
    for nc, bits in ((256, 8), (4096, 12), (65536, 16)):
        g = cases.gen(nc + rows)
        cb = (torch.randn(nc, 8, generator=g) * 0.05).half().to(gpu)
        idx = torch.randint(0, nc, (n, width // 8), generator=g)
        packed, w = IndexPacking.pack(idx.reshape(-1), bits).to(gpu), cb[idx.to(gpu)].reshape(n, width)[:, :k]
        for m in (1, 5, 16, 29, 70):
            x = torch.randn(m, k, generator=g).half().to(gpu)
            _close(kernels.vq_linear_blocks(x, packed, cb, bits, n, width=width), x, w)
    for ncr in (256, 65536):
        L = cases.rvq_layer(ncr + rows, n, width, 65536, ncr, zipf=False)
        pm, pr, cm, cr, sc, rb = (L[name].to(gpu) for name in ("pm", "pr", "cbm", "cbr", "scale", "wbias"))
        w = kernels.rvq_dequant(pm, L["bm"], pr, L["br"], cm, cr, sc, rb, n, width, torch.float16)[:, :k]
        for m in (1, 5, 16, 29, 70):
            x = torch.randn(m, k, generator=cases.gen(m)).half().to(gpu)
            _close(kernels.rvq_linear_blocks(x, pm, L["bm"], pr, L["br"], cm, cr, sc, rb, n, width=width), x, w)


def _close(y, x, w):
    """One rounding of the output and f32 sums of K products in some order."""
    ref, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert bool(((y.double() - ref).abs() <= ref.abs() * 2.0**-10 + size * w.shape[1] * 2.0**-24 + 2.0**-24).all())
