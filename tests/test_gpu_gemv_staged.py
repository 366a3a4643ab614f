"""Activations of the VQ GEMV staged through LDS, as many tokens as there are: the same bits as operands straight from memory
(same products in the same order) with the codebook in LDS or in memory, one and two row tiles, K in parts over the
columns of a tile, odd token counts, ragged K, rows of x at a stride."""

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture
def staged(monkeypatch):
    from neuropress_amd import _lib

    def force(mode):
        monkeypatch.setenv("NPAMD_GEMV_XSTAGE", str(mode))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.undo()
    _lib.load().npamd_diag_reload_tuning()


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nc,bits", [(256, 8), (4096, 12), (65536, 16)])
def test_staged_activations(gpu, staged, nc, bits, act):
    from neuropress_amd import _lib, kernels

    g = cases.gen(nc)
    cb = (torch.randn(nc, 8, generator=g) * 0.05).to(act).to(gpu)
    seen = set()
    for n, k, tokens in ((4096, 64, (3, 16)), (4080, 320, (1, 5, 16)), (4096, 2176, (4, 9)), (5888, 1088, (8, 9, 13, 16)), (3088, 8512, (1, 2)),
                         (256, 512, (3, 8)), (1024, 2240, (2, 4)), (4100, 576, (17, 31))):  # fmt: skip
        packed = torch.randint(0, 256, (n * (k // 8) * bits // 8,), generator=g, dtype=torch.uint8).to(gpu)
        for m in tokens:
            x = torch.randn(m, k + 64, generator=g).to(act).to(gpu)[:, :k]
            out = []
            for mode in (0, 1, 2):
                staged(mode)
                out.append(kernels.vq_linear(x, packed, cb, bits, 8, None, n))
                if mode == 1:
                    seen.add(_lib.load().npamd_diag_last_gemv_staged())
            assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2]), (n, k, m)
    assert seen == {0, 1}


def test_staged_activations_with_fewer_waves(gpu, staged):
    """4096 x 14336 at 16 tokens: LDS does not hold the areas of all waves next to the table, so fewer of them walk more steps."""
    from neuropress_amd import kernels

    g = cases.gen(7)
    n, k, m = 4096, 14336, 16
    cb = (torch.randn(4096, 8, generator=g) * 0.05).half().to(gpu)
    packed = torch.randint(0, 256, (n * (k // 8) * 12 // 8,), generator=g, dtype=torch.uint8).to(gpu)
    x = torch.randn(m, k, generator=g).half().to(gpu)
    staged(0)
    plain = kernels.vq_linear(x, packed, cb, 12, 8, None, n).double()
    staged(1)
    y = kernels.vq_linear(x, packed, cb, 12, 8, None, n).double()
    # two orders of f32 sums of k products, each rounded to fp16
    assert bool(((y - plain).abs() <= 2.0 ** -10 * plain.abs() + 1e-3).all())


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", ["none", "scale", "both"])
def test_residual_index_lines(gpu, staged, rows, act):
    """Residual layers of one row tile per block load their indices four lanes to a row and turn them through LDS: rows and K
    around the tiles, with the activations straight from memory and staged, against the decoded weight."""
    from neuropress_amd import kernels

    g = cases.gen(11)
    cb, cr = ((torch.randn(c, 8, generator=g) * 0.05).half().to(gpu) for c in (5000, 256))
    for n, k, m in ((3073, 64, 1), (3088, 320, 2), (4099, 2240, 1), (40, 576, 9), (3100, 448, 16), (17, 1088, 31)):
        idx = torch.randint(0, 5000, (n * k // 8,), generator=g)
        main = idx.to(torch.int16).view(torch.uint8).to(gpu)
        res = torch.randint(0, 256, (n * k // 8,), generator=g, dtype=torch.uint8).to(gpu)
        scale = (torch.rand(n, generator=g) + 0.5).half().to(gpu) if rows != "none" else None
        bias = (torch.randn(n, generator=g) * 0.01).half().to(gpu) if rows == "both" else None
        x = torch.randn(m, k, generator=g).to(act).to(gpu)
        w = cb.cpu()[idx].view(n, k) + cr.cpu()[res.cpu().long()].view(n, k)  # each step rounded to fp16, as the format has it
        if scale is not None:
            w = w * scale.cpu()[:, None]
        if bias is not None:
            w = w + bias.cpu()[:, None]
        w = w.to(act).double()
        ref = x.double().cpu() @ w.T
        tol = 2.0 ** (-10 if act == torch.float16 else -7)  # the rounding of the output; f32 sums of k products
        slack = 2.0 ** -22 * (x.double().cpu().abs() @ w.abs().T)
        for mode in (0, 2):
            staged(mode)
            y = kernels.rvq_linear(x, main, 16, res, 8, cb, cr, scale, bias, n).double().cpu()
            assert bool(((y - ref).abs() <= tol * ref.abs() + slack + 1e-6).all()), (n, k, m, mode)
