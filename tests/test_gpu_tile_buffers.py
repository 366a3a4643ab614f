"""The tile GEMM with two x tiles in LDS (129 to 256 tokens next to a table, more than 256 in any case), on rows long enough for reads and transfers to meet:
every call against the decoded weight in float64."""

import pytest
import torch

from neuropress_amd.transforms.vq_packing import IndexPacking
from tests import cases

pytestmark = pytest.mark.gpu


def _calls(fn, x, w, calls):
    ref, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = ref.abs() * 2.0**-10 + size * w.shape[1] * 2.0**-24 + 2.0**-24  # one rounding of the output and f32 sums
    for _ in range(calls):
        assert bool(((fn().double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("n,k,m,nc,bits", [(7494, 13568, 163, 4096, 12), (2593, 9984, 165, 4096, 12), (4955, 8192, 158, 4096, 16), (5000, 8192, 250, 1500, 16),
                                           (7494, 13568, 300, 256, 8), (3000, 9984, 384, 4096, 12)])  # fmt: skip
def test_vq(gpu, n, k, m, nc, bits):
    from neuropress_amd import kernels

    g = cases.gen(n)
    cb = (torch.randn(nc, 8, generator=g) * 0.02).half().to(gpu)
    idx = torch.randint(0, nc, (n * (k // 8),), generator=g)
    packed = IndexPacking.pack(idx, bits).to(gpu)
    w = cb[idx.to(gpu)].reshape(n, k)
    x = torch.randn(m, k, generator=g).half().to(gpu)
    _calls(lambda: kernels.vq_gemm_tile(x, packed, cb, bits, n), x, w, 8)


@pytest.mark.parametrize("m", [270, 384])
def test_residual_and_int4(gpu, m):
    from neuropress_amd import kernels

    n, k = 3000, 8192
    R, Q = cases.rvq_layer(7, n, k, zipf=False), cases.q4_layer(8, n, k)
    x = torch.randn(m, k, generator=cases.gen(m)).half().to(gpu)
    rvq = [R[name].to(gpu) for name in ("pm", "pr", "cbm", "cbr", "scale", "wbias")]
    pm, pr, cm, cr, sc, rb = rvq
    w = kernels.rvq_dequant(pm, R["bm"], pr, R["br"], cm, cr, sc, rb, n, k, torch.float16)
    _calls(lambda: kernels.rvq_linear(x, pm, R["bm"], pr, R["br"], cm, cr, sc, rb, n, None, tile=True), x, w, 6)
    blob, scale = Q["blob"].to(gpu), Q["scale"].to(gpu)
    _calls(lambda: kernels.q_gemm_tile(x, blob, scale, 4, 32), x, kernels.q_dequant(blob, scale, 4, 32, None, torch.float16), 6)
