"""Layers whose K is not a whole number of 64-column chunks: the index stream is padded once, the activations per
call (together with the column permutation), and every band then computes with zeros past K."""

import pytest
import torch

import neuropress_amd.nn.np_vq_linear as vqmod
from neuropress_amd.nn import NPVQLinear, VQProxy
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [0, 8, 24])
@pytest.mark.parametrize("k", [8, 40, 1000, 2184, 33000])
def test_gather_columns(gpu, k, width):
    from neuropress_amd import kernels

    g = cases.gen(k)
    wide = (k + 7) // 8 * 8 + width
    big = torch.randn(3, k + 5, generator=g).half().to(gpu)
    perm = torch.randperm(k, generator=g).to(gpu)
    for x in (big[:, :k].contiguous(), big[:, 5:]):  # 16-byte aligned rows, and rows that are not
        for p in (None, perm):
            out = kernels.gather_columns(x, None if p is None else p.int(), wide)
            assert torch.equal(out[:, :k], x if p is None else x[:, p]) and not out[:, k:].any()


@pytest.mark.parametrize("rows", [255, 400, 600, 1023, 1025])
@pytest.mark.parametrize("k", [40, 2056, 5003, 16384, 16392, 32768])
def test_gather_columns_of_many_rows(gpu, k, rows):
    """Whole rows per block, and two rows per block where LDS holds them: an odd last row, rows around the LDS limits."""
    from neuropress_amd import kernels

    g = torch.Generator(device=gpu).manual_seed(k)
    x = torch.randint(-30000, 30000, (rows, k), generator=g, device=gpu, dtype=torch.int16).view(torch.half)
    big = torch.zeros(k + 4, dtype=torch.int32, device=gpu)
    big[1 : k + 1] = torch.randperm(k, generator=g, device=gpu)
    for perm in (big[1 : k + 1].clone(), big[1 : k + 1]):  # 16-byte aligned, and not
        out = kernels.gather_columns(x, perm, (k + 63) // 64 * 64)
        assert torch.equal(out[:, :k].view(torch.int16), x.view(torch.int16)[:, perm.long()]) and not out[:, k:].any()


@pytest.mark.parametrize("rows,k", [(3, 40), (1025, 40), (3, 33000)])
def test_gather_columns_reads_only_columns_that_exist(gpu, rows, k):
    from neuropress_amd import kernels

    x = torch.randn(rows, k, generator=cases.gen(k)).half().to(gpu)
    perm = torch.arange(k, dtype=torch.int32)
    perm[[0, 9, 17, 30, k - 1]] = torch.tensor([k, -1, -(2**31), 2**31 - 1, k + 8], dtype=torch.int32)
    out = kernels.gather_columns(x, perm.to(gpu), (k + 7) // 8 * 8)
    there = ((perm >= 0) & (perm < k)).to(gpu)
    assert torch.equal(out[:, :k][:, there], x[:, there]) and not out[:, :k][:, ~there].any()


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k,nc,vl,perm", [(70, 8, 16, 8, False), (130, 200, 1000, 8, True), (257, 1000, 4096, 4, False),
                                            (64, 2184, 65536, 8, True), (96, 1544, 300, 8, False)])  # fmt: skip
def test_ragged_k_runs_the_fused_bands(gpu, n, k, nc, vl, perm, act, monkeypatch):
    from neuropress_amd import kernels

    monkeypatch.setattr(vqmod, "_TILE_MIN_GRID_FRACTION", 0.0)  # small layers: force the tile band
    monkeypatch.setattr(vqmod, "_TILE_WIDE_SMALL_MAX_TOKENS", 128)
    L = cases.vq_layer(n + k, n, k, nc, vl=vl, bias=True, act=act, std=0.05)
    cp = torch.randperm(k, generator=cases.gen(k)) if perm else None
    layer = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, vl, "cuda_wmma", bias=L["bias"].float(),
                       column_perm=cp).to(gpu)  # fmt: skip
    w = L["cb"][L["idx"]].reshape(n, k).to(act).float()
    used = []
    for m in (1, 3, 17, 40, 100, 400):
        x = torch.randn(m, k, generator=cases.gen(m)).to(act)
        ref = torch.nn.functional.linear((x if cp is None else x[:, cp]).float(), w, L["bias"].float())
        for call in range(2):  # the first call and the planned one
            y = layer(x.to(gpu)).float().cpu()
            err = (y - ref).abs()
            assert bool((err <= 1e-2 + 1e-2 * ref.abs()).all()), (m, call, float(err.max()))
        # rows of x with a stride, and the wrappers in place of the plan
        with monkeypatch.context() as mp:
            for name in ("vq_linear", "vq_gemm_tile"):
                real = getattr(kernels, name)
                mp.setattr(kernels, name, lambda *a, _r=real, _n=name, **kw: (used.append((m, _n)), _r(*a, **kw))[1])
            xs = torch.zeros(m, k + 3, dtype=act)
            xs[:, :k] = x
            y2 = layer(xs.to(gpu)[:, :k]).float().cpu()
            assert bool(((y2 - ref).abs() <= 1e-2 + 1e-2 * ref.abs()).all()), m
    assert used == [(1, "vq_linear"), (3, "vq_linear"), (17, "vq_linear"), (40, "vq_gemm_tile"), (100, "vq_gemm_tile")]


@pytest.mark.parametrize("nc,bad", [(1000, (0, 1, 999)), (65536, (0, 65535)), (40000, tuple(range(39000)))])
def test_infinities_in_the_codebook_stay_what_they_are(gpu, nc, bad, monkeypatch):
    """Padded columns multiply zeros with a finite codebook row, so that an infinite output does not turn into NaN."""
    monkeypatch.setattr(vqmod, "_TILE_MIN_GRID_FRACTION", 0.0)
    monkeypatch.setattr(vqmod, "_TILE_WIDE_SMALL_MAX_TOKENS", 128)
    monkeypatch.setattr(vqmod, "_TILE_WIDE_TINY_WEIGHTS", 0)
    n, k = 70, 200
    L = cases.vq_layer(nc, n, k, nc, bits=16, std=0.05)
    idx = torch.randint(max(bad) + 1 if len(bad) > 3 else 2, nc - 1, (n, k // 8), generator=cases.gen(1))
    idx[0, -1], idx[3, 2], idx[69, -1] = bad[0], bad[-1], bad[1]
    L["cb"][list(bad), 3] = float("inf")
    layer = NPVQLinear(VQProxy(torch.zeros_like(L["cb"])).to(gpu), vqmod.IndexPacking.pack(idx.reshape(-1), 16), 16, n, k, 8, "cuda_wmma").to(gpu)
    layer(torch.zeros(3, k, dtype=torch.half, device=gpu))
    layer.proxy.centroids.copy_(L["cb"])  # written in place: another row may be the finite one
    w = L["cb"][idx].reshape(n, k).float()
    for m in (3, 40, 400):
        x = torch.randn(m, k, generator=cases.gen(m)).half()
        ref = torch.nn.functional.linear(x.float(), w)
        for call in range(2):
            y = layer(x.to(gpu)).float().cpu()
            assert torch.equal(y[:, [0, 3, 69]], ref[:, [0, 3, 69]]) and bool(torch.isinf(ref[:, [0, 3, 69]]).all()), (m, call)
            fine = torch.isfinite(ref)
            assert bool(((y - ref)[fine].abs() <= 1e-2 + 1e-2 * ref[fine].abs()).all()), (m, call)


def test_layers_prepare_before_their_codebook_arrives(gpu):
    L = cases.vq_layer(3, 70, 200, 1000, std=0.05)
    proxy = VQProxy(L["cb"])
    layer = NPVQLinear(proxy, L["packed"], L["bits"], 70, 200, 8, "cuda_wmma").to(gpu)
    layer.prepare()
    proxy.to(gpu)
    x = torch.randn(3, 200, generator=cases.gen(1)).half()
    ref = torch.nn.functional.linear(x.float(), L["cb"][L["idx"]].reshape(70, 200).float())
    assert torch.allclose(layer(x.to(gpu)).float().cpu(), ref, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits,nc", [(8, 200), (12, 900), (16, 65536)])
@pytest.mark.parametrize("m,k,perm", [(1, 72, True), (77, 2184, True), (1023, 456, False), (300, 5000, True), (5, 8200, False), (1030, 264, True)])
def test_decode_and_gather_in_one_launch(gpu, dtype, bits, nc, m, k, perm):
    """What the one launch writes is what the decode and the gather write one after the other: rows shorter and longer than a
    block's 2048 columns, one and many, rows at a distance, the most rows it takes and more (the two calls), a weight of a
    ragged number of vectors."""
    from neuropress_amd import _lib, kernels
    from neuropress_amd.transforms.vq_packing import IndexPacking

    n, width = 37, (k + 63) // 64 * 64
    g = torch.Generator().manual_seed(m + k + bits)
    packed = IndexPacking.pack(torch.randint(0, nc, (n * width // 8,), generator=g), bits).to(gpu)
    cb = torch.randn(nc, 8, generator=g).half().to(gpu)
    x = torch.randn(m, k + 8, generator=g).to(dtype).to(gpu)[:, :k]
    p = torch.randperm(k, generator=g).int().to(gpu) if perm else None
    w = torch.full((n, width), 7.0, dtype=dtype, device=gpu)
    out = torch.full((m, width), 7.0, dtype=dtype, device=gpu)
    code = _lib.F16 if dtype == torch.float16 else _lib.BF16
    _lib.call("npamd_vq_dequant_gather", packed.data_ptr(), packed.numel(), bits, cb.data_ptr(), nc, 8, n * width // 8, w.data_ptr(), code,
              x.data_ptr(), x.stride(0), p.data_ptr() if perm else None, out.data_ptr(), width, m, k,
              torch.cuda.current_stream().cuda_stream)  # fmt: skip
    assert torch.equal(w, kernels.vq_dequant(packed, cb, bits, n, width, dtype))
    assert torch.equal(out, kernels.gather_columns(x, p, width))


@pytest.mark.parametrize("bits,nc,n", [(8, 200, 1024), (8, 200, 1025), (16, 65536, 2048), (16, 65536, 2049)])
@pytest.mark.parametrize("k", [16384, 16380])
def test_decode_and_gather_on_both_sides_of_the_line_for_long_rows(gpu, bits, nc, n, k):
    """The longest rows the one launch takes, layers up to its line and one row past it (the two calls): the same bytes."""
    from neuropress_amd import _lib, kernels
    from neuropress_amd.transforms.vq_packing import IndexPacking

    m, width = 5, 16384
    assert _lib.load().npamd_diag_gather_fits_decode(bits, n * width // 8, k, 1) == (n in (1024, 2048))
    g = torch.Generator().manual_seed(n + k)
    packed = IndexPacking.pack(torch.randint(0, nc, (n * width // 8,), generator=g), bits).to(gpu)
    cb = torch.randn(nc, 8, generator=g).half().to(gpu)
    x = torch.randn(m, k, generator=g).half().to(gpu)
    p = torch.randperm(k, generator=g).int().to(gpu)
    w = torch.full((n, width), 7.0, dtype=torch.half, device=gpu)
    out = torch.full((m, width), 7.0, dtype=torch.half, device=gpu)
    _lib.call("npamd_vq_dequant_gather", packed.data_ptr(), packed.numel(), bits, cb.data_ptr(), nc, 8, n * width // 8, w.data_ptr(),
              _lib.F16, x.data_ptr(), x.stride(0), p.data_ptr(), out.data_ptr(), width, m, k,
              torch.cuda.current_stream().cuda_stream)  # fmt: skip
    assert torch.equal(w, kernels.vq_dequant(packed, cb, bits, n, width, torch.half))
    assert torch.equal(out, kernels.gather_columns(x, p, width))
