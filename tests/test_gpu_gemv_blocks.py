"""The fused GEMVs with a workgroup per 32 tokens: token counts around the blocks' edges, tables in LDS (one and two row tiles, large and
small) and in memory, K of one chunk up to several steps per wave, rows of x that end inside the last chunk, rows at a
stride; against the decoded weight in float64.  And the calls that lowered layers send there."""

import pytest
import torch

import neuropress_amd.nn.np_linear as qmod
import neuropress_amd.nn.np_vq_linear as vqmod
from neuropress_amd.nn import NPLinear, NPVQLinear, VQProxy
from neuropress_amd.transforms.vq_packing import IndexPacking
from tests import cases

pytestmark = pytest.mark.gpu
TOKENS = (17, 32, 33, 63, 64, 65, 130)


def _check(y, x, w, bias=None):
    """One rounding of the output, and f32 sums of K products in some order."""
    x, w = x.double(), w.double()
    ref, size = x @ w.T, x.abs() @ w.abs().T
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    bound = ref.abs() * (2.0**-10 if y.dtype == torch.float16 else 2.0**-7) + size * w.shape[1] * 2.0**-24 + 2.0**-24
    assert bool(((y.double() - ref).abs() <= bound).all())


def _rows(m, k, act, gpu, g):
    return torch.randn(m, k + 24, generator=g).to(act).to(gpu)[:, :k]


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nc,bits", [(16, 4), (256, 8), (1000, 16), (4096, 12), (65536, 16)])
def test_vq(gpu, nc, bits, act):
    from neuropress_amd import kernels

    g = cases.gen(nc)
    cb = (torch.randn(nc, 8, generator=g) * 0.05).to(act).to(gpu)
    for n, k, short in ((259, 64, 0), (256, 2112, 8), (1030, 1088, 56), (2064, 2048, 0), (300, 4224, 24), (4112, 576, 40)):
        idx = torch.randint(0, nc, (n, k // 8), generator=g)
        packed = IndexPacking.pack(idx.reshape(-1), bits).to(gpu)
        w = cb[idx.to(gpu)].reshape(n, k)[:, : k - short]
        bias = torch.randn(n, generator=g).to(gpu)
        for m in TOKENS + ((1, 3, 9, 16, 300) if short else (300,)):
            x = _rows(m, k - short, act, gpu, g)
            _check(kernels.vq_linear_blocks(x, packed, cb, bits, n, bias, width=k), x, w, bias)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nc,bits", [(256, 8), (4096, 12)])
def test_two_row_tiles_next_to_a_table_walk_several_steps(gpu, nc, bits, act, monkeypatch):
    """More row tiles than compute units and long rows, which the table GEMM takes unless it is off: each wave stages its activations again
    for every step."""
    from neuropress_amd import _lib, kernels

    lib = _lib.load()
    monkeypatch.setenv("NPAMD_TABLE_TILE", "-1")
    lib.npamd_diag_reload_tuning()
    g = cases.gen(nc)
    cb = (torch.randn(nc, 8, generator=g) * 0.05).to(act).to(gpu)
    for n, k, short in ((4112, 4096, 0), (4130, 8512, 24)):
        idx = torch.randint(0, nc, (n, k // 8), generator=g)
        packed = IndexPacking.pack(idx.reshape(-1), bits).to(gpu)
        w = cb[idx.to(gpu)].reshape(n, k)[:, : k - short]
        bias = torch.randn(n, generator=g).to(gpu)
        for m in (17, 24, 32):
            x = _rows(m, k - short, act, gpu, g)
            y = kernels.vq_linear_blocks(x, packed, cb, bits, n, bias, width=k)
            assert (lib.npamd_diag_last_table_tile(), lib.npamd_diag_last_gemv_staged()) == (-1, 1)
            _check(y, x, w, bias)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nc,ncr", [(65536, 256), (4096, 256), (65536, 65536)])
def test_residual(gpu, nc, ncr, act):
    from neuropress_amd import kernels

    for n, k, short in ((259, 64, 0), (256, 2112, 8), (1030, 1088, 56), (2064, 2048, 0), (6000, 576, 16)):
        L = cases.rvq_layer(n, n, k, nc, ncr, zipf=False)
        pm, pr, cm, cr, sc, rb = (L[name].to(gpu) for name in ("pm", "pr", "cbm", "cbr", "scale", "wbias"))
        w = kernels.rvq_dequant(pm, L["bm"], pr, L["br"], cm, cr, sc, rb, n, k, act)[:, : k - short]
        g = cases.gen(n)
        for m in TOKENS + ((1, 2, 5, 16) if short else ()):
            x = _rows(m, k - short, act, gpu, g)
            _check(kernels.rvq_linear(x, pm, L["bm"], pr, L["br"], cm, cr, sc, rb, n, width=k), x, w)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits,zero_point", [(4, False), (4, True), (8, False), (8, True)])
def test_group_quantized(gpu, bits, zero_point, act):
    from neuropress_amd import kernels

    for n, k, group in ((258, 64, 32), (256, 2112, 64), (1030, 1024, 128), (2064, 512, 32), (4112, 320, 64), (257, 192, 64)):
        L = cases.q4_layer(n + k, n, k, nbits=bits, gs=group, asym=zero_point)
        blob, sc, zp = (None if L[name] is None else L[name].to(gpu) for name in ("blob", "scale", "zp"))
        w = kernels.q_dequant(blob, sc, bits, group, zp, act)
        g = cases.gen(n)
        for m in TOKENS + (300,):
            x = _rows(m, k, act, gpu, g)
            _check(kernels.q_linear_blocks(x, blob, sc, bits, group, zp), x, w)


def test_what_the_entries_refuse(gpu):
    from neuropress_amd import kernels

    cb = torch.zeros(256, 8, dtype=torch.half, device=gpu)
    packed = torch.zeros(256 * 16, dtype=torch.uint8, device=gpu)
    x = torch.zeros(40, 128, dtype=torch.half, device=gpu)
    for columns, width in ((64, 128), (124, 128), (128, 120)):  # a whole chunk missing, no whole piece, no whole chunk
        with pytest.raises(RuntimeError):
            kernels.vq_linear_blocks(x[:, :columns].contiguous(), packed, cb, 8, 256, width=width)
    with pytest.raises(RuntimeError):
        kernels.vq_linear(x, packed, cb, 8, 8, None, 256)  # more than 32 tokens


def _layers(gpu, n, k, perm):
    L = cases.vq_layer(n + k, n, k, 1000, bias=True)
    cp = torch.randperm(k, generator=cases.gen(k)) if perm else None
    yield vqmod, "_BLOCKS_MAX_TOKENS", lambda: NPVQLinear(
        VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, 8, "cuda_wmma", bias=L["bias"].float(), column_perm=cp).to(gpu)  # fmt: skip
    if not perm:
        Q = cases.q4_layer(n + k, n, k, bias=True)
        yield qmod, "_Q_BLOCKS_MAX_TOKENS", lambda: NPLinear(
            Q["blob"], Q["scale"], n, k, 32, 4, "sym", "cuda", bias=Q["bias"].float()).to(gpu)  # fmt: skip
        R = cases.rvq_layer(n + k, n, k)
        yield vqmod, "_BLOCKS_MAX_TOKENS", lambda: NPVQLinear(
            VQProxy(R["cbm"]).to(gpu), R["pm"], R["bm"], n, k, 8, "cuda_wmma", residual_proxy=VQProxy(R["cbr"]).to(gpu),
            packed_residual=R["pr"], residual_bits=R["br"], row_scale=R["scale"], row_bias=R["wbias"]).to(gpu)  # fmt: skip


@pytest.mark.parametrize("perm", [False, True])
def test_layers_against_the_other_bands(gpu, perm, monkeypatch):
    """Layers that take the blocks, on the first call, the planned one, with rows at odd addresses and under capture, against the same
    layers without them; a bias that asks for a gradient keeps it."""
    for module, name, make in _layers(gpu, 512, 2048, perm):
        layer = make()
        for m in (40, 100):
            base = torch.randn(m, 2048 + 3, generator=cases.gen(m)).half().to(gpu)
            x = base[:, :2048].contiguous()
            assert layer._blocks_win(m) and layer._band(x, m) in ("blocks", "tile") and layer._band(x, m, True) != "blocks"
            first, again, strided = layer(x), layer(x), layer(base[:, :2048])
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                captured = layer(x)
            for _ in range(3):
                captured.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(captured, first)
            assert torch.equal(first, again) and torch.equal(first, strided)
            with monkeypatch.context() as mp:
                mp.setattr(module, name, 0)
                assert layer._band(x, m) not in ("blocks", "fused")
                other = layer(x)
            assert torch.allclose(first.float(), other.float(), rtol=2e-3, atol=2e-3)  # two orders of the same f32 sums, each rounded once
        if getattr(layer, "bias", None) is not None and layer._band(x, m) == "blocks":
            layer.bias.requires_grad_()
            assert layer(x).requires_grad


def test_replaced_wrappers_get_the_arguments_they_document(gpu, monkeypatch):
    """A caller's function in the place of one that the blocks entries now and then stand in for is called with the arguments it has always
    had, and undone again the layer is what it was."""
    from neuropress_amd import kernels

    monkeypatch.setattr(vqmod, "_TILE_MIN_GRID_FRACTION", 0.0)  # the tile GEMM's band without the blocks
    monkeypatch.setattr(qmod, "_Q_TILE_MIN_GRID_FRACTION", 0.0)
    seen = []

    def spy(name, real):
        def vq_gemm_tile(x, packed_indices, centroids, bits, out_features, bias=None):
            seen.append(name)
            return real(x, packed_indices, centroids, bits, out_features, bias)

        def q_gemm_tile(x, w_pack, scale, nbits, group_size, zero_point=None, bias=None):
            seen.append(name)
            return real(x, w_pack, scale, nbits, group_size, zero_point, bias)

        def rvq_linear(x, packed_main, bits_main, packed_res, bits_res, centroids_main, centroids_res, row_scale, row_bias, out_features,
                       bias=None, tile=None):  # fmt: skip
            seen.append(name)
            return real(x, packed_main, bits_main, packed_res, bits_res, centroids_main, centroids_res, row_scale, row_bias, out_features,
                        bias, tile=tile)  # fmt: skip

        def dense_linear(x, w, bias=None):
            seen.append(name)
            return real(x, w, bias)

        def rvq_dequant(*args):
            seen.append(name)
            return real(*args)

        return {f.__name__: f for f in (vq_gemm_tile, q_gemm_tile, rvq_linear, dense_linear, rvq_dequant)}[name]

    n, k = 1024, 4096
    L = cases.vq_layer(1, n, k, 4096)
    plain = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, 8, "cuda_wmma").to(gpu)
    R = cases.rvq_layer(1, n, k, 4096, 256, zipf=False)
    res = NPVQLinear(VQProxy(R["cbm"]).to(gpu), R["pm"], R["bm"], n, k, 8, "cuda_wmma", residual_proxy=VQProxy(R["cbr"]).to(gpu),
                     packed_residual=R["pr"], residual_bits=R["br"], row_scale=R["scale"], row_bias=R["wbias"]).to(gpu)  # fmt: skip
    Q = cases.q4_layer(1, n, k)
    q = NPLinear(Q["blob"], Q["scale"], n, k, 32, 4, "sym", "cuda").to(gpu)
    S = cases.vq_layer(2, n, 2184, 65536)
    ragged = NPVQLinear(VQProxy(S["cb"]).to(gpu), S["packed"], S["bits"], n, 2184, 8, "cuda_wmma").to(gpu)
    T = cases.rvq_layer(2, n, 2184, 4096, 256, zipf=False)
    ragged_res = NPVQLinear(VQProxy(T["cbm"]).to(gpu), T["pm"], T["bm"], n, 2184, 8, "cuda_wmma", residual_proxy=VQProxy(T["cbr"]).to(gpu),
                            packed_residual=T["pr"], residual_bits=T["br"], row_scale=T["scale"], row_bias=T["wbias"]).to(gpu)  # fmt: skip
    for layer, name, m, kk in ((plain, "vq_gemm_tile", 40, k), (q, "q_gemm_tile", 40, k), (res, "rvq_linear", 40, k), (res, "rvq_linear", 24, k),
                               (ragged, "dense_linear", 600, 2184), (ragged_res, "rvq_dequant", 24, 2184), (ragged_res, "rvq_dequant", 600, 2184)):  # fmt: skip
        x = torch.randn(m, kk, generator=cases.gen(m)).half().to(gpu)
        before = layer(x)
        seen.clear()
        with monkeypatch.context() as mp:
            mp.setattr(kernels, name, spy(name, getattr(kernels, name)))
            during = layer(x)
        assert seen == [name], (name, m, kk)
        assert torch.allclose(before.float(), during.float(), rtol=2e-3, atol=2e-3), name
        assert torch.equal(layer(x), before), name


def test_a_blocks_entry_that_fails_leaves_the_tile_gemm_alone(gpu, monkeypatch):
    """Where fallbacks are allowed: the call goes to decode + product, other layers keep the tile GEMM."""
    from neuropress_amd import kernels

    monkeypatch.setattr(vqmod, "_ALLOW_FALLBACK", True)
    monkeypatch.setattr(vqmod, "_tile_failed", False)
    monkeypatch.setattr(kernels, "_warned_fallbacks", set())

    def fails(*args, **more):
        raise RuntimeError("no such kernel")

    n, k = 1024, 4096
    for residual, kk, m in ((False, k, 40), (True, k, 40), (True, 2184, 3)):
        L = cases.rvq_layer(1, n, kk, 4096, 256, zipf=False) if residual else cases.vq_layer(1, n, kk, 4096)
        cb, packed, bits = (L["cbm"], L["pm"], L["bm"]) if residual else (L["cb"], L["packed"], L["bits"])
        more = dict(residual_proxy=VQProxy(L["cbr"]).to(gpu), packed_residual=L["pr"], residual_bits=L["br"], row_scale=L["scale"],
                    row_bias=L["wbias"]) if residual else {}  # fmt: skip
        layer = NPVQLinear(VQProxy(cb).to(gpu), packed, bits, n, kk, 8, "cuda_wmma", **more).to(gpu)
        x = torch.randn(m, kk, generator=cases.gen(m)).half().to(gpu)
        assert layer._band(x, m) == "blocks"
        before = layer(x)
        with monkeypatch.context() as mp:
            mp.setattr(kernels, "rvq_linear_blocks" if residual else "vq_linear_blocks", fails)
            assert torch.allclose(layer(x).float(), before.float(), rtol=2e-3, atol=2e-3)
        assert not vqmod._tile_failed and torch.equal(layer(x), before)


def _at_odd_addresses(t):
    """The same values in a contiguous tensor that starts 4 bytes behind a 16-byte address."""
    flat = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)
    out = flat[4 // t.element_size():][: t.numel()].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("odd", ["packed", "codebook", "residual"])
def test_vq_weights_at_any_address(gpu, odd):
    """Buffers that start between two 16-byte addresses, at every band, planned or not."""
    for n, k, residual in ((512, 2048, False), (512, 2048, True), (512, 2040, False), (512, 2040, True)):
        if odd == "residual" and not residual:
            continue
        move = lambda t, name: _at_odd_addresses(t.to(gpu)) if odd == name else t.to(gpu)
        if residual:
            L = cases.rvq_layer(n + k, n, k, 4096, 256, zipf=False)
            w = ((L["cbm"][L["im"]] + L["cbr"][L["ir"]]).reshape(n, k) * L["scale"][:, None] + L["wbias"][:, None]).float()
            layer = NPVQLinear(VQProxy(move(L["cbm"], "codebook")), move(L["pm"], "packed"), L["bm"], n, k, 8, "cuda_wmma",
                               residual_proxy=VQProxy(move(L["cbr"], "residual")), packed_residual=move(L["pr"], "residual"),
                               residual_bits=L["br"], row_scale=L["scale"].to(gpu), row_bias=L["wbias"].to(gpu))  # fmt: skip
        else:
            L = cases.vq_layer(n + k, n, k, 1000)
            w = L["cb"][L["idx"]].reshape(n, k).float()
            layer = NPVQLinear(VQProxy(move(L["cb"], "codebook")), move(L["packed"], "packed"), L["bits"], n, k, 8, "cuda_wmma")
        for m in (1, 20, 40, 100, 300):
            x = torch.randn(m, k, generator=cases.gen(m)).half()
            ref = x.float() @ w.T
            for _ in range(2):
                err = (layer(x.to(gpu)).float().cpu() - ref).abs()
                assert bool((err <= 1e-2 + 1e-2 * ref.abs()).all()), (k, residual, m, float(err.max()))


@pytest.mark.parametrize("bits", [4, 8])
def test_group_quantized_weights_at_any_address(gpu, bits):
    n, k = 512, 2048
    Q = cases.q4_layer(n + k, n, k, nbits=bits)
    layer = NPLinear(_at_odd_addresses(Q["blob"].to(gpu)), Q["scale"].to(gpu), n, k, 32, bits, "sym", "cuda")
    assert layer.u8_blob.data_ptr() % 16
    w = ((Q["codes"].float() - (1 << (bits - 1))).reshape(n, k // 32, 32) * Q["scale"].float().reshape(n, k // 32, 1)).reshape(n, k).half().float()
    for m in (1, 20, 40, 100, 300):
        x = torch.randn(m, k, generator=cases.gen(m)).half()
        ref = x.float() @ w.T
        for _ in range(2):
            err = (layer(x.to(gpu)).float().cpu() - ref).abs()
            assert bool((err <= 1e-2 + 1e-2 * ref.abs()).all()), (m, float(err.max()))


@pytest.mark.parametrize("form,n,k,m,band", [("vq", 1157, 680, 471, "dense"), ("rvq", 1157, 680, 471, "dense"), ("vq", 1024, 4096, 600, "dense"),
                                             ("table", 512, 2048, 100, "blocks"), ("rvq", 512, 2048, 40, "blocks"), ("rvq", 512, 680, 3, "blocks"),
                                             ("q", 512, 2048, 40, "blocks"), ("q", 1024, 4096, 900, "dense")])  # fmt: skip
def test_rows_at_odd_addresses_stay_with_the_plan(gpu, form, n, k, m, band):
    """The package's product and the blocks entries read whole 16 bytes: a planned call copies rows at other addresses or distances first."""
    if form == "q":
        L = cases.q4_layer(n, n, k)
        layer = NPLinear(L["blob"], L["scale"], n, k, 32, 4, "sym", "cuda").to(gpu)
    elif form == "rvq":
        L = cases.rvq_layer(n, n, k, 4096, 256, zipf=False)
        layer = NPVQLinear(VQProxy(L["cbm"]).to(gpu), L["pm"], L["bm"], n, k, 8, "cuda_wmma", residual_proxy=VQProxy(L["cbr"]).to(gpu),
                           packed_residual=L["pr"], residual_bits=L["br"], row_scale=L["scale"], row_bias=L["wbias"]).to(gpu)  # fmt: skip
    else:
        L = cases.vq_layer(n, n, k, 4096 if form == "table" else 65536)
        layer = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, 8, "cuda_wmma").to(gpu)
    base = torch.randn(m, k + 3, generator=cases.gen(m)).half().to(gpu)
    x = base[:, :k]
    assert layer._band(x, m) == band and (band == "blocks" or layer._own_product(m, x.dtype))
    expect = layer(x.contiguous())
    shifted = torch.empty(m * k + 1, dtype=x.dtype, device=gpu)[1:].view(m, k).copy_(x)
    for given in (x, shifted):  # at an odd distance, from an odd address
        planned = layer._plan.run(given)
        assert planned is not None and torch.equal(planned, expect) and torch.equal(layer(given), expect)


def test_rows_too_far_apart_for_tiles_are_copied(gpu):
    """A layer routed to the table GEMM keeps it: its rows' offsets have 32 bits, the GEMV in its place would decode the weight per 32 tokens."""
    n, k, m, apart = 4096, 2048, 100, 1 << 22
    L = cases.vq_layer(n, n, k, 4096)
    layer = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"], L["bits"], n, k, 8, "cuda_wmma").to(gpu)
    far = torch.empty(m * apart, dtype=torch.half, device=gpu).view(m, apart)[:, :k].copy_(torch.randn(m, k, generator=cases.gen(m)))
    expect = layer(far.contiguous())
    planned = layer._plan.run(far)
    assert layer._band(far, m) == "blocks" and planned is not None and torch.equal(planned, expect)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):  # not by the plan
        captured = layer(far)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(captured, expect)
