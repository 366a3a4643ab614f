"""The slice GEMM (csrc/slice_gemm.hip): codebook slices in LDS, up to 32 tokens, partial sums added by a second kernel."""

import pytest
import torch

from neuropress_amd import kernels
from oracle import oracle as orc
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture
def plan(monkeypatch):
    """force(tiles, parts): row tiles per wave and parts of K of the kernel for one test."""
    from neuropress_amd import _lib

    def force(tiles: int, parts: int):
        monkeypatch.setenv("NPAMD_SLICE_TILES", str(tiles))
        monkeypatch.setenv("NPAMD_SLICE_PARTS", str(parts))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.delenv("NPAMD_SLICE_TILES", raising=False)
    monkeypatch.delenv("NPAMD_SLICE_PARTS", raising=False)
    _lib.load().npamd_diag_reload_tuning()


def _layer(gpu, n, k, nc, m, act, seed=0, bias=True):
    L = cases.vq_layer(seed + n + k + nc + m, n, k, nc, bits=16, act=act, m=m, bias=bias, std=0.05)
    return L, L["x"].to(gpu), L["packed"].to(gpu), L["cb"].to(act).to(gpu), L["bias"].to(gpu) if bias else None


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 7, 16, 17, 32])
@pytest.mark.parametrize(
    "n,k,nc,tiles,parts",
    [(70, 64, 4097, 0, 0), (64, 576, 8192, 1, 2), (300, 1088, 8193, 2, 1), (257, 2048, 20000, 4, 3), (130, 1600, 65536, 0, 0),
     (520, 1024, 65535, 4, 1), (33, 512, 40000, 1, 1)],
)  # fmt: skip
def test_slice_gemm_against_the_oracle(gpu, oracle_lib, plan, act, m, n, k, nc, tiles, parts):
    """One slice and several, the last of them short; K of one chunk, of whole and ragged super-steps, in one part and more;
    N ragged against 16-row tiles and against four columns; one and two token tiles."""
    plan(tiles, parts)
    L, x, pk, cb, bias = _layer(gpu, n, k, nc, m, act)
    y = kernels.vq_slice_gemm(x, pk, cb, n, bias)
    code = orc.torch_dtype_code(act)
    w = oracle_lib.vq_decode(L["packed"].numpy(), 16, orc.to_bits(L["cb"]), n, k, code)
    ref = oracle_lib.linear_f64(orc.to_bits(L["x"]), code, w, code, orc.to_bits(L["bias"]), code)
    ok, max_abs, excess = cases.within_tol(y.float().cpu().numpy(), ref)
    assert ok, f"max abs err {max_abs:.3e}, {excess:.2f}x the 1e-2 bound"
    assert torch.equal(y, kernels.vq_slice_gemm(x, pk, cb, n, bias))


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nc", [8192, 65536])
def test_slice_gemm_reads_codebook_rows_exactly(gpu, plan, act, nc):
    """One-hot activations: every output is one codebook value, whichever slice and part it comes from."""
    n, k = 200, 1600
    L, _, pk, cb, _ = _layer(gpu, n, k, nc, 1, act, bias=False)
    wt = kernels.vq_dequant(pk, L["cb"].to(gpu), 16, n, k, act).t()
    eye = torch.eye(k, dtype=act, device=gpu)
    for rows in (slice(0, 32), slice(510, 526), slice(1570, 1600)):
        assert torch.equal(kernels.vq_slice_gemm(eye[rows].contiguous(), pk, cb, n), wt[rows])


@pytest.mark.parametrize("m", [3, 16, 29])
@pytest.mark.parametrize("nc", [5000, 65536])
def test_slice_gemm_keeps_infinities_where_they_belong(gpu, plan, m, nc):
    """Indices outside a slice read zeros, and zero times an infinity is not zero: infinite and NaN activations reach their own
    token only, with the values that the GEMV over memory gives; infinite codebook rows reach the rows that use them."""
    n, k = 150, 1664
    plan(2, 2)
    _, x, pk, cb, _ = _layer(gpu, n, k, nc, m, torch.float16, bias=False)
    x[1, 5], x[2, 1600], x[2, 70] = float("inf"), float("-inf"), float("nan")
    y, ref = kernels.vq_slice_gemm(x, pk, cb, n), kernels.vq_linear(x, pk, cb, 16, 8, None, n)
    assert torch.isfinite(ref[0]).all() and not torch.isfinite(ref[1:3]).any()
    torch.testing.assert_close(y, ref, rtol=2e-3, atol=2e-3, equal_nan=True)
    x = torch.randn(m, k, dtype=torch.float16, device=gpu)
    cb[: nc // 50, 3] = float("inf")
    y, ref = kernels.vq_slice_gemm(x, pk, cb, n), kernels.vq_linear(x, pk, cb, 16, 8, None, n)
    assert not torch.isfinite(ref).all()
    torch.testing.assert_close(y, ref, rtol=2e-3, atol=2e-3, equal_nan=True)


def test_slice_gemm_hands_other_forms_on(gpu, plan):
    """What the kernel does not take -- rows at an odd address, few codebook rows, more than 32 tokens -- is the tile GEMM's."""
    n, k = 96, 640
    for nc, m, shift in ((65536, 5, 1), (300, 5, 0), (65536, 40, 0)):
        _, x, pk, cb, bias = _layer(gpu, n, k, nc, m, torch.float16)
        wide = torch.zeros(m, k + 8, dtype=torch.float16, device=gpu)
        wide[:, shift : shift + k] = x
        y = kernels.vq_slice_gemm(wide[:, shift : shift + k], pk, cb, n, bias)
        assert torch.equal(y, kernels.vq_gemm_tile(wide[:, shift : shift + k], pk, cb, 16, n, bias))


@pytest.mark.parametrize("perm", [False, True])
def test_module_takes_the_slice_gemm_where_it_was_timed_faster(gpu, monkeypatch, perm):
    """Layers whose times say so, with and without a column permutation, against decode + GEMM; calls that record a gradient
    do not take it, nor do layers that were not timed."""
    from neuropress_amd import AutoKernelLowering
    from neuropress_amd.qweights import VQWeight, attach_quantized_weight

    n, k, nc = 256, 1024, 8192
    L = cases.vq_layer(5, n, k, nc, act=torch.float16, m=12, std=0.05)
    order = torch.randperm(k) if perm else None
    linear = attach_quantized_weight(torch.nn.Linear(k, n, bias=False, device="meta"),
                                     VQWeight.from_indices(L["idx"], L["cb"], n, k, column_permutation=order))  # fmt: skip
    model = torch.nn.Sequential(linear)
    AutoKernelLowering().apply(model)
    layer = model.to(gpu)[0]
    x = L["x"].to(gpu)
    assert not layer._slice_gemm_wins(12)
    key = (layer.packed_indices.device, layer.packed_indices.data_ptr(), layer.packed_indices._version)
    layer._derived["sliced"] = (key, (None, 0, ((1, 1e3, 1e3),)))  # as if both GEMVs had taken a millisecond
    layer._plan = None
    assert layer._slice_gemm_wins(12) and layer._band(x, 12) == "slice" and layer._band(x, 12, True) != "slice"
    w = kernels.vq_dequant(layer.packed_indices, L["cb"].to(gpu), layer.bits, n, k, torch.float16).float()
    ref = (x if order is None else x[:, order.to(gpu)]).float() @ w.t()
    for _ in range(2):  # the second call is the plan's
        torch.testing.assert_close(layer(x).float(), ref, rtol=2e-3, atol=5e-3)
    layer._derived["sliced"] = (key, (None, 0, ((1, 1.0, 1.0),)))
    assert not layer._slice_gemm_wins(12)


def _timed_module(gpu, n, k, nc, act, perm=False, bias=False, seed=5):
    """A lowered layer as if both GEMVs had been timed at a millisecond, so that the slice GEMM serves up to 32 tokens; and its
    weight as torch multiplies it (columns of x in their own order), in float32."""
    from neuropress_amd import AutoKernelLowering
    from neuropress_amd.qweights import VQWeight, attach_quantized_weight

    L = cases.vq_layer(seed + n + k, n, k, nc, act=act, m=1, bias=True, std=0.05)
    order = torch.randperm(k, generator=cases.gen(seed)) if perm else None
    weight = VQWeight.from_indices(L["idx"], L["cb"], n, k, column_permutation=order)
    linear = attach_quantized_weight(torch.nn.Linear(k, n, bias=False, device="meta"), weight)
    if bias:
        linear.bias = torch.nn.Parameter(L["bias"], requires_grad=False)
    model = torch.nn.Sequential(linear)
    AutoKernelLowering().apply(model)
    layer = model.to(gpu)[0]
    packed = layer.packed_indices
    layer._derived["sliced"] = ((packed.device, packed.data_ptr(), packed._version), (None, 0, ((1, 1e3, 1e3),)))
    layer._plan = None
    w = kernels.vq_dequant(packed, L["cb"].to(gpu), layer.bits, n, k, act).float()
    if order is not None:
        w = w[:, torch.argsort(order).to(gpu)]
    return layer, w, L["bias"].to(gpu).float() if bias else torch.zeros(n, device=gpu)


def _near(y, x, w, b, act):
    """Sums are f32 and the output is rounded once: half an ulp of it, and 2^-20 of the products' absolute values."""
    ref = x.double() @ w.double().t() + b.double()
    tol = 2.0 ** (-11 if act == torch.float16 else -8) * ref.abs() + 2.0 ** -20 * (x.double().abs() @ w.double().abs().t()) + 1e-6
    return bool(((y.double() - ref).abs() <= 1.01 * tol).all())


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,perm,bias", [(1000, False, True), (1000, True, False), (584, False, False), (1024, True, True)])
def test_module_slice_band_eager_planned_captured_and_on_two_streams(gpu, act, k, perm, bias):
    """K that is no whole number of 64-column chunks (rows padded with zeros), columns permuted, a bias: the module's first
    call, the calls its plan issues, a captured call replayed between eager work, and calls on two streams at once, each with
    a workspace of its own."""
    n, nc, m = 300, 9000, 12
    layer, w, b = _timed_module(gpu, n, k, nc, act, perm, bias)
    xs = [torch.randn(m, k, generator=cases.gen(i)).to(act).to(gpu) for i in range(4)]
    assert layer._band(xs[0], m) == "slice"
    eager = [layer(x) for x in xs]
    assert layer._plan is not None
    for x, y in zip(xs, eager):
        assert _near(y, x, w, b, act)
        assert torch.equal(layer(x), y)
    static, s = xs[0].clone(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        layer(static)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = layer(static)
    for i in (1, 2, 3, 0):
        static.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager[i]), f"replay on input {i}"
        assert torch.equal(layer(xs[i]), eager[i])
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    for turn in range(8):
        for j, st in enumerate(streams):
            with torch.cuda.stream(st):
                got.append((2 * j + turn % 2, layer(xs[2 * j + turn % 2])))
    torch.cuda.synchronize()
    assert all(torch.equal(y, eager[i]) for i, y in got)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
def test_module_with_real_lists_takes_the_slice_gemm(gpu, act):
    """A layer large enough for slice lists, prepared and timed as a program prepares it: one token goes to the lists, sixteen to
    the slice GEMM (16 against 37 us for lookups in memory on a layer of this size), and every count to the kernel of its
    band whichever count came first."""
    from neuropress_amd.nn import NPVQLinear, VQProxy

    n, k, nc = 8192, 4096, 16384
    L = cases.vq_layer(11, n, k, nc, bits=16, act=act, m=1, std=0.05)
    layer = NPVQLinear(VQProxy(L["cb"]).to(gpu), L["packed"].to(gpu), 16, n, k, 8, "cuda_wmma").to(gpu)
    assert layer.prepare_sliced()
    counts = layer._slice_gemm_counts()
    assert 16 in counts and 1 not in counts
    w = kernels.vq_dequant(layer.packed_indices, L["cb"].to(gpu), 16, n, k, act).float()
    b = torch.zeros(n, device=gpu)
    for m in (1, 16, 2, 3, 7, 32, 5, 1):
        x = torch.randn(m, k, generator=cases.gen(m)).to(act).to(gpu)
        assert (layer._band(x, m) == "slice") == (m in counts)
        first = layer(x)
        assert _near(first, x, w, b, act), m
        if m in counts:  # partial sums in a fixed order, and nothing but this kernel gives these bits
            assert torch.equal(first, kernels.vq_slice_gemm(x, layer.packed_indices, layer.proxy.centroids_as(act), n))
        assert torch.equal(layer(x), first)
