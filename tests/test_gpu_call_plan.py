"""The native call path (CallPlan): a layer's later calls give what its first one gives, and the plan steps aside
when anything it was built from changes."""

import copy

import pytest
import torch

import neuropress_amd.nn.np_linear as qmod
import neuropress_amd.nn.np_vq_linear as vqmod
from neuropress_amd.nn import NPLinear, NPVQLinear, VQProxy
from tests import cases

pytestmark = pytest.mark.gpu


def _layer(kind, gpu, act):
    n, k = 96, 512
    if kind == "q4":
        Q = cases.q4_layer(5, n, k, act=act, bias=True)
        return NPLinear(Q["blob"], Q["scale"], n, k, 32, 4, "sym", "cuda", bias=Q["bias"]).to(gpu)
    if kind == "rvq":
        R = cases.rvq_layer(6, n, k, act=act)
        layer = NPVQLinear(VQProxy(R["cbm"]), R["pm"], R["bm"], n, k, 8, "cuda_wmma", residual_proxy=VQProxy(R["cbr"]),
                           packed_residual=R["pr"], row_scale=R["scale"], row_bias=R["wbias"])  # fmt: skip
    else:
        nc, bits = {"vq8": (256, 8), "vq16": (20000, 16)}[kind.split("-")[0]]
        V = cases.vq_layer(7, n, k, nc, bits=bits, act=act, bias=True, std=0.05)
        perm = torch.randperm(k, generator=cases.gen(8)) if kind.endswith("perm") else None
        layer = NPVQLinear(VQProxy(V["cb"]), V["packed"], bits, n, k, 8, "cuda_wmma", bias=V["bias"], column_perm=perm)
    layer.proxy.to(gpu)
    if layer.residual_proxy is not None:
        layer.residual_proxy.to(gpu)
    return layer.to(gpu)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["vq8", "vq8-perm", "vq16", "vq16-perm", "rvq", "q4"])
def test_planned_calls_equal_first_calls_and_follow_the_module(gpu, kind, act, monkeypatch):
    monkeypatch.setattr(vqmod, "_SLICED_MIN_INDICES", 1)
    monkeypatch.setattr(vqmod, "_TILE_MAX_TOKENS", 64)
    monkeypatch.setattr(vqmod, "_TILE_MIN_GRID_FRACTION", 0.0)
    monkeypatch.setattr(qmod, "_Q_TILE_MAX_TOKENS", 64)
    monkeypatch.setattr(qmod, "_Q_TILE_MIN_GRID_FRACTION", 0.0)
    layer = _layer(kind, gpu, act)
    k = layer.in_features
    for m in (1, 2, 9, 40, 130):  # every band
        x = torch.randn(m, k, generator=cases.gen(m)).to(act).to(gpu)
        layer._plan = None
        first = layer(x)
        plan = layer._plan
        assert plan is not None and not plan.stale(layer)
        assert torch.equal(layer(x), first)
        assert torch.equal(plan(layer, x), first)  # the plan itself answers
        assert torch.equal(plan(layer, x.reshape(m, 1, 1, k)), first.reshape(m, 1, 1, -1))
        wide = torch.zeros(m, 3, k, dtype=act, device=gpu)
        wide[:, 2] = x
        strided = plan(layer, wide[:, 2:]).reshape(m, -1)  # rows at a stride; torch's dense product may sum in another order
        assert torch.equal(strided, first) if m < 130 else torch.allclose(strided, first, rtol=2e-2, atol=2e-2)
        if m > 1:
            assert plan(layer, wide[:, :2]) is None  # two row distances: not a stack of rows
        assert plan(layer, x.cpu()) is None and plan(layer, x.double()) is None and plan(layer, x[:, : k // 2]) is None
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            side.wait_stream(torch.cuda.current_stream())
            torch.cuda.synchronize()
            assert torch.equal(layer(x), first) and torch.equal(layer(x), first)
        torch.cuda.synchronize()
        copied = copy.deepcopy(layer)
        assert copied._plan is None  # it may run another kernel: the slice lists are not its buffers'
        assert torch.allclose(copied(x), first, rtol=2e-2, atol=2e-2)
        layer.bias = None if layer.bias is None else layer.bias + 1  # another tensor in the buffer's place
        if layer.bias is not None:
            assert plan.stale(layer) and plan(layer, x) is None
            assert not torch.equal(layer(x), first)
            layer.bias = layer.bias - 1
        backend, layer.backend = layer.backend, layer.backend.__class__("default")
        assert plan(layer, x) is None
        layer(x)
        layer.backend = backend


def test_planned_norm_and_lookups(gpu):
    from neuropress_amd.nn.np_embedding import NPEmbedding
    from neuropress_amd.nn.np_rms_norm import NPRMSNorm
    from neuropress_amd.nn.np_vq_embedding import NPVQEmbedding

    g = cases.gen(9)
    norm = NPRMSNorm(torch.rand(320, generator=g).half() + 0.5, 1e-5).to(gpu)
    for m in (1, 77):
        x = torch.randn(m, 320, generator=g).half().to(gpu)
        first = norm(x)
        assert torch.equal(norm._plan(norm, x), first)
    norm.eps = 1.0
    assert norm._plan(norm, x) is None and not torch.equal(norm(x), first)
    Q = cases.q4_layer(10, 300, 256)
    proxy = VQProxy((torch.randn(1000, 8, generator=g) * 0.05).half()).to(gpu)
    tab = torch.randint(0, 1000, (300, 32), generator=g)
    for emb in (NPVQEmbedding(tab, proxy, 256, 8, out_dtype=torch.bfloat16).to(gpu),
                NPEmbedding(Q["blob"], Q["scale"], 300, 256, 32, 4, "sym", "cuda", padding_idx=3).to(gpu)):  # fmt: skip
        for shape in ((1,), (3, 5)):
            ids = torch.randint(0, 300, shape, generator=g).to(gpu)
            first = emb(ids)
            assert first.shape == (*shape, 256) and torch.equal(emb._plan(emb, ids), first)
            assert emb._plan(emb, ids.int()) is None and torch.equal(emb(ids.int()), first)


@pytest.mark.parametrize("kind", ["vq8", "q4"])
def test_module_call_takes_the_long_way_when_something_stands_between(gpu, kind, monkeypatch):
    """``module(x)`` skips torch's module call only while that would do nothing but call the class's own forward."""
    layer = _layer(kind, gpu, torch.float16)
    x = torch.randn(1, layer.in_features, generator=cases.gen(1)).half().to(gpu)
    first = layer(x)
    assert torch.equal(layer(x), first) and type(layer).__call__ is not torch.nn.Module.__call__
    seen = []
    for register in (layer.register_forward_pre_hook, layer.register_forward_hook,
                     torch.nn.modules.module.register_module_forward_hook):  # fmt: skip
        handle = register(lambda *args: seen.append(1))
        assert torch.equal(layer(x), first) and len(seen) == 1
        handle.remove()
        assert torch.equal(layer(x), first) and len(seen) == 1
        seen.clear()
    own = layer.forward
    layer.forward = lambda t: own(t) + 1
    assert torch.equal(layer(x), first + 1)
    del layer.forward
    monkeypatch.setattr(type(layer), "forward", lambda self, t: type(self)._planned_forward(self, t) + 2)
    assert torch.equal(layer(x), first + 2)
    monkeypatch.undo()
    torch_call = torch.nn.Module.__call__
    monkeypatch.setattr(torch.nn.Module, "__call__", lambda self, *a, **k: seen.append(1) or torch_call(self, *a, **k))
    assert torch.equal(layer(x), first) and len(seen) == 1
    monkeypatch.undo()
    assert torch.equal(layer(x), first) and len(seen) == 1
    copied = copy.deepcopy(layer)
    assert torch.equal(copied(x), copied(x))
    with pytest.raises(TypeError):
        layer()


def _small_bands(monkeypatch):
    """Every band on small layers: 1-7 tokens sliced, to 32 GEMV, to 64 tile, then decode + product."""
    monkeypatch.setattr(vqmod, "_SLICED_MIN_INDICES", 1)
    for module, prefix in ((vqmod, "_TILE"), (qmod, "_Q_TILE")):
        monkeypatch.setattr(module, prefix + "_MAX_TOKENS", 64)
        monkeypatch.setattr(module, prefix + "_MIN_GRID_FRACTION", 0.0)


@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["vq8", "vq8-perm", "vq16", "vq16-perm", "rvq", "q4", "norm"])
def test_expanded_inputs_equal_their_copies(gpu, kind, act, monkeypatch):
    """One row for a whole batch, one row per beam, one prompt for every beam: rows at distance 0 or at several, on the
    first call and on the planned ones."""
    from neuropress_amd.nn.np_rms_norm import NPRMSNorm

    _small_bands(monkeypatch)
    k = 512
    layer = NPRMSNorm(torch.rand(k, generator=cases.gen(1)).to(act), 1e-5).to(gpu) if kind == "norm" else _layer(kind, gpu, act)
    for rows in (3, 9, 20, 65):  # times two: every band
        base = torch.randn(rows, k, generator=cases.gen(rows)).to(act).to(gpu)
        for x in (base[:1].expand(2 * rows, k), base[:, None].expand(rows, 2, k), base[None].expand(2, rows, k),
                  base[0].expand(1, k), base[0].expand(2, rows, k)):  # fmt: skip
            for call in range(2):
                y, ref = layer(x), layer(x.clone(memory_format=torch.contiguous_format))
                assert y.shape == ref.shape
                # the dense products may sum in another order
                assert torch.equal(y, ref) if rows < 65 else torch.allclose(y, ref, rtol=2e-2, atol=2e-2), (rows, x.stride(), call)


@pytest.mark.parametrize("kind", ["vq8", "vq8-perm", "rvq", "q4"])
def test_inputs_at_odd_addresses(gpu, kind, monkeypatch):
    """Dense rows that do not start at a 16-byte boundary (a slice of a flat buffer), in every band."""
    _small_bands(monkeypatch)
    layer, k = _layer(kind, gpu, torch.float16), 512
    for m in (20, 40, 130) if kind == "vq8-perm" else (2, 20, 40, 130):  # the GEMV that gathers columns refuses them
        x = torch.randn(m * k + 1, generator=cases.gen(m)).half().to(gpu)[1:].view(m, k)
        ref = layer(x.clone())
        for call in range(2):
            assert torch.allclose(layer(x), ref, rtol=2e-2, atol=2e-2), (m, call)


@pytest.mark.parametrize("cast", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["vq8", "vq16", "rvq"])
def test_cast_codebooks(gpu, kind, cast, monkeypatch):
    """``model.to(dtype)`` on a lowered model casts the codebooks: the bands that look rows up in a copy of the
    activations' type serve them, the decodes read fp16 and say so."""
    _small_bands(monkeypatch)
    layer, k = _layer(kind, gpu, torch.float16), 512
    xs = {m: torch.randn(m, k, generator=cases.gen(m)).half().to(gpu) for m in (2, 20, 40, 130)}
    before = {m: layer(x) for m, x in xs.items()}
    for module in (layer, layer.proxy, layer.residual_proxy):
        if module is not None:
            module.to(cast)
    for m, x in xs.items():
        for call in range(2):
            if kind == "rvq" or m == 130:
                with pytest.raises(RuntimeError, match="must be float16"):
                    layer(x)
            else:
                assert torch.allclose(layer(x), before[m], rtol=2e-2, atol=2e-2), (m, call)


@pytest.fixture
def dense_tile(monkeypatch):
    from neuropress_amd import _lib

    def force(tile):
        monkeypatch.setenv("NPAMD_DENSE_TILE", str(tile))
        _lib.load().npamd_diag_reload_tuning()

    yield force
    monkeypatch.delenv("NPAMD_DENSE_TILE", raising=False)
    _lib.load().npamd_diag_reload_tuning()


def _dense_cases():
    # name, format, n, k, tokens: calls the library's product serves when a gradient is asked for
    return [
        ("own product", "vq8", 96, 512, 130), ("own product", "q4", 96, 512, 130), ("own product", "rvq", 96, 512, 130),
        ("library product", "vq8-perm", 96, 512, 130), ("own product", "vq8-perm", 96, 512, 130), ("odd K, gemv", "vq8", 96, 200, 3), ("odd K, tile", "vq8-perm", 96, 200, 40),
        ("half grid", "vq8", 8320, 512, 100), ("half grid", "q4", 8320, 512, 100), ("half grid", "rvq", 8320, 512, 100),
        ("tight grid", "vq8", 5504, 2048, 40), ("tight grid", "q4", 5504, 4096, 40), ("long K", "vq8", 2048, 6144, 200),
        ("wide tile", "vq16", 3072, 4096, 200),
    ]  # fmt: skip


def _weight_layer(kind, n, k, gpu):
    """A layer and its dense weight in float64."""
    g = cases.gen(n + k)
    if kind == "q4":
        Q = cases.q4_layer(5, n, k)
        layer = NPLinear(Q["blob"], Q["scale"], n, k, 32, 4, "sym", "cuda").to(gpu)
        return layer, (Q["codes"].double() - 8) * Q["scale"].double().reshape(n, -1).repeat_interleave(32, 1)
    if kind == "rvq":
        R = cases.rvq_layer(6, n, k, nc_main=4096, zipf=False)
        proxies = VQProxy(R["cbm"]).to(gpu), VQProxy(R["cbr"]).to(gpu)
        layer = NPVQLinear(proxies[0], R["pm"], R["bm"], n, k, 8, "cuda_wmma", residual_proxy=proxies[1], packed_residual=R["pr"],
                           row_scale=R["scale"], row_bias=R["wbias"]).to(gpu)  # fmt: skip
        w = ((R["cbm"][R["im"]] + R["cbr"][R["ir"]]).reshape(n, k) * R["scale"][:, None] + R["wbias"][:, None]).double()
        return layer, w
    nc, bits = {"vq8": (256, 8), "vq16": (20000, 16)}[kind.split("-")[0]]
    V = cases.vq_layer(7, n, k, nc, bits=bits, std=0.05)
    perm = torch.randperm(k, generator=g) if kind.endswith("perm") else None
    layer = NPVQLinear(VQProxy(V["cb"]).to(gpu), V["packed"], bits, n, k, 8, "cuda_wmma", column_perm=perm).to(gpu)
    w = V["cb"][V["idx"]].reshape(n, k).double()
    return layer, w if perm is None else torch.zeros_like(w).index_copy_(1, perm, w)  # y = x[:, perm] @ w.T


@pytest.mark.parametrize("name,kind,n,k,m", _dense_cases())
def test_gradients_where_the_library_product_had_them(gpu, dense_tile, name, kind, n, k, m, monkeypatch):
    monkeypatch.setattr(vqmod, "_SLICED_MAX_TOKENS", 0)  # no slice lists to build and time
    if name == "library product":
        dense_tile(-1)  # never the package's own
    layer, w = _weight_layer(kind, n, k, gpu)
    x = torch.randn(m, k, generator=cases.gen(m)).half().to(gpu)
    dy = torch.randn(m, n, generator=cases.gen(m + 1)).half()
    ref = (dy.double() @ w).float()
    for call in range(2):  # without a plan, and with one the call below has made
        leaf = x.clone().requires_grad_()
        y = layer(leaf)
        assert y.requires_grad
        y.backward(dy.to(gpu))
        err = (leaf.grad.float().cpu() - ref).norm() / ref.norm()
        assert float(err) < 4e-3, (call, float(err))  # the rounding of dy @ w to fp16, of w in fp16
        with torch.no_grad():
            assert torch.allclose(layer(leaf), y, rtol=2e-2, atol=2e-2) and not layer(leaf).requires_grad
        assert not layer(x).requires_grad


@pytest.mark.parametrize("name,kind,n,k,m", _dense_cases()[:10])
def test_forward_mode_and_vmap_where_the_library_product_had_them(gpu, dense_tile, name, kind, n, k, m):
    import torch.autograd.forward_ad as fwad
    from torch.utils.flop_counter import FlopCounterMode

    if name == "library product":
        dense_tile(-1)  # never the package's own

    layer, w = _weight_layer(kind, n, k, gpu)
    x, t = (torch.randn(2, m, k, generator=cases.gen(m + i)).half().to(gpu) for i in range(2))
    tangent, primal = ((v.cpu().double() @ w.T).float() for v in (t, x))

    def close(a, ref):
        assert float((a.float().cpu() - ref).norm() / ref.norm()) < 4e-3

    for call in range(2):
        with fwad.dual_level():
            out = fwad.unpack_dual(layer(fwad.make_dual(x[0], t[0])))
            assert out.tangent is not None
            close(out.tangent, tangent[0])
        close(torch.func.vmap(layer)(x), primal)
        with FlopCounterMode(display=False) as flops:
            layer(x[0])
        assert flops.get_total_flops() == 2 * m * n * k
        close(layer(x[0]), primal[0])  # makes the plan the second pass meets


def test_out_of_memory_keeps_its_type(gpu):
    """Callers catch torch.OutOfMemoryError to retry with less: an allocation that fails inside a plan raises it too."""
    from neuropress_amd.nn.np_embedding import NPEmbedding

    k = 8192
    blob = torch.zeros(16, k // 2, dtype=torch.uint8, device=gpu)
    emb = NPEmbedding(blob, torch.ones(16 * k // 32, dtype=torch.half, device=gpu), 16, k, 32, 4, "sym", "cuda").to(gpu)
    emb(torch.zeros(4, dtype=torch.int64, device=gpu))
    ids = torch.zeros(1, dtype=torch.int64, device=gpu).expand(1 << 26).contiguous()  # an output of 1 TiB
    for call in range(2):
        with pytest.raises(torch.OutOfMemoryError):
            emb(ids)


@pytest.mark.parametrize("kind", ["vq8", "q4"])
def test_sparse_inputs_are_refused_by_python(gpu, kind):
    """A tensor whose layout queries throw is the module's to refuse, with a plan and without."""
    layer = _layer(kind, gpu, torch.float16)
    x = torch.zeros(1, layer.in_features, dtype=torch.half, device=gpu)
    for call in range(2):
        with pytest.raises(RuntimeError):
            layer(x.to_sparse_csr())
        layer(x)


@pytest.mark.parametrize("act", [torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["vq8-perm", "vq16-perm"])
def test_column_permutations_with_negative_entries_and_past_the_end(gpu, kind, act, monkeypatch):
    """As torch's indexing reads them, in every band: counted from the end, and reported."""
    _small_bands(monkeypatch)
    layer, k = _layer(kind, gpu, torch.float16), 512
    perm = layer.column_perm.clone()
    xs = {m: torch.randn(m, k, generator=cases.gen(m)).to(act).to(gpu) for m in (2, 20, 40, 130)}
    ref = {m: layer(x) for m, x in xs.items()}
    layer.column_perm[::3] -= k
    for m, x in xs.items():
        assert torch.equal(layer(x), ref[m]) and torch.equal(layer(x), ref[m]), m
    layer.column_perm[5] = k
    for x in xs.values():
        for call in range(2):
            with pytest.raises(IndexError, match="out of range"):
                layer(x)
    layer.prepare()  # says nothing: the buffer may be about to be loaded
    layer.column_perm.copy_(perm)
    for m, x in xs.items():
        assert torch.equal(layer(x), ref[m]), m


@pytest.mark.parametrize("kind", ["vq8", "rvq", "q4"])
def test_plans_follow_the_band_lines(gpu, kind, monkeypatch):
    """Every line the choice between the bands reads: a plan made under another value is stale."""
    from neuropress_amd.nn import backends

    layer = _layer(kind, gpu, torch.float16)
    x = torch.randn(40, 512, generator=cases.gen(1)).half().to(gpu)
    module = qmod if kind == "q4" else vqmod
    for owner, name in [(backends, n) for n in backends.BAND_LINES] + [(module, n) for n in module._PLAN_THRESHOLDS]:
        y = layer(x)
        plan = layer._plan
        assert not plan.stale(layer)
        with monkeypatch.context() as mp:
            value = getattr(owner, name)
            mp.setattr(owner, name, dict(value) if isinstance(value, dict) else not value if isinstance(value, bool) else value * 1.0)
            assert plan.stale(layer) and plan(layer, x) is None, name
        assert torch.equal(layer(x), y)


@pytest.mark.parametrize("kind", ["vq8", "vq8-perm", "rvq", "q4"])
def test_autocast_decides_the_type_of_the_dense_bands(gpu, kind):
    layer = _layer(kind, gpu, torch.float16)
    x = torch.randn(130, 512, generator=cases.gen(1)).half().to(gpu)
    ref = layer(x)
    for call in range(2):
        for dtype in (torch.float16, torch.bfloat16):
            with torch.autocast("cuda", dtype=dtype):
                y = layer(x)
                assert y.dtype == dtype and torch.allclose(y.float(), ref.float(), rtol=2e-2, atol=5e-2)
                assert layer(x[:4]).dtype == torch.float16  # the fused kernels answer in x's type
                assert layer(x.float()).dtype == dtype


@pytest.mark.parametrize("kind", ["vq8", "rvq", "q4"])
def test_replaced_products_are_called(gpu, dense_tile, kind, monkeypatch):
    """The product of the dense band, the package's own and the library's: instrumentation put in its place sees every call."""
    from neuropress_amd import kernels

    layer = _layer(kind, gpu, torch.float16)
    x = torch.randn(130, 512, generator=cases.gen(1)).half().to(gpu)
    for tile, owner, name in ((0, kernels, "dense_linear"), (-1, torch.nn.functional, "linear")):
        dense_tile(tile)
        layer._plan = None
        ref = layer(x)
        real, seen = getattr(owner, name), []
        with monkeypatch.context() as mp:
            mp.setattr(owner, name, lambda *a, **k: seen.append(1) or real(*a, **k))
            assert torch.equal(layer(x), ref) and torch.equal(layer(x), ref) and len(seen) == 2
        assert torch.equal(layer(x), ref) and len(seen) == 2


@pytest.mark.parametrize("tile", [0, -1])
@pytest.mark.parametrize("kind", ["vq8", "vq8-perm", "q4"])
def test_bias_gradients_where_the_library_product_had_them(gpu, dense_tile, kind, tile):
    """A bias that is trained on its own: the input asks for no gradient."""
    dense_tile(tile)
    layer = _layer(kind, gpu, torch.float16)
    x = torch.randn(130, 512, generator=cases.gen(1)).half().to(gpu)
    dy = torch.randn(130, 96, generator=cases.gen(2)).half().to(gpu)
    for call in range(2):
        layer(x)  # without a gradient asked for: a plan
        layer.bias.requires_grad_()
        y = layer(x)
        assert y.requires_grad
        (grad,) = torch.autograd.grad(y, layer.bias, dy)
        assert torch.allclose(grad.float(), dy.float().sum(0), rtol=1e-2, atol=2e-2)
        with torch.no_grad():
            assert not layer(x).requires_grad
        layer.bias.requires_grad_(False)
        assert not layer(x).requires_grad
