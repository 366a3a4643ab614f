"""Tensors a module derives on its first call, read by a call on another stream."""

import pytest
import torch

from neuropress_amd.nn import NPVQLinear, VQProxy
from neuropress_amd.nn.np_rms_norm import NPRMSNorm
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["norm", "bias"])
def test_calls_on_another_stream_wait_for_what_the_first_call_made(gpu, kind, monkeypatch):
    """The first call casts a weight or bias behind other work of its stream; a second call on a second stream, with nothing
    in between, must not read the cast before it is made."""
    from neuropress_amd import _lib

    monkeypatch.setenv("NPAMD_DENSE_TILE", "-1")  # the library's product: its bias is cast to the activations' type
    _lib.load().npamd_diag_reload_tuning()
    try:
        k = 512
        if kind == "norm":
            layer = NPRMSNorm(torch.rand(k, generator=cases.gen(1)) + 0.5, 1e-5).to(gpu)
        else:
            V = cases.vq_layer(7, k, k, 256, bias=True, std=0.05)
            layer = NPVQLinear(VQProxy(V["cb"]).to(gpu), V["packed"], 8, k, k, 8, "cuda_wmma", bias=V["bias"].float()).to(gpu)
        x = torch.randn(600, k, generator=cases.gen(2)).half().to(gpu)
        work = torch.randn(8192, 8192, device=gpu).half()
        first, second, third = (torch.cuda.Stream() for _ in range(3))
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            del_me = torch.zeros(k, dtype=torch.half, device=gpu)  # the cast will lie here
            del del_me
            for _ in range(30):  # some 30 ms
                torch.mm(work, work)
            a = layer(x)
        with torch.cuda.stream(second):
            b = layer(x)
        with torch.cuda.stream(third):
            c = layer(x), layer(x)
        torch.cuda.synchronize()
        assert layer._plan is not None
        assert torch.equal(a, b) and torch.equal(a, c[0]) and torch.equal(a, c[1]) and bool(a.any())
    finally:
        monkeypatch.undo()
        _lib.load().npamd_diag_reload_tuning()
