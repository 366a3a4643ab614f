"""The native call path's decisions that need no GPU: which layouts it reads in place."""

import pytest
import torch

from neuropress_amd import _lib


def _rows(x):
    """Storage offsets of the rows of x, row by row."""
    lead = x.shape[:-1]
    return [sum(i * s for i, s in zip(index, x.stride())) for index in torch.cartesian_prod(*[torch.arange(n) for n in lead]).reshape(-1, len(lead)).tolist()]


_BASE = torch.arange(4096.0).half()


@pytest.mark.parametrize(
    "size, stride",
    [
        ((8, 64), (64, 1)), ((8, 64), (96, 1)), ((1, 64), (0, 1)), ((4, 8, 64), (512, 64, 1)), ((4, 1, 64), (200, 64, 1)),
        ((8, 64), (0, 1)), ((4, 8, 64), (64, 0, 1)), ((4, 8, 64), (0, 64, 1)), ((1, 8, 64), (64, 0, 1)), ((4, 8, 64), (0, 0, 1)),
        ((8, 64), (32, 1)), ((8, 64), (63, 1)), ((2, 3, 64), (64, 64, 1)), ((2, 3, 64), (256, 64, 1)), ((2, 2, 64), (64, 128, 1)),
        ((64, 8), (1, 64)), ((3, 64), (64, 2)), ((2, 1, 3, 64), (240, 7, 80, 1)), ((2, 4, 3, 64), (0, 240, 80, 1)), ((64,), (1,)),
    ],
)  # fmt: skip
def test_rows_read_in_place_are_the_rows_of_x(size, stride):
    """Where the plan takes a layout, row r lies r distances from the first; anything else it leaves alone: expanded
    inputs (one token for every beam, one mask row for a batch), overlapping and permuted rows."""
    x = torch.as_strided(_BASE, size, stride)
    ldx = _lib.host().row_distance(x)
    rows = _rows(x) if x.dim() > 1 else [0]
    taken = x.stride(-1) == 1 and (len(rows) == 1 or (rows[1] >= x.shape[-1] and rows == [r * rows[1] for r in range(len(rows))]))
    if not taken:
        assert ldx is None
    else:
        assert ldx >= x.shape[-1] and rows == [r * ldx for r in range(len(rows))]


def test_tracked_tensors():
    """Calls that torch follows are not for a plan: it would drop what is followed, or read a tensor without storage."""
    import torch.autograd.forward_ad as fwad
    from torch.utils.flop_counter import FlopCounterMode

    tracked = _lib.host().tracked
    x = torch.randn(3, 8)
    assert not tracked(x) and not tracked(x[1:, ::2]) and not tracked(x.half())
    with torch.inference_mode():
        assert not tracked(x) and not tracked(torch.ones(2))
    assert not tracked(torch.nn.Parameter(x, requires_grad=False))
    leaf = x.clone().requires_grad_()
    assert tracked(leaf) and tracked(leaf * 2)
    with torch.no_grad():
        assert not tracked(leaf)
    with fwad.dual_level():
        assert tracked(fwad.make_dual(x, x)) and not tracked(x)
    assert not tracked(x)
    for dtype in (torch.bfloat16, torch.float16):
        with torch.autocast("cpu", dtype=dtype):
            assert tracked(x.half()) == (dtype != torch.half) and not tracked(x) and not tracked(x.long())
    seen = []
    torch.func.vmap(lambda t: seen.append(tracked(t)) or t)(x)
    torch.func.grad(lambda t: seen.append(tracked(t)) or t.sum())(x)
    torch.func.jvp(lambda t: seen.append(tracked(t)) or t, (x,), (x,))
    torch.jit.trace(lambda t: seen.append(tracked(t)) or t + 1, (x,), check_trace=False)
    with FlopCounterMode(display=False):
        seen.append(tracked(x))
    seen += [tracked(torch._neg_view(x)), tracked(x.to_sparse()), tracked(x.to_mkldnn())]
    assert seen == [True] * len(seen)


def test_exceptions_of_torch_reach_python():
    """A query that throws (a sparse row-compressed tensor has no strides) raises; nothing unwinds through the interpreter."""
    with pytest.raises(RuntimeError):
        _lib.host().row_distance(torch.ones(2, 3).to_sparse_csr())
