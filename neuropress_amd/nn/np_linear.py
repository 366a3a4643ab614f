"""NPLinear: ``nn.Linear`` replacement with a packed n-bit group-quantized weight.

Same surface as the reference (neuropress/nn/np_linear.py:426-871):
``NPLinear(u8_blob, scale, out_features, in_features, group_size, nbits, qtype,
backend, bias, zero_point, ...)``, ``from_linear``, ``set_backend``,
``to_qtensor``, ``linearize_qtensor_weights`` and the helpers ``_unpack_u8`` /
``_pack_u8`` / ``_q_dequant_linear``.

Dequantisation rule (neuropress/nn/np_linear.py:333-353):

    ``q = (blob[n, k // vpb] >> ((k % vpb) * nbits)) & mask``
    ``w = (float(q) - zp) * float(scale[n, k // group_size])``   (f32),
    ``zp = 2**(nbits-1)`` when symmetric

The ``cuda`` backend runs the HIP kernels: a fused dequant GEMV up to 16
tokens (32 where it reads whole lines), a fused dequant MFMA GEMM up to ``_Q_TILE_MAX_TOKENS``, and decode +
dense GEMM above.  bf16 activations are computed natively (the reference casts
them to fp16 first, np_linear.py:748-749).
"""

from __future__ import annotations

import logging
import os

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import _lib
from ..qweights import ScalarQScheme, ScalarQWeight, is_scalar_qweight
from ..t2n.packing import BitPacking
from .backends import Backend, LinearBackend, is_hip_backend_available, tensor_version, tile_band_ok

log = logging.getLogger(__name__)

# Most tokens of the GEMV with a workgroup per 32 tokens, which serves small layers past the GEMV's own (kernels.gemv_blocks_preferred).
_Q_BLOCKS_MAX_TOKENS: int = int(os.environ.get("NEUROPRESS_Q_BLOCKS_MAX_TOKENS", "65536"))
# Upper end of the fused-GEMM band for the int4 path; above it decode + GEMM.
# Measured on one MI355X (14336 x 4096, group 32): fused GEMM 35-40 us up to 128
# tokens and 56 us at 256 against 56-64 / 80 us for decode + GEMM; 83-84 vs 78-84 us at
# 320-384, 158 vs 93 us at 512.
_Q_TILE_MAX_TOKENS: int = int(os.environ.get("NEUROPRESS_Q_TILE_MAX_TOKENS", "256"))
# Long reductions (K >= _Q_TILE_SPLIT_LONG_K), where the dense GEMM is slow, keep the fused
# GEMM up to this many tokens: 4096 x 14336 80 vs 105-109 us at 320-384, 148 vs 120 us at 512.
_Q_TILE_LONG_K_MAX_TOKENS: int = 384
# Layers of at least _Q_TILE_WIDE_MIN_FEATURES output or input features run the 128-column fused GEMM
# (256-row blocks past 384 tokens): 14336 x 4096 61 us at 384 tokens and 78-82 at 512 against 86 and 93 us
# for decode + GEMM, 150 against about 140 at 1024; 4096 x 14336 68 / 82 us at 384 / 512.
_Q_TILE_WIDE_MAX_TOKENS: int = int(os.environ.get("NEUROPRESS_Q_TILE_WIDE_MAX_TOKENS", "512"))
_Q_TILE_WIDE_MIN_FEATURES: int = 8192
# As for the VQ path: the fused GEMM splits the reduction when the layer has few
# output features; a layer that still leaves most compute units idle takes decode +
# GEMM.  Measured (fused vs decode + GEMM): 4096 x 14336 41-57 vs 93-115 us from 128 to
# 256 tokens; 4096 x 4096 19 vs 22 us at 64, 23 vs 23 at 128, 27 vs 25 at 192, 30 vs 27 at 256;
# 8192 x 2048 24 vs 21 at 128; 1024 x 4096 (not enough workgroups even when split) 17 vs 14 us at 64.
_Q_TILE_MIN_GRID_FRACTION: float = 0.7
_Q_TILE_SPLIT_MAX_TOKENS: int = 144
# The same against decode + the library's product, which calls that record a gradient take: 4096 x 4096 24-31 vs 37-45 us
# from 128 to 256 tokens, 39-41 vs 39-40 us at 320-384.  Where it serves a call, gradients flow: the line is part of
# what the module does and stays where it is.
_Q_TILE_SPLIT_LIBRARY_MAX_TOKENS: int = 256
_Q_TILE_SPLIT_LONG_K: int = 8192
# Grids of more than half the compute units that are too large to split (8193 to 11456 output features): the fused GEMM
# from this K on, below it up to 256 tokens without zero points.  Decode + GEMM / fused, us at 36 / 100 / 256 / 384 tokens:
# 11008 x 4096 40 / 42 / 51 / 61 against 26 / 29 / 39 / 52, 8320 x 12288 93 / 108 / 132 / 151 against 48 / 56 / 81 / 114; 10240 x 2048
# 20 / 22 / 27 / 31 against 17 / 20 / 25 / 34, with zero points 20 / 22 / 27 / 32 against 22 / 23 / 29 / 39.
_Q_TILE_HALF_GRID_K: int = 4096
_Q_FUSED_MAX_TOKENS: int = 16
# 17..32 tokens: the GEMV reuses every dequantized operand for two 16-token tiles and beats the fused GEMM at any K where
# it reads whole lines (us at 24 / 32 tokens against the fused GEMM at 33: int4 14336 x 4096 20.6 / 21.2, 28; 4096 x 14336
# 19.8 / 21.6, 31; int8 14336 x 4096 22 / 24, 30; 4096 x 14336 24 / 25, 35), elsewhere while x is small (_gemv_max_tokens):
_Q_FUSED_WIDE_MAX_TOKENS: int = 32
_Q_FUSED_WIDE_MAX_ACTIVATIONS = {4: 1 << 18, 8: 1 << 17}  # tokens x in_features, by bit width
_Q_FUSED_WIDE_INT8_MAX_K: int = 8192

_ALLOW_FALLBACK: bool = os.environ.get("NEUROPRESS_ALLOW_KERNEL_FALLBACK", "").strip() in (
    "1", "true", "yes",
)  # fmt: skip


def _unpack_u8(u8_blob: torch.Tensor, nbits: int) -> torch.Tensor:
    """``[N, K/vpb]`` packed bytes -> ``[N, K]`` one value per byte (np_linear.py:78-97)."""
    return BitPacking(nbits).decompress(u8_blob)


def _pack_u8(values: torch.Tensor, nbits: int) -> torch.Tensor:
    """Inverse of :func:`_unpack_u8` (np_linear.py:100-118)."""
    return BitPacking(nbits).compress(values.to(torch.uint8))


def _kernel_blob(weight_q) -> torch.Tensor:
    """The weight's codes in the kernels' ``[N, K // vpb]`` layout (np_linear.py:121-138).

    A blob already bit-packed at the scheme's width has that layout and is reused.
    """
    nbits = weight_q.qscheme.n_bits
    comps = getattr(weight_q, "u8_compressors", None) or []
    if (
        len(comps) == 1
        and getattr(comps[0], "nbits", None) == nbits
        and weight_q.u8_blob.dim() == 2
    ):
        return weight_q.u8_blob
    return _pack_u8(weight_q.decompress_to_u8(), nbits)


def _resolve_backend(
    backend: str | LinearBackend | None,
    nbits: int | None = None,
    group_size: int | None = None,
) -> LinearBackend:
    """Resolve an alias to a concrete :class:`LinearBackend` (np_linear.py:166-213).

    ``"auto"``: ``CUDA`` (the HIP kernels) when a GPU and the kernel library
    are available, else ``COMPILE``.  The third-party GemLite backend the
    reference prefers is not part of this package; asking for it explicitly
    raises ``ValueError`` at construction.
    """
    if backend is None or backend == "torch":
        return LinearBackend.DEFAULT
    if isinstance(backend, (LinearBackend, Backend)):
        backend = backend.value
    if backend != "auto":
        return LinearBackend(backend)  # ValueError for unknown strings
    if torch.cuda.is_available() and is_hip_backend_available():
        return LinearBackend.CUDA
    return LinearBackend.COMPILE


def _q_dequant_weight(
    u8_blob: torch.Tensor,
    scale: torch.Tensor,
    nbits: int,
    group_size: int,
    zero_point: torch.Tensor | None,
) -> torch.Tensor:
    """f32 ``[N, K]`` weight with torch ops (the decode half of np_linear.py:333-351)."""
    n = u8_blob.shape[0]
    vals = _unpack_u8(u8_blob, nbits).to(torch.float32)
    k = vals.shape[1]
    g = k // group_size
    vals = vals.reshape(n, g, group_size)
    sc = scale.to(torch.float32).reshape(n, g, 1)
    zp = (
        zero_point.to(torch.float32).reshape(n, g, 1)
        if zero_point is not None
        else float(1 << (nbits - 1))
    )
    return ((vals - zp) * sc).reshape(n, k)


def _q_dequant_linear(
    x: torch.Tensor,
    u8_blob: torch.Tensor,
    scale: torch.Tensor,
    nbits: int,
    group_size: int,
    zero_point: torch.Tensor | None,
    bias: torch.Tensor | None,
) -> torch.Tensor:
    """Generic n-bit group-quantized dequant + linear with torch ops (np_linear.py:298-353)."""
    w = _q_dequant_weight(u8_blob, scale, nbits, group_size, zero_point)
    return F.linear(x, w.to(x.dtype), bias)


# What the choice of a kernel reads besides the buffers: a call plan is valid while these are unchanged.
_PLAN_ATTRIBUTES = ("backend", "out_features", "in_features", "group_size", "nbits", "zero_point", "bias")
_PLAN_THRESHOLDS = ("_Q_TILE_MAX_TOKENS", "_Q_TILE_LONG_K_MAX_TOKENS", "_Q_TILE_WIDE_MAX_TOKENS", "_Q_TILE_WIDE_MIN_FEATURES",
                    "_Q_TILE_MIN_GRID_FRACTION", "_Q_TILE_SPLIT_MAX_TOKENS", "_Q_TILE_SPLIT_LONG_K", "_Q_TILE_HALF_GRID_K",
                    "_Q_FUSED_MAX_TOKENS", "_Q_BLOCKS_MAX_TOKENS",
                    "_Q_FUSED_WIDE_MAX_TOKENS", "_Q_FUSED_WIDE_MAX_ACTIVATIONS", "_Q_FUSED_WIDE_INT8_MAX_K")  # fmt: skip


class NPLinear(nn.Module):
    """Linear layer with a packed n-bit quantized weight and a pluggable backend."""

    _plan = None  # CallPlan of the calls made so far (see forward)

    def __init__(
        self,
        u8_blob: torch.Tensor,
        scale: torch.Tensor,
        out_features: int,
        in_features: int,
        group_size: int,
        nbits: int,
        qtype: str,
        backend: str | LinearBackend | None,
        bias: torch.Tensor | None = None,
        zero_point: torch.Tensor | None = None,
        weight_q=None,
        qtensor_meta: dict[str, str] | None = None,
        compute_dtype: torch.dtype = torch.float16,
    ) -> None:
        super().__init__()
        if qtype not in ("sym", "asym"):
            raise ValueError(f"qtype must be 'sym' or 'asym', got {qtype!r}")
        self._qtensor_meta = qtensor_meta
        self.out_features = out_features
        self.in_features = in_features
        self.group_size = group_size
        self.nbits = nbits
        self.qtype = qtype
        self.backend = _resolve_backend(backend, nbits=nbits, group_size=group_size)
        if self.backend == LinearBackend.GEMLITE:
            raise ValueError("backend 'gemlite' is a third-party kernel not included in this package")
        self._compute_dtype = compute_dtype
        if weight_q is not None:
            object.__setattr__(self, "_weight_q", weight_q)

        self.register_buffer("u8_blob", u8_blob.contiguous())
        self.register_buffer("scale", scale.to(torch.float16).reshape(-1).contiguous())
        if zero_point is not None:
            self.register_buffer("zero_point", zero_point.to(torch.float16).reshape(-1).contiguous())
        else:
            self.zero_point = None
        if bias is not None:
            self.register_buffer("bias", bias.contiguous())
        else:
            self.bias = None
        self._derived: dict = {}

    def _apply(self, fn, recurse: bool = True):
        result = super()._apply(fn, recurse)
        self._derived = {}
        self._plan = None
        return result

    @classmethod
    def from_linear(
        cls, linear: nn.Linear, backend: str | LinearBackend | None = LinearBackend.AUTO
    ) -> NPLinear:
        """Build from an ``nn.Linear`` with a scalar-quantized weight (np_linear.py:539-607)."""
        wq = linear.weight
        if not is_scalar_qweight(wq):
            raise TypeError(
                f"Unsupported weight type {type(wq).__name__!r}. Expected a scale-only "
                "(symmetric) or scale+zero-point (asymmetric) quantized weight."
            )
        qs = wq.qscheme
        zp = None
        if getattr(qs, "zero_point", None) is not None:
            zp = qs.per_group_zero_point().detach() if hasattr(qs, "per_group_zero_point") else qs.zero_point
        bias = linear.bias.detach().clone() if linear.bias is not None else None
        return cls(
            u8_blob=_kernel_blob(wq),
            scale=qs.scale.detach().clone(),
            out_features=linear.out_features,
            in_features=linear.in_features,
            group_size=qs.group_size,
            nbits=qs.n_bits,
            qtype="sym" if zp is None else "asym",
            backend=backend,
            bias=bias,
            zero_point=zp,
            weight_q=wq,
            qtensor_meta={"dequant_to_dtype": str(getattr(wq, "dequant_to_dtype", torch.float16))},
            compute_dtype=getattr(wq, "dequant_to_dtype", torch.float16),
        )

    def to_qtensor(self) -> ScalarQWeight:
        """Rebuild the quantized weight; the packed blob is preserved bit for bit
        (the property tested at tests/test_quantized_weight_regressions.py:79-92 of the reference)."""
        if self._qtensor_meta is None:
            raise RuntimeError(
                "Cannot reconstruct QTensor: no serde metadata stored. "
                "Build via NPLinear.from_linear() to enable to_qtensor()."
            )
        scheme = ScalarQScheme(self.nbits, self.group_size, self.scale, self.zero_point)
        return ScalarQWeight(self.u8_blob, scheme, self._compute_dtype)

    def set_backend(self, backend: str | LinearBackend | None) -> NPLinear:
        """Switch backend in place; ``"auto"`` re-resolves now (np_linear.py:651-696)."""
        bk = _resolve_backend(backend, nbits=self.nbits, group_size=self.group_size)
        if bk == LinearBackend.GEMLITE:
            raise RuntimeError("backend 'gemlite' is not available in this package")
        self.backend = bk
        return self

    # ------------------------------------------------------------------

    def _bias_f32(self) -> torch.Tensor | None:
        if self.bias is None:
            return None
        # Keyed on the buffer's device, address and version counter: load_state_dict or an in-place
        # copy_ into `bias` makes a new fp32 copy.  Not stored inside a graph capture (a tensor made
        # there holds data only after a replay).
        src = self.bias
        key = (src.device, src.data_ptr(), tensor_version(src))
        hit = self._derived.get("bias_f32")
        if hit is not None and hit[0] == key:
            return hit[1]
        b = src.detach().to(torch.float32).contiguous()
        if not (src.is_cuda and torch.cuda.is_current_stream_capturing()):
            self._derived["bias_f32"] = (key, b)
        return b

    def _bias_as(self, dtype: torch.dtype) -> torch.Tensor | None:
        if self.bias is None or self.bias.dtype == dtype:
            return self.bias
        return self.bias.to(dtype)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        plan = self._plan
        if plan is not None:  # a call made before: same token count, dtype and buffers
            y = plan(self, x)
            if y is not None:
                return y
        if self.backend == LinearBackend.CUDA:
            return self._forward_cuda(x)
        # default / compile: the torch-op specification of the layer.
        return self._forward_compile(x)

    _planned_forward = forward  # module(x) may go straight to the plan (kernels/plans.py)

    def _forward_compile(self, x: torch.Tensor) -> torch.Tensor:
        return _q_dequant_linear(
            x, self.u8_blob, self.scale, self.nbits, self.group_size, self.zero_point,
            self._bias_as(x.dtype),
        )

    def _mfma_layer(self) -> bool:
        ok = self._derived.get("mfma_layer")
        if ok is None:
            from .. import kernels

            ok = kernels.q_fused_supported(self.in_features, self.nbits, self.group_size)
            self._derived["mfma_layer"] = ok
        return ok

    def _compute_units(self) -> int:
        cus = self._derived.get("cus")
        if cus is None:
            cus = torch.cuda.get_device_properties(self.u8_blob.device).multi_processor_count
            self._derived["cus"] = cus
        return cus

    def _tile_grid_fills_gpu(self, x: torch.Tensor, m: int, tracked: bool = False) -> bool:
        cus = self._compute_units()
        if tracked:
            return tile_band_ok(m, self.out_features, self.in_features, cus, _Q_TILE_MIN_GRID_FRACTION,
                                _Q_TILE_SPLIT_LIBRARY_MAX_TOKENS, _Q_TILE_SPLIT_LONG_K, library=True)  # fmt: skip
        return tile_band_ok(
            m, self.out_features, self.in_features, cus,
            _Q_TILE_MIN_GRID_FRACTION, _Q_TILE_SPLIT_MAX_TOKENS, _Q_TILE_SPLIT_LONG_K, _Q_FUSED_WIDE_MAX_TOKENS,
            self.in_features >= _Q_TILE_HALF_GRID_K or (self.zero_point is None and m <= 256),
            4096 if self.zero_point is None else 6144,
        )  # fmt: skip

    def _gemv_max_tokens(self, m: int, tracked: bool = False) -> int:
        """End of the GEMV band for a call of *m* tokens: 16, or 32 where a GEMV stays ahead of the fused GEMM.  *tracked*: as it
        is against decode + the library's product, which such calls take past it."""
        if _Q_FUSED_MAX_TOKENS < m <= _Q_FUSED_WIDE_MAX_TOKENS:
            from .. import kernels

            scales = (None, None) if tracked else (self.scale, self.zero_point)  # tracked: storage may be a trace's
            lines, staged = kernels.q_gemv_staging(m, self.out_features, self.in_features, self.nbits, self.group_size, *scales)
            # The GEMV that reads whole lines stays ahead of the tile GEMM at any K (GEMV at 24 / 32 tokens, tile GEMM at 33, us:
            # 4096 x 14336 int4 19.6 / 21.3, 30.7, int8 24.0 / 24.7, 35; 5888 x 7168 int4 15.7 / 16.6).  The other GEMV serves layers
            # with an odd count of scales or scales that start between two dwords.  Against the tile GEMM, us at 24 tokens:
            # int4 14336 x 14336 65.8 / 76.3, 4096 x 14336 22.9 / 26.8; int8, whose codes are twice the bytes, where no compute
            # unit has two row tiles and K is short, or too few have none for the tile GEMM to gain by its parts of K:
            # 4096 x 8192 17.2 / 19.3, 3584 x 14336 26.4 / 27.6, 1536 x 8192 13.9 / 14.5 and x 10240 16.5 / 14.9, 3072 x 14336
            # 26.0 / 24.5, 4904 x 8192 29.7 / 24.0, 14336 x 8192 52.8 / 47.5.
            tiles, cus = -(-self.out_features // 16), self._compute_units()
            if not tracked and (lines or self.nbits == 4 or (
                staged and tiles <= cus and (self.in_features <= _Q_FUSED_WIDE_INT8_MAX_K or 5 * tiles >= 4 * cus)
            )):  # fmt: skip
                return _Q_FUSED_WIDE_MAX_TOKENS
            # Calls that record a gradient, where the line is part of what the module does: while x is small, past that
            # int4 where the other GEMV stages its activations.
            cap = _Q_FUSED_WIDE_MAX_ACTIVATIONS.get(self.nbits, 0)
            if self.zero_point is not None and self.nbits == 4:
                cap = 1 << 30  # the fused GEMM pays for the zero points per tile: GEMV at any K
            if m * self.in_features <= cap or (staged and self.nbits == 4):
                return _Q_FUSED_WIDE_MAX_TOKENS
        return _Q_FUSED_MAX_TOKENS

    def _forward_cuda(self, x: torch.Tensor) -> torch.Tensor:
        """HIP path by token count; takes the place of np_linear.py:731-761."""
        if not x.is_cuda:
            return self._forward_compile(x)
        from .. import kernels

        m = x.numel() // self.in_features
        try:
            tracked = kernels.tracked(x, self.bias)
            band = self._band(x, m, tracked)
            if not tracked and not torch.cuda.is_current_stream_capturing():
                y = self._planned(x, m, band)
                if y is not None:
                    return y
            if band == "blocks" and kernels.replaced("q_gemm_tile", "q_dequant", "dense_linear"):
                band = self._band(x, m, tracked, blocks=False)  # whose function a caller has put another in the place of
            if band != "dense":
                fn = {"fused": kernels.q_linear, "blocks": kernels.q_linear_blocks}.get(band, kernels.q_gemm_tile)
                return fn(x, self.u8_blob, self.scale, self.nbits, self.group_size, self.zero_point, self._bias_f32())
            w = kernels.q_dequant(
                self.u8_blob, self.scale, self.nbits, self.group_size, self.zero_point, x.dtype
            )
        except RuntimeError as exc:
            if not _ALLOW_FALLBACK:
                raise
            kernels.warn_kernel_fallback("q_linear", "torch dequant + matmul", exc)
            return self._forward_compile(x)
        if self._own_product(m, x.dtype) and not tracked:
            return kernels.dense_linear(x.reshape(-1, self.in_features), w, self._bias_f32()).reshape(*x.shape[:-1], self.out_features)
        return F.linear(x, w, self._bias_as(x.dtype))

    def _own_product(self, m: int, dtype: torch.dtype) -> bool:
        """Whether the dense product of a decode + GEMM call is the package's own kernel."""
        from .. import kernels

        return dtype in (torch.float16, torch.bfloat16) and kernels.dense_preferred(m, self.out_features, self.in_features)

    def _band(self, x: torch.Tensor, m: int, tracked: bool = False, blocks: bool = True) -> str:
        """Which kernel serves a call of *m* tokens: ``fused`` (GEMV), ``blocks`` (GEMV, a workgroup per 32 tokens), ``tile`` (fused GEMM) or ``dense`` (decode + GEMM).
        *tracked* (``kernels.tracked(x)``): the dense product is the library's, and so are the limits against it.  *blocks* False: what ``blocks``
        takes the place of."""
        # Layers the MFMA kernels do not take (1 / 2 / 8 bits, odd group sizes) would run an
        # element-wise kernel, slower at every token count than decoding once and calling the
        # dense GEMM (14336 x 4096, 8 bits: 99 us against 57 us at one token, 452 against 57 at 16).
        if x.dtype not in (torch.float16, torch.bfloat16) or not self._mfma_layer():
            return "dense"
        if m <= self._gemv_max_tokens(m, tracked):
            return "fused"
        limit = _Q_TILE_MAX_TOKENS
        if self.in_features >= _Q_TILE_SPLIT_LONG_K:
            limit = max(limit, _Q_TILE_LONG_K_MAX_TOKENS)
        if limit > 0 and max(self.in_features, self.out_features) >= _Q_TILE_WIDE_MIN_FEATURES:
            limit = max(limit, _Q_TILE_WIDE_MAX_TOKENS)
        tile = m <= limit and self._tile_grid_fills_gpu(x, m, tracked)
        if blocks and not tracked and self._blocks_win(m, tile):
            return "blocks"
        return "tile" if tile else "dense"

    def _blocks_win(self, m: int, tile: bool = True) -> bool:
        """Whether the GEMV with a workgroup per 32 tokens is ahead of the fused GEMM (*tile*) and of decode + GEMM.  Layers of fewer than
        256 output features, the least that the estimates were checked on, keep those (NPVQLinear._blocks_win), though most would gain: decode +
        GEMM / this, int4, us at 64 tokens 64 x 512 7.8 / 4.2, 200 x 4096 11.8 / 6.6, at 1024 tokens 128 x 8192 14.2 / 21.1."""
        from .. import kernels

        if not 16 < m <= _Q_BLOCKS_MAX_TOKENS or self.out_features < 256 or min(_Q_FUSED_MAX_TOKENS, _Q_TILE_MAX_TOKENS) <= 0:
            return False
        # By sizes first: every token count a layer meets asks, and most of them get their answer there.
        if not kernels.gemv_blocks_preferred(m, self.out_features, self.in_features, self.nbits, tile=tile):
            return False
        if self.u8_blob.data_ptr() % 16:
            return False  # a slice of a larger buffer, say: the entry refuses it, the kernels it takes the place of serve it
        lines, _ = kernels.q_gemv_staging(
            _lib.GEMV_MAX_M, self.out_features, self.in_features, self.nbits, self.group_size, self.scale, self.zero_point
        )
        return lines

    def _planned(self, x: torch.Tensor, m: int, band: str):
        """Add this call to the layer's plan and let the plan issue it; None where it cannot."""
        from ..kernels import plans

        n, k = self.out_features, self.in_features
        if m < 1 or x.dtype not in plans.DTYPE_CODES or x.device != self.u8_blob.device or (
            self.u8_blob.dtype != torch.uint8 or self.scale.dtype != torch.float16
            or tuple(self.u8_blob.shape) != (n, k * self.nbits // 8) or self.scale.numel() * self.group_size != n * k
            or (self.zero_point is not None
                and (self.zero_point.numel() != self.scale.numel() or self.zero_point.dtype != torch.float16))
        ):  # fmt: skip
            return None
        plan = self._plan
        if plan is None or plan.stale(self):
            plan = plans.make(self, _PLAN_ATTRIBUTES, globals(), _PLAN_THRESHOLDS,
                              sources=(self.u8_blob, self.scale, self.zero_point, self.bias))  # fmt: skip
            if plan is None:
                return None
        code = plans.DTYPE_CODES[x.dtype]
        if band == "dense" and self._own_product(m, x.dtype):
            band = "product"
        number = plan.names.get((band, x.dtype))
        if number is None:
            kind = {"fused": plans.Q_GEMV, "blocks": plans.Q_BLOCKS, "tile": plans.Q_TILE}.get(band, plans.Q_DENSE)
            args = (self.u8_blob, self.scale, self.zero_point, self._bias_f32(), 0, 0, self.nbits, self.group_size, code)
            bias = self._bias_as(x.dtype) if band == "dense" else self._bias_f32() if band == "product" else None
            number = plan.names[band, x.dtype] = plans.template(plan, kind, n, k, args, x.dtype, bias=bias, leaf=self.bias, own=band == "product")
        scratch = {"tile": plans.tile_scratch, "product": plans.product_scratch}.get(band)
        plan.route(code, m, number, scratch(m, n, k) if scratch else 0)
        self._plan = plan
        return None if plan.wrapped() else plan.run(x)

    def extra_repr(self) -> str:
        return (
            f"in={self.in_features}, out={self.out_features}, "
            f"nbits={self.nbits}, group_size={self.group_size}, "
            f"qtype={self.qtype}, backend={self.backend.value}"
        )


def linearize_qtensor_weights(
    model: nn.Module,
    backend: str | LinearBackend | None = LinearBackend.AUTO,
) -> nn.Module:
    """Replace every ``nn.Linear`` carrying a scalar-quantized weight with an :class:`NPLinear`.

    Follows neuropress/nn/np_linear.py:796-871; VQ weights are left to
    :func:`~neuropress_amd.nn.np_vq_linear.linearize_vq_weights`.
    """
    replacements: list[tuple[str, NPLinear]] = []
    for name, module in model.named_modules():
        if not isinstance(module, nn.Linear) or not is_scalar_qweight(module.weight):
            continue
        try:
            layer = NPLinear.from_linear(module, backend)
        except (TypeError, ValueError) as exc:
            log.warning("linearize_qtensor_weights: skipping %s — %s", name, exc)
            continue
        replacements.append((name, layer))

    for name, layer in replacements:
        if "." in name:
            parent_name, attr = name.rsplit(".", 1)
            parent = model.get_submodule(parent_name)
        else:
            parent, attr = model, name
        setattr(parent, attr, layer)

    counts: dict[str, int] = {}
    for _, layer in replacements:
        counts[layer.backend.value] = counts.get(layer.backend.value, 0) + 1
    summary = ", ".join(f"{v}x{k}" for k, v in sorted(counts.items()))
    log.info(
        "linearize_qtensor_weights: replaced %d layer(s) [%s]", len(replacements), summary or "none"
    )
    return model
