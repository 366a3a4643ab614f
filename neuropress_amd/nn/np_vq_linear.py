"""NPVQLinear: drop-in ``nn.Linear`` replacement with a VQ-compressed weight.

The weight is a packed stream of codebook indices plus a codebook shared
through a :class:`VQProxy`:

    ``W[n, g*VL + v] = centroids[idx[n * n_groups + g], v]``

Same module surface as the reference (neuropress/nn/np_vq_linear.py:399-1517):
``VQProxy``, ``NPVQLinear(proxy, packed_indices, bits, out_features, in_features,
vector_len, backend, bias, column_perm, ...)``, ``from_qtensor_linear``,
``to_qtensor``, ``forward``, ``linearize_vq_weights``.  What differs is what runs
underneath: hand-written gfx950 kernels instead of CUDA/Triton, selected by
token count ``m = x.numel() // in_features``:

====================  ==============================  ==========================
band                  condition                        kernel
====================  ==============================  ==========================
(a) fused GEMV        ``m <= _FUSED_MAX_TOKENS``, or   ``kernels.vq_linear``
                      ``m <= 32`` while x is small
    slice GEMM        up to 32 tokens of large tables, ``kernels.vq_slice_gemm``
                      where timed lists say so (one
                      token: only where they lost)
(b) tile-decode GEMM  ``m <= _TILE_MAX_TOKENS``        ``kernels.vq_gemm_tile``
    table GEMM        past 16 tokens where its         ``kernels.vq_linear_blocks``
                      estimate is the least (up to
                      4096 rows; small layers: a GEMV
                      with a workgroup per 32 tokens)
(c) decode + GEMM     otherwise                        ``kernels.vq_dequant`` + ``kernels.dense_linear`` or ``F.linear``
====================  ==============================  ==========================

Only band (c) with ``F.linear`` carries gradients, tangents and the like: calls that ask for them
(``kernels.tracked``) take it instead of ``dense_linear``, at the token counts where it was the faster one against
the other bands.

The dispatch rule itself is the reference's (np_vq_linear.py:1014-1058); the
thresholds are re-derived for one MI355X and stay overridable through the same
environment variables.  Prefix-coded index formats (tiered / n-tier /
zero-escape) are expanded to the fixed-width stream once, at construction.
"""

from __future__ import annotations

import logging
import os
import weakref

import torch
import torch.nn as nn
import torch.nn.functional as F

from ..qweights import VQScheme, VQWeight, is_vq_weight
from ..transforms.vq_entropy_packing import decode_to_flat
from ..transforms.vq_packing import (
    IndexPacking,
    NTieredIndexPacking,
    TieredIndexPacking,
    ZeroEscapePacking,
)
from . import backends
from .backends import Backend, VQBackend, is_hip_backend_available, tensor_version, tile_band_ok

log = logging.getLogger(__name__)

_unprepared_warned = False


def _warn_unprepared_once() -> None:
    """One WARNING per process when a layer meant for the slice-list GEMV runs without its lists."""
    global _unprepared_warned
    if not _unprepared_warned:
        _unprepared_warned = True
        log.warning(
            "NPVQLinear: a layer with a codebook of more than 4096 rows has no slice lists for its current "
            "buffers (never prepared, or its indices were reloaded): decode steps run the slower fused GEMV.  "
            "Call neuropress_amd.prepare_decode(model) once the model is on its GPU."
        )


def _env_int(names: tuple[str, ...], default: int) -> int:
    for name in names:
        v = os.environ.get(name)
        if v is not None and v.strip():
            return int(v)
    return default


# Token-count bands (tokens = rows of the flattened input), read once at import
# like the reference's (np_vq_linear.py:73-87).  The fused GEMV issues the
# contraction as 16-row MFMA tiles, so 1..16 tokens cost the same: the fused
# band ends at 16 here (2 in the reference, whose GEMV re-reads the weight per token).
_FUSED_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_FUSED_MAX_TOKENS",), 16)
# 17..32 tokens: the GEMV reuses every decoded operand for two 16-token tiles.  Each of its
# workgroups reads all of x from L2, so it wins while x is small (tokens x in_features at most
# _FUSED_WIDE_MAX_ACTIVATIONS).  Measured, GEMV vs tile GEMM at 17 / 24 / 32 tokens, bf16:
# 14336 x 4096, 4096-row codebook 15.7 / 16.7 / 15.1 vs 22 us, 65536-row 39.2 / 40.2 / 41.6 vs 39 us;
# 4096 x 4096 7.1 / 7.6 / 9.6 vs 12.7 us; 4096 x 14336 15.7 / 17.3 / 24.0 vs 22.4 / 22.8 / 23.5 us.  Residual
# layers 31-32 vs 32 us (14336 x 4096): GEMV at any length.
_FUSED_WIDE_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_FUSED_WIDE_MAX_TOKENS",), 32)
_FUSED_WIDE_MAX_ACTIVATIONS: int = 1 << 18
_GEMV_KERNEL_MAX_TOKENS: int = 32  # what the GEMV entry points accept (NPAMD_GEMV_MAX_M)

# Decode steps (1-7 tokens) of layers whose codebook is too large to sit in a
# compute unit's LDS next to the GEMV's buffers (more than 4096 rows): the fused
# GEMV then pays one L2 lookup per index (34-35 us on a 14336 x 4096 layer with a
# 65536-row codebook, any token count up to 16), while the slice-list GEMV
# (kernels.vq_linear_sliced) keeps 4096-row codebook slices in LDS: 10.3-10.9 / 14.2 /
# 20.3 / 30.9 us at 1 / 2 / 4 / 7 tokens; an eighth token needs a second pass over the
# entries.  The slice lists are built on the host by prepare_sliced() / prepare_decode(),
# never by forward() (about 26 MB per such layer, on top of the packed stream the other
# bands keep reading).  0 disables the path.
_SLICED_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_SLICED_MAX_TOKENS",), 7)
_SLICED_MIN_CENTROIDS: int = 4097
_SLICED_MIN_INDICES: int = _env_int(("NEUROPRESS_VQ_SLICED_MIN_INDICES",), 1 << 20)
# The slice GEMM (kernels.vq_slice_gemm) for the same layers: whole 8192-row slices of the codebook in LDS, up to 32 tokens at
# once.  Its time does not depend on the indices, that of the kernels that look rows up in memory does: which one is
# faster is asked of the times taken when the slice lists were made.  Slice GEMM / fused GEMV or tile GEMM, us at 3 / 16 / 32
# tokens: 4096 x 14336 with 65536 rows 26 / 28 / 39 against 36 / 39 / 41, with 16384 14.6 / 16.6 / 20.6 against 33.7 / 36.9 / 38.5,
# 14336 x 4096 with 8192 rows 13.1 / 14.9 / 18.6 against 29.5 / 33.4 / 34.3; 4096 x 4096 with 65536 rows 12.8 / 15 / 20.5 against
# 12 / 13 / 14, with 8192 8.2 / 8.9 / 11.2 against 10.4 / 11.3 / 12.3.
_SLICE_GEMM_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_SLICE_GEMM_MAX_TOKENS",), 32)
_SLICE_GEMM_GATHER_US: float = 3.0  # of a column permutation, which the slice lists and some fused GEMVs apply themselves

# Whether a module that reaches a GPU through .to() / .cuda() / load_state_dict() builds the tensors
# its kernels derive from the buffers there and then (slice lists: a host round trip per layer).
_PREPARE_ON_MOVE: bool = _env_int(("NEUROPRESS_VQ_PREPARE_ON_MOVE",), 1) != 0

# cuda_lut layers: 0 = always decode + GEMM, the reference's default routing.
_LUT_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_LUT_MAX_TOKENS",), 0)

# Most tokens of the GEMV with a workgroup per 32 tokens, which serves small layers past 16 of them, and of the table GEMM behind the same
# entry point, which serves layers of any size with a codebook of up to 4096 rows (kernels.gemv_blocks_preferred).
_BLOCKS_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_BLOCKS_MAX_TOKENS",), 1 << 16)
# Upper end of the tile-decode GEMM band.  NEUROPRESS_VQ_TRITON_MAX_TOKENS is the
# reference's name for the same knob and is honoured too.  0 disables the band.
# Measured on one MI355X (14336 x 4096 layer): the tile GEMM beats decode + GEMM
# from 17 to about 320 tokens (58 vs 67 us at 64, 74 vs 86 us at 256, 100 vs 96 us
# at 384, 190 vs 101 us at 512, where a second row block re-decodes the weight).
_TILE_MAX_TOKENS: int = _env_int(
    ("NEUROPRESS_VQ_TILE_MAX_TOKENS", "NEUROPRESS_VQ_TRITON_MAX_TOKENS"), 256
)

# Layers whose codebook LDS does not hold (more than 4096 rows of eight) run the 128-column tile GEMM,
# which splits the reduction by itself and stays ahead of decode + GEMM up to a token count that goes
# with the layer's weights and with K (us at 96 / 144 / 230 / 384 tokens, tile against decode + dense product):
# 4096 x 14336 44 / 50 / 57 / 73 against 66 / 81 / 78 / 97; 3152 x 7296 26 / 31 / 36 / 47 against 45 / 42 / 46 / 53,
# 2048 x 10752 24 / 30 / 34 / 43 against 33 / 35 / 38 / 46; 1024 x 8192 16 / 21 / 23 / 29 against 20 / 22 / 24 / 27;
# 4096 x 4096 24 / 27 / 29 / 37 against 27 / 26 / 30 / 35, 2048 x 4096 16 / 21 / 23 / 28 against 19 / 20 / 22 / 24; and at
# 64 / 128 / 256 tokens 8192 x 2048 22 / 29 / 35 against 23 / 25 / 30, 3008 x 2240 15 / 19 / 26 against 15 / 16 / 18,
# 1024 x 4096 15 / 19 / 24 against 15 / 16 / 17, 2048 x 2048 13 / 15 / 22 against 12 / 12 / 13.
_TILE_WIDE_MAX_TOKENS: int = _env_int(("NEUROPRESS_VQ_TILE_WIDE_MAX_TOKENS",), 384)
_TILE_WIDE_MIN_WEIGHTS: int = 1 << 25  # below: 384 tokens only with _MID_LAYER_K features on _MID_LAYER_WEIGHTS
# Column blocks that nearly fill the GPU by themselves (K in two or three parts): 256 tokens.  At 200 tokens, tile / decode +
# product: 11008 x 2048 31.6 / 35.1, 10000 x 3072 40.7 / 46.5, 14336 x 2048 35.3 / 39.8; 8192 x 2048 33 / 27.
_TILE_WIDE_BROAD_WEIGHTS: int = 1 << 24
_TILE_WIDE_BROAD_FEATURES: int = 9216
_TILE_WIDE_TINY_WEIGHTS: int = 5_000_000  # below: 32 tokens, where the GEMV ends
_TILE_WIDE_LONG_MAX_TOKENS: int = 256  # _MID_LAYER_WEIGHTS and K of 4096, or _SMALL_LAYER_WEIGHTS and K of _TILE_SPLIT_LONG_K
_TILE_WIDE_MID_MAX_TOKENS: int = 128  # _SMALL_LAYER_WEIGHTS and K of 4096
_TILE_WIDE_SMALL_MAX_TOKENS: int = 64  # all others
# Against decode + the library's product, which calls that record a gradient take: layers of _TILE_WIDE_BROAD_WEIGHTS, half
# of it below (us at 128 / 256 / 384 tokens, tile against decode + library product: 6144 x 4096 32 / 41 / 56 against 47 / 61 / 55,
# 8192 x 2048 28 / 34 / 46 against 34 / 40 / 38; 1024 x 4096 18 / 24 / 29 against 20 / 21 / 22).  Where that product
# serves a call, gradients flow: the line is part of what the module does and stays where it is.
_TILE_WIDE_LIBRARY_MAX_TOKENS: int = 256

# The tile GEMM gives each workgroup 64 output columns (and up to 384 rows).  When
# that grid covers less than this fraction of the compute units the kernel splits
# the reduction over up to 16 workgroups per tile (at least 512 input features
# each); a layer that still cannot cover the fraction takes decode + GEMM.
_TILE_MIN_GRID_FRACTION: float = 0.7

# Upper end of the band for layers that need the split.  Measured on one MI355X,
# tile GEMM vs decode + GEMM: 4096 x 14336 layer 51-60 vs 75-113 us up to 128
# tokens and 82 vs 101 us at 256; 4096 x 4096 layer 25-31 vs 30-39 us up to 128
# tokens, 39 vs 36 us at 256.
_TILE_SPLIT_MAX_TOKENS: int = 128
# Small layers (fewer than 8 M weights) decode in 4-8 us and leave the band earlier; residual ones at 32 tokens.
_TILE_SMALL_LAYER_MAX_TOKENS: int = 64
# Grids of more than half the compute units that are too large to split (8193 to 11456 output features): the tile GEMM up
# to 256 tokens, fewer on very long reductions.  Decode + GEMM / tile, us at 36 / 100 / 256 tokens: 11008 x 4096 with a
# 256-row codebook 44 / 46 / 53 against 18 / 20 / 36, with 4096 rows 38 / 40 / 50 against 21 / 24 / 43, residual 43 / 45 / 55
# against 34 / 39 / 51; 8320 x 12288 with 256 rows 69 / 76 / 105 against 43 / 53 / 109, residual 121 / 127 / 152 against 83 / 107 / 164.
_TILE_HALF_GRID_MAX_ACTIVATIONS: int = 5 << 19  # tokens x K
_TILE_SPLIT_LONG_K: int = 8192  # from this many input features on, _TILE_MAX_TOKENS applies
# Layers of at least this many indices time their slice-list GEMV against the fused one when the
# lists are built (NPVQLinear._sliced_token_limit).
_SLICED_TUNE_MIN_INDICES: int = 1 << 20
# Residual layers take the tile band under the same grid rule as plain ones.  Measured, tile
# GEMM vs decode + GEMM, bf16, 33 / 128 / 256 tokens: 14336 x 4096 53 / 56 / 72 against 75 / 76 /
# 92 us; 4096 x 4096 26 / 31 / 40 against 33 / 42 / 41 us; 4096 x 14336 54 / 63 / 84 against
# 78 / 107 / 100 us; 1024 x 4096 (too few column blocks, decode + GEMM by the grid rule) 20 / 22 /
# 27 against 24 / 21 / 22 us.

# Opt-in: when a HIP kernel call fails, warn once and run torch ops instead (the
# reference's behaviour).  Off by default so a missing or broken kernel library
# is an error, not a silent slow path.
_ALLOW_FALLBACK: bool = os.environ.get("NEUROPRESS_ALLOW_KERNEL_FALLBACK", "").strip() in (
    "1", "true", "yes",
)  # fmt: skip

# Backends that run the HIP bands.  The three per-format members name, in the reference, kernels
# that decode a prefix-coded stream inside the GEMV; here such layers are expanded to the fixed-width
# stream at construction, so the members are labels that route like CUDA_WMMA.
_CODED_BACKENDS = frozenset({VQBackend.CUDA_TIERED, VQBackend.CUDA_NTIER, VQBackend.CUDA_ZERO_ESCAPE})
_FUSED_BACKENDS = frozenset({VQBackend.CUDA_WMMA, VQBackend.CUDA_LUT, VQBackend.CUDA}) | _CODED_BACKENDS

# What the band decision reads besides the buffers: a call plan is valid while these are unchanged.
_PLAN_ATTRIBUTES = ("backend", "proxy", "residual_proxy", "out_features", "in_features", "vector_len", "bits", "residual_bits",
                    "bias", "column_perm", "packed_residual", "row_scale", "row_bias")  # fmt: skip
_PLAN_THRESHOLDS = ("_FUSED_MAX_TOKENS", "_FUSED_WIDE_MAX_TOKENS", "_FUSED_WIDE_MAX_ACTIVATIONS", "_SLICED_MAX_TOKENS",
                    "_SLICED_MIN_CENTROIDS", "_SLICED_MIN_INDICES", "_SLICE_GEMM_MAX_TOKENS", "_SLICE_GEMM_GATHER_US", "_LUT_MAX_TOKENS", "_BLOCKS_MAX_TOKENS", "_TILE_MAX_TOKENS", "_TILE_WIDE_MAX_TOKENS",
                    "_TILE_WIDE_MIN_WEIGHTS", "_TILE_WIDE_BROAD_WEIGHTS", "_TILE_WIDE_BROAD_FEATURES",
                    "_TILE_WIDE_TINY_WEIGHTS", "_TILE_WIDE_MID_MAX_TOKENS",
                    "_TILE_WIDE_LONG_MAX_TOKENS", "_TILE_WIDE_SMALL_MAX_TOKENS", "_TILE_SMALL_LAYER_MAX_TOKENS",
                    "_TILE_MIN_GRID_FRACTION", "_TILE_SPLIT_MAX_TOKENS", "_TILE_SPLIT_LONG_K",
                    "_TILE_HALF_GRID_MAX_ACTIVATIONS", "_tile_failed")  # fmt: skip

# Latched once the tile GEMM fails with fallback allowed, so later calls go
# straight to decode + GEMM (reference: np_vq_linear.py:91-93).
_tile_failed: bool = False

# Index widths the fast kernels stream directly; other widths are widened to
# 16 bits once, on first GPU use.
_FAST_BITS = frozenset({4, 8, 12, 16})


def _fused_max_tokens(backend: VQBackend) -> int:
    """Largest token count for which *backend*'s fused kernel is used."""
    return _LUT_MAX_TOKENS if backend == VQBackend.CUDA_LUT else _FUSED_MAX_TOKENS


def _resolve_vq_backend(
    backend: str | VQBackend | Backend | None,
    use_tiered: bool = False,
    use_ntier: bool = False,
    use_zero_escape: bool = False,
    bits: int = 8,
    out_features: int = 0,
    num_centroids: int = 0,
    vector_len: int = 8,
) -> VQBackend:
    """Resolve a backend alias to a concrete :class:`VQBackend` (never ``AUTO``).

    Signature and alias handling follow the reference
    (neuropress/nn/np_vq_linear.py:101-170): ``None`` / ``"torch"`` ->
    ``DEFAULT``, unknown strings raise ``ValueError``.  ``"auto"`` on a machine
    where the HIP library can run resolves to ``CUDA_WMMA`` -- the three-band
    path -- for every codebook size and vector length: the reference's detours
    (vector_len != 4 -> COMPILE, bits > 12 -> CUDA_LUT) exist because its
    tensor-core kernels are fixed to VL = 4 and a 4096-entry shared-memory
    codebook; the kernels here have neither limit.  Without a GPU ``"auto"``
    resolves to ``COMPILE`` as in the reference.
    """
    if backend is None or backend == "torch":
        return VQBackend.DEFAULT
    if isinstance(backend, (VQBackend, Backend)):
        val = backend.value
    elif isinstance(backend, str):
        val = backend
    else:
        val = str(backend)
    if val != "auto":
        return VQBackend(val)  # raises ValueError for unknown strings
    if not (torch.cuda.is_available() and is_hip_backend_available()):
        return VQBackend.COMPILE
    # Same precedence as the reference (np_vq_linear.py:158-163); all four run the same kernels.
    if use_zero_escape:
        return VQBackend.CUDA_ZERO_ESCAPE
    if use_ntier:
        return VQBackend.CUDA_NTIER
    if use_tiered:
        return VQBackend.CUDA_TIERED
    return VQBackend.CUDA_WMMA


def _vq_dequant_linear(
    x: torch.Tensor,
    packed_indices: torch.Tensor,
    centroids: torch.Tensor,
    bits: int,
    n_vectors: int,
    out_features: int,
    in_features: int,
    bias: torch.Tensor | None,
) -> torch.Tensor:
    """Unpack, gather, ``F.linear`` with torch ops: the specification of the layer.

    Follows neuropress/nn/np_vq_linear.py:178-211.  Runs on whatever device the
    buffers live on; used by the ``default`` / ``compile`` backends.
    """
    indices = IndexPacking.unpack(packed_indices, bits, n_vectors)
    w = centroids[indices].reshape(out_features, in_features)
    return F.linear(x, w.to(x.dtype), bias)


# ---------------------------------------------------------------------------
# VQProxy — shared codebook
# ---------------------------------------------------------------------------


class VQProxy(nn.Module):
    """Shared VQ codebook holder (reference: neuropress/nn/np_vq_linear.py:399-455).

    Holds ``centroids`` ``[num_centroids, vector_len]`` as a float16 buffer.
    One instance is shared by every :class:`NPVQLinear` of a quantization group
    and is registered on the model root, not on each layer.
    """

    centroids: torch.Tensor

    def __init__(self, centroids: torch.Tensor) -> None:
        super().__init__()
        self.register_buffer("centroids", centroids.to(torch.float16))
        self._cast_cache: dict = {}
        # Layers that read this codebook (weakly held, not copied or pickled with the proxy): told
        # when the codebook moves or is reloaded, because a parent's .to() may move a layer first.
        self._users: weakref.WeakSet = weakref.WeakSet()
        self.register_load_state_dict_post_hook(VQProxy._after_load_state_dict)

    def _bind(self, user: nn.Module) -> None:
        self._users.add(user)

    def _notify_users(self) -> None:
        for user in list(self._users):
            if user.proxy is self or user.residual_proxy is self:
                user._prepare_after_move()

    def _apply(self, fn, recurse: bool = True):
        result = super()._apply(fn, recurse)
        self._cast_cache = {}
        self._notify_users()
        return result

    @staticmethod
    def _after_load_state_dict(module, incompatible_keys) -> None:
        module._cast_cache = {}
        module._notify_users()

    def __getstate__(self):
        state = self.__dict__.copy()
        state.pop("_users", None)
        return state

    def __setstate__(self, state):
        super().__setstate__(state)
        self._users = weakref.WeakSet()

    @property
    def num_centroids(self) -> int:
        return self.centroids.shape[0]

    @property
    def vector_len(self) -> int:
        return self.centroids.shape[1]

    def centroids_as(self, dtype: torch.dtype) -> torch.Tensor:
        """The codebook cast to *dtype*, cached until the buffer moves or changes.

        A bf16 model multiplies by bf16-rounded codebook rows (that is what
        ``W.to(x.dtype)`` means); casting the table once keeps that conversion
        out of the kernels' inner loops.
        """
        c = self.centroids
        if dtype == c.dtype:
            return c
        key = (dtype, c.device, c.data_ptr(), tensor_version(c))
        hit = self._cast_cache.get("entry")
        if hit is None or hit[0] != key:
            hit = (key, c.to(dtype).contiguous())
            self._cast_cache["entry"] = hit
        return hit[1]

    def extra_repr(self) -> str:
        return f"num_centroids={self.num_centroids}, vector_len={self.vector_len}"

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        raise RuntimeError(
            "VQProxy.forward() should not be called.  Access centroids "
            "directly via self.proxy.centroids."
        )


# ---------------------------------------------------------------------------
# NPVQLinear
# ---------------------------------------------------------------------------


class NPVQLinear(nn.Module):
    """Linear layer with a VQ-compressed weight and a shared codebook proxy.

    Constructor arguments up to ``zesc_row_offsets`` are the reference's
    (neuropress/nn/np_vq_linear.py:493-513).  With ``use_tiered`` / ``tier_bits`` /
    ``zero_escape`` the buffer passed as ``packed_indices`` is a prefix-coded one
    (``transforms/vq_entropy_packing.py``): it is expanded once, here, into the
    fixed-width stream all kernels read (``self.packed_indices``, ``self.bits`` wide),
    so these layers run the same three bands as any other; the ``*_row_offsets``
    arguments, which the reference's per-format kernels need, are accepted and
    unused, and :meth:`to_qtensor` packs the indices back.  The
    ``residual_*`` / ``row_*`` arguments add an optional residual codebook and
    a per-output-row fp16 scale and bias on the decoded weight:

        ``W[n, :] = ((Cm[im] + Cr[ir]) * row_scale[n]) + row_bias[n]``

    each operation rounded to fp16 (the benchmark's residual-VQ configuration; not in the reference).
    """

    _plan = None  # CallPlan of the calls made so far (see forward)

    def __init__(
        self,
        proxy: VQProxy,
        packed_indices: torch.Tensor,
        bits: int,
        out_features: int,
        in_features: int,
        vector_len: int,
        backend: str | VQBackend | None,
        bias: torch.Tensor | None = None,
        column_perm: torch.Tensor | None = None,
        use_tiered: bool = False,
        cold_bits: int = 8,
        hot_row_offsets: torch.Tensor | None = None,
        cold_row_offsets: torch.Tensor | None = None,
        qtensor_meta: dict[str, str] | None = None,
        tier_bits: list[int] | None = None,
        ntier_row_offsets: list[torch.Tensor] | None = None,
        zero_escape: bool = False,
        zesc_row_offsets: list[torch.Tensor] | None = None,
        residual_proxy: VQProxy | None = None,
        packed_residual: torch.Tensor | None = None,
        residual_bits: int = 0,
        row_scale: torch.Tensor | None = None,
        row_bias: torch.Tensor | None = None,
    ) -> None:
        super().__init__()
        if in_features % vector_len:
            raise ValueError(f"in_features={in_features} not divisible by vector_len={vector_len}")
        if proxy.vector_len != vector_len:
            raise ValueError(f"vector_len={vector_len} does not match the codebook ({proxy.vector_len})")
        self._qtensor_meta = qtensor_meta
        self.out_features = out_features
        self.in_features = in_features
        self.vector_len = vector_len
        self.bits = bits
        self.n_vectors = out_features * (in_features // vector_len)
        # Same precedence as the reference's scheme (neuropress/transforms/vq.py:220-247).
        self.zero_escape = bool(zero_escape)
        self.tier_bits = None if zero_escape or tier_bits is None else list(tier_bits)
        self.use_tiered = bool(use_tiered) and not zero_escape and tier_bits is None
        self.cold_bits = cold_bits
        self._hot_bits = TieredIndexPacking.DEFAULT_HOT_BITS
        self._coded_bits = bits
        if self.zero_escape or self.tier_bits is not None or self.use_tiered:
            packed_indices, bits = self._expand_prefix_coded(packed_indices, proxy.num_centroids)
            self.bits = bits
        self.backend = _resolve_vq_backend(
            backend,
            use_tiered=self.use_tiered,
            use_ntier=self.tier_bits is not None,
            use_zero_escape=self.zero_escape,
            bits=bits,
            out_features=out_features,
            num_centroids=proxy.num_centroids,
            vector_len=vector_len,
        )
        need = IndexPacking.packed_nbytes(self.n_vectors, bits)
        if packed_indices.numel() < need:
            raise ValueError(
                f"packed_indices holds {packed_indices.numel()} bytes, {need} needed for "
                f"{self.n_vectors} indices of {bits} bits"
            )

        # The proxy is a plain attribute, not a sub-module: it must not appear
        # once per layer in state_dict (reference: np_vq_linear.py:588-590).
        object.__setattr__(self, "proxy", proxy)
        object.__setattr__(self, "residual_proxy", residual_proxy)
        self._bind_proxies()

        self.register_buffer("packed_indices", packed_indices.contiguous())
        self._register_optional("bias", bias)
        self._register_optional(
            "column_perm", None if column_perm is None else column_perm.to(torch.int64)
        )
        self.residual_bits = residual_bits
        if residual_proxy is not None:
            if packed_residual is None:
                raise ValueError("residual_proxy given without packed_residual")
            if residual_proxy.vector_len != vector_len:
                raise ValueError("residual codebook must have the same vector length")
            self.residual_bits = residual_bits or IndexPacking.bits_for(residual_proxy.num_centroids)
        self._register_optional("packed_residual", packed_residual)
        self._register_optional("row_scale", None if row_scale is None else row_scale.to(torch.float16))
        self._register_optional("row_bias", None if row_bias is None else row_bias.to(torch.float16))
        # Derived, rebuilt on demand: f32 bias for the kernels, widened index stream.
        self._derived: dict = {}
        # load_state_dict() copies into the buffers in place: what was derived from them is stale.
        self.register_load_state_dict_post_hook(NPVQLinear._after_load_state_dict)

    def _expand_prefix_coded(self, coded: torch.Tensor, num_centroids: int) -> tuple[torch.Tensor, int]:
        """Prefix-coded buffer -> ``(fixed-width stream, its bit width)``.

        The reference keeps such layers in their coded form and decodes prefixes in
        every GEMV (np_vq_linear.py:644-801, kernels/vq_linear_tiered.cu); here the
        coded form is a storage format only.
        """
        self._coded_bits = self.bits  # the width argument as given (the reference's cold-tier width)
        if self.use_tiered:
            _, _, self.cold_bits, self._hot_bits, _ = TieredIndexPacking._parse_header(coded)
        elif self.zero_escape:
            self.cold_bits = ZeroEscapePacking._parse_header(coded)[1]
        idx = decode_to_flat(
            coded, use_tiered=self.use_tiered, tier_bits=self.tier_bits, zero_escape=self.zero_escape
        )
        if idx.numel() != self.n_vectors:
            raise ValueError(
                f"prefix-coded buffer holds {idx.numel()} indices, the layer needs {self.n_vectors}"
            )
        if idx.numel() and int(idx.max().item()) >= num_centroids:
            raise ValueError("prefix-coded buffer names a codebook row past the end of the codebook")
        width = IndexPacking.bits_for(num_centroids)
        if width == 4 and idx.numel() % 2:
            width = 8  # a 4-bit stream needs an even count
        return IndexPacking.pack(idx, width), width

    def _coded_indices(self) -> torch.Tensor:
        """The layer's indices packed back into the prefix-coded format it was built from."""
        idx = IndexPacking.unpack(self.packed_indices.cpu(), self.bits, self.n_vectors)
        if self.zero_escape:
            return ZeroEscapePacking.pack(idx, self.cold_bits)
        if self.tier_bits is not None:
            return NTieredIndexPacking.pack(idx, self.tier_bits)
        return TieredIndexPacking.pack(idx, self.cold_bits, self._hot_bits)

    def _register_optional(self, name: str, t: torch.Tensor | None) -> None:
        if t is not None:
            self.register_buffer(name, t.contiguous())
        else:
            setattr(self, name, None)

    def _bind_proxies(self) -> None:
        for proxy in (self.proxy, self.residual_proxy):
            if proxy is not None:
                proxy._bind(self)

    def _buffer_places(self) -> tuple:
        return tuple((b.device, b.data_ptr(), b.dtype) for b in self._buffers.values() if b is not None)

    def _apply(self, fn, recurse: bool = True):
        """``.to()`` / ``.cuda()`` / ``.half()``: the derived tensors belong to the old buffers.  A move
        is already a heavy host operation, so when the module arrives on a GPU the tensors its
        kernels derive from the buffers -- the slice lists included -- are made here (or, when the
        shared codebook arrives after the layer, by the codebook's own move): ``lower on the CPU ->
        model.to("cuda") -> forward`` reaches the fast decode kernel with no further call, as a
        caller of the reference expects (neuropress/t2n/model_io.py:590-596).
        ``NEUROPRESS_VQ_PREPARE_ON_MOVE=0`` leaves that to :func:`neuropress_amd.prepare_decode`."""
        before = self._buffer_places()
        result = super()._apply(fn, recurse)
        if self._buffer_places() != before:
            self._derived = {}
        self._plan = None
        self._bind_proxies()  # a copied or unpickled proxy starts with no users
        self._prepare_after_move()
        return result

    def _prepare_after_move(self) -> None:
        if not _PREPARE_ON_MOVE or not self.packed_indices.is_cuda or self.backend not in _FUSED_BACKENDS:
            return
        if torch.cuda.is_current_stream_capturing():
            return
        # The shared codebooks are sub-modules of the model root, not of this layer, and may still be
        # on their way: they call back when they arrive.
        for proxy in (self.proxy, self.residual_proxy):
            if proxy is not None and proxy.centroids.device != self.packed_indices.device:
                return
        try:
            if not self.prepare_sliced():
                self.prepare()
        except RuntimeError as exc:  # no kernel library on this machine: forward will say so
            if not _ALLOW_FALLBACK:
                raise
            self._fallback("prepare", "unprepared kernels", exc)

    @staticmethod
    def _after_load_state_dict(module, incompatible_keys) -> None:
        module._derived = {}
        module._plan = None
        module._prepare_after_move()

    # ------------------------------------------------------------------
    # Factory / inverse
    # ------------------------------------------------------------------

    @classmethod
    def from_qtensor_linear(
        cls,
        linear: nn.Linear,
        proxy: VQProxy,
        backend: str | VQBackend | None = VQBackend.AUTO,
        residual_proxy: VQProxy | None = None,
    ) -> NPVQLinear:
        """Build from an ``nn.Linear`` whose ``weight`` is a VQ weight.

        Follows neuropress/nn/np_vq_linear.py:831-921.  Raises ``TypeError``
        (message naming ``QTensorTractVQ``, as the reference does) when the
        weight is not vector-quantized.
        """
        weight_q = linear.weight
        if not is_vq_weight(weight_q):
            raise TypeError(
                f"Expected a VQ weight (QTensorTractVQ / VQWeight), got {type(weight_q).__name__!r}."
            )
        qs = weight_q.qscheme
        bias = linear.bias.detach().clone() if linear.bias is not None else None
        perm = getattr(qs, "column_permutation", None)
        res_c = getattr(qs, "residual_centroids", None)
        if res_c is not None and residual_proxy is None:
            residual_proxy = VQProxy(res_c)
        row_scale = getattr(qs, "row_scale", None)
        row_bias = getattr(qs, "row_bias", None)
        return cls(
            proxy=proxy,
            packed_indices=weight_q.u8_blob.detach().clone(),
            bits=qs.is_packed_indices,
            out_features=linear.out_features,
            in_features=linear.in_features,
            vector_len=qs.vector_len,
            backend=backend,
            bias=bias,
            column_perm=perm.detach().clone() if perm is not None else None,
            use_tiered=bool(getattr(qs, "use_tiered", False)),
            tier_bits=getattr(qs, "tier_bits", None),
            zero_escape=bool(getattr(qs, "zero_escape", False)),
            qtensor_meta={"original_shape": tuple(getattr(qs, "original_shape", ()))},
            residual_proxy=residual_proxy,
            packed_residual=getattr(weight_q, "residual_blob", None),
            residual_bits=getattr(qs, "residual_bits", 0),
            row_scale=row_scale,
            row_bias=row_bias,
        )

    def to_qtensor(self) -> VQWeight:
        """Rebuild the VQ weight this module was lowered from (for unlowering / saving).

        Same contract as neuropress/nn/np_vq_linear.py:977-1008: raises
        ``RuntimeError`` when the module was not built by :meth:`from_qtensor_linear`.
        """
        if self._qtensor_meta is None:
            raise RuntimeError(
                "Cannot reconstruct QTensor: no serde metadata stored. "
                "Build via NPVQLinear.from_qtensor_linear() to enable to_qtensor()."
            )
        coded = self.use_tiered or self.tier_bits is not None or self.zero_escape
        scheme = VQScheme(
            centroids=self.proxy.centroids,
            original_shape=(self.out_features, self.in_features),
            is_packed_indices=self._coded_bits if coded else self.bits,
            column_permutation=self.column_perm,
            use_tiered=self.use_tiered,
            tier_bits=self.tier_bits,
            zero_escape=self.zero_escape,
            residual_centroids=None if self.residual_proxy is None else self.residual_proxy.centroids,
            residual_bits=self.residual_bits,
            row_scale=self.row_scale,
            row_bias=self.row_bias,
        )
        blob = self._coded_indices().to(self.packed_indices.device) if coded else self.packed_indices
        return VQWeight(blob, scheme, self.packed_residual)

    # ------------------------------------------------------------------
    # Derived buffers
    # ------------------------------------------------------------------

    @property
    def is_residual(self) -> bool:
        return self.residual_proxy is not None or self.row_scale is not None or self.row_bias is not None

    def _derive(self, name: str, source: torch.Tensor, build, *more: torch.Tensor):
        """``build()`` cached under *name* until *source* (or one of *more*) moves, is replaced or is written to.

        Every tensor derived from a buffer (a widened index stream, the slice lists, the fp32
        bias, the int32 permutation) is keyed on the buffer's device, address and version
        counter, so ``load_state_dict`` or an in-place ``copy_`` into the buffer invalidates it.
        Inside a graph capture nothing is stored: a tensor made there lives in the graph's
        private pool and holds data only after a replay, so a later eager call must make its own.
        """
        key = (source.device, source.data_ptr(), tensor_version(source))
        for t in more:
            key += (t.data_ptr(), tensor_version(t))
        hit = self._derived.get(name)
        if hit is not None and hit[0] == key:
            return hit[1]
        value = build()
        if not (source.is_cuda and torch.cuda.is_current_stream_capturing()):
            self._derived[name] = (key, value)
        return value

    def _derived_hit(self, name: str, source: torch.Tensor):
        """The cached value of :meth:`_derive`, or None when it is missing or stale."""
        hit = self._derived.get(name)
        if hit is not None and hit[0] == (source.device, source.data_ptr(), tensor_version(source)):
            return hit[1]
        return None

    def _bias_f32(self) -> torch.Tensor | None:
        if self.bias is None:
            return None
        return self._derive("bias_f32", self.bias, lambda: self.bias.detach().to(torch.float32).contiguous())

    def _bias_as(self, dtype: torch.dtype) -> torch.Tensor | None:
        """Bias in the activation dtype for the torch GEMM (``F.linear`` wants one dtype)."""
        if self.bias is None or self.bias.dtype == dtype:
            return self.bias
        return self.bias.to(dtype)

    def _kernel_stream(self) -> tuple[torch.Tensor, int]:
        """Index stream and width the fused kernels read.

        Widths outside {4, 8, 12, 16}, and layers whose K is not a whole number of
        64-column chunks, are widened to a 16-bit stream once per
        device so they take the vectorised index loads (precedent: the
        reference re-lays index streams out at construction, np_vq_linear.py:644-696).
        Rows of the latter are padded to :meth:`_kernel_k` columns with the index of the codebook row of the smallest
        values: the activations are zero there, and zero times an infinity is not (a codebook none of whose rows is
        finite can turn an infinite output into NaN).
        """
        pad = (self._kernel_k() - self.in_features) // self.vector_len
        if (self.bits in _FAST_BITS or self.bits > 16) and pad == 0:
            return self.packed_indices, self.bits
        from .. import kernels

        def widen() -> torch.Tensor:
            wide = kernels.widen_indices_u16(self.packed_indices, self.n_vectors, self.bits)
            if pad:
                rows = wide.view(torch.int16).reshape(self.out_features, -1)
                # bits of a value without its sign: infinities and NaN are the largest
                size = self.proxy.centroids.to(wide.device, torch.float16).view(torch.int16) & 0x7FFF
                filler = size.amax(1).argmin().to(torch.int16)  # bits of the unsigned index
                wide = torch.cat([rows, filler.expand(self.out_features, pad)], 1).reshape(-1).view(torch.uint8)
            return wide

        return self._derive("wide", self.packed_indices, widen, *((self.proxy.centroids,) if pad else ())), 16

    def _kernel_res_stream(self) -> tuple[torch.Tensor, int]:
        """The residual stream next to :meth:`_kernel_stream`: 8 or 16 bits wide and padded where that is padded, with index 0: no row
        is sure to be finite together with the main one and the row's scale, so nothing may multiply the padding."""
        pad = (self._kernel_k() - self.in_features) // self.vector_len
        stream, bits = self._res_stream(), self._res_bits()
        if pad == 0:
            return stream, bits
        from .. import kernels

        def widen() -> torch.Tensor:
            wide = stream if bits == 8 else kernels.widen_indices_u16(stream, self.n_vectors, bits)
            size = 1 if bits == 8 else 2  # bytes
            rows = wide.reshape(-1)[: self.n_vectors * size].reshape(self.out_features, -1)
            return torch.nn.functional.pad(rows, (0, pad * size)).reshape(-1)

        return self._derive("wide_res", stream, widen), 8 if bits == 8 else 16

    def _kernel_k(self) -> int:
        """Columns the MFMA kernels contract: K, rounded up to whole 64-column chunks where the layer is otherwise
        of a form they take (vector length 8, or 4 without a residual stream, at most 16 bits per index)."""
        k = self.in_features
        if k % 64 == 0 or self.vector_len not in (4, 8) or self.bits > 16 or self.n_vectors == 0:
            return k
        if self.is_residual and (self.vector_len != 8 or self._res_bits() > 16):
            return k
        return k + 64 - k % 64

    # ------------------------------------------------------------------
    # Forward
    # ------------------------------------------------------------------

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """Band dispatch by token count (reference: neuropress/nn/np_vq_linear.py:1014-1058).

        A call this layer has made before -- same token count, dtype and buffers -- is issued by its plan."""
        plan = self._plan
        if plan is not None:
            y = plan(self, x)
            if y is not None:
                return y
        return self._forward(x)

    _planned_forward = forward  # module(x) may go straight to the plan (kernels/plans.py)

    def _forward(self, x: torch.Tensor) -> torch.Tensor:
        from .. import kernels

        m = x.numel() // self.in_features
        tracked = x.is_cuda and self.backend in _FUSED_BACKENDS and kernels.tracked(x, self.bias)
        band = self._band(x, m, tracked)
        if x.is_cuda and not tracked and not torch.cuda.is_current_stream_capturing():
            y = self._planned(x, m, band)
            if y is not None:
                return y
        if band == "blocks" and kernels.replaced("vq_linear", "vq_gemm_tile", "vq_dequant", "rvq_linear", "rvq_dequant", "dense_linear"):
            band = self._band(x, m, tracked, blocks=False)  # whose function a caller has put another in the place of
        if band == "sliced":
            return self._forward_sliced(x, self._sliced_for(m))  # applies column_perm inside the kernel
        if band == "gemv_perm":
            return self._fused(x, tile=False, perm=self._perm_i32(x.device))
        if self.column_perm is not None:
            x = x[..., self.column_perm]
        if band == "dense":
            return self._forward_dequant_gemm(x)
        if band == "tile":
            return self._forward_tile_gemm(x)
        if band == "slice":
            return self._forward_slice_gemm(x)
        if band == "blocks":
            return self._forward_blocks(x)
        if self.backend == VQBackend.CUDA_LUT:
            return self._forward_cuda_lut(x)
        if self.backend == VQBackend.CUDA_WMMA or self.backend in _CODED_BACKENDS:
            return self._forward_cuda_wmma(x)
        if self.backend == VQBackend.CUDA:
            return self._forward_cuda(x)
        if self.backend == VQBackend.COMPILE:
            return self._forward_compile(x)
        return self._forward_default(x)

    def _band(self, x: torch.Tensor, m: int, tracked: bool = False, blocks: bool = True) -> str:
        """Which kernel serves a call of *m* tokens: ``sliced``, ``gemv_perm`` (the GEMV that gathers x's columns),
        ``fused`` (the backend's GEMV), ``blocks`` (it with a workgroup per 32 tokens and for rows of x that end inside the last 64
        columns, or the table GEMM), ``slice`` (the slice GEMM), ``tile``, ``dense`` (decode + GEMM) or ``torch``.

        *tracked* (``kernels.tracked(x)``): the dense product is the library's, columns are gathered by torch and none
        are padded; the limits are those against that.  What it serves carries gradients, the other kernels do not.
        *blocks* False: what ``blocks`` takes the place of."""
        if self.backend not in _FUSED_BACKENDS:
            return "torch"
        if x.dtype not in (torch.float16, torch.bfloat16):
            return "dense"  # fp32 activations: decode + GEMM
        sliced = m <= min(_SLICED_MAX_TOKENS, _fused_max_tokens(self.backend)) and x.is_cuda and self._sliced_for(m) is not None
        if x.is_cuda and not tracked and self._slice_gemm_wins(m):
            return "slice"
        if sliced:
            return "sliced"
        if self.column_perm is not None and self._perm_fusable(x, m):
            return "gemv_perm"
        ragged = self._kernel_k() != self.in_features
        if x.is_cuda and (not self._mfma_layer() or (ragged and (tracked or (self.is_residual and not (blocks and self._blocks_read()))))):
            # Shapes without an MFMA kernel (vector lengths other than 8 and 4, K not a
            # multiple of 64): the element-wise GEMV is slower than decoding once and calling
            # the dense GEMM at every token count (14336 x 4096: 99 us against 57 us at one token).
            return "dense"
        if m > self._gemv_max_tokens(m):
            tile = self.backend != VQBackend.CUDA_LUT and m <= self._tile_max_tokens(tracked) and self._tile_band_ok(x, m, tracked)
            if blocks and x.is_cuda and not tracked and self._blocks_win(m, tile):
                return "blocks"
            return "tile" if tile else "dense"
        # Ragged rows, where they are whole 16 bytes, are read where they lie.  Those that a permutation copies are padded on the way: the GEMV on
        # whole chunks is ahead (us per call, read as ragged rows / padded: 8000 x 4104 with 256 rows 7.9 / 7.4 at one token, 8.1 / 7.8 at 4).
        # Residual rows are never padded, see _kernel_res_stream, nor given to the tile GEMM (past 32 tokens, a raised band).
        short = ragged and (self.is_residual or (self.in_features % 8 == 0 and self.column_perm is None and m <= _GEMV_KERNEL_MAX_TOKENS))
        return "blocks" if blocks and x.is_cuda and short and self._blocks_read() else "fused"

    # -- call plan ---------------------------------------------------------

    def _planned(self, x: torch.Tensor, m: int, band: str):
        """Add this call to the layer's plan and let the plan issue it; None where it cannot."""
        from .. import kernels
        from ..kernels import plans

        plan = self._plan
        if plan is not None and plan.stale(self):
            self._plan = plan = None
        if plan is not None and band == "sliced" and (band, x.dtype) in plan.names:
            return kernels.SlicedCallPlan(plan).run(x)  # the wrapper functions have been replaced
        if m < 1 or band == "torch" or (band == "tile" and _tile_failed) or x.dtype not in plans.DTYPE_CODES or (
            x.device != self.packed_indices.device or not self._kernel_types(band)
        ):  # fmt: skip
            return None
        if plan is None:
            plan = self._new_plan()
            if plan is None:
                return None
        self._add_route(plan, x.dtype, m, band)
        self._plan = plan
        return None if plan.wrapped() else plan.run(x)

    def _kernel_types(self, band: str) -> bool:
        """Whether the buffers have the types the kernels of *band* read them as.  ``model.to(dtype)`` casts codebooks and
        row tensors; the bands of plain layers that look rows up in a copy of x's type take any codebook."""
        if self.packed_indices.dtype != torch.uint8:
            return False
        if not self.is_residual:
            return band != "dense" or self.proxy.centroids.dtype == torch.float16
        f16 = (self.proxy.centroids, self._res_centroids(), self.row_scale, self.row_bias)
        return self._res_stream().dtype == torch.uint8 and all(t is None or t.dtype == torch.float16 for t in f16)

    def _new_plan(self):
        from ..kernels import plans

        try:
            return plans.make(
                self, _PLAN_ATTRIBUTES, globals(), _PLAN_THRESHOLDS,
                holders=[p for p in (self.proxy, self.residual_proxy) if p is not None],
                sources=(self.packed_indices, self.proxy.centroids, self.bias, self.column_perm, self.packed_residual,
                         self.row_scale, self.row_bias, None if self.residual_proxy is None else self.residual_proxy.centroids),
            )  # fmt: skip
        except RuntimeError as exc:
            self._fallback("call_plan", "the Python call path", exc)
            return None

    def _add_route(self, plan, dtype: torch.dtype, m: int, band: str) -> None:
        from ..kernels import plans

        tile = band == "tile" or (band == "fused" and m > _GEMV_KERNEL_MAX_TOKENS)
        kind = "tile" if tile else "product" if band == "dense" and self._own_product(m, dtype) else band
        number = plan.names.get((kind, dtype))
        if number is None:
            number = plan.names[kind, dtype] = self._template(plan, dtype, kind)
        code = plans.DTYPE_CODES[dtype]
        if band == "sliced":
            sl, limit, _ = self._derived_hit("sliced", self.packed_indices)
            most = min(limit, _SLICED_MAX_TOKENS, _fused_max_tokens(self.backend))
            others = self._slice_gemm_counts()
            for tokens in range(1, most + 1):
                if tokens not in others or tokens > _SLICE_GEMM_MAX_TOKENS:
                    plan.route(code, tokens, number, sl.workspace_bytes(tokens))
        elif band == "slice":
            plan.route(code, m, number, plans.slice_scratch(m, self.out_features, self._kernel_k(), self.proxy.num_centroids))
        else:
            scratch = plans.tile_scratch if tile else plans.product_scratch if kind == "product" else None
            plan.route(code, m, number, scratch(m, self.out_features, self._kernel_k()) if scratch else 0)

    def _template(self, plan, dtype: torch.dtype, kind: str) -> int:
        from ..kernels import plans

        n, k, vl = self.out_features, self.in_features, self.vector_len
        code = plans.DTYPE_CODES[dtype]
        packed, proxy = self.packed_indices.reshape(-1), self.proxy
        perm = None
        if self.column_perm is not None and kind not in ("sliced", "gemv_perm"):
            perm = self._perm_i64(packed.device) if dtype == torch.float32 else self._perm_i32(packed.device)
        if kind == "sliced":
            sl, _, _ = self._derived_hit("sliced", self.packed_indices)
            i32 = None if self.column_perm is None else self._perm_i32(packed.device)
            plan.hold(sl)  # the plan passes the address of its header
            args = (i32, sl.header_ptr, sl.blob, proxy.centroids_as(dtype), code, self._bias_f32(), code)
            return plans.template(plan, plans.SLICED, n, k, args, dtype)
        # In the place of the dense product, which carries the bias's gradient: past the GEMV's band, and for all calls of ragged rows that ask for one.
        leaf = self.bias if kind == "blocks" or self._kernel_k() != k else None
        if self.is_residual:
            dense = kind in ("dense", "product")
            (main, bits), (res, res_bits) = ((packed, self.bits), (self._res_stream(), self._res_bits())) if dense else (
                self._kernel_stream(), self._kernel_res_stream())  # fmt: skip
            main, res, cr = main.reshape(-1), res.reshape(-1), self._res_centroids()
            args = (main, main.numel(), bits, res, res.numel(), res_bits, proxy.centroids, proxy.num_centroids,
                    cr, cr.shape[0], self.row_scale, self.row_bias, vl)  # fmt: skip
            if kind in ("dense", "product"):
                own = kind == "product"
                bias = self._bias_f32() if own else self._bias_as(dtype)
                return plans.template(plan, plans.RVQ_DENSE, n, k, args, dtype, perm=perm, bias=bias, leaf=self.bias, own=own)
            kind_code = {"tile": plans.RVQ_TILE, "blocks": plans.RVQ_BLOCKS}.get(kind, plans.RVQ_GEMV)
            return plans.template(plan, kind_code, n, self._kernel_k(), (*args, self._bias_f32(), code), dtype, k_in=k, perm=perm, leaf=leaf)
        stream, bits = self._kernel_stream()
        stream = stream.reshape(-1)
        if kind in ("dense", "product"):
            own = kind == "product"
            bias = self._bias_f32() if own else self._bias_as(dtype)
            # The library's product takes any K; the package's own any whole 16 bytes, but what a permutation copies is padded.
            width = self._kernel_k() if own and (perm is not None or k % 8) else k
            if width == k and self._kernel_k() != k:
                stream, bits = packed, self.bits
            args = (stream, stream.numel(), bits, proxy.centroids, proxy.num_centroids, vl, n * (width // vl))
            return plans.template(plan, plans.VQ_DENSE, n, width, args, dtype, k_in=k, perm=perm, bias=bias, leaf=self.bias, own=own)
        args = (stream, stream.numel(), bits, proxy.centroids_as(dtype), code, proxy.num_centroids, vl, self._bias_f32(), code)
        if kind == "gemv_perm":
            return plans.template(plan, plans.VQ_GEMV_PERM, n, k, (*args, self._perm_i32(stream.device)), dtype)
        kind_code = {"tile": plans.VQ_TILE, "slice": plans.VQ_SLICE, "blocks": plans.VQ_BLOCKS}.get(kind, plans.VQ_GEMV)
        return plans.template(plan, kind_code, n, self._kernel_k(), args, dtype, k_in=k, perm=perm, leaf=leaf)

    # -- slice-list GEMV ---------------------------------------------------

    def _sliced_eligible(self) -> bool:
        return (
            _SLICED_MAX_TOKENS > 0
            and not self.is_residual
            and self.vector_len == 8
            and self.proxy.num_centroids >= _SLICED_MIN_CENTROIDS
            and self.n_vectors >= _SLICED_MIN_INDICES
        )

    def prepare_sliced(self) -> bool:
        """Build the slice-list form of the indices for the module's current device.

        Host work (the stream is copied to the host, re-laid there and uploaded; then both decode
        GEMVs are timed on the layer's own indices), so it is never done by ``forward``: call it --
        or :func:`neuropress_amd.prepare_decode` for a whole model -- after the module has reached
        its GPU and before the first decode step or graph capture.  Returns False when the layer
        does not use the path.
        """
        if not (self._sliced_eligible() and self.packed_indices.is_cuda):
            return False
        if torch.cuda.is_current_stream_capturing():
            raise RuntimeError("NPVQLinear.prepare_sliced() copies to the host and back: call it before the capture")
        self._derive("sliced", self.packed_indices, self._build_sliced)
        self._slice_gemm_counts()  # a first call asks it
        self._plan = None  # it may hold routes of the fused GEMV for the token counts the lists serve
        self.prepare()
        return True

    def prepare(self) -> None:
        """Make every tensor the kernels derive from the module's buffers (widened index stream,
        fp32 bias, int32 permutation, the codebook in the usual activation dtypes) for the current
        device, so that a first call inside a graph capture finds them."""
        if not self.packed_indices.is_cuda:
            return
        self._kernel_stream()
        self._bias_f32()
        if self.column_perm is not None:
            try:
                self._perm_i32(self.packed_indices.device)
            except (IndexError, RuntimeError):  # e.g. materialised and not loaded yet: a call says so
                pass
        for dtype in (torch.float16, torch.bfloat16):
            self.proxy.centroids_as(dtype)
        if self.is_residual:
            self._res_stream()
            self._kernel_res_stream()
            self._res_centroids()
        if self.backend in _FUSED_BACKENDS and (self._plan is None or self._plan.stale(self)):
            self._plan = self._new_plan()  # still without routes: every call adds its own

    def _build_sliced(self):
        """(slice lists, most tokens for which they beat the fused GEMV on this layer, the times that say so)."""
        from .. import kernels

        sl = kernels.vq_slice_indices(
            self.packed_indices, self.bits, self.out_features, self.in_features,
            self.vector_len, self.proxy.num_centroids,
        )  # fmt: skip
        kernels.sliced_workspace(sl.blob.device, sl.workspace_bytes(_SLICED_MAX_TOKENS))
        return sl, *self._sliced_token_limit(sl)

    def _sliced_token_limit(self, sl) -> tuple[int, tuple]:
        """Most tokens for which this layer's slice-list GEMV beats its fused GEMV, and what was timed: (tokens, us of
        the slice lists, us of the fused GEMV), up to the first token count at which the lists lose.

        With indices spread evenly over the codebook the slice lists win up to
        ``_SLICED_MAX_TOKENS`` by a wide margin.  A skewed index distribution (one codebook
        slice holding most of the indices) does two things: the hot slice's workgroups
        carry more of the work, or outnumber the compute units, and the fused GEMV's
        lookups start hitting in L1.  Which one wins then depends on the layer, so every
        layer of the size the path is meant for is timed here, once, when its lists are
        built (by ``prepare_sliced``, never by ``forward``)."""
        if self.n_vectors < _SLICED_TUNE_MIN_INDICES:
            return _SLICED_MAX_TOKENS, ()
        dev = sl.blob.device
        from .. import kernels

        dt = torch.float16
        cb = self.proxy.centroids_as(dt)
        stream, bits = self._kernel_stream()

        def timed(fn) -> float:
            # GPU time, not issue time: eight calls captured in a HIP graph and replayed (launched
            # eagerly, both kernels finish faster than Python can issue them).
            side = torch.cuda.Stream(device=dev)
            side.wait_stream(torch.cuda.current_stream(dev))
            with torch.cuda.stream(side):
                fn()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    for _ in range(8):
                        fn()
                graph.replay()
                t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                t0.record()
                for _ in range(3):
                    graph.replay()
                t1.record()
                t1.synchronize()
            torch.cuda.current_stream(dev).wait_stream(side)
            return t0.elapsed_time(t1) * 1e3 / 24

        limit, times = 0, []
        try:
            for m in (1, 2, 4, _SLICED_MAX_TOKENS):
                if m > _SLICED_MAX_TOKENS:
                    break
                x = torch.ones(m, self.in_features, dtype=dt, device=dev)
                ws = torch.zeros(sl.workspace_bytes(m) // 4, dtype=torch.float32, device=dev)
                t_sliced = timed(lambda: kernels.vq_linear_sliced(x, sl, cb, workspace=ws))
                xf = kernels.gather_columns(x, None, self._kernel_k()) if self._kernel_k() != self.in_features else x
                t_fused = timed(lambda: kernels.vq_linear(xf, stream, cb, bits, self.vector_len, None, self.out_features))
                times.append((m, t_sliced, t_fused))
                if t_sliced >= t_fused:
                    break
                limit = m
        except RuntimeError:
            # e.g. another thread of the process is capturing a graph: keep the measured default
            return _SLICED_MAX_TOKENS, ()
        return limit, tuple(times)

    def _sliced_for(self, m: int):
        """The slice lists when they exist for the buffer as it is now and win at *m* tokens, else None.

        A lookup only: an eligible layer whose lists were never built (or whose indices were
        reloaded since) runs the fused GEMV, and says so once."""
        hit = self._derived_hit("sliced", self.packed_indices)
        if hit is None:
            if self._sliced_eligible():
                _warn_unprepared_once()
            return None
        sl, limit, _ = hit
        return sl if m <= limit else None

    def _slice_gemm_wins(self, m: int) -> bool:
        """Whether the slice GEMM is the fastest kernel for *m* tokens."""
        return m <= _SLICE_GEMM_MAX_TOKENS and m in self._slice_gemm_counts()

    def _slice_gemm_counts(self) -> frozenset[int]:
        """The token counts at which the slice GEMM is the fastest kernel: its estimate against what was timed on this layer's
        own indices, the slice lists (between two timed token counts: on the line through them) or, past them, the fused GEMV
        at the most tokens it was timed with (it does not get faster, and the tile GEMM of 17 to 32 tokens is level with
        it).  One token stays with the lists where they won it.  Layers that were not timed -- lists never built, or fewer
        than 2^20 indices -- do not take it."""
        if self.proxy.num_centroids <= 4096 or self.bits > 16 or self.backend == VQBackend.CUDA_LUT or _FUSED_MAX_TOKENS <= 0:
            return frozenset()
        hit = self._derived_hit("sliced", self.packed_indices)
        if hit is None or not hit[2]:
            return frozenset()
        cached = self._derived.get("slice_gemm")
        if cached is None or cached[0] is not hit:
            counts = frozenset(m for m in range(min(hit[1], 1) + 1, 33) if self._slice_gemm_ahead(m, hit))
            cached = self._derived["slice_gemm"] = (hit, counts)
        return cached[1]

    def _slice_gemm_ahead(self, m: int, timed) -> bool:
        from .. import kernels

        us = kernels.slice_gemm_us(m, self.out_features, self._kernel_k(), self.proxy.num_centroids)
        us += _SLICE_GEMM_GATHER_US if us and self.column_perm is not None else 0.0
        _, limit, times = timed
        if m <= limit:
            (m0, t0), (m1, t1) = next(
                ((a[0], a[1]), (b[0], b[1])) for a, b in zip((times[0], *times), times) if b[0] >= m or b is times[-1]
            )  # fmt: skip
            other = t1 if m1 == m0 else t0 + (t1 - t0) * (m - m0) / (m1 - m0)
        else:
            other = times[-1][2]
        return 0 < us < other

    def _perm_i32(self, device: torch.device) -> torch.Tensor:
        """``column_perm`` as the int32 device tensor the kernels read (cached): in range, negative entries wrapped as
        torch's indexing does.  The check waits for the device, once per buffer contents."""

        def build() -> torch.Tensor:
            perm, k = self.column_perm.to(device), self.in_features
            if tuple(perm.shape) != (k,):
                raise RuntimeError(f"NPVQLinear: column_perm must hold in_features={k} entries, got {tuple(perm.shape)}")
            low, high = -k, k - 1
            if perm.is_cuda and torch.cuda.is_current_stream_capturing():
                perm = perm.clamp(low, high)  # not to be looked at here: nothing the kernels could read past x with
            elif k:
                low, high = torch.stack(torch.aminmax(perm)).tolist()
            if low < -k or high >= k:
                raise IndexError(f"NPVQLinear: column_perm has entries out of range for in_features={k}")
            return (perm if low >= 0 else torch.where(perm < 0, perm + k, perm)).to(torch.int32).contiguous()

        return self._derive("perm_i32", self.column_perm, build)

    def _perm_i64(self, device: torch.device) -> torch.Tensor:
        """The same for torch's gather of 32-bit activations inside a call plan, which wraps nothing."""
        return self._derive("perm_i64", self.column_perm, lambda: self._perm_i32(device).to(torch.int64))

    def _gemv_max_tokens(self, m: int) -> int:
        """End of band (a) for a call of *m* tokens: the fused limit, or 32 while x stays small."""
        limit = _fused_max_tokens(self.backend)
        if limit == 16 and 16 < m <= min(_FUSED_WIDE_MAX_TOKENS, 32):
            if self.is_residual or m * self.in_features <= _FUSED_WIDE_MAX_ACTIVATIONS:
                return 32
            if self._gemv_stages_activations(m) and not self._tile_ahead_from_17():
                return 32
        return limit

    def _blocks_win(self, m: int, tile: bool = True) -> bool:
        """Whether the GEMV with a workgroup per 32 tokens (or the table GEMM behind the same entry) is ahead of
        the tile GEMM (*tile*) and of decode + GEMM.  Layers of fewer than 256 output features, the least that
        the estimates were checked on, keep those.  Many would gain, those with long rows or a large codebook lose: decode +
        GEMM / this, us at 64 tokens, 4096 rows 128 x 1024 7.9 / 4.9, 200 x 4096 11.8 / 9.4, 128 x 8192 11.8 / 15.9, 65536 rows
        128 x 1024 8.1 / 5.4, 64 x 4096 11.7 / 14.4, 128 x 8192 12.3 / 23.0, residual 128 x 2048 10.5 / 9.6, 200 x 4096 12.7 / 16.0."""
        if not 16 < m <= _BLOCKS_MAX_TOKENS or self.out_features < 256 or min(_FUSED_MAX_TOKENS, _TILE_MAX_TOKENS) <= 0 or self.backend == VQBackend.CUDA_LUT:
            return False
        if self.vector_len != 8 or self.proxy.centroids.dtype != torch.float16 or not self._mfma_layer() or (
            self.is_residual and self._kernel_k() == self.in_features
            and (self.bits if self.bits in _FAST_BITS else 16, self._res_bits()) not in ((16, 8), (16, 16), (12, 8), (8, 8))
        ):  # fmt: skip
            return False
        from .. import kernels

        return kernels.gemv_blocks_preferred(m, self.out_features, self._kernel_k(), int(self.is_residual), self.proxy.num_centroids,
                                             self.column_perm is not None, tile) and self._blocks_read()  # fmt: skip

    def _blocks_read(self) -> bool:
        """Whether the buffers start at 16-byte addresses (not slices of larger ones, say): the blocks entries refuse others, the kernels
        they take the place of serve them."""
        buffers = [self.packed_indices, self.proxy.centroids]
        if self.is_residual:
            buffers += [self._res_stream(), self._res_centroids()]
        return all(t.data_ptr() % 16 == 0 for t in buffers)

    def _tile_ahead_from_17(self) -> bool:
        """Large layers with at least twice as many output as input features and a codebook kept in memory: the
        128-column tile GEMM is level with the staged GEMV at 17 tokens and ahead at 24-32 (tile vs GEMV at
        17 / 24 / 32 tokens: 14336 x 4096 40.3 / 39.0 / 40.4 vs 41.0 / 42.2 / 43.1 us, 11008 x 4096 35.4 / 35.8 / 36.1
        vs 35.6 / 36.9 / 39.2); on 8192 x 8192 they tie, on 4096 x 14336 (44 vs 39-41.5 us) and on small layers
        (4096 x 4096: 20.6-21.3 vs 13.3-14.0) the GEMV stays ahead."""
        return (
            _TILE_MAX_TOKENS > 0
            and self._wide_tile_layer()
            and self.out_features >= 2 * self.in_features
            and self.in_features * self.out_features >= _TILE_WIDE_MIN_WEIGHTS
        )

    def _gemv_stages_activations(self, m: int) -> bool:
        """Layers of one row tile per workgroup whose lookups go to memory run the GEMV that stages
        its activations through LDS, which stays ahead of the tile GEMM at any K (65536-row
        codebook, GEMV vs tile GEMM at 17 / 24 / 32 tokens: 4096 x 14336 39.8 / 39.7 / 42.0 vs
        48.7-49.6 us, 4096 x 8192 24.2 / 24.1 / 24.8 vs 33.8-34.8 us; with a 4096-row table, which
        the GEMV looks up in LDS, it does not: 23.4 / 28.4 / 33.4 vs 24.6-25.8 us)."""
        hit = self._derived.get("stages")
        if hit is None or hit[0] != m:
            from .. import kernels

            rows = max(1, self.proxy.num_centroids * self.vector_len // 8)  # table size in rows of eight
            hit = (m, kernels.gemv_stages_activations(m, self.out_features, self._kernel_k(), rows))
            self._derived["stages"] = hit
        return hit[1]

    def _perm_fusable(self, x: torch.Tensor, m: int) -> bool:
        """Whether the fused GEMV gathers ``x[..., column_perm]`` itself for this call."""
        if not x.is_cuda or self.is_residual or m > min(_fused_max_tokens(self.backend), 16):
            return False
        if self.bits > 16 or not self._mfma_layer():
            return False  # index widths the fused kernel does not stream (codebooks beyond 65536 rows)
        from .. import kernels

        bits = self.bits if self.bits in _FAST_BITS else 16  # as _kernel_stream
        return kernels.vq_linear_perm_supported(
            m, self.out_features, self.in_features, self.proxy.num_centroids, self.vector_len, bits
        )

    def _forward_sliced(self, x: torch.Tensor, sliced) -> torch.Tensor:
        from .. import kernels

        *leading, _ = x.shape
        perm = self._perm_i32(x.device) if self.column_perm is not None else None
        if x.device != self.packed_indices.device:
            raise RuntimeError(f"NPVQLinear: input on {x.device}, weights on {self.packed_indices.device}")
        x2d = kernels._rows(x.reshape(-1, self.in_features))
        try:
            # forward() has checked x's dtype and device; the other tensors come out of this
            # module's caches in the form the kernel reads.
            y = kernels.vq_linear_sliced_checked(
                x2d, sliced, self.proxy.centroids_as(x.dtype), self._bias_f32(), perm
            )
        except RuntimeError as exc:
            self._fallback("vq_linear_sliced", "decode + GEMM", exc)
            if self.column_perm is not None:
                x = x[..., self.column_perm]
            return self._forward_dequant_gemm(x)
        return y.reshape(*leading, self.out_features)

    def _mfma_layer(self) -> bool:
        """Whether the MFMA kernels take this layer's shape."""
        ok = self._derived.get("mfma_layer")
        if ok is None:
            from .. import kernels

            k = self._kernel_k()
            bits = self.bits if k == self.in_features and (self.bits in _FAST_BITS or self.bits > 16) else 16  # as _kernel_stream
            ok = kernels.vq_fused_supported(k, self.vector_len, bits)
            self._derived["mfma_layer"] = ok
        return ok

    def _wide_tile_layer(self) -> bool:
        """Whether the tile GEMM of this layer is the 128-column kernel (codebook kept in memory)."""
        return (
            not self.is_residual
            and self.vector_len == 8
            and 12 < self.bits <= 16  # read as a 16-bit stream (see _kernel_stream)
            and self.proxy.num_centroids * self.vector_len * 2 > 65536
        )

    def _tile_max_tokens(self, tracked: bool = False) -> int:
        """Upper end of the tile-decode GEMM band for this layer."""
        if _TILE_MAX_TOKENS > 0 and self._wide_tile_layer():
            weights = self.in_features * self.out_features
            k = self.in_features
            if weights >= _TILE_WIDE_MIN_WEIGHTS:
                return max(_TILE_MAX_TOKENS, _TILE_WIDE_MAX_TOKENS)
            if tracked:
                broad = weights >= _TILE_WIDE_BROAD_WEIGHTS
                return min(_TILE_WIDE_MAX_TOKENS, _TILE_WIDE_LIBRARY_MAX_TOKENS if broad else _TILE_WIDE_LIBRARY_MAX_TOKENS // 2)
            if weights >= backends._MID_LAYER_WEIGHTS and k >= 4096:
                return _TILE_WIDE_MAX_TOKENS if k >= backends._MID_LAYER_K else min(_TILE_WIDE_MAX_TOKENS, _TILE_WIDE_LONG_MAX_TOKENS)
            if weights >= _TILE_WIDE_BROAD_WEIGHTS and self.out_features >= _TILE_WIDE_BROAD_FEATURES:
                return min(_TILE_WIDE_MAX_TOKENS, _TILE_WIDE_LONG_MAX_TOKENS)
            if weights >= backends._SMALL_LAYER_WEIGHTS and k >= 4096:
                return min(_TILE_WIDE_MAX_TOKENS, _TILE_WIDE_LONG_MAX_TOKENS if k >= _TILE_SPLIT_LONG_K else _TILE_WIDE_MID_MAX_TOKENS)
            if weights < _TILE_WIDE_TINY_WEIGHTS and _TILE_MIN_GRID_FRACTION > 0:
                return min(_TILE_WIDE_MAX_TOKENS, _GEMV_KERNEL_MAX_TOKENS)
            return min(_TILE_WIDE_MAX_TOKENS, _TILE_WIDE_SMALL_MAX_TOKENS)
        return _TILE_MAX_TOKENS

    def _tile_band_ok(self, x: torch.Tensor, m: int, tracked: bool = False) -> bool:
        """True when the tile GEMM's grid (64 columns x up to 384 rows per workgroup,
        times the reduction splits the kernel adds for layers with few output
        features) covers at least ``_TILE_MIN_GRID_FRACTION`` of the compute units."""
        if not x.is_cuda:
            return True
        if not self._mfma_layer() or (self.is_residual and self._kernel_k() != self.in_features):
            return False  # the tile entry point would run its element-wise fallback, or ask for padded columns
        if self._wide_tile_layer():
            return True  # the 128-column kernel fills the GPU by splitting the reduction; its band is a token count
        cus = self._derived.get("cus")
        if cus is None:
            cus = torch.cuda.get_device_properties(x.device).multi_processor_count
            self._derived["cus"] = cus
        if tracked:
            return tile_band_ok(m, self.out_features, self.in_features, cus, _TILE_MIN_GRID_FRACTION, _TILE_SPLIT_MAX_TOKENS,
                                _TILE_SPLIT_LONG_K, library=True)  # fmt: skip
        return tile_band_ok(
            m, self.out_features, self._kernel_k(), cus,
            _TILE_MIN_GRID_FRACTION, _TILE_SPLIT_MAX_TOKENS, _TILE_SPLIT_LONG_K,
            32 if self.is_residual else _TILE_SMALL_LAYER_MAX_TOKENS,
            m <= 256 and m * self._kernel_k() <= _TILE_HALF_GRID_MAX_ACTIVATIONS, 4096 if self.is_residual else 2048,
        )  # fmt: skip

    # -- torch-op paths ---------------------------------------------------

    def _dense_weight_torch(self, dtype: torch.dtype) -> torch.Tensor:
        idx = IndexPacking.unpack(self.packed_indices, self.bits, self.n_vectors)
        w = self.proxy.centroids[idx]
        if self.is_residual:
            if self.residual_proxy is not None:
                ir = IndexPacking.unpack(self.packed_residual, self.residual_bits, self.n_vectors)
                w = w + self.residual_proxy.centroids[ir]
            w = w.reshape(self.out_features, self.in_features)
            if self.row_scale is not None:
                w = w * self.row_scale[:, None]
            if self.row_bias is not None:
                w = w + self.row_bias[:, None]
        return w.reshape(self.out_features, self.in_features).to(dtype)

    def _forward_default(self, x: torch.Tensor) -> torch.Tensor:
        """Follows neuropress/nn/np_vq_linear.py:1091-1095."""
        if self.is_residual:
            return F.linear(x, self._dense_weight_torch(x.dtype), self._bias_as(x.dtype))
        return _vq_dequant_linear(
            x, self.packed_indices, self.proxy.centroids, self.bits, self.n_vectors,
            self.out_features, self.in_features, self._bias_as(x.dtype),
        )  # fmt: skip

    def _forward_compile(self, x: torch.Tensor) -> torch.Tensor:
        """The reference compiles the gather path with a tracing compiler
        (np_vq_linear.py:1150-1160); here the same ops run eagerly."""
        return self._forward_default(x)

    # -- HIP paths --------------------------------------------------------

    def _fallback(self, kernel: str, fallback: str, exc: Exception) -> None:
        """Re-raise unless fallbacks were opted into; then warn once per kernel."""
        if not _ALLOW_FALLBACK:
            raise exc
        from .. import kernels

        kernels.warn_kernel_fallback(kernel, fallback, exc)

    def _forward_dequant_gemm(self, x: torch.Tensor) -> torch.Tensor:
        """Band (c): decode the weight in one kernel pass, then a dense GEMM.

        Follows neuropress/nn/np_vq_linear.py:1127-1148.  The decoded ``[N, K]``
        weight is a temporary returned to the allocator after the matmul.
        """
        from .. import kernels

        try:
            own = self._own_product(x.numel() // self.in_features, x.dtype) and not kernels.tracked(x, self.bias)
            # Ragged rows as they are only where nothing has taken the place of the product: one that has is given whole 64-column chunks.
            padded = self._kernel_k() != self.in_features and (self.in_features % 8 or kernels.replaced("dense_linear"))
            own = own and not (padded and self.is_residual)
            if self.is_residual:
                w = kernels.rvq_dequant(
                    self.packed_indices, self.bits, self._res_stream(), self._res_bits(),
                    self.proxy.centroids, self._res_centroids(), self.row_scale, self.row_bias,
                    self.out_features, self.in_features, x.dtype,
                )  # fmt: skip
            elif own and padded:
                stream, bits = self._kernel_stream()
                w = kernels.vq_dequant(stream, self.proxy.centroids, bits, self.out_features, self._kernel_k(), x.dtype)
            else:
                w = kernels.vq_dequant(
                    self.packed_indices, self.proxy.centroids, self.bits,
                    self.out_features, self.in_features, x.dtype,
                )  # fmt: skip
            if own:
                x2d = x.reshape(-1, self.in_features)
                if w.shape[1] != self.in_features:
                    x2d = kernels.gather_columns(x2d, None, w.shape[1])
                more = {"ragged": True} if w.shape[1] % 64 else {}
                return kernels.dense_linear(x2d, w, self._bias_f32(), **more).reshape(*x.shape[:-1], self.out_features)
        except RuntimeError as exc:
            self._fallback("vq_dequant", "the gather path", exc)
            return self._forward_compile(x)
        return F.linear(x, w, self._bias_as(x.dtype))

    def _own_product(self, m: int, dtype: torch.dtype) -> bool:
        """Whether the dense product of a decode + GEMM call is the package's own kernel."""
        from .. import kernels

        return dtype in (torch.float16, torch.bfloat16) and kernels.dense_preferred(m, self.out_features, self._kernel_k())

    def _forward_tile_gemm(self, x: torch.Tensor) -> torch.Tensor:
        """Band (b): MFMA GEMM decoding weight tiles in-kernel.

        Takes the place of the reference's Triton band (np_vq_linear.py:1097-1125).
        """
        global _tile_failed
        if _tile_failed or x.dtype not in (torch.bfloat16, torch.float16):
            return self._forward_dequant_gemm(x)
        try:
            y = self._fused(x, tile=True)
        except RuntimeError as exc:
            self._fallback("vq_gemm_tile", "decode + GEMM", exc)
            _tile_failed = True
            return self._forward_dequant_gemm(x)
        return y

    def _forward_slice_gemm(self, x: torch.Tensor) -> torch.Tensor:
        """Up to 32 tokens on large layers with codebooks of more than 4096 rows (:meth:`_slice_gemm_wins`)."""
        from .. import kernels

        *leading, _ = x.shape
        x2d = x.reshape(-1, self.in_features)
        if self._kernel_k() != self.in_features:
            x2d = kernels.gather_columns(x2d, None, self._kernel_k())
        try:
            y = kernels.vq_slice_gemm(x2d, self._kernel_stream()[0], self.proxy.centroids_as(x.dtype), self.out_features, self._bias_f32())
        except RuntimeError as exc:
            self._fallback("vq_slice_gemm", "decode + GEMM", exc)
            return self._forward_dequant_gemm(x)
        return y.reshape(*leading, self.out_features)

    def _res_stream(self) -> torch.Tensor:
        if self.packed_residual is not None:
            return self.packed_residual
        dev = self.packed_indices.device
        return self._derive("zero_res", self.packed_indices, lambda: torch.zeros(self.n_vectors, dtype=torch.uint8, device=dev))

    def _res_bits(self) -> int:
        return self.residual_bits if self.packed_residual is not None else 8

    def _res_centroids(self) -> torch.Tensor:
        if self.residual_proxy is not None:
            return self.residual_proxy.centroids
        dev = self.packed_indices.device
        return self._derive(
            "zero_cb", self.packed_indices, lambda: torch.zeros((1, self.vector_len), dtype=torch.float16, device=dev)
        )

    def _forward_blocks(self, x: torch.Tensor) -> torch.Tensor:
        """Any number of tokens and rows that end inside the last 64 columns: the GEMV with a workgroup per 32 tokens, or the table GEMM."""
        from .. import kernels

        x2d, width = x.reshape(-1, self.in_features), self._kernel_k()
        main, bits = self._kernel_stream()
        try:
            if self.is_residual:
                y = kernels.rvq_linear_blocks(
                    x2d, main, bits, *self._kernel_res_stream(), self.proxy.centroids, self._res_centroids(), self.row_scale,
                    self.row_bias, self.out_features, self._bias_f32(), width=width,
                )  # fmt: skip
            else:
                y = kernels.vq_linear_blocks(x2d, main, self.proxy.centroids_as(x.dtype), bits, self.out_features, self._bias_f32(), width=width)
        except RuntimeError as exc:
            self._fallback("rvq_linear_blocks" if self.is_residual else "vq_linear_blocks", "decode + GEMM", exc)
            return self._forward_dequant_gemm(x)
        return y.reshape(*x.shape[:-1], self.out_features)

    def _fused(self, x: torch.Tensor, tile: bool, perm: torch.Tensor | None = None) -> torch.Tensor:
        from .. import kernels

        *leading, _ = x.shape
        x2d = x.reshape(-1, self.in_features)
        if self.is_residual:
            (main, bits), (res, res_bits) = self._kernel_stream(), self._kernel_res_stream()
            y = kernels.rvq_linear(
                x2d, main, bits, res, res_bits,
                self.proxy.centroids, self._res_centroids(), self.row_scale, self.row_bias,
                self.out_features, self._bias_f32(), tile=tile,
            )  # fmt: skip
        else:
            stream, bits = self._kernel_stream()
            if self._kernel_k() != self.in_features:
                x2d = kernels.gather_columns(x2d, None, self._kernel_k())
            cb = self.proxy.centroids_as(x.dtype)
            fn = kernels.vq_gemm_tile if tile else kernels.vq_linear
            if tile:
                y = fn(x2d, stream, cb, bits, self.out_features, self._bias_f32())
            else:
                y = fn(x2d, stream, cb, bits, self.vector_len, self._bias_f32(), self.out_features,
                       column_perm=perm)  # fmt: skip
        return y.reshape(*leading, self.out_features)

    def _forward_cuda(self, x: torch.Tensor) -> torch.Tensor:
        """Band (a) (reference: np_vq_linear.py:1173-1187).  Above the kernel's
        32-token limit (reachable only with a raised threshold) the tile GEMM runs."""
        m = x.numel() // self.in_features
        return self._fused(x, tile=m > _GEMV_KERNEL_MAX_TOKENS)

    def _forward_cuda_wmma(self, x: torch.Tensor) -> torch.Tensor:
        """GEMV / GEMM by token count (reference: np_vq_linear.py:1250-1267)."""
        m = x.numel() // self.in_features
        return self._fused(x, tile=m > _GEMV_KERNEL_MAX_TOKENS)

    def _forward_cuda_lut(self, x: torch.Tensor) -> torch.Tensor:
        """Reached only when ``_LUT_MAX_TOKENS`` was raised above 0.

        The reference's LUT kernel (np_vq_linear.py:1192-1248) builds an
        ``[M, n_groups, NC]`` table, which for the codebooks it is chosen for is
        larger than the weight and loses at every M (np_vq_linear.py:75-79);
        it is not rebuilt.  The same result is produced by the fused kernels.
        """
        m = x.numel() // self.in_features
        return self._fused(x, tile=m > _GEMV_KERNEL_MAX_TOKENS)

    # ------------------------------------------------------------------

    def extra_repr(self) -> str:
        perm_str = ", perm=True" if self.column_perm is not None else ""
        res_str = ", residual=True" if self.is_residual else ""
        if self.zero_escape:
            tiered_str = ", zero_escape=True"
        elif self.tier_bits is not None:
            tiered_str = f", ntier={self.tier_bits}"
        elif self.use_tiered:
            tiered_str = f", tiered=True(cold={self.cold_bits})"
        else:
            tiered_str = ""
        return (
            f"in={self.in_features}, out={self.out_features}, "
            f"vector_len={self.vector_len}, "
            f"num_centroids={self.proxy.num_centroids}, "
            f"bits={self.bits}, backend={self.backend.value}"
            f"{perm_str}{tiered_str}{res_str}"
        )


# ---------------------------------------------------------------------------
# Model-level transform
# ---------------------------------------------------------------------------


def linearize_vq_weights(
    model: nn.Module,
    backend: str | VQBackend | None = VQBackend.AUTO,
) -> nn.Module:
    """Replace every ``nn.Linear`` carrying a VQ weight with an :class:`NPVQLinear`.

    Follows neuropress/nn/np_vq_linear.py:1432-1517: layers whose codebook is
    the same tensor object share one :class:`VQProxy`; each unique proxy is
    registered on the model root as ``_vq_proxy_<i>`` (residual codebooks as
    ``_vq_res_proxy_<i>``).  The model is mutated in place and returned.
    """
    proxy_cache: dict[int, VQProxy] = {}
    res_cache: dict[int, VQProxy] = {}
    replacements: list[tuple[str, NPVQLinear]] = []

    for name, module in model.named_modules():
        if not isinstance(module, nn.Linear) or not is_vq_weight(module.weight):
            continue
        qs = module.weight.qscheme
        cid = id(qs.centroids)
        if cid not in proxy_cache:
            proxy_cache[cid] = VQProxy(qs.centroids)
        res_proxy = None
        res_c = getattr(qs, "residual_centroids", None)
        if res_c is not None:
            if id(res_c) not in res_cache:
                res_cache[id(res_c)] = VQProxy(res_c)
            res_proxy = res_cache[id(res_c)]
        try:
            layer = NPVQLinear.from_qtensor_linear(module, proxy_cache[cid], backend, res_proxy)
        except (TypeError, ValueError, NotImplementedError) as exc:
            log.warning("linearize_vq_weights: skipping %s — %s", name, exc)
            continue
        replacements.append((name, layer))

    if not replacements:
        log.info("linearize_vq_weights: no VQ-weight linear layers found.")
        return model

    for i, proxy in enumerate(proxy_cache.values()):
        model.add_module(f"_vq_proxy_{i}", proxy)
    for i, proxy in enumerate(res_cache.values()):
        model.add_module(f"_vq_res_proxy_{i}", proxy)

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
        "linearize_vq_weights: replaced %d layer(s) [%s], %d unique proxy/ies",
        len(replacements),
        summary,
        len(proxy_cache),
    )
    return model
