"""Backend enumerations for the quantized inference modules.

String values are the reference's (neuropress/nn/backends.py:102-159) so that
recipes, YAML lowering configs and saved checkpoints keep working.  The names
that say "cuda" select the HIP kernels of this package:

===================  =========================================================
``cuda`` / ``cuda_wmma``  fused decode GEMV -> tile-decode MFMA GEMM -> decode + GEMM,
                          by token count
``cuda_lut``              decode + GEMM at every token count unless the LUT
                          threshold is raised (the routing the reference gives
                          large-codebook layers)
``compile`` / ``default`` gather + ``F.linear`` with torch ops (CPU or GPU)
===================  =========================================================

``is_cuda_jit_available`` keeps its name; here it answers "can the HIP kernel
library run": the shared object loads and a GPU is visible.
"""

from __future__ import annotations

import enum
import logging
import os

_log = logging.getLogger(__name__)

_hip_ok: bool | None = None


def is_hip_backend_available() -> bool:
    """True when ``libnpamd.so`` loads and torch sees a GPU.  Cached.

    ``NEUROPRESS_FORCE_CUDA_JIT=1`` skips the probe and answers True, as the
    reference's switch of the same name does (neuropress/nn/backends.py:40).
    """
    global _hip_ok
    if _hip_ok is not None:
        return _hip_ok
    if os.environ.get("NEUROPRESS_FORCE_CUDA_JIT", "").strip() in ("1", "true", "yes"):
        _hip_ok = True
        return True
    import torch

    from .. import _lib

    if not torch.cuda.is_available():
        _hip_ok = False
        return False
    _hip_ok = _lib.is_available()
    if not _hip_ok:
        _log.warning(
            "libnpamd.so could not be loaded; HIP backends disabled, falling back to torch ops"
        )
    return _hip_ok


# Name kept for drop-in compatibility with code written against the reference.
is_cuda_jit_available = is_hip_backend_available


class _StrEnum(str, enum.Enum):
    """``enum.StrEnum`` for Python < 3.11: members compare and format as their value."""

    def __str__(self) -> str:
        return str(self.value)

    def __format__(self, spec: str) -> str:
        return format(str(self.value), spec)


class LinearBackend(_StrEnum):
    """Valid backends for scalar-quantized ``nn.Linear`` (:class:`.NPLinear`)."""

    AUTO = "auto"
    DEFAULT = "default"
    COMPILE = "compile"
    CUDA = "cuda"
    GEMLITE = "gemlite"


class EmbeddingBackend(_StrEnum):
    """Valid backends for scalar-quantized ``nn.Embedding`` (:class:`.NPEmbedding`)."""

    AUTO = "auto"
    DEFAULT = "default"
    COMPILE = "compile"
    CUDA = "cuda"


class NormBackend(_StrEnum):
    """Valid backends for RMSNorm modules (:class:`.NPRMSNorm`)."""

    AUTO = "auto"
    DEFAULT = "default"
    CUDA = "cuda"


class VQBackend(_StrEnum):
    """Valid backends for vector-quantized ``nn.Linear`` (:class:`.NPVQLinear`)."""

    AUTO = "auto"
    DEFAULT = "default"
    COMPILE = "compile"
    CUDA = "cuda"
    CUDA_WMMA = "cuda_wmma"
    CUDA_LUT = "cuda_lut"
    CUDA_TIERED = "cuda_tiered"
    CUDA_NTIER = "cuda_ntier"
    CUDA_ZERO_ESCAPE = "cuda_zero_escape"


class Backend(_StrEnum):
    """Superset enum kept for backward compatibility."""

    DEFAULT = "default"
    COMPILE = "compile"
    CUDA = "cuda"
    CUDA_WMMA = "cuda_wmma"
    CUDA_LUT = "cuda_lut"
    CUDA_TIERED = "cuda_tiered"
    CUDA_NTIER = "cuda_ntier"
    CUDA_ZERO_ESCAPE = "cuda_zero_escape"
    GEMLITE = "gemlite"
    AUTO = "auto"


def tensor_version(t) -> int:
    """``t._version`` for cache keys, or -1 for tensors that keep no version counter.

    Tensors created or moved under ``torch.inference_mode()`` raise on ``_version``; they
    cannot be written in place outside inference mode either, so device and address identify them.
    """
    try:
        return t._version
    except RuntimeError:
        return -1


# Layers of fewer weights than this decode in 4-8 us, and the dense product that follows is the faster kernel: they
# leave the tile GEMM earlier (tile_band_ok).  Long reductions of fewer weights than the last leave it past 256 tokens, and
# so do those of at least _MID_LAYER_K features on layers of at least the second.
_SMALL_LAYER_WEIGHTS: int = 8_000_000
_MID_LAYER_WEIGHTS: int = 12_000_000
_MID_LAYER_K: int = 6144
_LARGE_LAYER_WEIGHTS: int = 1 << 25
# Decode + GEMM / tile, us at 36 / 128 tokens: 5632 x 2048 with a 256-row codebook 14.0 / 15.9 against 11.5 / 14.7, residual 17.1 / 18.9
# against 16.9 / 21.6, int4 14.0 / 16.3 against 15.8 / 19.4; 5632 x 4096 int4 22.3 / 25.7 against 20.4 / 23.3, with zero points
# 22.4 / 25.7 against 24.9 / 27.7; 5504 x 8192 int4 41.6 / 48.3 against 29.5 / 36.3, 256-row codebook 43.4 / 50.2 against 20.7 / 27.1.
_TIGHT_GRID_FRACTION: float = 0.66
# What a call plan's choice of a kernel read here (it is valid while these are unchanged).
BAND_LINES = ("_SMALL_LAYER_WEIGHTS", "_MID_LAYER_WEIGHTS", "_MID_LAYER_K", "_LARGE_LAYER_WEIGHTS", "_TIGHT_GRID_FRACTION")


def tile_band_ok(
    m: int, n: int, k: int, cus: int, min_fraction: float, split_max_tokens: int, long_k: int,
    small_max_tokens: int = 1 << 30, half_ok: bool = False, tight_k: int = 1 << 30, library: bool = False,
) -> bool:
    """Whether the tile-decode GEMM has enough workgroups for ``m`` tokens on an
    ``n x k`` layer.  Mirrors the kernel's own plan: without a split when the
    (64 columns x up to 384 rows) grid covers ``min_fraction`` of ``cus`` compute
    units; otherwise up to 16 reduction splits of at least 512 input features.  *half_ok*: a grid of more than half
    the compute units, too large to split, will do.  From *tight_k* input features on 0.66 of them will do for a split
    grid (86 to 89 column blocks, in two parts).  *library*: against decode + the library's product, the alternative of
    calls that torch has to follow, as measured with int4 weights: 4096 x 4096 24-31 us against 37-45 from 128 to 256
    tokens; 1024 x 4096 (not enough workgroups even when split) 17-19 against 16-20.

    Measured, us, tile GEMM / decode + dense product: 3008 x 2240 with a 4096-row codebook 13.7 / 14.1 at 33 tokens,
    14.4 / 14.2 at 64, 17.5 / 15.2 at 128, with int4 weights 15.8 / 13.1 at 33; 6144 x 1024 int4 13.9 / 10.9 at 33;
    2048 x 8192 int4 29.6 / 30.2 at 256, 39.3 / 35.4 at 384; 4096 x 14336 int4 68 / 104 at 384.  At 230 tokens: 2432 x 7936
    int4 29.0 / 31.2, with a 256-row codebook 25.1 / 35.8, residual VQ 31.9 / 40.1; 4096 x 6144 30.5 / 34.3, 28.2 / 34.2,
    35.9 / 40.7; 4096 x 4096 26.1 / 24.6, 26.7 / 25, 28.8 / 28.6."""
    blocks = -(-n // 64) * -(-m // 384)
    if blocks >= min_fraction * cus or (half_ok and 2 * blocks > cus):
        return True
    splits = max(1, min(cus // blocks, k // 512, 16))
    if library:
        return splits * blocks >= min_fraction * cus and (m <= split_max_tokens or k >= long_k)
    if splits * blocks < min_fraction * cus and not (splits > 1 and k >= tight_k and splits * blocks >= _TIGHT_GRID_FRACTION * cus):
        return False
    if n * k < _SMALL_LAYER_WEIGHTS and m > small_max_tokens:
        return False
    if m <= split_max_tokens or (k >= _MID_LAYER_K and n * k >= _MID_LAYER_WEIGHTS and m <= 256):
        return True
    return k >= long_k and (n * k >= _LARGE_LAYER_WEIGHTS or m <= 256)
