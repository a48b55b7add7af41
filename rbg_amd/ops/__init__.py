"""rbg_amd.ops — dispatch layer over the CDNA4 HIP kernels.

On a GPU the compiled in-tree extension (_hip_ops, built by setup.py for
gfx950) is MANDATORY: a missing extension raises instead of silently running
an eager fallback, so GPU tests always exercise the native path.  On CPU
(unit tests, GPU-less CI) the fp32 torch references in ops.reference serve
as the implementation.
"""
from __future__ import annotations

import functools
import heapq
import importlib
from dataclasses import dataclass
from typing import Any, Dict, List, Optional, Tuple

import numpy as np
import torch

from ..utils import hip_build
from ..utils.upload import upload
from . import reference

# Extension modules by name, loaded as far as they are built; a process needs
# those that its model runs on (utils/hip_build.py EXTENSIONS_OF).
EXTENSIONS: Dict[str, Any] = {}
_errors: Dict[str, Exception] = {}
for _name in hip_build.HIP_SOURCES:
    try:
        EXTENSIONS[_name] = importlib.import_module("." + _name, __name__)
    except Exception as e:  # noqa: BLE001
        _errors[_name] = e

_hip = EXTENSIONS.get("_hip_ops")
HAVE_HIP = _hip is not None


def _check_stale() -> None:
    """Fail loudly on a GPU box if a shipped .so predates its kernel sources
    (stale-binary guard; the stamps are written by utils/hip_build.py)."""
    for name in EXTENSIONS:
        if hip_build.is_stale(name):
            raise RuntimeError(
                f"rbg_amd HIP extension {name} is STALE: kernel sources "
                "changed after the last build.  Rebuild in-tree: "
                "PYTORCH_ROCM_ARCH=gfx950 python setup.py build_ext "
                "--inplace")


if EXTENSIONS and torch.cuda.is_available():
    _check_stale()


def require(*names: str):
    """The first of these extensions that is built."""
    for name in names:
        if name in EXTENSIONS:
            return EXTENSIONS[name]
    errors = "; ".join(f"{n}: {_errors[n]!r}" for n in names)
    raise RuntimeError(
        f"rbg_amd HIP extension {' or '.join(names)} is not built but a GPU "
        "tensor was passed.  Build it in-tree: PYTORCH_ROCM_ARCH=gfx950 "
        f"python setup.py build_ext --inplace (import error: {errors})")


def _require_hip():
    return _hip if _hip is not None else require("_hip_ops")


def _require_mix():
    return require("_hip_mix")


def _require_latent():
    return require("_hip_latent")


def _require_moe():
    return require("_hip_moe")


def _require_hyper():
    return require("_hip_hyper")


def _require_experts():
    return require("_hip_experts")


def _require_gated():
    return require("_hip_gated")


def _on_gpu(t: torch.Tensor) -> bool:
    return t.is_cuda


# 0: products go to hipBLASLt, not to the hand-written GEMMs
SKINNY_GEMM = int(__import__("os").environ.get("RBG_SKINNY_GEMM", "1"))


def _skinny(rows: int, n: int, k: int, parts: bool = False) -> bool:
    """Does the hand-written decode GEMM (hip/skinny_gemm.hip) take a
    [rows, k] x [n, k] product, rather than hipBLASLt?  ``parts``: its reader
    adds up the parts of a split k, which saves a launch.  Measured over the
    whole range with cold weights (us, own / library): the library is uneven.

    Up to 10240 columns, as it splits k and the library does not: long ones at
    any decode batch (4096 x 4096: 96 rows 19 / 25, 129 rows 22.1 / 22.1;
    4096 x 14336: 192 rows 47 / 103, 256 rows 63 / 62; 5120 x 25600: 256 rows
    121 / 261), short ones for few rows (4096 x 2048: 32 rows 11.3 / 13.6, 64
    rows 15.3 / 14.5; 1024 x 4096: 64 rows 12.2 / 14.7, 128 rows 16.5 / 12.0).

    Beyond, up to 64 rows where its workgroups fill the chip: from 16384 columns
    (24576 x 3072: 5 rows 28 / 51, 64 rows 35 / 38; 32768 x 5120: 48 rows 66 / 87,
    64 rows 68 / 70; 36864 x 4096: 68 / 73 and 80 / 82; 65536 x 4096: 92 / 124 and
    103 / 136), except between its whole rounds for rows that are no multiple of 4
    KB apart or long, which the library reads as well (36864 x 3072: 16 rows 52 /
    53, 48 rows 61 / 56; 49152 x 5120: 32 rows 105 / 98; 49152 x 8192: 5 rows 148 /
    172, 32 rows 165 / 156).  Of fewer columns two thirds of the chip are enough for
    short k (12288 x 1536: 48 rows 16.2 / 16.9, 64 rows 17.7 / 17.0; x 4096: 64 rows
    28.7 / 28.9; not x 5120: 16 rows 30.7 / 29.2).  From 65 rows the library's tiles
    are as good (24576 x 2048: 64 rows 24.7 / 30.0, 96 rows 30 / 32, 128 rows 36 /
    34)."""
    if rows < 1 or n % 32 or k % 512:
        return False
    if n <= 10240:
        if k <= 2048:
            return rows <= (64 if parts or k <= 1024 and n >= 8192 else 32)
        if n <= 2048 and not parts:
            return rows <= min(256, k // 64)
        return rows <= (256 if k > 16384 else 192 if k >= 12288 else 128)
    if rows <= 4:
        return k % 2048 == 0 or n <= 24576 and k <= 4096
    if n <= 12288 and k > 16384:
        return 16 < rows <= 256
    if rows > 64 or _uneven(rows, n, k, parts):
        return False
    if n < 16384 and k <= 6144:
        return (k <= 1024 or k % 2048 == 0 and (n > 12288 or k <= 4096) or
                k <= 4096 and (rows <= 48 or parts and n <= 12288))
    if n < 16384 or k > 8192:
        return (k % 2048 == 0 and not 32768 < n < 49152 and
                (n > 16384 or k >= 12288))
    if n >= 65536:
        return _after_rounds(rows, n, k)
    return not (32768 < n < 65536 and rows > 16 and
                (k > 2560 if k % 2048 else k > 6144 and n <= 53248))


def _uneven(rows: int, n: int, k: int, parts: bool) -> bool:
    """Widths that _skinny gives away: a little above whole rounds of the decode GEMM's
    workgroups, 32768 columns or with 32 rows of W a wave 65536 (own / library, us: 33152
    x 4096, 48 rows 82.7 / 75.0, 32 rows even; 66048 x 3584, 64 rows 118 / 110, x 2560 56
    rows 0.84; 102400 x 7168, 48 rows 312 / 270, 56 rows 0.94), 50304 to 52224, whose
    second round is half full (x 5120: 5 rows 104 / 96, 16 rows 0.93; x 7168: 16 rows 141 /
    131), and short ones where the library's tiles of 64 rows fill the chip (13696 x 1024,
    64 rows 12.3 / 10.3; 15232 x 1536, 48 rows 15.5 / 14.7; 22016 x 7168, 24 rows 66 /
    63)."""
    if n < 16384:
        return not parts and (rows > 56 if k <= 1024 else
                              rows > 32 and k < 2048)
    if 20480 < n < 24576:
        return rows > 16 and k % 2048 > 0 and k > 6144
    if 32768 < n < 36864 and rows > 40:
        return 2048 < k <= 4096
    if 40960 < n < 54272 and rows <= 16:
        return k % 2048 > 0 and k > 4096 and (rows <= 8 or k > 6144)
    if 65536 < n < 73728:
        return k % 4096 > 0 and k > 2048 and (
            rows > 56 or rows > 32 and 2560 < k < 4096)
    return (98304 < n < 110592 and rows > 32 and rows % 16 == 0 and
            k > (6144 if rows > 48 else 4096))


def _after_rounds(rows: int, n: int, k: int) -> bool:
    """The decode GEMM from 65536 columns and to 8192 k, where its workgroups make
    whole rounds and a part of one (of the library's time: 4096 and 6144 k 0.83 to 1;
    73728 x 5120: 32 rows 0.90, 64 rows 1.14; 77824 x 8192: 16 rows 0.89, 32 rows 1.07;
    98304 x 8192 0.74 to 0.89)."""
    if k <= 6144:
        return k <= 4096 or k % 2048 == 0 or rows <= 32 or n >= 77824
    return n >= 90112 or rows <= 16 and n >= 77824


def _takes_skinny(x: torch.Tensor, w: torch.Tensor,
                  parts: bool = False) -> bool:
    return (SKINNY_GEMM and _on_gpu(x) and x.dim() == 2 and w.dim() == 2 and
            x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and
            _skinny(x.shape[0], w.shape[0], x.shape[1], parts) and
            _plain(x, w))


def _plain(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Not what only the library takes: strides, rows that begin between
    multiples of 16 bytes, gradients."""
    return (w.is_contiguous() and
            (x.data_ptr() | w.data_ptr()) % 16 == 0 and
            not (torch.is_grad_enabled() and
                 (x.requires_grad or w.requires_grad)))


def _stream(rows: int, n: int, k: int) -> bool:
    """Does the GEMM of up to 4 rows (hip/stream_rows.hip) take a [rows, k] x [n, k]
    product?  Of 268 of 1024 to 128256 columns and 1024 to 25600 k, 1 to 4 rows with
    cold weights, it takes 0.82 of the time of what is taken without it, and of 7 of
    them, of 25600 k, 0.2 to 3% more.  Not the widest of 2048 k, which the decode GEMM takes as one
    turn (us, 1 row: 128256 x 2048 84.6 / 90.6, 65536 x 2048 44.9 / 46.3, 49152 x 2048
    33.5 / 33.8, 65536 x 1024 27.4 / 22.5)."""
    return (1 <= rows <= 4 and n >= 1024 and n % 32 == 0 and k >= 1024 and
            k % 256 == 0 and (n <= 49152 or k > 2048 or k == 1024))


def _takes_stream(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (SKINNY_GEMM and _hip is not None and _on_gpu(x) and x.dim() == 2 and
            w.dim() == 2 and x.dtype == torch.bfloat16 and
            w.dtype == torch.bfloat16 and x.shape[1] == w.shape[1] and
            _stream(x.shape[0], w.shape[0], x.shape[1]) and _plain(x, w))


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """Projection GEMM: decode shapes take the hand-written kernels,
    prefill-sized ones the library."""
    if _takes_stream(x, w):
        return _hip.stream_linear(x.contiguous(), w)
    if _takes_skinny(x, w):
        # one of these is there whatever the model
        return require("_hip_ops", "_hip_mix", "_hip_gated", "_hip_moe",
                       "_hip_hyper").skinny_gemm(
            x if x.is_contiguous() else x.contiguous(), w)
    return torch.nn.functional.linear(x, w)


def linear_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear(x, w).float(): the decode GEMM stores its rounded results so (a
    launch of 2 to 4 us less), the GEMM of prompts its sums."""
    if _takes_stream(x, w):
        return _hip.stream_linear(x.contiguous(), w, 1)
    if _takes_skinny(x, w):
        return require("_hip_ops", "_hip_mix", "_hip_gated", "_hip_moe",
                       "_hip_hyper").skinny_gemm(
            x if x.is_contiguous() else x.contiguous(), w, wide=True)
    if _hip is not None and _takes_tile(x, w, _tile_f32):
        return _hip.tile_f32(x.contiguous(), w)
    return linear(x, w).float()


def _tile_f32(rows: int, n: int, k: int) -> bool:
    """Does the GEMM of prompts take a product in f32, rather than hipBLASLt and a
    conversion (a launch and its result once more)?  From 65 rows, where the decode GEMM
    ends, of wide matrices, as for fewer columns it would have to split k.  Own /
    library, in us, over 2030 sizes of 65 to 256 rows, 16384 to 128256 columns and 1024 to
    10240 k: what the rule takes 0.85 of the time (128 rows of 32768 x 4096 67.6 / 71.8,
    32768 x 8192 120 / 151, 128256 x 4096 220 / 268, 65536 x 8192 224 / 234; 129 rows of
    65536 x 5120 150 / 170, 192 rows even), 18 of 1148 slower by 3 to 6% (49152 x 2560: 80
    rows 71.0 / 67.7).  The lines lie where they were drawn for stores that took up
    to 5 us a tile longer: not k that is no multiple of 2048 from 4096 on (24576 x 5120:
    128 rows 78.3 / 75.2), nor where its tiles begin a round that the library's do not
    (66048 x 4096: 128 rows 166 / 161, 80 rows 146 / 158; 102400 x 2560: 80 rows 144 /
    135).  Of what they leave to the library it would now take 0.92 of the time on
    average, by 0.68 to 1.37 (34048 x 1536: 129 rows 36 / 53; 16384 x 4096: 128 rows 41 /
    45)."""
    if k < 1024 or k > 8192 or k % 64 or n % 64 or not _tile_fits(rows, n, k):
        return False
    if rows > 128:
        return rows <= 256 and n >= 49152 and k <= 6144
    if rows <= 64 or n < 24576:
        return False
    if k < 2048:
        return not 32768 < n < 41984
    fourth = rows >= 80 and 98304 < n < 126976
    if k % 2048:
        return k <= 4096 and not (49152 < n < 65536 or fourth or
                                  rows > 112 and 65536 < n < 71680)
    if rows > 112 and (32768 < n < 36864 and k == 4096 or
                       65536 < n < 71680 and k > 2048):
        return False
    return k <= 4096 or not fourth


def _tile_fits(rows: int, n: int, k: int) -> bool:
    """Sizes that the GEMM of prompts has numbers for: offsets within W's halves of
    32 bits, 2^24 tiles (hip/tile_bindings.h check_tile refuses others)."""
    return ((n // 2 + 256) * k < 2 ** 31 and rows < 2 ** 24 and
            -(-rows // 128) * -(-n // 128) < 2 ** 24)


def _tile(rows: int, n: int, k: int) -> bool:
    """Does the GEMM of prompts (hip/tile_gemm.hip) take a [rows, k] x [n, k]
    product whose reader adds up parts, rather than the decode GEMM or
    hipBLASLt?  It splits k where its tiles are few, which the library does not,
    and picks a tile by the shape.  Of 17000 shapes of 65 to 9500 rows, 1024 to 16384
    columns and 1024 to 28672 k, with the norm that reads the sums, it takes 0.6 to 0.8
    of the better of both from 8192 k, 0.85 to 0.95 of shorter (us: 5120 x 8192: 200 rows
    55 / 36; 2048 x 5632: 128 rows 18.5 / 15.9; 6144 x 4096: 704 rows 57 / 45; 4096 x
    4096: 1200 rows 55 / 47; 8192 x 28672: 400 rows 420 / 200).  The rule takes 0.4%
    more than the fastest of each.  Left to the others is a short k of a small result,
    which the library's smaller tiles end sooner (2048 x 2048: 200 rows 12.8 / 13.1, 640
    rows 17.2 / 16.5; 3072 x 2048: 150 rows 13.0 / 14.9, 704 rows 21 / 19; 1408 x 2560:
    300 rows 14.2 / 19.0), of up to 256 rows only if it is a multiple of 128 (1984 x 6144:
    113 rows 23 / 16) or below 1536; rows longer than the norm takes sums of; and what
    _whole_sooner says."""
    if (rows <= 64 or k < 1024 or k % 64 or not 1024 <= n <= 16384 or
            n % 64 or not _tile_fits(rows, n, k)):
        return False
    if rows > 256 and k < 5120:
        return rows * n > 1_000_000 and not _whole_sooner(rows, n, k)
    return (k > 2048 or k > 1536 and k % 128 > 0 or n > 8192 or
            rows * n > 1_200_000)


def _whole_sooner(rows: int, n: int, k: int) -> bool:
    """Is the library sooner than the tiles, of more than 256 rows and a k that those do
    not split (hip/tile_bindings.h pick_tile_parts)?  Over 3200 sizes of 257 to 1000 rows,
    2048 to 16384 columns and 2304 to 4608 k, with the norm, the tiles take 0.93 of its
    time and more of it where its own make whole rounds (library / tiles, us): to 288 rows
    of 5632 to 6400 columns 1.07 to 1.22 times (6144 x 4096: 257 rows 33.0 / 37.7, 288
    rows 34.0 / 40.1, 289 rows 34.5 / 33.7) and of 8704 to 10752 1.00 to 1.08; of 321 to
    384 rows, 3328 to 4096 columns 0.98 to 1.14 (4096 x 4096: 336 rows 28.7 / 30.0, 384
    rows 29.6 / 33.0, 385 rows 30.2 / 27.9) and more than 10752 columns 1.02 to 1.13
    (12288 x 4096: 300 rows 63 / 57, 380 rows 62 / 67; 16384 themselves stay with the
    tiles at 1.04 to 1.10, so that of them rows once taken stay taken); of 513 to 576
    rows, 3328 to 3584 and 8704 to 10752 columns 1.00 to 1.16.  A k between multiples of
    128 slows the library down (3840 x 4160: 365 rows 0.79)."""
    if k >= 4736 or k <= 2048 or k % 128:
        return False
    if rows <= 288:
        return 5376 < n <= 6400 or k >= 2560 and 8448 < n <= 10752
    if 320 < rows <= 384:
        return 10752 < n < 16384 or k >= 3072 and 3200 < n <= 4096
    return k >= 2560 and 512 < rows <= 576 and (3200 < n <= 3584 or
                                                8448 < n <= 10752)


def _takes_tile(x: torch.Tensor, w: torch.Tensor, rule) -> bool:
    return (SKINNY_GEMM and _on_gpu(x) and x.dim() == 2 and w.dim() == 2 and
            x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and
            x.shape[1] == w.shape[1] and
            rule(x.shape[0], w.shape[0], x.shape[1]) and _plain(x, w))


def linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear for a reader that adds up: where the GEMM splits k, or perhaps has few
    rows, f32 sums [parts, T, N] before their reduction, else [T, N] in x's dtype."""
    if _takes_stream(x, w):
        # in bf16, which the next norm reads in half the time (3 sequences of up to
        # 15000 tokens, six layers: 814 us, of sums 852), where the decode GEMM has
        # them so; the others keep their f32
        rows, k = x.shape
        once = k % 2048 == 0 or rows <= 2 and k <= 8192 and w.shape[0] <= 12288
        return _hip.stream_linear(x.contiguous(), w, 0 if once else 2)
    if x.shape[0] > 64 and _takes_tile(x, w, _tile):
        return _require_hip().tile_parts(x.contiguous(), w)
    if _takes_skinny(x, w, parts=True):
        return _require_hip().skinny_parts(
            x if x.is_contiguous() else x.contiguous(), w)
    return torch.nn.functional.linear(x, w)


def _glu(rows: int, n: int, k: int) -> bool:
    """Does a gate/up product apply silu in the decode GEMM, which then
    cannot split k?  Where its workgroups fill the chip all the same.  Against the
    product, by linear_parts or the library or in tiles, and silu_mul, at 1500
    shapes of 5 to 64 rows, 4096 to 131072 columns and 1024 to 10240 k (us): any
    from 11264 or 16384 columns (24576 x 4096: 5 rows 33.4 / 34.8, 64 rows 37.6 /
    38.8; 51200 x 5120 95 / 102), fewer of short k (4096 x 1024: 5 rows 7.2 / 8.7; 8192 x
    2048, 48 rows 13.0 / 13.1; 11264 x 4096: 32 rows even, 64 rows 9% more; 13312 x
    8192: 16 rows 0.96, 64 rows 1.07), 0.83 to 1.0 of the time but 5% more between
    those lines.  Not long k of 32769 to 40959 (36864 x 10240: 16 rows 1.07, 45056
    0.96).

    Up to 4 rows what the GEMM for them leaves: k below 1024, few columns."""
    if rows < 1 or n % 64 or k % 256 or k < 512:
        return False
    if rows <= 4:
        return k % 512 == 0 and (k % 2048 == 0 or n <= 24576 and k <= (
            8192 if rows <= 2 and n <= 12288 else 1536))
    if rows > 64:
        return False
    if n < 4096:
        return k <= (1536 if rows <= 32 else 1024)
    if k <= 2048:
        return True
    if n < 16384:
        few = rows <= 32
        return n >= 11264 and (k <= (4096 if few else 3072) or
                               few and n >= 13312 and k <= 8192)
    if k > 8192:
        return (n >= 18432 and not 32768 < n < 40960 and
                (n <= 65536 or k % 2048 == 0))
    return n < 65536 or _after_rounds(rows, n, k)


def _tile_few(rows: int, n: int, k: int) -> bool:
    """Does the GEMM of prompts take gate/up of 5 to 64 rows, in tiles of 64?  Asked
    after the decode GEMM (_glu), which reads its weights as well and leaves k that is
    no multiple of 256, and 65536 x 8192, where both and the library are even.  Of odd k
    it takes 0.3 to 1.0 of the library and silu_mul over 16640 to 57344 columns, 2112 to
    7232 k (us: 16640 x 4160: 5 rows 0.38, 64 rows 0.81; 36864 x 6080: 5 rows 1.01, 48
    rows 0.87), 0.5 to 1.04 to 98304 columns, but of long k up to 32 rows only (73728 x
    8000: 32 rows 271 / 370, 48 rows 273 / 232); not beyond (131072 x 4160: 5 rows 216 /
    184)."""
    if not 4 < rows <= 64 or k < 2048 or k > 8192 or n <= 16384:
        return False
    if k % 2048 == 0:       # a CU has about one tile; of these _glu leaves one size
        return n <= 26624 or 32768 < n <= 65536
    return k % 256 > 0 and (n <= 57344 or
                            n <= 98304 and (k <= 7232 or rows <= 32))


def _tile_glu(rows: int, n: int, k: int) -> bool:
    """Does it take a gate/up product, with silu?  Against what linear_swiglu would take
    instead, over 4400 shapes of 65 to 9500 rows, 2048 to 65536 columns and 1024 to 28672
    k: 0.75 to 0.9 of the time to 2048 k and 0.9 to 0.95 of the longer, where its tiles
    fill the chip (us: 28672 x 4096: 300 rows 82 / 72, 640 rows 147 / 127, 2048 rows 381 /
    342; 11264 x 2048: 96 rows 21.1 / 18.4, 1600 rows 95 / 68), which by the size of the
    result they have to do the more the longer k is.

    Instead of it stand, to 16384 columns, the parts of linear_parts, which silu cannot
    have here and which fill the chip with a small result (4096 x 8192: 320 rows 1.8 times,
    1500 rows 1.1); they keep f32 too, up to sizes that the rule knows.  Of more columns
    it is the library and silu_mul, which round gate and up to bf16.  What is taken there
    by its range is 0.94 of that time over 97 sizes where the result alone would not tell
    (24576 x 4096: 65 rows 54.8 / 44.9, 80 rows 54.6 / 45.9, 96 rows 51.6 / 47.5; 23552 x
    16512: 623 rows 0.58) and up to 1.15 for some of long k (36480 x 8704: 256 rows 1.11;
    32704 x 12608: 170 rows 1.15).  Left to the library are a part of a second round
    (36864 x 8192: 320 rows 1.09) and few rows of the widest (51200 x 5120: 65 to 99 rows
    117 / 127)."""
    if (k < 1024 or k % 64 or n < 2048 or n % 64 or
            not _tile_fits(rows, n, k)):
        return False
    if rows <= 64:
        return _tile_few(rows, n, k)
    if k <= 1536:
        return True
    if n > 16384:
        if k <= n and (24576 <= n <= 32768 if rows <= 128 else
                       not 256 < rows <= 384):
            return True
    elif k <= n:        # where linear_parts has no sums, but one rounded product
        if n > 12288 and rows > 256 and (
                k < 4736 or (rows > 512 or k < 10240) and
                rows * n > (6_300_000 if k >= 8192 else 5_500_000)):
            return True
        if n >= 8192 and rows > 128 and k < 3584 and rows * n > 1_590_000:
            return True
    if 24576 < n <= 32768 and k <= 8192 or n > 49152 and k > 6144:
        return True
    if k > 4096 and (20480 < n <= 24576 and rows <= 384 or
                     32768 < n <= 40960 and rows <= 320):
        return False
    return rows * n >= k * (400 if k <= 2048 else 600 if k <= 4096 else 1000)


def linear_swiglu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x Wg^T) * (x Wu^T), w = [Wg; Wu]."""
    if _takes_stream(x, w):
        return _hip.stream_swiglu(x.contiguous(), w)
    if _takes_tile(x, w, _glu):
        return _require_hip().skinny_swiglu(x.contiguous(), w)
    if x.shape[0] > 4 and _takes_tile(x, w, _tile_glu):
        return _require_hip().tile_swiglu(x.contiguous(), w)
    return silu_mul(linear_parts(x, w))


def place_inputs(fields, tables, new_fields, new_tables) -> None:
    """A captured decode step's inputs from new ones on its device: ``fields``, and
    ``tables`` [rows, width] with page 0 beyond ``new_tables`` [seqs, used]."""
    n, used = new_tables.shape
    fields.copy_(new_fields)
    tables.zero_()
    tables[:n, :used].copy_(new_tables)


def place_host_inputs(fields, tables, new_fields: np.ndarray,
                      new_tables: np.ndarray) -> None:
    """place_inputs of what the host has: int64 fields, int32 tables.  One launch that
    reads pinned memory, without a copy before it, of 4 us and a wait of 6 (steps of
    128 sequences 1931 -> 1910 us, of 45 1044 -> 1028)."""
    if _on_gpu(fields) and _hip is not None:
        _hip.place_host_inputs(fields, tables, torch.from_numpy(new_fields),
                               torch.from_numpy(new_tables))
        return
    place_inputs(fields, tables,
                 *upload([new_fields, new_tables], fields.device))


def _route(rows: int, n: int, k: int, glu: bool) -> int:
    if glu and _glu(rows, n, k):
        return 3
    if glu and _tile_glu(rows, n, k):
        return 4
    if rows > 64 and _tile(rows, n, k):
        return 2
    return 1 if _skinny(rows, n, k, True) else 0


@functools.lru_cache(maxsize=1024)
def _own_routes(rows: int, first, second, glu: bool) -> Tuple[int, int]:
    return _route(rows, *first, glu), _route(rows, *second, False)


def block_routes(rows: int, first, second, glu: bool) -> Tuple[int, int]:
    """What linear_parts, or linear_swiglu for the first, takes for products of
    that many rows and weights of these two shapes, as numbers of bindings.cpp's
    Route."""
    return (_own_routes(rows, first, second, glu) if SKINNY_GEMM
            else (0, 0))


def prompt_attention_block(src, residual, weight, eps: float, wqkv, wo,
                           heads: int, q_norm, k_norm, key_cache, value_cache,
                           cos_sin, positions, slot_mapping, scale: float,
                           plan, slots=None) -> Optional[torch.Tensor]:
    """norm_heads, prefill_attention by ``plan`` and linear_parts in one native
    call, which adds to ``residual`` in place; None, and nothing done, for what
    it does not take."""
    if not _on_gpu(residual) or plan is None or PREFILL_SWZ < 16:
        return None
    return _require_hip().prompt_attention_block(
        src, residual, weight, eps, wqkv, wo,
        block_routes(residual.shape[0], wqkv.shape, wo.shape, False), heads,
        q_norm, k_norm, key_cache, value_cache, cos_sin, positions,
        slot_mapping, scale, plan.blocks, plan.lens, plan.items, plan.joins,
        plan.parts, slots)


def swiglu_block(src, residual, weight, eps: float, w_gate_up,
                 w_down) -> Optional[torch.Tensor]:
    """norm_swiglu and linear_parts in one native call, which adds to
    ``residual`` in place; None, and nothing done, for what it does not take."""
    if not _on_gpu(residual):
        return None
    return _require_hip().swiglu_block(
        src, residual, weight, eps, w_gate_up, w_down,
        block_routes(residual.shape[0], w_gate_up.shape, w_down.shape, True))


def embed_rows(ids: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
    """table[ids]; NaN for an id outside where the kernel takes the call (1.8 us
    for a row of 4096, the indexing kernel 3.0; 128 rows 2.0 both)."""
    if (_on_gpu(table) and table.dtype == torch.bfloat16 and
            table.dim() == 2 and ids.dim() == 1 and
            table.is_contiguous() and table.shape[1] % 8 == 0 and
            table.data_ptr() % 16 == 0):
        return _require_hip().embed_rows(ids.long().contiguous(), table)
    return table[ids.long()]


def rows_at(x: torch.Tensor, rows: List[int]) -> torch.Tensor:
    """x[rows] of rows that the host names: one launch, which reads them from pinned
    memory, in place of a copy and the indexing kernel, 14 us with the wait between
    them (a prompt of 37 tokens, which its host bounds, 397 -> 383 us)."""
    if (_on_gpu(x) and _hip is not None and x.dtype == torch.bfloat16 and
            x.dim() == 2 and x.is_contiguous() and x.shape[1] % 8 == 0 and
            x.shape[1] > 0 and x.data_ptr() % 16 == 0):
        return _hip.rows_at(x, rows)
    return x[upload([np.array(rows, dtype=np.int64)], x.device)[0]]


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if _on_gpu(x):
        return _require_hip().rmsnorm(x, weight, eps)
    return reference.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float) -> None:
    if _on_gpu(x):
        _require_hip().fused_add_rmsnorm(x, residual, weight, eps)
        return
    reference.fused_add_rmsnorm(x, residual, weight, eps)


def add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                weight: torch.Tensor, eps: float) -> torch.Tensor:
    """residual += x (in place); returns its RMS norm, perhaps in x.  x may be
    linear_parts' sums."""
    if _on_gpu(x):
        # a workgroup per row with the row in registers: of many rows only few
        # run at a time (4096 wide: 256 rows 3.4 us against 3.5 of the other, 1024
        # rows 7.1 against 5.9)
        if x.dtype == torch.float32 or (
                x.shape[0] <= 256 and x.shape[-1] <= 16384):
            return _require_hip().add_rmsnorm(x, residual, weight, eps)
    fused_add_rmsnorm(x, residual, weight, eps)
    return x


def silu_mul(x: torch.Tensor) -> torch.Tensor:
    if _on_gpu(x):
        return _require_hip().silu_mul(x)
    return reference.silu_mul(x)


def rope_store_kv(q, k, v, key_cache, value_cache, cos_sin, positions,
                  slot_mapping) -> None:
    if _on_gpu(q):
        _require_hip().rope_store_kv(q, k, v, key_cache, value_cache,
                                     cos_sin, positions, slot_mapping)
        return
    reference.rope_store_kv(q, k, v, key_cache, value_cache, cos_sin,
                            positions, slot_mapping)


def rope_heads(proj, heads: int, q_norm, k_norm, eps: float, key_cache,
               value_cache, cos_sin, positions, slot_mapping) -> torch.Tensor:
    """rope_store_kv of a fused projection [T, q | k | v] (in place) or of
    linear_parts' sums, with RMS norms of the query and key heads before it
    (None: without); returns the projection in bf16."""
    dim, kvh = key_cache.shape[3], key_cache.shape[1]
    if _on_gpu(proj) and dim == 128 and proj.is_contiguous():
        return _require_hip().rope_heads(
            proj, heads, q_norm, k_norm, eps, key_cache, value_cache, cos_sin,
            positions, slot_mapping)
    if proj.dim() == 3:
        proj = proj.sum(0).to(key_cache.dtype)
    q, k, v = proj.split([heads * dim, kvh * dim, kvh * dim], dim=1)
    if q_norm is not None:
        for part, w in ((q, q_norm), (k, k_norm)):
            part.copy_(rmsnorm(part.reshape(-1, dim), w,
                               eps).view(part.shape))
    rope_store_kv(q, k, v, key_cache, value_cache, cos_sin, positions,
                  slot_mapping)
    return proj


def _takes_rows(src, residual: torch.Tensor, weight: torch.Tensor,
                w: torch.Tensor) -> bool:
    """Can norm and GEMM of up to 4 rows be one launch (hip/stream_rows.hip)?  Its
    waves hold an eighth of k of the rows, a sixteenth above 5120, in registers.  Of 184
    shapes of 1536 to 12288 columns and 1024 to 8192 k it takes 0.74 of the time of what
    was taken before, with silu of 4096 to 57344 columns 0.81 of 192; slower by 1 to
    1.5% are two of 6144 k, with silu."""
    return (_takes_stream(residual, w) and residual.shape[1] <= 8192 and
            residual.is_contiguous() and weight.data_ptr() % 16 == 0 and
            (src is None or (src.numel() == residual.numel() and
                             src.dtype in (torch.bfloat16, torch.float32) and
                             src.is_contiguous() and
                             src.data_ptr() % 16 == 0)))


def _normed(src, residual, weight, eps: float) -> torch.Tensor:
    if src is None:
        return rmsnorm(residual, weight, eps)
    return add_rmsnorm(src, residual, weight, eps)


def _norm_project(src, residual, weight, eps: float, w):
    """The projection by ``w`` of the RMS norm of residual + src, and the new
    residual, perhaps in the old one's memory."""
    if _takes_rows(src, residual, weight, w):
        return _require_hip().norm_rows(src, residual, weight, eps, w, 2)
    return linear_parts(_normed(src, residual, weight, eps), w), residual


def norm_heads(src, residual, weight, eps: float, w, heads: int, q_norm,
               k_norm, key_cache, value_cache, cos_sin, positions,
               slot_mapping):
    """rope_heads of the projection by ``w`` of the RMS norm of residual + src
    (src: linear_parts' result, or None).  Returns the projection in bf16 and
    the new residual, perhaps in the old one's memory."""
    proj, residual = _norm_project(src, residual, weight, eps, w)
    return rope_heads(proj, heads, q_norm, k_norm, eps, key_cache, value_cache,
                      cos_sin, positions, slot_mapping), residual


def norm_decode(src, residual, weight, eps: float, w, heads: int, q_norm,
                k_norm, key_cache, value_cache, cos_sin, positions,
                slot_mapping, block_tables, context_lens, scale: float,
                num_splits: int = 0, tickets=None):
    """decode_attention of norm_heads' queries, and the new residual."""
    proj, residual = _norm_project(src, residual, weight, eps, w)
    return decode_heads(proj, heads, q_norm, k_norm, eps, key_cache,
                        value_cache, cos_sin, positions, slot_mapping,
                        block_tables, context_lens, scale, num_splits,
                        tickets), residual


def norm_swiglu(src, residual, weight, eps: float, w):
    """linear_swiglu of the RMS norm of residual + src, and the new residual."""
    # of more rows than one where the norm does not cost more than its launch
    # (hip/stream_rows.hip launch_norm_rows)
    if _takes_rows(src, residual, weight, w):
        rows, k = residual.shape
        if rows == 1 or (src is None or src.dtype == torch.bfloat16) and (
                rows == 2 or k <= 4096):
            return _require_hip().norm_rows(src, residual, weight, eps, w, 1)
    return linear_swiglu(_normed(src, residual, weight, eps), w), residual


def _decode_span(pairs: int) -> Tuple[int, int]:
    """Keys of a part, and the most parts of a sequence, for that many
    (sequence, key head) pairs.  Few pairs need short parts to fill the chip,
    many need long ones, which start less often (us, 256 / 512 / 1024 / 2048
    keys: 8 pairs of 2048 10 / 13 / 18 / 26; 56 pairs of up to 3000 18.9 / 21.7 /
    19.7 / 29.8; 128 pairs of up to 2048 31 / 26 / 24 / 29; 360 pairs of up to
    2500 63 / 59 / 58 / 68; 512 pairs of up to 2048, 8 query heads each, 98 / 89 /
    84 / 76; 1024 pairs of 2080 224 / 191 / 177 / 174).  With
    tickets and no more sequences than 64 and than CUs for a key head the kernel finds
    the parts by the lengths, at most this many of a sequence (hip/decode_join.h)."""
    if pairs <= 64:
        return 256, 32
    if pairs <= 96:
        return 512, 16
    if pairs <= 384:
        return 1024, 8
    # Pairs alone fill the chip here: parts only even out ragged lengths, and
    # every workgroup without keys costs its start (128 sequences of 2080, 4 /
    # 8 / 20 / 64 parts: 184 / 179 / 191 / 218 us; one of 60000 beside 48 of 500,
    # 8 / 16 / 64 parts: 187 / 113 / 77 us).  8192 workgroups at most, as the sums
    # of each are 512 bytes a query head.
    return 2048, max(1, min(16, 8192 // pairs))


def pick_decode_splits(num_seqs: int, num_kv_heads: int,
                       max_context: int, variant: int = -1,
                       page_size: int = 16) -> int:
    """Fill the chip: MI355X has 256 CUs / 8 XCDs; measured optimum is
    ~1024 workgroups for BOTH kernels (profiles/decode_breakdown r59
    sweep: V4 B128 peaks at splits=2 = 1024 WGs, B64 at splits=4 = 1024).
    The MFMA kernel packs 2 sequences per WG, so its base WG count is
    half the dot2 kernel's at equal splits."""
    if variant < 0:
        variant = DECODE_VARIANT
    # Pages of other sizes take the dot2 form, whatever the variant.  Few pairs
    # gain by short parts there too (pages of 32, 8 heads, 32 / 16 parts: 1 x
    # 2048 12.4 / 16.0 us, 1 x 30000 85 / 159; 8 / 5: 45 of up to 2500 100 / 108),
    # many do not (8 / 2: 128 x 2080 311 / 307).
    if variant == 7 and page_size != 16 and num_seqs * num_kv_heads > 384:
        variant = 4
    if variant == 7:
        # as many as the table's capacity may need of _decode_span, or up to a
        # limit, above which parts grow with the sequence (hip/decode_pages.hip)
        span, most = _decode_span(num_seqs * num_kv_heads)
        return max(1, min((max_context + span - 1) // span, most))
    if variant >= 4:
        # v4/v5 pack 2 seqs per WG; v6 runs 1 seq per (2-wave) WG
        per_wg = 2 if variant in (4, 5) else 1
        base = num_kv_heads * ((num_seqs + per_wg - 1) // per_wg)
        by_ctx = max(1, max_context // 32)      # >= one page pair per split
    else:
        base = num_seqs * num_kv_heads
        by_ctx = max(1, max_context // 256)
    if base >= 1024:
        return 1
    want = max(1, 1024 // max(base, 1))
    return int(min(want, by_ctx, 16))


DECODE_VARIANT = int(__import__("os").environ.get("RBG_DECODE_VARIANT", "7"))  # decode_pages.hip: 6.1 TB/s against 5.5 of 4 (128 x 2080)
PREFILL_SWZ = int(__import__("os").environ.get("RBG_PREFILL_SWZ", "16"))  # prefill_flash.hip; below 16: the forms of attn_prefill.hip


def decode_attention(q, key_cache, value_cache, block_tables, context_lens,
                     scale: float, num_splits: int = 0,
                     variant: int = -1, tickets=None) -> torch.Tensor:
    """``tickets``: int32 zeros, one for every sequence and key head, which only
    this stream uses and which are zeros again afterwards: the parts of a sequence
    are then added up without a launch of their own."""
    if _on_gpu(q):
        if num_splits <= 0:
            if (DECODE_VARIANT if variant < 0 else variant) == 7:
                max_ctx = block_tables.shape[1] * key_cache.shape[2]
            else:
                max_ctx = (int(context_lens.max().item())
                           if context_lens.numel() else 1)
            num_splits = pick_decode_splits(q.shape[0], key_cache.shape[1],
                                            max_ctx, variant,
                                            key_cache.shape[2])
        if variant < 0:
            variant = DECODE_VARIANT
        return _require_hip().decode_attention(
            q, key_cache, value_cache, block_tables, context_lens, scale,
            num_splits, variant,
            _decode_span(q.shape[0] * key_cache.shape[1])[0], tickets)
    return reference.decode_attention(q, key_cache, value_cache, block_tables,
                                      context_lens, scale)


def decode_heads(proj, heads: int, q_norm, k_norm, eps: float, key_cache,
                 value_cache, cos_sin, positions, slot_mapping, block_tables,
                 context_lens, scale: float, num_splits: int = 0,
                 tickets=None) -> torch.Tensor:
    """decode_attention of rope_heads of one new token of every sequence, which
    context_lens count and whose slot no other sequence reads.  One launch where
    the attention has the kernel for pages of 16 (the rotation's own: 3 us)."""
    dim, kvh = key_cache.shape[3], key_cache.shape[1]
    if (_on_gpu(proj) and DECODE_VARIANT == 7 and dim == 128 and
            key_cache.shape[2] == 16 and heads % kvh == 0 and
            heads // kvh in (1, 2, 4, 8) and proj.is_contiguous() and
            key_cache.is_contiguous() and value_cache.is_contiguous() and
            block_tables.is_contiguous()):
        rows = proj.shape[-2]
        if num_splits <= 0:
            num_splits = pick_decode_splits(rows, kvh,
                                            block_tables.shape[1] * 16)
        return _require_hip().decode_heads(
            proj, heads, q_norm, k_norm, eps, key_cache, value_cache, cos_sin,
            positions, slot_mapping, block_tables, context_lens, scale,
            num_splits, _decode_span(rows * kvh)[0], tickets)
    qkv = rope_heads(proj, heads, q_norm, k_norm, eps, key_cache, value_cache,
                     cos_sin, positions, slot_mapping)
    q = qkv[:, :heads * dim].view(-1, heads, dim)
    return decode_attention(q, key_cache, value_cache, block_tables,
                            context_lens, scale, num_splits, tickets=tickets)


@dataclass
class PrefillPlan:
    """Workgroups of prompt attention (bindings.cpp prefill_flash)."""
    blocks: torch.Tensor        # [n, 4] int32
    lens: torch.Tensor          # [n] int32
    # where blocks are cut by keys: [m, 4] and [c, 3] int32, parts in all
    items: Optional[torch.Tensor] = None
    joins: Optional[torch.Tensor] = None
    parts: int = 0


def _cut_prefill(tiles: np.ndarray, kv_heads: int):
    """Work of blocks of so many tiles of 64 keys, most first, as equal shares
    of the chip's CUs: (items, joins, parts), or None where whole blocks are as
    good.

    A CU's share holds whole blocks as far as they fit, and other blocks are cut
    to fill it.  Times in us are those of hip/prefill_flash.hip: a tile takes 1.2
    by itself on a CU and 1.0 where its CU has others too; a part leaves 64 KB of sums, which
    are written and read at 5 TB/s, and the launch that adds them up takes 5.
    Whole blocks and cut ones, 32 heads of 8 (us): 40 rows after 9000 keys 140 / 27,
    512 after 4000 79 / 55, 1500 after 9000 294 / 249.  Not cut: 2048 rows, whose
    longest workgroups run beside the shortest (51), nor more blocks than four a
    CU, which even out by themselves."""
    cus = max(1, 256 // kv_heads)           # of a key head
    n, work = len(tiles), int(tiles.sum())
    if n == 0 or n > 4 * cus:
        return None
    share = max(-(-work // cus), 4)
    part_time = kv_heads * 0.026
    tile_time = 1.2 if n <= cus else 1.0
    least = tile_time * share + 5 + part_time * 2 * int((tiles > share).sum())
    tiles = tiles.tolist()
    whole = 1.2 * tiles[0]
    if n > cus:
        load = [t for t in reversed(tiles[:cus])]       # a heap: they ascend
        for t in tiles[cus:]:
            heapq.heapreplace(load, load[0] + t)
        whole = max(whole, max(load))
    if least > 0.95 * whole:
        return None
    items, joins, cut, parts = [], [], [], 0
    room = [-share] * cus                               # negative: a heap
    for b, t in enumerate(tiles):
        if t <= -room[0]:
            heapq.heapreplace(room, room[0] + t)
            items.append((b, 0, t, -1))
        else:
            cut.append(b)
    room = sorted(-r for r in room)                     # the most last
    over = max(2, share // 8)       # a share may be this much more
    for b in cut:
        done, first = 0, parts
        while done < tiles[b]:
            left = tiles[b] - done
            take = left
            if room and left > room[-1] + over:
                take = room[-1]
            if room:
                room[-1] -= take
                if room[-1] <= over:
                    room.pop()
                    if room and room[-1] <= over:
                        room.clear()
            items.append((b, done, done + take, parts))
            parts += 1
            done += take
        if parts == first + 1:      # whole after all
            items[-1] = items[-1][:3] + (-1,)
            parts = first
        else:
            joins.append((b, first, parts - first))
    longest = max(i[2] - i[1] for i in items)
    cost = max(1.2 * longest, tile_time * share) + 5 + part_time * parts
    if not joins or cost > 0.95 * whole:
        return None
    return np.array(items), np.array(joins), parts


def _turn_round(order: np.ndarray, kv_heads: int) -> np.ndarray:
    """Most work first.  Where all run at once, two per CU (256 CUs), the second
    half is turned round, so that the longest share with the shortest (2048
    tokens of 32 heads: 61 -> 56 us)."""
    if len(order) * kv_heads <= 512:
        half = 256 // kv_heads
        order = np.concatenate([order[:half], order[half:][::-1]])
    return order


def prefill_plan(cu, cu_k, heads: int, kv_heads: int, device) -> PrefillPlan:
    """``cu`` and ``cu_k``: where each sequence's query and kv rows begin, on
    the host.  For a GPU by hip/prefill_plan.h; what follows below, with _cut_prefill and
    _turn_round, states its steps and reasons, is its oracle in the tests, number by
    number, and plans for other devices.  A change to one is a change to both."""
    if torch.device(device).type == "cuda":
        return PrefillPlan(*_require_hip().prefill_plan(
            *(x if isinstance(x, list) else np.asarray(x).tolist()
              for x in (cu, cu_k)), heads, kv_heads, torch.device(device)))
    tokens = 128 // (heads // kv_heads)
    cu, cu_k = np.asarray(cu), np.asarray(cu_k)
    rows, lens = np.diff(cu), np.diff(cu_k)
    count = (rows + tokens - 1) // tokens
    seq = np.repeat(np.arange(len(rows)), count)
    nth = np.arange(len(seq)) - np.repeat(np.cumsum(count) - count, count)
    past = (lens - rows)[seq]
    need = np.minimum(past + (nth + 1) * tokens, lens[seq])
    order = np.argsort(-need, kind="stable")
    tiles = np.maximum((need[order] + 63) // 64, 0)
    cut = _cut_prefill(tiles, kv_heads)
    if cut is None:
        order = _turn_round(order, kv_heads)
    info = np.stack([cu[:-1][seq], nth, cu_k[:-1][seq], past], axis=1)
    arrays = [info[order], lens[seq][order]]
    if cut is not None:
        items, joins, parts = cut
        by_work = np.argsort(items[:, 1] - items[:, 2], kind="stable")
        arrays += [items[_turn_round(by_work, kv_heads)], joins]
    dev = upload([a.astype(np.int32) for a in arrays], device)
    return PrefillPlan(*dev, parts) if cut is not None else PrefillPlan(*dev)


def prefill_attention(q, k, v, cu_seqlens, scale: float, cu_seqlens_k=None,
                      plan: Optional[PrefillPlan] = None,
                      slots=None) -> torch.Tensor:
    """Varlen causal attention; q [Tq, QH, D], k/v [Tkv, KVH, D], or pages
    [pages, KVH, page_size, D] of which ``slots`` [Tkv] (page * page_size +
    place) names the rows.  ``plan``: prefill_plan of the same sequences, made
    once for all layers of a step."""
    if _on_gpu(q):
        kvh = k.shape[1]
        group = q.shape[1] // kvh
        if (PREFILL_SWZ >= 16 and q.shape[1] % kvh == 0 and group <= 128 and
                (slots is None or k.shape[2] & (k.shape[2] - 1) == 0)):
            if plan is None:
                cu = cu_seqlens.tolist()
                plan = prefill_plan(
                    cu, cu if cu_seqlens_k is None else cu_seqlens_k.tolist(),
                    q.shape[1], kvh, q.device)
            return _require_hip().prefill_flash(
                q, k, v, plan.blocks, plan.lens, scale, slots, plan.items,
                plan.joins, plan.parts)
    if slots is not None:
        at = slots.long()
        pages, place = at // k.shape[2], at % k.shape[2]
        k, v = k[pages, :, place], v[pages, :, place]
    if _on_gpu(q):
        # bit 2 = 8-wave 16x16 blocks; bit 3 = 4-wave 32x32 blocks
        swz = PREFILL_SWZ if PREFILL_SWZ < 16 else 6
        qtile = 128 if (swz & 12) else 64
        block_info, seq_lens = reference.prefill_block_info(
            cu_seqlens.cpu(), qtile=qtile,
            cu_seqlens_k=None if cu_seqlens_k is None else cu_seqlens_k.cpu())
        return _require_hip().prefill_attention(
            q, k, v, block_info.to(q.device), seq_lens.to(q.device), scale,
            swz)
    return reference.prefill_attention(q, k, v, cu_seqlens, scale,
                                       cu_seqlens_k)


build_cos_sin_table = reference.build_cos_sin_table


# -- f32 residual stream ----------------------------------------------------


def embed_stream(tokens, table, scale: float, copies: int = 1) -> torch.Tensor:
    """f32 stream [T, W] = table[tokens] * scale; [T, copies * W] of equal
    streams."""
    if _on_gpu(table):
        # linked into every extension of designs that scale
        return require("_hip_mix", "_hip_gated", "_hip_hyper").embed_stream(
            tokens, table, scale, copies)
    return reference.embed_stream(tokens, table, scale, copies)


def stream_norm(x, delta, w1, w2, groups: int, eps: float, dtype):
    """x += delta (in place, f32); returns the grouped RMS norms of x under
    w1 and w2 (None without w2) in ``dtype``."""
    if _on_gpu(x):
        out = _require_mix().stream_norm(x, delta, w1, w2, groups, eps,
                                         dtype == torch.float32, None, None,
                                         None, None)
        return out[0], (out[1] if w2 is not None else None)
    return reference.stream_norm(x, delta, w1, w2, groups, eps, dtype)


def stream_norm_conv(x, delta, w1, w2, groups: int, eps: float, dtype,
                     conv_w, conv_state, slots, positions):
    """Decode form of stream_norm + causal_conv, one token per sequence: the
    first result is convolved with its slot's history, which moves on."""
    if _on_gpu(x):
        out = _require_mix().stream_norm(x, delta, w1, w2, groups, eps,
                                         dtype == torch.float32, conv_w,
                                         conv_state, slots, positions)
        return out[0], (out[1] if w2 is not None else None)
    n1, n2 = reference.stream_norm(x, delta, w1, w2, groups, eps, dtype)
    cu = torch.arange(n1.shape[0] + 1, dtype=torch.int32)
    return reference.causal_conv(n1, conv_w, conv_state, cu, positions,
                                 slots), n2


CONV_TILE = 16


def causal_conv(x, conv_w, conv_state, tiles, cu_seqlens, starts, slots):
    """x + causal depthwise convolution over varlen sequences; conv_w is
    [taps, W], conv_state [slots, taps-1, W] (advanced in place)."""
    if _on_gpu(x):
        return _require_mix().causal_conv(x, conv_w, conv_state, tiles,
                                          cu_seqlens, starts, slots,
                                          max(CONV_TILE, conv_w.shape[0]))
    return reference.causal_conv(x, conv_w, conv_state, cu_seqlens, starts,
                                 slots)


# -- gates ------------------------------------------------------------------


def gelu_mul(x, out) -> None:
    """out (may be a column slice) = gelu_tanh(x[:, :F]) * x[:, F:]."""
    if _on_gpu(x):
        require("_hip_mix", "_hip_hyper").gelu_mul(x, out)
        return
    reference.gelu_mul(x, out)


def clamped_glu(gate, up, limit: float, out) -> None:
    """out = g sigmoid(1.702 g) (u + 1), g = min(gate, limit), u = up within
    +-limit; gate and up are column slices of one buffer."""
    if _on_gpu(gate):
        _require_hyper().clamped_glu(gate, up, limit, out)
        return
    reference.clamped_glu(gate, up, limit, out)


def tanh_rows(x) -> torch.Tensor:
    if _on_gpu(x):
        return _require_mix().tanh_rows(x)
    return torch.tanh(x.float()).to(x.dtype)


# -- generalized delta rule ---------------------------------------------------


DELTA_CHUNK = 16        # tokens per chunk of the prompt kernels


def delta_rule(proj, z, w2, w0, a_bias, norm_w, state, slots, cu_seqlens,
               starts, out, offs, decay_scale: float, unit_eps: float,
               norm_eps: float, chunks=None) -> None:
    """Gated delta rule over varlen rows (cu_seqlens None: one row per
    sequence), with the head norm and the output gate; ``offs`` are the
    columns of r, k, v, a, g and the low-rank decay input in ``proj``.  The
    decay logit is ``z``, or W2 tanh(low) formed in the kernel when None.
    With ``chunks`` = (tiles, chunk_cu) of DELTA_CHUNK tokens and a ``z``, the
    rows go through the matrix cores a chunk at a time."""
    if _on_gpu(proj):
        mix = _require_mix()
        args = (proj, z, w2, w0, a_bias, norm_w, state, slots, cu_seqlens,
                starts, out, offs, decay_scale, unit_eps, norm_eps)
        # the chunk form scales by e^(DELTA_CHUNK * decay_scale)
        if (chunks is not None and z is not None and state.shape[-1] <= 128
                and decay_scale * DELTA_CHUNK <= 60.0):
            mix.delta_chunk(*args, *chunks)
        else:
            mix.delta_step(*args)
        return
    reference.delta_rule(proj, z, w2, w0, a_bias, norm_w, state, slots,
                         cu_seqlens, starts, out, offs, decay_scale, unit_eps,
                         norm_eps)


# -- latent attention -----------------------------------------------------------


@dataclass
class Rotary:
    """Rotary positions of a step's rows: table [positions, dims] = [cos | sin]
    (models/rotary.py); pairs are neighbours (interleaved) or half the dims
    apart."""
    table: torch.Tensor
    positions: torch.Tensor     # [T] int32
    interleaved: bool

    def rows(self, part: slice) -> "Rotary":
        return Rotary(self.table, self.positions[part], self.interleaved)

    @property
    def dims(self) -> int:
        return self.table.shape[1]


def _rotary(rot: Optional[Rotary]):
    return (None, None, False) if rot is None else (rot.table, rot.positions,
                                                    rot.interleaved)


def latent_store(x, w, cache, slots, eps: float,
                 rot: Optional[Rotary] = None, second=None):
    """c = rms_norm(x) * w, written to the paged latents; returns c.  With
    ``rot`` x's last columns are no latent but a key part: rotated, it follows
    in the cache and in c.  ``second`` = (x2, w2), another latent of the same
    rows: its norm is returned beside c."""
    if _on_gpu(x):
        out = _require_latent().latent_store(x, w, cache, slots, eps,
                                             *_rotary(rot),
                                             *(second or (None, None)))
    else:
        out = reference.latent_store(x, w, cache, slots, eps, rot, second)
    return out[0] if second is None else out


def rotate_rows(x, rot: Rotary) -> None:
    """Rotates x [T, H, rot.dims] in place."""
    if _on_gpu(x):
        _require_latent().rotate_rows(x, *_rotary(rot))
        return
    x.copy_(reference.rotate(x, rot))


def window_attention(q, k, v, gate, out, view, scale: float, window: int,
                     shared=None, sink=None) -> None:
    """Causal attention over the last ``window`` positions (0: all), q/k
    [T, H, D], v [T, H, Dv]; ``view`` locates each query among the keys
    (engine/batch.py WindowView).  out = o * sigmoid(gate).  ``shared`` [T, D2]
    are the last dims of every head's key (k then has the others); ``sink`` [H]
    f32 is a logit per head without key and value."""
    if _on_gpu(q):
        _require_latent().window_attention(q, k, v, gate, out, view.row_info,
                                           view.seq_info, view.blocks, scale,
                                           window, shared, sink)
        return
    reference.window_attention(q, k, v, gate, out, view.row_info, scale,
                               window, shared, sink)


def pick_latent_splits(num_seqs: int, num_heads: int, max_keys: int) -> int:
    """Key splits of latent_decode: two workgroups per CU, one for small
    batches (the splits' sums cost more than they hide there), at least one
    64-key step each.  Depends on sizes only, so a captured decode step keeps
    its value."""
    base = num_seqs * ((num_heads + 15) // 16)
    want = 512 if base >= 64 else 256
    steps = (max_keys + 63) // 64
    return int(max(1, min((want + base - 1) // base, steps, 64)))


def latent_decode(q, cache, block_tables, context_lens, scale: float,
                  window: int, rank: int = 0, sink=None) -> torch.Tensor:
    """q [S, H, D] absorbed queries against the paged latents [.., D], whose
    first ``rank`` columns (0: all) are the value; returns [S, H, rank].
    ``sink`` as in window_attention."""
    rank = rank or q.shape[2]
    if _on_gpu(q):
        keys = block_tables.shape[1] * cache.shape[1]
        splits = pick_latent_splits(q.shape[0], q.shape[1],
                                    min(keys, window) if window else keys)
        return _require_latent().latent_decode(q, cache, block_tables,
                                               context_lens, scale, window,
                                               splits, rank, sink)
    return reference.latent_decode(q, cache, block_tables, context_lens,
                                   scale, window, rank, sink)


def head_linear(x, w, gate=None, out=None, tail=None,
                rot: Optional[Rotary] = None) -> torch.Tensor:
    """out[s, h, j] = sum_k x[s, h, k] w[h, j, k], times sigmoid(gate); ``out``
    [S, H * n] may be a column slice.  With ``tail`` [S, H, rot.dims] each head
    of out ends in its rotation: out [S, H, n + dims]."""
    heads, n = w.shape[0], w.shape[1]
    full = n + (rot.dims if rot is not None else 0)
    if out is None:
        out = x.new_empty((x.shape[0], heads * full))
    o = out.unflatten(1, (heads, full))
    if _on_gpu(x):
        _require_latent().head_linear(x, w, gate, o, tail, *_rotary(rot))
    else:
        reference.head_linear(x, w, gate, o[..., :n])
        if rot is not None:
            o[..., n:] = reference.rotate(tail, rot)
    return out if rot is None else o


# -- sandwich norms, paged attention, sparse experts ---------------------------


@dataclass
class Routing:
    """Which experts a step's tokens go to: T * top (token, choice) pairs,
    stored in expert order and cut into tiles of one expert each."""
    top: int
    tile: int                   # most rows of a tile
    weights: torch.Tensor       # [T, top] f32
    inv: torch.Tensor           # [T * top] int32: a pair's row
    rows: torch.Tensor          # [T * top] int32: a row's token
    tiles: torch.Tensor         # [n, 3] int32: expert, first row, rows
    count: Optional[torch.Tensor] = None    # GPU: how many tiles are used


def embed_pairs(tokens, prev, table, pairs, mul_prev: int,
                mul_cur: int) -> torch.Tensor:
    """f32 stream: table[token] + pairs[(prev * mul_prev + token * mul_cur) mod
    buckets], the last row of ``pairs`` where prev is -1."""
    if _on_gpu(table):
        return _require_moe().embed_pairs(tokens, prev, table, pairs, mul_prev,
                                          mul_cur)
    return reference.embed_pairs(tokens, prev, table, pairs, mul_prev, mul_cur)


def sandwich_norm(x, pending, w, eps: float, dtype):
    """x += RMS norm of what is pending under its weight (in place, f32; None:
    nothing); returns the RMS norm of x under w in ``dtype`` (None without w).
    ``pending`` = (rows, routing or None, weight); rows with a routing are
    weighed and summed first."""
    rows = route = wb = None
    if pending is not None:
        rows, route, wb = pending
    if _on_gpu(x):
        return _require_moe().sandwich_norm(
            x, rows, route.inv if route else None,
            route.weights if route else None, wb, w, eps,
            dtype == torch.float32)
    return reference.sandwich_norm(x, rows, route, wb, w, eps, dtype)


def moe_combine(y, route) -> torch.Tensor:
    """Weighed sums of each token's expert rows, in y's dtype."""
    if _on_gpu(y):
        return _require_experts().moe_combine(y, route.inv, route.weights)
    return reference.moe_combine(y, route).to(y.dtype)


def rope_store_paged(proj, bias, cos_sin, positions, slots, heads: int,
                     dim: int, k, v, offs) -> None:
    """Adds the biases (None: none) of a fused projection, rotates the leading
    dimensions of its queries (in place) and keys by cos_sin [positions, dims]
    = [cos | sin] (None: not), and writes keys and values to the pages [pages,
    kv heads, page_size, size].  ``offs`` are the columns of q, k, v; of q
    alone when the keys are another layer's."""
    if _on_gpu(proj):
        _require_moe().rope_store_paged(proj, bias, cos_sin, positions, slots,
                                        heads, dim, k, v, offs)
        return
    reference.rope_store_paged(proj, bias, cos_sin, positions, slots, heads,
                               dim, k, v, offs)


@dataclass
class Difference:
    """Differential heads: a head's query and key are two, whose softmaxes o1
    and o2 over the same values become (o1 - lam o2) / rms * scale."""
    lam: torch.Tensor           # [1] f32
    scale: float
    eps: float                  # inside the root


def _difference(diff: Optional[Difference]):
    return (None, 1.0, 0.0) if diff is None else (diff.lam, diff.scale,
                                                  diff.eps)


def paged_prefill(q, k, v, view, out, scale: float, softcap: float,
                  sink: bool, window: int = 0,
                  diff: Optional[Difference] = None) -> None:
    """Causal attention of portions [R, H, D] over the pages; ``view`` is the
    step's engine/batch.py PagedView.  Scores are scale * q.k, then softcap *
    tanh(score / softcap) (0: as they are); ``sink`` adds a key of score 0 and
    no value; ``window`` is how many keys a row sees, itself included (0: all
    before it).  With ``diff`` q and k hold two maps of half the size."""
    if _on_gpu(q):
        _require_moe().paged_prefill(q, k, v, view.tables, view.seq_info,
                                     view.row_info, view.blocks, out, scale,
                                     softcap, sink, window,
                                     *_difference(diff))
        return
    reference.paged_rows(q, k, v, view.tables, view.row_info, out, scale,
                         softcap, sink, window, diff)


def pick_paged_splits(num_seqs: int, kv_heads: int, max_keys: int) -> int:
    """Key splits of paged_decode: two workgroups per CU, at least one
    128-key step each.  Depends on sizes only, so that a captured decode step
    keeps its value."""
    base = max(1, num_seqs * kv_heads)
    steps = (max_keys + 127) // 128
    return int(max(1, min((512 + base - 1) // base, steps, 64)))


def paged_decode(q, k, v, tables, context_lens, out, scale: float,
                 softcap: float, sink: bool, splits: int = 0, window: int = 0,
                 diff: Optional[Difference] = None) -> None:
    """One query row per sequence, [S, H, D]; scores as in paged_prefill."""
    if _on_gpu(q):
        if splits <= 0:
            keys = tables.shape[1] * k.shape[2]
            # a window may begin anywhere in its first step
            splits = pick_paged_splits(
                q.shape[0], k.shape[1],
                min(keys, window + 127) if window else keys)
        _require_moe().paged_decode(q, k, v, tables, context_lens, out, scale,
                                    softcap, sink, window,
                                    *_difference(diff), splits)
        return
    info = torch.stack([torch.arange(q.shape[0], dtype=torch.int32),
                        context_lens - 1], dim=1)
    reference.paged_rows(q, k, v, tables, info, out, scale, softcap, sink,
                         window, diff)


def router_logits(x, w) -> torch.Tensor:
    """x W^T in 32-bit, [T, experts] f32."""
    if _on_gpu(x):
        return _require_experts().router_logits(x, w)
    return x.float() @ w.float().T


def expert_tile(x, w, top: float) -> int:
    """Rows per tile that suit x [T, K] through experts w [E, N, K], ``top`` of
    them a token on average."""
    pairs = x.shape[0] * top
    rows = pairs / w.shape[0]                   # per expert, on average
    if (not _on_gpu(x) or x.dtype == torch.float32 or w.shape[1] % 8 or
            w.shape[2] % 8 or
            # the chip would not be full of 64-column pieces
            pairs * ((w.shape[1] + 63) // 64) < 256):
        return 16
    return 32 if rows <= 20 else 64 if rows <= 40 else 128


def moe_route(logits, correction, groups: int, keep: int, top: int,
              tile: int, softmax: bool = False, share: Optional[float] = None,
              identity: int = 0) -> Routing:
    """Chooses the ``top`` experts of each token by sigmoid(logit) + correction
    among the ``keep`` groups with the largest sums of their two best, and lays
    the pairs out by expert.  Weights are the sigmoids.  ``softmax``: the
    choice is by logit + correction, the weights are the softmax of the
    chosen.  ``share``: the scores are the softmax of all, the weights the
    chosen ones' shares of their scores times ``share``.  The last ``identity``
    experts return their input: their pairs are weighed but get no row."""
    if _on_gpu(logits):
        mod = _require_experts()
        mode = (mod.ROUTE_SHARE if share is not None else
                mod.ROUTE_CHOSEN if softmax else mod.ROUTE_SIGMOID)
        weights, inv, rows, tiles, count = mod.moe_route(
            logits, correction, groups, keep, top, tile, mode, identity,
            1.0 if share is None else share)
        return Routing(top, tile, weights, inv, rows, tiles, count)
    ids, weights = reference.moe_choose(logits, correction, groups, keep, top,
                                        softmax, share)
    return Routing(top, tile, weights, *reference.moe_tiles(
        ids, logits.shape[1] - identity, tile))


def interleave_glu(gate, up) -> torch.Tensor:
    """Rows of two matrices [.., F, K] (F even) as expert_linear's ``swiglu``
    reads them: two of the gate, two of the up matrix, and so on."""
    f, k = gate.shape[-2:]
    pair = [t.unflatten(-2, (f // 2, 2)) for t in (gate, up)]
    return torch.cat(pair, dim=-2).flatten(-3, -2)


def expert_linear(x, w, route, gather: bool = False, relu2: bool = False,
                  swiglu: bool = False,
                  limit: Optional[float] = None) -> torch.Tensor:
    """Rows in expert order times their expert's w [E, N, K]; ``gather`` takes
    x's rows by token, ``relu2`` applies max(0, .)^2, ``swiglu`` takes w's rows
    as interleave_glu lays them and gives silu(gate) * up, [.., N / 2]; with
    ``limit`` it is clamped_glu."""
    if _on_gpu(x):
        mod = _require_experts()
        act = (mod.EXPERT_RELU2 if relu2 else mod.EXPERT_NONE if not swiglu
               else mod.EXPERT_SILU_GLU if limit is None else
               mod.EXPERT_CLAMPED_GLU)
        return mod.expert_linear(
            x, w, route.rows if gather else None, route.tiles, route.count,
            route.rows.numel(), route.tile, act, limit or 0.0)
    return reference.expert_linear(x, w, route, gather, relu2, swiglu, limit)


# -- hyper-connections -----------------------------------------------------------


@dataclass
class TanhNorm:
    """Dynamic tanh: tanh(alpha * x) * w + b, no statistics of the row."""
    alpha: torch.Tensor         # [1] f32
    w: torch.Tensor             # [W] f32
    b: torch.Tensor             # [W] f32


@dataclass
class Stir:
    """A sublayer's output on its way into the streams: x_t becomes
    sum_s mix[s, t] x_s + mult * out[t] * y, y = rows plus, with a routing, the
    weighed sum of the token's expert rows (``self_rows``: of experts that
    return their input)."""
    conn: torch.Tensor          # [S * S + S] f32 = mix[from, to] | out
    mult: float
    rows: Optional[torch.Tensor] = None         # [T, W]
    experts: Optional[torch.Tensor] = None      # [T * top, W]
    route: Optional[Routing] = None
    self_rows: Optional[torch.Tensor] = None    # [T, W]


def hyper_norm(x, streams: int, stir: Optional[Stir], read,
               norm: Optional[TanhNorm], dtype):
    """x [T, streams * W] f32 takes what is pending (in place); returns the
    norm of sum_s read[s] x_s in ``dtype`` (None without a norm)."""
    if _on_gpu(x):
        s = stir or Stir(None, 1.0)
        n = norm or TanhNorm(None, None, None)
        return _require_hyper().hyper_norm(
            x, streams, s.conn, s.rows, s.experts,
            s.route.inv if s.route else None,
            s.route.weights if s.route else None, s.self_rows, s.mult, read,
            n.w, n.b, n.alpha, dtype == torch.float32)
    return reference.hyper_norm(x, streams, stir, read, norm, dtype)


# -- gated branches, gated delta rule -------------------------------------------


@dataclass
class Branch:
    """What a layer leaves to be added to the stream: (rows + bias) * scale *
    sigmoid(logits + gate_bias), rows of tokens or (with a routing) of their
    chosen experts, weighed and summed."""
    rows: torch.Tensor          # [T, W], or expert rows
    logits: torch.Tensor        # [T, W]
    gate_bias: torch.Tensor     # [W] f32
    scale: torch.Tensor         # [W] f32
    bias: Optional[torch.Tensor] = None         # [W] f32
    route: Optional[Routing] = None


def gate_norm(x, branches, w, eps: float, dtype):
    """x += the branches (in place, f32; at most two); returns the RMS norm of
    x under w, one number or one per coordinate, in ``dtype`` (None without
    w)."""
    if _on_gpu(x):
        return _require_gated().gate_norm(
            x, [(b.rows, b.route.inv if b.route else None,
                 b.route.weights if b.route else None, b.logits, b.gate_bias,
                 b.scale, b.bias) for b in branches], w, eps,
            dtype == torch.float32)
    return reference.gate_norm(x, branches, w, eps, dtype)


def silu_glu(gate, up, gate_bias, up_bias, out) -> None:
    """out = silu(gate + gate_bias) * (up + up_bias); gate and up are column
    slices of one buffer, the biases may be None."""
    if _on_gpu(gate):
        _require_gated().silu_glu(gate, up, gate_bias, up_bias, out)
        return
    reference.silu_glu(gate, up, gate_bias, up_bias, out)


def short_conv(x, conv_w, ring, tiles, cu_seqlens, starts, slots):
    """silu of the causal depthwise convolution of varlen rows (a column
    slice); conv_w [taps, W], the last tap the current token's; ring [slots,
    taps, W] holds a sequence's last inputs, position p's at p % taps."""
    if _on_gpu(x):
        return _require_gated().short_conv(x, conv_w, ring, tiles, cu_seqlens,
                                           starts, slots,
                                           max(CONV_TILE, conv_w.shape[0]))
    return reference.short_conv(x, conv_w, ring, cu_seqlens, starts, slots)


@dataclass
class GatedDelta:
    """Constants of a gated delta rule (gated_delta)."""
    a_log: torch.Tensor         # [H] f32
    dt_bias: torch.Tensor       # [H] f32, or [H*D]: a decay per key channel
    norm: torch.Tensor          # [E] f32
    kv_heads: int
    silu: bool                  # output gate: silu, else sigmoid
    q_scale: float
    unit_eps: float             # inside the root of q's and k's norms
    norm_eps: float             # inside the root of the head norm's


def gated_delta(p: GatedDelta, qkv, offs, beta, decay, gate, state, slots,
                cu_seqlens, starts, out, conv=None, chunks=None) -> None:
    """Gated delta rule over varlen rows (cu_seqlens None: one row per
    sequence) with the head norm and the output gate.  ``offs`` are the columns
    of q, k [kv_heads, D], v [H, E] in ``qkv``; state [slots, H, D, E].
    Per token, with unit q (times q_scale) and k, g = exp(-exp(a_log) *
    softplus(decay + dt_bias)):
      S <- g S;  u = sigmoid(beta) (v - S^T k);  S <- S + k u^T;  o = S^T q.
    ``conv`` = (conv_w, ring): decode rows, whose q, k, v are first convolved
    as by short_conv, over the columns from q's on.  With ``chunks`` = (tiles,
    chunk_cu) of DELTA_CHUNK tokens the rows go through the matrix cores."""
    if _on_gpu(qkv):
        mod = _require_gated()
        args = (qkv, beta, decay, gate, p.a_log, p.dt_bias, p.norm, state,
                slots, cu_seqlens, starts, out, offs, p.kv_heads, p.silu,
                p.q_scale, p.unit_eps, p.norm_eps)
        if chunks is not None and state.shape[2] <= mod.CHUNK_MAX_DIM:
            assert mod.CHUNK == DELTA_CHUNK
            mod.gated_chunk(*args, *chunks)
        else:
            mod.gated_step(*args, *(conv or (None, None)))
        return
    if conv is not None:
        n = slots.numel()
        width = conv[0].shape[1]
        x = reference.short_conv(
            qkv[:, offs[0]:offs[0] + width], *conv,
            torch.arange(n + 1, dtype=torch.int32), starts, slots)
        qkv, offs = x, [o - offs[0] for o in offs]
    reference.gated_delta(p, qkv, offs, beta, decay, gate, state, slots,
                          cu_seqlens, starts, out)
