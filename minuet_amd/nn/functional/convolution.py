"""Gather-GEMM-Scatter forward and its stage timers (mirrors
minuet/nn/functional/convolution.py)."""
from typing import Optional

import torch

from . import _C
from ..kernel_map import KernelMap

__all__ = ["cuda_time_gather", "cuda_time_scatter", "sparse_convolution_forward",
           "cuda_time_gemm", "set_gemm_parallel_level", "Epilogue", "pack_weights",
           "prefers_implicit", "prefers_streamed", "prefers_hits", "implicit_rows_limit", "hits_rows_limit",
           "hits_rows_from", "streamed_rows_limit", "implicit_rows_from", "implicit_rows_few", "layer_form",
           "prefers_implicit_over",
           "pieces_rows_limit", "channel_pieces"]

pack_weights = _C.pack_weights

Epilogue = _C.Epilogue

GEMM_PARALLEL_LEVEL = 4
DATAFLOWS = ("auto", "gather_gemm_scatter", "implicit", "list_driven")


def set_gemm_parallel_level(level: int):
    """Kept for compatibility (reference: convolution.py:15-25).  The reference
    spreads per-bucket GEMMs over this many streams; here all offsets run in
    one grouped launch, so the value has no effect."""
    global GEMM_PARALLEL_LEVEL
    GEMM_PARALLEL_LEVEL = level


def layer_form(stride, dilation, transposed: bool) -> str:
    """What the rules below ask of a layer beside its shape, because it decides how
    many of its offsets have a source: ``"plain"`` (stride 1), ``"dilated"`` (stride 1),
    ``"strided"`` and ``"transposed"`` (stride 2 at most, no dilation), or ``"other"``."""
    if all(s == 1 for s in stride):
        return "plain" if all(d == 1 for d in dilation) else "dilated"
    if any(s > 2 for s in stride) or any(d != 1 for d in dilation):
        return "other"
    return "transposed" if transposed else "strided"


def prefers_implicit(num_offsets: int, num_source_features: int, num_target_features: int,
                     dtype: torch.dtype, form: str = "plain") -> bool:
    """Whether ``dataflow="auto"`` takes the single-kernel form for a layer of
    this shape: it must fit that kernel, and it must be the faster one, which
    measurements say it is for 16-bit features with source rows of up to 128
    bytes and up to 128 output channels, and for rows of up to 256 bytes with up
    to 64 output channels under kernels of more than 8 offsets (beyond that its
    matrix work on empty (offset, target) pairs outweighs the buffer traffic it
    saves).  With rows of up to 64 bytes there is so little of that work that up to
    36 offsets take any number of output channels, and 5x5x5 over few rows and over
    many (``implicit_rows_few``, ``implicit_rows_from``): a second 128 of them
    cost as much as the first, the three kernels' product rows more (us, three
    kernels and here: 3x3x3 24 -> 256 over 200 000 voxels of a LiDAR scan 326 / 66, 32
    -> 160 over 5 000 of a room 19 / 10, over 1 000 15 / 11; 2x2x2 16 -> 160 over 50 000
    28 / 16; over 290 layers of 8 to 36 offsets, strided and transposed ones among them,
    1 000 to 300 000 voxels of three kinds of scene, 0.76 times as long at most).  Not
    kernels in between, where a target has a smaller share of
    its offsets (4x4x4 32 -> 160 over 50 000 of a room 53 / 64), nor larger ones
    (6x6x6 32 -> 256 over 50 000 155 / 200), nor strides of 3 and more (3x3x3 32 -> 512
    transposed 1.2 to 1.3 times as long over 30 000).  An fp32 layer of more than one offset goes by its rows instead
    (``hits_rows_limit``); without rows to go by, this says yes to the narrow
    ones with strided 2^D kernels, whose (offset, target) pairs are mostly hits."""
    if not _C.implicit_forward_supported(num_source_features, num_target_features, dtype, num_offsets):
        return False
    if dtype != torch.float32:
        row_bytes = num_source_features * dtype.itemsize
        if row_bytes <= 128:
            return num_target_features <= 128 or (row_bytes <= 64 and form != "other"
                                                  and (num_offsets <= 36 or num_offsets == 125))
        return row_bytes <= 256 and num_target_features <= 64 and num_offsets > 8
    return num_offsets <= 8 and num_source_features * num_target_features <= 1024


def prefers_streamed(num_offsets: int, num_source_features: int, num_target_features: int,
                     dtype: torch.dtype) -> bool:
    """Whether ``dataflow="auto"`` takes the single-kernel form for a layer too wide
    for ``prefers_implicit``: 16-bit rows of 144 to 512 bytes (or of 80 and more
    under more than 128 output channels), whose rows and weights stream through
    LDS.  Against three kernels or offset groups, us a layer: 128 -> 128 channels
    over 6 850 voxels 23.0 and 11.8, over 18 600 of a LiDAR level 27.7 and 17.3,
    256 -> 256 over 2 000 27.1 and 16.8, over 25 600 of a scan 39.5 and 37.1.  Not
    rows of more than 384 bytes under up to 96 output channels and more than 8
    offsets, which have four stages an offset and few product bytes to save: 256 ->
    64 over 23 100 24.2 and 30.7, 256 -> 96 over 10 400 21.6 and 26.2, 256 -> 32 over
    18 800 19.5 and 27.7 (the other way round over few voxels, 256 -> 32 over 2 300
    22.6 and 16.9; 192 -> 64 over 22 000 24.0 and 24.0, over 13 800 19.7 and 15.9).
    Nor more than 36 offsets, most of which a target has no source under and which
    are walked all the same: 4x4x4 and 5x5x5, 256 -> 128 over 9 000 of a scan 29 and
    94, 192 -> 224 over 20 000 of a room 73 and 203, 192 -> 64 over 26 000 23 and 49,
    128 -> 128 over 40 000 66 and 99 (96 -> 128 over 4 000 28 and 19; over 55 layers,
    with tiles and without, 1.36 times as long; 3x3x4 over 33 layers 0.89).

    What stays slower: fp16 layers of few sources a target just before they get
    tiles (160 -> 128 over 12 000 of a LiDAR scan 17.2 and 20.3), and strided layers
    of many targets whose map is kept for many calls (256 -> 160 onto 20 000 19 and 30,
    256 -> 256 onto 46 000 47 and 50).  On new clouds, where the other forms have rank
    tables to build, those take 0.67 times as long (of 209 the slowest two 1.12)."""
    if num_offsets > 36 or (num_offsets > 8 and num_source_features > 192 and num_target_features <= 96):
        return False
    return _C.streamed_forward_supported(num_offsets, num_source_features, num_target_features, dtype)


def streamed_rows_limit(num_offsets: int, num_source_features: int, num_target_features: int,
                        dtype: torch.dtype) -> int:
    """The most source rows of which ``prefers_streamed`` holds.

    Streamed workgroups take 128 output channels at a time, and fp16 3x3x3 layers of
    more than 192 input channels whose last 128 are at least half empty do without
    once workgroups of 64 x 64 no longer fit the chip in one go (offset groups and
    streamed, us: 256 -> 160 over 26 000 with dilation 2 31 and 39, 224 -> 144 over
    60 000 62 and 102, 224 -> 192 over 20 000 31 and 39, 208 -> 160 over 12 000 21 and
    25; below, 256 -> 192 over 3 000 21 and 18, over 700 18 and 14).  In bf16 the
    groups take longer: 256 -> 129 to 192 over 6 layers 0.85 times as long streamed."""
    if (num_offsets == 27 and num_source_features > 192 and num_target_features > 128
            and (num_target_features - 1) % 128 < 64 and dtype == torch.float16):
        return 256 // -(-num_target_features // 64) * 64
    return (1 << 63) - 1


def implicit_rows_from(num_offsets: int, num_source_features: int, num_target_features: int,
                       dtype: torch.dtype, form: str = "plain") -> int:
    """The fewest source rows past ``implicit_rows_few`` over which ``dataflow="auto"``
    takes the single-kernel form for a 16-bit layer that is not in its shape the
    faster one over any number of them (``prefers_implicit``, ``prefers_streamed``); one
    more than ``implicit_rows_limit``: over none.

    5x5x5 layers whose product rows outgrow the caches: rows of up to 64 bytes and
    more than 128 output channels; rows of 80 to 128 bytes and
    more than 128 output channels, of which the second 128 cost as much as the
    first, so half of them more than a whole, and rows of up to 256 bytes and 97 to
    128 output channels.  us, three kernels and here, the slowest and the fastest
    kind of scene: 32 -> 256 over 100 000 voxels 0.3 times as long of a LiDAR scan and
    0.4 of a room (over 50 000 1.5 and 1.2); 64 -> 256 over 100 000 of a room 312 / 239, of a LiDAR scan 333
    / 178 (over 30 000 of a room 72 / 84), 64 -> 160 over 150 000 333 / 278 and 447 / 205
    (over 100 000 of a room 219 / 234), 128 -> 128 over 150 000 282 / 264 and 369 / 185
    (over 100 000 of a room 172 / 215).  Not 128 -> 160 (250 000 of a room 570 / 666) nor
    128 -> 256 (481 / 496 over 150 000).  Strided layers have targets of fewer sources: 64 -> 160
    over 150 000 takes 0.75 to 1.13 times as long as in three kernels, 128 -> 128 over 250 000
    0.5 to 1.12, with a dilation of 2 0.4 to 1.06 and 0.4 to 1.15, so these two are for
    plain and transposed layers (0.35 to 0.6); 64 -> 256 strided 0.6 to 0.84, dilated 0.5 to 0.92."""
    far = implicit_rows_limit(num_source_features, dtype) + 1
    if (dtype == torch.float32 or num_offsets != 125 or form == "other"
            or not _C.implicit_forward_supported(num_source_features, num_target_features, dtype, num_offsets)):
        return far
    row_bytes = num_source_features * dtype.itemsize
    dense = form in ("plain", "transposed")
    if row_bytes <= 128 and num_target_features > 128 and (row_bytes <= 64 or (num_target_features - 1) % 128 >= 64):
        return min(far, 100_000)
    if dense and ((row_bytes <= 128 and num_target_features > 128)
                  or (128 < row_bytes <= 256 and 96 < num_target_features <= 128)):
        return min(far, 150_000)
    return far


def implicit_rows_few(num_offsets: int, num_source_features: int, num_target_features: int,
                      dtype: torch.dtype, form: str = "plain") -> int:
    """The most source rows short of ``implicit_rows_from`` over which ``auto`` takes
    the single-kernel form for the layer spoken of there (-1: over none).

    5x5x5, rows of up to 64 bytes, more than 128 output channels: a workgroup walks
    all 125 offsets whatever the number of rows, which costs less than two more launches
    while the chip is not full, and more from then on until product rows outgrow the
    caches.  Times as long as in three kernels, LiDAR / room / object: 32 -> 256 over 3 000
    0.86 / 0.51 / 0.46, 6 000 0.88 / 0.57 / 0.50, 12 000 1.07 / 0.83 / 0.71, 20 000 1.53 / 1.06 /
    0.80, 50 000 1.54 / 1.21 / 0.51; 32 -> 512 over 6 000 1.09 / 0.74 / 0.61; 32 -> 256 with a
    dilation of 2 over 12 000 1.12 / 0.92 / 0.94, transposed over 9 000 1.22 / 1.02 / 1.05,
    strided over 12 000 0.93 / 0.70 / 0.52."""
    if (num_offsets != 125 or dtype == torch.float32 or num_target_features <= 128
            or not prefers_implicit(num_offsets, num_source_features, num_target_features, dtype, form)):
        return -1
    return (20_000 if form in ("plain", "strided") else 12_000) // -(-num_target_features // 128)


def implicit_rows_limit(num_source_features: int, dtype: torch.dtype) -> int:
    """The most source rows of which the single-kernel form takes any: it addresses
    them through 32-bit buffer offsets, so features of 4 GiB and more go to the
    three kernels or the offset groups, which do not."""
    return (_C.IMPLICIT_MAX_SOURCE_BYTES - 1) // (num_source_features * dtype.itemsize)


def prefers_implicit_over(num_offsets: int, num_source_features: int, num_target_features: int,
                          dtype: torch.dtype, num_rows: int, form: str = "plain") -> bool:
    """``prefers_implicit`` over ``num_rows`` source rows."""
    layer = (num_offsets, num_source_features, num_target_features, dtype, form)
    most, begin = implicit_rows_limit(num_source_features, dtype), implicit_rows_from(*layer)
    return (prefers_implicit(*layer) and num_rows <= most
            and not (begin <= most and implicit_rows_few(*layer) < num_rows < begin))


def hits_rows_limit(num_offsets: int, num_source_features: int, num_target_features: int,
                    dtype: torch.dtype, form: str = "plain") -> int:
    """The most source rows over which ``dataflow="auto"`` takes the single-kernel
    form for an fp32 layer of more than one offset (-1: over none).

    That form multiplies hits only, 16 of one offset at a time, and reads the
    weights again for every 16; the three kernels read them once per 128 rows
    of their lists but write and read product rows.  So the line goes by rows x
    channels in x channels out.  It lies at 2.1 thousand million of them over
    the number of offsets, because rows have more hits the more offsets there
    are, and at 110 million at most: over 160 to 190 layers each of 2x2x2
    strided, 3x3x3 and 5x5x5 (three kinds of scene, 500 to 300 000 voxels, 24 to
    256 channels) the layers chosen by it take 0.7, 0.7 and 1.7 % longer than by
    the better choice for each.  Hits only against three kernels, us: 2x2x2 64 ->
    128 over 10 000 voxels 10.9 / 14.5, 64 -> 64 over 30 000 15.8 / 14.7; 3x3x3 64
    -> 64 over 10 000 12.3 to 21.0 / 13.0 to 20.6, over 20 000 26.4 / 21.7, 128 ->
    128 over 3 000 19.0 / 21.3, over 10 000 40.8 / 25.2; 5x5x5 64 -> 64 over 1 000
    17.7 / 19.4, over 10 000 32.6 to 67 / 25.3 to 40.6.  Up to 32 x 32 channels it
    is the faster one at any size (3x3x3 over 200 000 52 / 76, 5x5x5 over 100 000
    63 / 76), or about even (2x2x2 over 300 000 31.5 / 31.7 and, transposed, 36.9
    / 33.6).

    So it is for at most 16 input channels under 27 to 125 offsets, where products
    cost next to nothing and product rows as much as ever (0.4 to 0.96 times as
    long over 120 layers of 64 to 512 output channels and 3 000 to 300 000 voxels;
    one of 1.02): 3x3x3 16 -> 96 over 40 000 voxels of a room 26 / 35, over 200 000
    of a LiDAR scan 113 / 236, 16 -> 256 over 100 000 of objects 148 / 311; 5x5x5 16 ->
    256 over 20 000 83 / 92.  That holds for odd kernel sizes (3x3x5, 3x5x5, 7x7x1, 3x3x9
    and 11x11x1 0.29 to 1.08 times as long, LiDAR scans of 30 000 to 60 000 voxels last), dilated
    (0.4 to 1.03) and strided (0.4 to 1.05), and for transposed 3x3x3 layers (0.6 to 1.07;
    5x5x5 0.57 to 1.13); not for even ones, where a LiDAR scan of 12 000 to 130 000 voxels takes
    1.1 to 1.3 times as long (3x3x4, 4x4x4, 5x5x4), nor for strides of 3 and more (3x3x3
    transposed 0.7 to 1.4).

    Never more than ``implicit_rows_limit``."""
    if (dtype != torch.float32 or num_offsets <= 1
            or not _C.implicit_forward_supported(num_source_features, num_target_features, dtype)):
        return -1
    most = implicit_rows_limit(num_source_features, dtype)
    work = num_source_features * num_target_features
    if work <= 1024 or (num_source_features <= 16 and 27 <= num_offsets <= 125 and num_offsets % 2 == 1
                        and (form in ("plain", "dilated", "strided") or (form == "transposed" and num_offsets == 27))):
        return most
    return min(most, min(110_000_000, 2_100_000_000 // num_offsets) // work)


def hits_rows_from(num_offsets: int, num_source_features: int, num_target_features: int,
                   dtype: torch.dtype, form: str = "plain") -> int:
    """The fewest source rows past ``hits_rows_limit`` over which ``dataflow="auto"``
    takes the single-kernel form again (one more than ``implicit_rows_limit``:
    over none).

    From some 100 million products on, product rows outgrow the caches and the
    three kernels slow down, the single-kernel form does not.  With up to 48 input
    channels it is then the faster one for every kind of scene, LiDAR first and
    rooms, whose voxels have the fewest neighbours, last; us here and in three
    kernels, 3x3x3: 48 -> 64 over 250 000 voxels of a room 128 / 137, over 200 000
    108 / 102, of objects 180 / 249; 32 -> 64 of a LiDAR scan 132 / 228; 5x5x5: 48 -> 64
    over 150 000 of a room 207 / 242, over 100 000 153 / 147, 32 -> 64 of a LiDAR scan
    177 / 297.  (64 input channels: over 300 000 of a LiDAR scan 259 / 386, of a room
    171 / 181, but 64 -> 48 164 / 156, and with the sums that ``compact_forward``
    keeps for these layers 8 % more.)  Times as long, 32 and 48 -> 64 to 256 over 250 000
    voxels: 3x3x5 0.66 to 0.95, 3x5x5 0.58 to 0.96, 7x7x1 0.48 to 0.92, 3x3x9 0.67 to 1.02; 5x5x5 over
    130 000 0.67 to 0.98.  Kernels of even sizes are slower there (3x3x4, 4x4x4, 5x5x4 0.74 to 1.29
    times) unless they have at most 16 input channels (0.55 to 0.91; over 130 000 up to 1.12).
    Dilated, strided and transposed layers never come back to it: targets that have fewer sources
    leave the 16 rows of a product emptier (3x3x3 with a dilation of 3 1.0 to 1.17 times as
    long over 250 000 voxels of objects, strided 0.94 to 1.06, 5x5x5 48 -> 256 1.11)."""
    far = implicit_rows_limit(num_source_features, dtype) + 1
    if (hits_rows_limit(num_offsets, num_source_features, num_target_features, dtype, form) < 0
            or form != "plain" or not 27 <= num_offsets <= 125
            or num_source_features > (48 if num_offsets % 2 == 1 else 16)):
        return far
    return min(far, 130_000 if num_offsets == 125 else 250_000)


def channel_pieces(num_source_features: int) -> int:
    """Into how many pieces an fp32 pointwise layer over few rows cuts its input
    channels: of 32, or of 16 where there are fewer than four of 32."""
    return num_source_features // (32 if num_source_features % 32 == 0 and num_source_features >= 128 else 16)


def pieces_rows_limit(num_source_features: int, num_target_features: int, dtype: torch.dtype) -> int:
    """The most rows over which ``dataflow="auto"`` cuts an fp32 pointwise layer into
    pieces (-1: over none).  They let a workgroup's wavefronts share a row, and
    every 16 rows read the weights again.  Where the kernel for one offset takes
    the layer otherwise (up to 128 channels, in and out) the line lies at 1.2
    million rows x output channels, which is when there are more workgroups than
    the chip holds: us there and in pieces 128 -> 128 over 700 rows 14.3 / 4.5, 96
    -> 128 over 9 000 12.6 / 8.6, 80 -> 48 over 20 000 8.1 / 7.8, over 26 000 8.3 /
    9.1, 96 -> 64 over 30 000 8.9 / 11.9, 64 -> 32 over 60 000 7.7 / 11.1.  Against
    the library and an output pass of its own it lies at 200 million rows x input
    x output channels: 256 -> 32 over 700 22 / 4.8, 256 -> 128 over 4 500 21.5 / 12.7,
    160 -> 128 over 9 000 22 / 13.3."""
    if (dtype != torch.float32 or num_source_features % 16 != 0 or num_source_features < 48
            or not _C.implicit_forward_supported(num_source_features, num_target_features, dtype)):
        return -1
    most = 200_000_000 // (num_source_features * num_target_features)
    if num_source_features <= 128 and num_target_features <= 128:
        most = min(most, 1_200_000 // num_target_features)
    return most


def prefers_hits(num_offsets: int, num_source_features: int, num_target_features: int, dtype: torch.dtype,
                 num_rows: int, form: str = "plain") -> bool:
    """Whether ``dataflow="auto"`` takes the single-kernel form for an fp32 layer
    over ``num_rows`` source rows (``hits_rows_limit``, ``hits_rows_from``)."""
    layer = (num_offsets, num_source_features, num_target_features, dtype, form)
    return num_rows <= hits_rows_limit(*layer) or (
        hits_rows_from(*layer) <= num_rows <= implicit_rows_limit(num_source_features, dtype))


def cuda_time_gather(weights: torch.Tensor, source_masks: torch.Tensor,
                     target_masks: torch.Tensor, kernel_map_sizes: torch.Tensor,
                     tile_size: int, allow_shortcut_matmul: bool = False,
                     threshold: Optional[float] = 0) -> float:
    """Milliseconds of one Gather with ``tile_size`` feature elements per lane
    (reference: convolution.py:28-53)."""
    return _C.cuda_time_gather(tile_size, allow_shortcut_matmul, threshold, weights,
                               source_masks, target_masks, kernel_map_sizes)


def cuda_time_scatter(weights: torch.Tensor, source_masks: torch.Tensor,
                      target_masks: torch.Tensor, kernel_map_sizes: torch.Tensor,
                      tile_size: int, allow_shortcut_matmul: bool = False,
                      threshold: Optional[float] = 0) -> float:
    """Milliseconds of one Scatter (reference: convolution.py:56-81)."""
    return _C.cuda_time_scatter(tile_size, allow_shortcut_matmul, threshold, weights,
                                source_masks, target_masks, kernel_map_sizes)


def cuda_time_gemm(weights: torch.Tensor, source_masks: torch.Tensor,
                   target_masks: torch.Tensor, kernel_map_sizes: torch.Tensor,
                   allow_shortcut_matmul: bool = False, parallel: Optional[int] = None,
                   threshold: Optional[float] = 0) -> float:
    """Milliseconds of the grouped GEMM (reference: convolution.py:84-107)."""
    if parallel is None:
        parallel = GEMM_PARALLEL_LEVEL
    return _C.cuda_time_gemm(allow_shortcut_matmul, parallel, threshold, weights, source_masks,
                             target_masks, kernel_map_sizes)


def sparse_convolution_forward(sources: torch.Tensor, weights: torch.Tensor,
                               source_masks: Optional[torch.Tensor] = None,
                               target_masks: Optional[torch.Tensor] = None,
                               kernel_map_order: Optional[torch.Tensor] = None,
                               kernel_map_sizes: Optional[torch.Tensor] = None,
                               gather_tile_size: int = 0, scatter_tile_size: int = 0,
                               allow_shortcut_matmul: bool = False,
                               parallel: Optional[int] = None,
                               threshold: Optional[float] = 0,
                               epilogue: Optional[_C.Epilogue] = None,
                               dataflow: str = "auto",
                               packed_weights: Optional[torch.Tensor] = None,
                               kernel_map=None) -> torch.Tensor:
    """Output features ``[N_out, C_out]`` of one sparse convolution
    (reference: convolution.py:110-155).

    The kernel map comes either as the reference's four tensors
    (``source_masks``, ``target_masks``, ``kernel_map_order``,
    ``kernel_map_sizes``; a 4-tuple from ``KernelMapCache.get_kernel_map``
    unpacks into them) or as ``kernel_map=`` a :class:`~minuet_amd.nn.KernelMap`,
    which is what ``KernelMapCache.get_kernel_map`` returns.  With the four
    tensors alone the call behaves like the reference: Gather, grouped GEMM and
    Scatter as separate kernels, and the sizes are read back from the device
    once per call.  A ``KernelMap`` carries host copies of sizes and order, the
    pair lists and the dense map, with which nothing is read back, the Gather
    is folded into the GEMM's operand load and ``dataflow`` has a choice:

    ``"gather_gemm_scatter"`` is the reference's dataflow, ``"implicit"`` the
    single-kernel output-stationary form (needs ``kernel_map.dense`` and
    ``weights`` in their original offset order, as a layer holds them) and
    ``"auto"`` takes the implicit form where it is the faster one: 16-bit
    features whose rows it can stage, and fp32 layers that are narrow, small or, with
    few input channels, large.

    ``"list_driven"`` is Gather-GEMM-Scatter without the rank tables: the GEMM
    reads its rows through the pair list and writes its products in
    target-major order (``KernelMap.row_ptr`` / ``out_pos``, built on first use
    from the dense map), so that Scatter reads them as one stream.  Scatter
    gains what the GEMM's scattered row writes lose, so ``"auto"`` never picks
    it; a layer's autotuner times it beside the other two.  Padding threshold,
    gather tile and the centre-offset shortcut have no meaning there.

    ``epilogue`` (:class:`Epilogue`) is applied to each output row before it is
    rounded to the feature dtype.  ``packed_weights`` (``pack_weights(weights)``,
    kept by the caller while the weights are unchanged) spares the packing pass
    that otherwise starts every call; it needs a ``KernelMap`` when the map is
    reordered (the host copy of the order) and is ignored without."""
    if not sources.is_cuda:
        raise NotImplementedError
    if dataflow not in DATAFLOWS:
        raise ValueError(f"dataflow must be one of {DATAFLOWS}")
    if kernel_map is None and isinstance(source_masks, KernelMap):
        kernel_map, source_masks = source_masks, None
    host_sizes = host_order = gather_index = dense = None
    if kernel_map is not None:
        source_masks, target_masks, kernel_map_order, kernel_map_sizes = kernel_map
        host_sizes, host_order = kernel_map.sizes_host, kernel_map.order_host
        gather_index = kernel_map.in_idx if host_sizes is not None else None
        dense = kernel_map.dense
    if dataflow == "implicit" and dense is None:
        raise ValueError("the implicit dataflow needs a KernelMap with its dense map")
    if dense is not None and dataflow in ("auto", "implicit"):
        rows, shape = sources.shape[0], (weights.shape[0], weights.shape[1], weights.shape[2], weights.dtype)
        # (what a map says of the layer's stride; a dilation it does not)
        form = "plain" if rows == dense.shape[1] else "strided" if rows > dense.shape[1] else "transposed"
        if dataflow == "implicit" or (prefers_hits(*shape, rows, form)
                                      if weights.dtype == torch.float32 and weights.shape[0] > 1
                                      else prefers_implicit_over(*shape, rows, form)):
            return _C.sparse_convolution_forward_implicit(sources, weights, dense, epilogue=epilogue,
                                                          packed_weights=packed_weights)
    if dataflow == "list_driven":
        if kernel_map is None or gather_index is None or not kernel_map.ensure_row_lists():
            raise ValueError("the list-driven dataflow needs a KernelMap with its dense map and pair lists")
        # list-driven form: Gather folded into the GEMM, products written in
        # target-major order, Scatter streams through them (no rank table read)
        return _C.sparse_convolution_forward_rows(
            sources, weights, host_sizes, host_order, gather_index, kernel_map.out_pos, kernel_map.row_ptr,
            scatter_tile_size=scatter_tile_size, epilogue=epilogue, packed_weights=packed_weights)
    if source_masks is None or target_masks is None or kernel_map_sizes is None:
        raise ValueError("the Gather-GEMM-Scatter dataflow needs the rank tables and sizes of the kernel map")
    if parallel is None:
        parallel = GEMM_PARALLEL_LEVEL
    if gather_index is not None and (kernel_map_order is None or host_order is not None):
        # the map brings host sizes and pair lists: what depends on it alone is checked once per map
        return _C.sparse_convolution_forward_map(
            sources, weights, kernel_map, gather_tile_size, scatter_tile_size, allow_shortcut_matmul,
            parallel, threshold, epilogue=epilogue, packed_weights=packed_weights)
    if kernel_map_order is not None:
        if host_order is None:
            packed_weights = None
        kernel_map_order = kernel_map_order.contiguous()
    return _C.cuda_sparse_convolution_forward(
        gather_tile_size, scatter_tile_size, allow_shortcut_matmul, parallel, threshold,
        sources.contiguous(), weights.contiguous(), source_masks.contiguous(),
        target_masks.contiguous(), kernel_map_order, kernel_map_sizes.contiguous(),
        kernel_map_sizes_host=host_sizes, gather_index=gather_index, epilogue=epilogue,
        packed_weights=packed_weights, kernel_map_order_host=host_order)
