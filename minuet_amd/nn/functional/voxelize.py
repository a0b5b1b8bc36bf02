"""Input preparation next to the convolution path: points -> voxels, and a
batch of clouds -> one SparseTensor (the step before the first layer)."""
from typing import Optional, Sequence

import torch

from minuet_amd.utils.helpers import as_tuple
from . import _C
from .hash import unique_coordinates

__all__ = ["voxelize", "collate"]


def voxelize(coordinates: torch.Tensor, voxel_size=1, dtype: torch.dtype = torch.int32,
             return_reverse_indices: bool = False):
    """Voxel coordinates ``floor(p / voxel_size)`` of the points ``p``, sorted and
    without duplicates; with ``return_reverse_indices`` also the row of the
    result each input point fell into.

    Same interface as the reference's ``voxelize`` (voxelize.py:11-35), which
    cannot run as written: it builds the voxel-size tensor on
    ``device=coordinates.dtype`` and hands unsorted rows to
    ``unique_coordinates``, which only merges neighbouring duplicates.  Here
    the rows are sorted first, so every voxel appears once."""
    if not coordinates.is_cuda:
        raise NotImplementedError
    ndim = coordinates.shape[1]
    if (coordinates.dtype in (torch.float32, torch.float64) and dtype in (torch.int32, torch.int64)
            and coordinates.shape[0] > 0 and 1 <= ndim <= 4):
        unique, reverse = _C.voxelize(coordinates.contiguous(), as_tuple(voxel_size, size=ndim, name="voxel_size"),
                                      dtype, return_reverse_indices)
        return (unique, reverse) if return_reverse_indices else unique
    size = torch.tensor(as_tuple(voxel_size, size=ndim, name="voxel_size"), dtype=coordinates.dtype,
                        device=coordinates.device)
    voxels = torch.floor(coordinates / size).to(dtype).contiguous()
    order, ordered = _C.sort_coordinates(voxels)
    unique, index = unique_coordinates(ordered)
    if not return_reverse_indices:
        return unique
    # index[i] = number of runs of equal rows that end before ordered row i,
    # which is the row of the result that ordered row i is written to
    reverse = torch.empty(voxels.shape[0], dtype=torch.int64, device=voxels.device)
    reverse[order.long()] = index[:-1].long()
    return unique, reverse


def _one_call(coordinates: Sequence[torch.Tensor], features: Optional[Sequence[torch.Tensor]]) -> bool:
    """Whether ``_C.collate`` takes these clouds: what it leaves out beside the
    general way's tensor expressions is nothing that anybody sees."""
    first = coordinates[0]
    if (len(coordinates) > _C.MAX_GATHER_SOURCES or not isinstance(first, torch.Tensor) or not first.is_cuda
            or first.dtype not in (torch.int32, torch.int64) or first.dim() != 2 or not 1 <= first.shape[1] <= 4
            or not _C.plain(coordinates)):
        return False
    device, dtype, ndim, total = first.device, first.dtype, first.shape[1], 0
    for c in coordinates:
        if (c.dtype != dtype or c.device != device or c.dim() != 2 or c.shape[1] != ndim or not c.is_contiguous()):
            return False
        total += c.shape[0]
    if not 0 < total <= 0x7FFFFFFF:
        return False
    if features is None:
        return True
    first = features[0]
    if (not isinstance(first, torch.Tensor) or first.dim() != 2 or first.shape[1] == 0
            or first.element_size() not in (2, 4, 8) or not _C.plain(features)
            or total * first.shape[1] * first.element_size() > _C.MAX_GATHER_BYTES):
        return False
    dtype, channels = first.dtype, first.shape[1]
    for f, c in zip(features, coordinates):
        if (f.dtype != dtype or f.device != device or f.dim() != 2 or f.shape[1] != channels
                or f.shape[0] != c.shape[0] or not f.is_contiguous()):
            return False
    return True


def collate(coordinates: Sequence[torch.Tensor], features: Optional[Sequence[torch.Tensor]] = None):
    """One batch from several clouds of voxel coordinates (each free of
    duplicates, in any order): ``(coordinates, batch_dims)`` with every cloud
    sorted inside its ``[batch_dims[g], batch_dims[g + 1])`` range, the layout
    ``SparseTensor`` and the batched kernels expect (tensors.py:38-95); with
    ``features`` also the feature rows in the same order."""
    if len(coordinates) == 0:
        raise ValueError("collate needs at least one cloud")
    if features is not None and len(features) != len(coordinates):
        raise ValueError("features and coordinates must list the same clouds")
    if _one_call(coordinates, features):
        ordered, batch_dims, rows = _C.collate(coordinates, features)
        return (ordered, batch_dims) if features is None else (ordered, batch_dims, rows)
    stacked = torch.cat(list(coordinates), dim=0).contiguous()
    if not stacked.is_cuda:
        raise NotImplementedError
    ends = [0]
    for cloud in coordinates:
        ends.append(ends[-1] + int(cloud.shape[0]))
    batch_dims = _C.upload_ints(ends, stacked.dtype, stacked.device)
    order, ordered = _C.sort_coordinates(stacked, batch_dims)
    if features is None:
        return ordered, batch_dims
    first = features[0]
    if (len(features) <= _C.MAX_GATHER_SOURCES and first.element_size() in (2, 4, 8) and _C.plain(features)
            and all(f.dim() == 2 and f.is_contiguous() and f.dtype == first.dtype and f.shape[1] == first.shape[1]
                    and f.device == stacked.device and f.shape[0] == c.shape[0]
                    for f, c in zip(features, coordinates)) and first.shape[1] > 0
            and ends[-1] * first.shape[1] * first.element_size() <= _C.MAX_GATHER_BYTES):
        return ordered, batch_dims, _C.gather_rows(features, order)
    return ordered, batch_dims, torch.cat(list(features), dim=0)[order.long()]
