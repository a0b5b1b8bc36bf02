"""Global pooling over each point cloud of a SparseTensor (mirrors
minuet/nn/functional/pooling.py).  Sums and means of all clouds are one library
call that reads the batch boundaries on the device; where gradients or tangents
are recorded, and for maxima, they are plain tensor reductions."""
import torch

from . import _C

__all__ = ["global_avg_pool", "global_max_pool", "global_sum_pool"]


def _per_cloud(x, reduce):
    if x.batch_dims is None:
        return reduce(x.F)
    bounds = x.batch_dims.tolist()
    return torch.stack([reduce(x.F[bounds[k]:bounds[k + 1]]) for k in range(x.batch_size)], dim=0)


def _native(x) -> bool:
    f, dims = x.F, x.batch_dims
    return (f.is_cuda and f.dim() == 2 and 0 < f.shape[1] <= _C.MAX_POOL_CHANNELS and f.shape[0] < 1 << 31
            and f.dtype in (torch.float32, torch.float16, torch.bfloat16) and f.is_contiguous()
            and (dims is None or (dims.device == f.device and dims.dtype in (torch.int32, torch.int64)
                                  and dims.is_contiguous() and dims.shape[0] - 1 <= _C.MAX_POOL_CLOUDS))
            and _C.plain((f,) if dims is None else (f, dims)))


def global_avg_pool(x):
    """Mean feature of every point cloud, stacked in batch order."""
    if _native(x):
        return _C.global_pool(x.F, x.batch_dims, True)
    return _per_cloud(x, lambda f: torch.mean(f, dim=0))


def global_sum_pool(x):
    """Feature sum of every point cloud, stacked in batch order."""
    if _native(x):
        return _C.global_pool(x.F, x.batch_dims, False)
    return _per_cloud(x, lambda f: torch.sum(f, dim=0))


def global_max_pool(x):
    """Channel-wise maximum of every point cloud, stacked in batch order."""
    return _per_cloud(x, lambda f: torch.max(f, dim=0)[0])
