"""Global pooling over each point cloud of a SparseTensor (mirrors
minuet/nn/functional/pooling.py).  Sums and means of all clouds are one library
call that reads the batch boundaries on the device; where gradients are
recorded, and for maxima, they are plain tensor reductions."""
import torch

from . import _C

__all__ = ["global_avg_pool", "global_max_pool", "global_sum_pool"]


def _per_cloud(x, reduce):
    if x.batch_dims is None:
        return reduce(x.F)
    bounds = x.batch_dims.tolist()
    return torch.stack([reduce(x.F[bounds[k]:bounds[k + 1]]) for k in range(x.batch_size)], dim=0)


def _native(x) -> bool:
    f = x.F
    return (f.is_cuda and f.dim() == 2 and f.shape[1] > 0 and f.is_contiguous()
            and f.dtype in (torch.float32, torch.float16, torch.bfloat16)
            and not (f.requires_grad and torch.is_grad_enabled())
            and (x.batch_dims is None or (x.batch_dims.is_contiguous()
                                          and x.batch_dims.dtype in (torch.int32, torch.int64))))


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
