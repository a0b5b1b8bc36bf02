"""ResNet-style sparse classifier, the second network family of the
reference's end-to-end benchmarks (its README names ResNet and UNet; the model
definitions live outside the reference tree, README.md:6): a 3x3x3 stem,
stride-2 stages of two residual blocks each, global average pooling over every
point cloud and a linear head.  Assembled from the public modules of this
package; in evaluation mode the BatchNorm / ReLU / residual-sum layers ride the
convolutions' output pass."""
import torch
import torch.nn.modules.module as module_state
from torch import nn

from minuet_amd.nn import BatchNorm, GlobalAvgPool, ReLU, SparseConv3d
from minuet_amd.nn.functional import _C
from minuet_amd.nn.fused import FusedSequential
from minuet_amd.tensors import SparseTensor
from minuet_amd.unet import ResidualBlock

__all__ = ["SparseResNet"]


def _seen(module: nn.Module) -> bool:
    """Whether a call of this module is watched, or its forward replaced."""
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                or module._backward_pre_hooks or module_state._global_forward_hooks
                or module_state._global_forward_pre_hooks or module_state._global_backward_hooks
                or module_state._global_backward_pre_hooks or "forward" in module.__dict__)


def _classify(head: nn.Module, rows: torch.Tensor) -> torch.Tensor:
    """``head(rows)``, by a kernel of this library where ``head`` is a plain linear
    layer with few products and nothing but its value is asked for."""
    if type(head) is nn.Linear and rows.is_cuda and rows.dim() == 2:
        weight, bias = head.weight, head.bias
        if (weight.dtype == rows.dtype and weight.device == rows.device and rows.shape[1] == weight.shape[1]
                and rows.dtype in (torch.float32, torch.float16, torch.bfloat16)
                and 0 < rows.shape[0] * weight.numel() <= _C.MAX_LINEAR_PRODUCTS
                and (bias is None or (bias.dtype == rows.dtype and bias.device == rows.device))
                and not _seen(head) and not torch.is_autocast_enabled()
                and _C.plain((rows, weight) if bias is None else (rows, weight, bias))):
            return _C.linear(rows, weight, bias)
    return head(rows)


class SparseResNet(nn.Module):
    """``in_channels`` features per voxel -> ``num_classes`` logits per point cloud."""

    def __init__(self, in_channels: int = 4, num_classes: int = 10, stem: int = 32,
                 stages=(64, 128, 256), dtype=None, device=None):
        super().__init__()
        factory = {"dtype": dtype, "device": device}
        self.stem = FusedSequential(SparseConv3d(in_channels, stem, 3, **factory),
                                    BatchNorm(stem, **factory), ReLU(inplace=True))
        self.down = nn.ModuleList()
        self.stages = nn.ModuleList()
        width = stem
        for out in stages:
            self.down.append(FusedSequential(SparseConv3d(width, out, 2, stride=2, **factory),
                                             BatchNorm(out, **factory), ReLU(inplace=True)))
            self.stages.append(nn.Sequential(ResidualBlock(out, out, **factory),
                                             ResidualBlock(out, out, **factory)))
            width = out
        self.pool = GlobalAvgPool()
        self.head = nn.Linear(width, num_classes, **factory)

    def forward(self, x: SparseTensor) -> torch.Tensor:
        x = self.stem(x)
        for down, stage in zip(self.down, self.stages):
            x = stage(down(x))
        pooled = self.pool(x)
        if pooled.dim() == 1:                      # a single cloud without batch_dims
            pooled = pooled.unsqueeze(0)
        return _classify(self.head, pooled)
