"""Voxel feature encoders of the data path (reference: sphconv/vfe.py)."""
import torch
from torch import nn

from . import _lib as L
from .utils import plain


class SimpleVoxel(nn.Module):
    """Mean of the points of a voxel (vfe.py:210-228)."""

    def __init__(self, num_input_features=4, use_norm=True, num_filters=(32, 128), with_distance=False,
                 voxel_size=(0.2, 0.2, 4), pc_range=(0, -40, -3, 70.4, 40, 1), name="VoxelFeatureExtractor"):
        super().__init__()
        self.name = name
        self.num_input_features = num_input_features

    def forward(self, features, num_voxels, coors):
        if (features.is_cuda and features.dtype == torch.float32 and num_voxels.dtype == torch.int32 and features.dim() == 3
                and num_voxels.shape == features.shape[:1] and not features.requires_grad and features.is_contiguous()
                and num_voxels.is_contiguous() and num_voxels.device == features.device
                and 0 < self.num_input_features <= features.shape[2] and features.shape[1] > 0 and plain(features) and plain(num_voxels)):
            return L.host().voxel_mean(features, num_voxels, self.num_input_features)      # one kernel
        # features [voxels, max_points, >=num_input_features], unused slots are zero
        points_mean = features[:, :, :self.num_input_features].sum(dim=1, keepdim=False) \
            / num_voxels.type_as(features).view(-1, 1)
        return points_mean.contiguous()
