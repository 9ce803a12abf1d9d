"""Test/benchmark input generation from LiDAR scans (reference: sphconv/datagen.py)."""
import numpy as np
import torch

from . import _lib as L
from .utils import plain
from .vfe import SimpleVoxel
from .voxelize import VoxelGeneratorV3

# entries of an example that are joined along their first axis as they are (datagen.py:62-64)
_CONCATENATED = frozenset(("voxels", "voxel", "num_points", "num_gt", "voxel_labels", "gt_names", "gt_classes",
                           "gt_boxes"))
# range, field of view and limits of the spherical grid the reference voxelises its KITTI scans on
# (datagen.py:81-86): point range (x, y, z), (r, azimuth, polar angle) range in metres / degrees,
# points per voxel, voxel budget
_POINT_RANGE = (6, -40, -3, 70.4, 40, 1)
_SPHERE_RANGE = (6, -45, 87.5, 70.4, 45, 100)
_MAX_PARTS = 64                        # SPH_MAX_BATCH_PARTS of the header
_POINTS_PER_VOXEL, _MAX_VOXELS = 2, 24000


def merge_batch_torch(batch_list):
    """Joins per-scan examples into one batch (same keys and error as datagen.py:53-74): every known entry is
    concatenated along axis 0, and each scan's 'coordinates' first get a leading column holding the scan's
    position in the batch.  An entry under any other name raises ValueError("unidentified key", key)."""
    names = []
    for example in batch_list:
        names += [k for k in example if k not in names]
    merged = {}
    for name in names:
        parts = [example[name] for example in batch_list if name in example]
        if name == "coordinates" and len(parts) <= _MAX_PARTS and all(
                c.is_cuda and c.dtype == torch.int32 and c.dim() == 2 and c.shape[1] == 3 and c.is_contiguous()
                and c.device == parts[0].device and plain(c) for c in parts):
            merged[name] = L.host().batch_coordinates(parts)                               # one kernel
            continue
        if name == "coordinates":
            parts = [torch.cat([torch.full((c.shape[0], 1), b, dtype=c.dtype, device=c.device), c], dim=1)
                     for b, c in enumerate(parts)]
        elif name not in _CONCATENATED:
            raise ValueError("unidentified key", name)
        merged[name] = torch.cat(parts, dim=0)
    return merged


class VoxelizationVFE():
    """Voxelisation + mean VFE of one scan file (datagen.py:77-108), both on the GPU when a device is given."""

    def __init__(self, resolution_HWD=[512, 512, 64]):
        self.resolution_HWD = resolution_HWD
        self.vfe = SimpleVoxel(4)
        self.voxel_generator = VoxelGeneratorV3(None, list(_POINT_RANGE), list(_SPHERE_RANGE), _POINTS_PER_VOXEL,
                                                _MAX_VOXELS, resolution_HWD, coord_system="spherical")

    def generate(self, file: str, device=None):
        points = np.fromfile(file, dtype=np.float32, count=-1).reshape([-1, 4])
        if device is not None:
            points = torch.from_numpy(points).to(device)
        res = self.voxel_generator.generate(points)
        voxels = self.vfe(res['voxels'], res['num_points_per_voxel'], res['coordinates'])
        return voxels, res['coordinates']
