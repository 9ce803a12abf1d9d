"""z_idx and the rows' columns of init_tensor, which come by rows or by columns (csrc/coo.hip, coo_by_columns): either side of
the line, columns of one and of several words, full ones, and a last workgroup that is not full."""
import pytest
import torch

from sphconv_amd import sphconv_cuda as ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,shape,n", [(1, (16, 64, 64), 255), (1, (16, 64, 64), 256), (2, (3, 5, 64), 1920), (3, (7, 11, 40), 300),
                                           (1, (9, 31, 130), 208), (1, (9, 31, 130), 210), (1, (5, 7, 200), 7000), (4, (64, 300, 65), 200000)])
def test_columns(batch, shape, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    lin = torch.randperm(batch * shape[0] * shape[1] * shape[2], generator=g, device="cuda")[:n]
    col, z = lin // shape[2], lin % shape[2]
    idx = torch.stack([col // (shape[0] * shape[1]), col // shape[1] % shape[0], col % shape[1], z], 1).int().contiguous()
    feat = torch.randn((n, 8), generator=g, device="cuda")
    out, z_idx, z_ptr, perm, cols = ext._init_tensor(feat, idx, batch, shape)
    order = lin.argsort()
    assert torch.equal(z_idx, z[order].int()) and torch.equal(cols, col[order].int()) and torch.equal(out, feat[order])
    assert torch.equal(perm.long()[order], torch.arange(n, device="cuda"))
    assert torch.equal(z_ptr.view(-1).long(), torch.bincount(col, minlength=z_ptr.numel()).cumsum(0))
