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
    _check(batch, shape, n, torch.randperm(batch * shape[0] * shape[1] * shape[2], generator=g, device="cuda")[:n])


@pytest.mark.parametrize("batch,shape,n", [(1, (64, 1024, 40), 65535), (1, (64, 1024, 40), 65536), (3, (31, 700, 64), 65537),
                                           (1, (64, 140, 250), 71680), (1, (64, 140, 250), 71681), (2, (64, 512, 256), 65536),
                                           (2, (64, 513, 256), 65537), (1, (64, 300, 257), 90000)])
@pytest.mark.parametrize("order", ["random", "sorted", "azimuth", "mostly sorted"])
def test_orders(batch, shape, n, order):
    """Rows in the columns' order, in another one, and in none, on grids on either side of the line."""
    g = torch.Generator(device="cuda").manual_seed(n)
    lin = torch.randperm(batch * shape[0] * shape[1] * shape[2], generator=g, device="cuda")[:n]
    if order == "azimuth":
        col = lin // shape[2]
        lin = lin[(col % shape[1] * shape[0] + col // shape[1]).argsort(stable=True)]
    elif order != "random":
        lin = lin.sort()[0]
    if order == "mostly sorted":                       # one workgroup of rows that the mark kernel looks at, one that it passes over
        lin = torch.cat([lin[:2048], lin[2048:2304].flip(0), lin[2304:2560], lin[2560:2816].flip(0), lin[2816:]])
    _check(batch, shape, n, lin)


def test_orders_with_rows_outside_and_rows_of_one_cell():
    """What the status reports, and the columns of what lies inside, as for short grids."""
    g = torch.Generator(device="cuda").manual_seed(1)
    shape, n = (64, 1024, 40), 70000
    lin = torch.randperm(shape[0] * shape[1] * shape[2], generator=g, device="cuda")[:n]
    col = lin // shape[2]
    idx = torch.stack([torch.zeros_like(col), col // shape[1], col % shape[1], lin % shape[2]], 1).int().contiguous()
    for bad in ([0, 64, 0, 0], [0, 0, 0, -1], idx[5].tolist()):
        wrong = idx.clone()
        wrong[40000] = torch.tensor(bad, dtype=torch.int32, device="cuda")
        with pytest.raises(ValueError):
            ext.init_tensor(torch.zeros((n, 4), device="cuda"), wrong, 1, shape)


def _check(batch, shape, n, lin):
    g = torch.Generator(device="cuda").manual_seed(n + 1)
    col, z = lin // shape[2], lin % shape[2]
    idx = torch.stack([col // (shape[0] * shape[1]), col // shape[1] % shape[0], col % shape[1], z], 1).int().contiguous()
    feat = torch.randn((n, 8), generator=g, device="cuda")
    out, z_idx, z_ptr, perm, cols = ext._init_tensor(feat, idx, batch, shape)
    order = lin.argsort()
    assert torch.equal(z_idx, z[order].int()) and torch.equal(cols, col[order].int()) and torch.equal(out, feat[order])
    assert torch.equal(perm.long()[order], torch.arange(n, device="cuda"))
    assert torch.equal(z_ptr.view(-1).long(), torch.bincount(col, minlength=z_ptr.numel()).cumsum(0))
