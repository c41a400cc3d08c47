"""Row-major GEMV: every choice of waves and rows per workgroup (rowGroup in gemv.hip), rows that end anywhere in a workgroup's slices and row
counts off the rows of a workgroup.  Small integers, so that every sum is exact in any order."""
import pytest
import torch

import rocwmma_amd as R

pytestmark = pytest.mark.gpu
# (m, bytes of a row): four rows a wave; a wave per row; one, two, four, eight waves a row; two rows on four and on eight waves
SHAPES = [(16386, 272), (16388, 2048), (1003 * 4, 1024), (300, 1040), (516, 5632), (20, 5648), (700, 9344), (12, 9360), (260, 30000), (8, 70000), (40, 131056),
          (4004, 20016), (2052, 16400), (9000, 20000), (20004, 16384)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,row", SHAPES)
@pytest.mark.parametrize("pad", [0, 4])
def test_rows_and_waves(dtype, m, row, pad):
    m, k = m // 4 * 4, row // dtype.itemsize // 4 * 4
    lda = k + pad
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    a = torch.randint(-3, 4, (m, lda), device="cuda", generator=gen).to(dtype)
    x = torch.randint(-3, 4, (k,), device="cuda", generator=gen).to(dtype)
    y = torch.randint(-50, 51, (m,), device="cuda", generator=gen).to(dtype)
    want = 2.0 * (a[:, :k].double() * x.double()).sum(dim=1) - y.double()
    out = torch.full((m + 16,), 7.0, dtype=dtype, device="cuda")
    (R.gemv if dtype == torch.float32 else R.dgemv)(R.ROW_MAJOR, m, k, a, x, y, out, 2.0, -1.0, lda=lda)
    assert torch.equal(out[:m].double(), want)
    assert bool((out[m:] == 7.0).all())
