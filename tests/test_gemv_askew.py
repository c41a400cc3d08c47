"""Col-major GEMV of matrices whose columns do not start on 128-byte boundaries (gemv.hip, BY_XCD): every length of run, with and without splits
of K, the last block of rows and the last split of any size.  Small integers, so that every sum is exact in any order."""
import pytest
import torch

import rocwmma_amd as R

pytestmark = pytest.mark.gpu
# runs of 64 bytes, 128, 256, 512 and 1 KiB; a single block; fewer columns than one trip of a workgroup; as many splits as the workspace holds
SHAPES = [(276, 460), (1164, 940), (332, 8924), (4, 4), (20, 300), (1104, 3772), (6044, 1548), (772, 15588), (8264, 2024), (14156, 1528), (4652, 10860),
          (11928, 5812), (5516, 6256), (6152, 11012), (11596, 6676), (260, 16388), (16388, 4)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,k", SHAPES)
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 0), (0, 4)])
def test_columns_off_cache_lines(dtype, m, k, pad, shift):
    es, lda = dtype.itemsize, m + pad
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    flat = torch.randint(-3, 4, (lda * k + shift,), device="cuda", generator=gen).to(dtype)
    a = flat[shift:]  # (shift: 16 or 32 bytes past an allocation's boundary)
    x = torch.randint(-3, 4, (k,), device="cuda", generator=gen).to(dtype)
    y = torch.randint(-50, 51, (m,), device="cuda", generator=gen).to(dtype)
    want = 2.0 * (a.view(k, lda)[:, :m].double() * x.double()[:, None]).sum(dim=0) - y.double()
    need = R.gemv_workspace_bytes(R.COL_MAJOR, m, k, es)
    call = R.gemv if dtype == torch.float32 else R.dgemv
    for offered in {0, need, need // 2}:
        out = torch.full((m + 16,), 7.0, dtype=dtype, device="cuda")
        ws = torch.full((offered + 64,), 0x5A, dtype=torch.uint8, device="cuda")
        call(R.COL_MAJOR, m, k, a, x, y, out, 2.0, -1.0, lda=lda, workspace=ws, workspace_bytes=offered)
        assert torch.equal(out[:m].double(), want), offered
        assert bool((out[m:] == 7.0).all()) and bool((ws[offered:] == 0x5A).all())
