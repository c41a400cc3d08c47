"""GPU parity of the col-major split GEMV where columns start off 128-byte boundaries: an XCD then takes a contiguous part of the
(block of rows, split) pairs.  Integer-valued operands: every sum is exact in any order, so y equals the product bit for bit.
Counts of workgroups off a multiple of the eight XCDs, a last block with few rows, every width of run, both element types, and
aligned columns beside them."""
import pytest
import torch

import rocwmma_amd as R


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,k,lda", [(6152, 5004, 6152), (1028, 8192, 1028), (260, 131072 + 4, 260), (68, 262144, 68), (132, 16384, 136), (2048, 8192, 2052),
                                     (2048, 8192, 2048), (4100, 8200, 4100)])
def test_split_sums_are_exact(dtype, m, k, lda):
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    a = torch.randint(-2, 3, (k, lda), device="cuda", generator=gen).to(dtype)
    x = torch.randint(-2, 3, (k,), device="cuda", generator=gen).to(dtype)
    need = R.gemv_workspace_bytes(R.COL_MAJOR, m, k, x.element_size())
    work = torch.full((need + 4096,), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.full((m + 16,), 7.0, device="cuda", dtype=dtype)
    call = R.gemv if dtype == torch.float32 else R.dgemv
    call(R.COL_MAJOR, m, k, a, x, None, y, lda=lda, workspace=work)
    want = (a[:, :m].double() * x.double()[:, None]).sum(dim=0)
    assert torch.equal(y[:m].double(), want) and bool((y[m:] == 7.0).all())
