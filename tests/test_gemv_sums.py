"""The col-major GEMV's sums (gemv.hip): the same bits wherever A lies in memory, but for its place in a cache line, and their error against float64."""
import pytest
import torch

import rocwmma_amd as R

pytestmark = pytest.mark.gpu


def _product(dtype, m, k, flat, x, offered):
    out = torch.full((m,), 7.0, dtype=dtype, device="cuda")
    ws = torch.empty(offered, dtype=torch.uint8, device="cuda") if offered else None
    (R.gemv if dtype == torch.float32 else R.dgemv)(R.COL_MAJOR, m, k, flat, x, None, out, 1.0, 0.0, workspace=ws, workspace_bytes=offered)
    return out


# columns a multiple of 128 bytes apart: on the plain launch, on the one for idle CUs, and split
@pytest.mark.parametrize("dtype,m,k", [(torch.float32, 8192, 1000), (torch.float32, 2048, 2048), (torch.float32, 864, 13476), (torch.float32, 8416, 8192),
                                       (torch.float64, 4096, 1000), (torch.float64, 1840, 2868)])
def test_bits_depend_on_the_start_in_a_line_alone(dtype, m, k):
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    values = torch.rand(m * k, device="cuda", generator=gen, dtype=dtype) - 0.5
    x = torch.rand(k, device="cuda", generator=gen, dtype=dtype) - 0.5
    room, piece = torch.empty(m * k + 64, device="cuda", dtype=dtype), 16 // dtype.itemsize
    exact = x.double() @ values.view(k, m).double()
    for offered in {0, R.gemv_workspace_bytes(R.COL_MAJOR, m, k, dtype.itemsize)}:
        for shifts in ((0, 8, 16), (1, 3, 9)):  # of 16 bytes: on a line of 128 bytes, inside one
            results = []
            for shift in shifts:
                at = shift * piece
                room[at:at + m * k] = values
                results.append(_product(dtype, m, k, room[at:at + m * k], x, offered))
            assert all(torch.equal(r, results[0]) for r in results)
            # (twice the forward bound of any order of k products: of these and, f64, of the reference)
            assert bool(((results[0].double() - exact).abs() <= (k + 4) * torch.finfo(dtype).eps * (x.double().abs() @ values.view(k, m).double().abs())).all())


# the norm of the error of sums in three levels, 1.2e-7 here; the same columns in one chain a lane have 3.2e-7, in sixteen waves of 32 to 128 columns each 1.6e-7
@pytest.mark.parametrize("m,k", [(6152, 11012), (2048, 2048)])
def test_error_of_the_sums(m, k):
    gen = torch.Generator(device="cuda").manual_seed(5)
    a = torch.rand(k, m, device="cuda", generator=gen) * 2 - 1
    x = torch.rand(k, device="cuda", generator=gen) * 2 - 1
    exact = x.double() @ a.double()
    for offered in {0, R.gemv_workspace_bytes(R.COL_MAJOR, m, k, 4)}:
        got = _product(torch.float32, m, k, a.view(-1), x, offered)
        assert float((got.double() - exact).norm() / exact.norm()) <= 1.45e-7
