"""GPU parity of the DLRM backward on 64 x 64 tiles, 16-bit types, around the rule that gives a launch the kernel for one workgroup a CU: 6 tiles of
features and more, and no more workgroups than CUs.  Integer-valued features, equal bit for bit."""
import pytest

import oraclelib as O
import rocwmma_amd as R
from test_dlrm_bwd_diagonal import test_pieces_cut_by_the_diagonal_hold_nothing_from_before_the_triangle as _before_the_triangle_poisoned
from test_dlrm_tiles import _backward_of_repeated_samples

pytestmark = pytest.mark.gpu

T64 = R.DLRM_KERNEL_TILED_64


# a last tile of 16, 32 and 64 rows and columns; as many workgroups as CUs (256) and more; the last shape without the kernel and the first with it
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(320, 64, 4), (336, 16, 1), (336, 64, 42), (336, 64, 43), (384, 48, 4), (480, 80, 2), (512, 64, 32), (512, 64, 33), (784, 400, 2),
                                       (1024, 64, 3), (1200, 240, 1)])
def test_backward_around_one_workgroup_a_cu(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T64)


@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(336, 16, 3), (512, 80, 5), (1024, 48, 4)])
def test_pieces_cut_by_the_diagonal(dtype, m, k, batch):
    _before_the_triangle_poisoned(dtype, m, k, batch, T64)
