"""GPU parity of the DLRM backward where a workgroup takes two or three 64 x 64 tiles of a row of tiles (16-bit types, launches of more than three
tiles a CU): whole and partial last groups, groups that reach past the last column, a last tile of 16, 32, 48 and 64 columns, the fewest K stages and
many.  Integer-valued features, equal bit for bit; the samples of a launch go round three."""
import pytest

import oraclelib as O
import rocwmma_amd as R
from test_dlrm_bwd_diagonal import test_pieces_cut_by_the_diagonal_hold_nothing_from_before_the_triangle as _before_the_triangle_poisoned
from test_dlrm_tiles import _backward_of_repeated_samples

pytestmark = pytest.mark.gpu

T64 = R.DLRM_KERNEL_TILED_64


# the last launch with one tile a workgroup and the first with two; then, on 256 CUs, two tiles of rows of 2, 4, 8, 13, 7, 2 and 4, and three of rows of 3, 6, 9, 11 and 15
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(80, 80, 192), (80, 80, 193), (80, 128, 280), (128, 208, 180), (688, 480, 16), (112, 800, 54), (336, 400, 30),
                                       (336, 80, 90), (208, 256, 64), (320, 192, 96), (144, 176, 120), (128, 336, 110), (112, 576, 60), (1008, 688, 11), (688, 960, 9)])
def test_backward_with_several_tiles_a_workgroup(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T64)


@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(80, 80, 193), (320, 176, 96), (848, 496, 11)])
def test_pieces_cut_by_the_diagonal(dtype, m, k, batch):
    _before_the_triangle_poisoned(dtype, m, k, batch, T64)
