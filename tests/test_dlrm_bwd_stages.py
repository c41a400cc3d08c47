"""GPU parity of the DLRM backward on macro tiles at every small number of K stages and with a partial last one (features beyond a multiple of 64;
f32: 32): a stage is requested while the one before it is multiplied or waits in registers.  Integer-valued features, equal bit for bit;
the samples of a launch go round three."""
import pytest

import oraclelib as O
import rocwmma_amd as R
from test_dlrm_tiles import _backward_of_repeated_samples

pytestmark = pytest.mark.gpu

T64, T128 = R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(64, 16, 700), (80, 80, 41), (128, 80, 60), (144, 80, 60), (192, 80, 60), (208, 48, 60), (256, 48, 40), (320, 192, 20),
                                       (336, 48, 20)])
def test_backward_at_every_stage_count(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T64)


@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(784, 400, 100), (1024, 1024, 64), (912, 528, 60)])
def test_backward_on_the_large_tile(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T128, distinct=2)
