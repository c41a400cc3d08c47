"""GPU parity of the diagonal tiles of the DLRM forward on macro tiles, whose two operands are one image in LDS: every remainder of the
six-stage K loop and its main part, a partial last stage, one diagonal tile and several, whole and cut.  Integer-valued features, equal bit
for bit; the samples of a launch go round three."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host
from test_dlrm_tiles import _small_integers

pytestmark = pytest.mark.gpu

T64, T128 = R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 7, 8, 14, 15])
@pytest.mark.parametrize("dtype,m,batch,kernel", [(O.F16, 64, 1500, T64), (O.BF16, 176, 60, T64), (O.F32, 112, 85, T64), (O.F16, 112, 1200, T128),
                                                  (O.BF16, 240, 300, T128)])
def test_diagonal_tiles_at_every_stage_count(dtype, m, batch, kernel, stages):
    store, distinct = O.NP_STORAGE[dtype], 3
    k = stages * 128 // np.dtype(store).itemsize - 16
    assert R.dlrm_kernel(dtype, m, k, batch) == kernel
    x, stride = _small_integers(51 + stages, distinct * m * k, dtype), k + m * (m - 1) // 2
    want = O.dlrm_fwd(dtype, x, m, k, distinct).reshape(distinct, stride)
    turn = np.arange(batch) % distinct
    dout = device_filled(batch * stride + 8, store, 0xEE)
    R.dlrm_fwd(dtype, to_device(x.reshape(distinct, m * k)[turn]), dout, m, k, batch)
    out = to_host(dout, store)
    assert np.all(out[batch * stride:].view(np.uint8) == 0xEE)
    assert np.array_equal(out[:batch * stride].view(np.uint8), want[turn].ravel().view(np.uint8))
