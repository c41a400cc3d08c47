"""GPU parity of the DLRM forward's stores of whole rows left of the diagonal tile: ordinary ones where a launch's input and result take up to
14 MB, nontemporal ones beyond.  Integer-valued features, equal bit for bit; the samples of a launch go round three."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host
from test_dlrm_tiles import _small_integers

pytestmark = pytest.mark.gpu

T64, T128 = R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128
LIMIT = 14000000


def _forward(dtype, m, k, batch, launch):
    store, stride, distinct = O.NP_STORAGE[dtype], k + m * (m - 1) // 2, 3
    x = _small_integers(71 + m + k, distinct * m * k, dtype)
    want = O.dlrm_fwd(dtype, x, m, k, distinct).reshape(distinct, stride)
    turn = np.arange(batch) % distinct
    dout = device_filled(batch * stride + 8, store, 0xEE)
    launch(to_device(x.reshape(distinct, m * k)[turn]), dout)
    out = to_host(dout, store)
    assert np.all(out[batch * stride:].view(np.uint8) == 0xEE)
    assert np.array_equal(out[:batch * stride].view(np.uint8), want[turn].ravel().view(np.uint8))


# the last batch of ordinary stores and the first of nontemporal ones: a last tile of 16, 64 and 128 rows, tiles of 64 and of 128
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("dtype,m,k,kernel", [(O.F16, 320, 192, T64), (O.BF16, 272, 80, T64), (O.F16, 144, 48, T64), (O.BF16, 512, 112, T128), (O.F16, 784, 368, T128),
                                              (O.F32, 272, 80, T64), (O.F32, 192, 128, T64)])
def test_rows_on_both_sides_of_the_store_rule(dtype, m, k, kernel, over):
    batch = LIMIT // ((m * k + k + m * (m - 1) // 2) * np.dtype(O.NP_STORAGE[dtype]).itemsize) + over
    assert R.dlrm_kernel(dtype, m, k, batch) == kernel
    _forward(dtype, m, k, batch, lambda x, out: R.dlrm_fwd(dtype, x, out, m, k, batch))
