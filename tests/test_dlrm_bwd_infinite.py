"""GPU parity of the DLRM backward for infinite features: S X with S zero on its diagonal only, so that an infinity in row j makes row j NaN and
every other row infinite (or NaN, where its own element of S is zero), whichever tile the row lies in and whichever kernel runs.  Integer-valued
features beside the infinities, equal value for value, NaN for NaN."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host
from test_dlrm_tiles import _small_integers

pytestmark = pytest.mark.gpu

WAVE, BLOCKED, T64, T128 = R.DLRM_KERNEL_BLOCK_PER_WAVE, R.DLRM_KERNEL_REGISTER_BLOCKED, R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


# a diagonal tile alone, cut by the last feature, among others; two diagonal stages a tile; the kernels without tiles
@pytest.mark.parametrize("dtype,m,k,batch,kernel", [(d, *c) for d in (O.F16, O.BF16) for c in ((64, 16, 700, T64), (80, 80, 41, T64), (144, 448, 17, T64),
                                                                                               (336, 48, 20, T64), (784, 400, 100, T128), (32, 176, 5, WAVE),
                                                                                               (80, 208, 1000, BLOCKED))]
                         + [(O.F32, 144, 448, 17, T64), (O.F32, 896, 384, 75, T128)])
def test_an_infinite_feature_makes_its_own_row_nan_and_the_others_infinite(dtype, m, k, batch, kernel):
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True) == kernel
    store, stride, distinct = O.NP_STORAGE[dtype], k + m * (m - 1) // 2, 2
    x, up = _small_integers(61 + m, distinct * m * k, dtype).reshape(distinct, m, k), _small_integers(62 + m, distinct * stride, dtype)
    inf, minus = O.f32_to_storage(np.array([np.inf, -np.inf], np.float32), dtype)
    # one to a column: the first and last row, rows around the tiles' edges and across their middle (of the last column: two of opposite sign)
    for col, row in enumerate(sorted({0, 5, 31, min(40, m - 1), min(63, m - 1), min(64, m - 1), m // 2, m - 9, m - 1})):
        x[0, row, col] = inf if col % 2 else minus
    x[1, 3, k - 1], x[1, m - 2, k - 1] = inf, minus
    _, want = O.dlrm_bwd(dtype, x.ravel(), up, m, k, distinct)
    turn = np.arange(batch) % distinct
    dmlp, dgrad = device_filled(batch * k, store, 0xEE), device_filled(batch * m * k, store, 0xEE)
    R.dlrm_bwd(dtype, to_device(x.reshape(distinct, m * k)[turn]), to_device(up.reshape(distinct, stride)[turn]), dmlp, dgrad, m, k, batch)
    got, want = to_host(dgrad, store), want.ravel()
    if dtype != O.F32:
        got, want = O.storage_to_f32(got, dtype), O.storage_to_f32(want, dtype)
    want = want.reshape(distinct, m * k)
    assert np.isinf(want).any() and np.isnan(want).any() and np.isfinite(want).any()
    assert np.array_equal(got.reshape(batch, m * k), want[turn], equal_nan=True)
