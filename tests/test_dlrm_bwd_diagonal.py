"""GPU parity of the diagonal tile of the DLRM backward on macro tiles, 16-bit types: its rows of the packed triangle are read in 16-byte
pieces that reach back over a row's start, for the first rows of a sample into the bottom-MLP gradient before the triangle.  Those elements
are NaN here: one that stays in a product shows in the whole row of the gradient.  Integer-valued features, equal bit for bit."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host
from test_dlrm_tiles import _small_integers

pytestmark = pytest.mark.gpu

T64, T128 = R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


# one tile whole and cut, two with the second cut after 16, several; the least width; two diagonal stages a tile
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch,kernel", [(64, 16, 700, T64), (80, 80, 41, T64), (112, 48, 600, T64), (144, 448, 17, T64), (784, 400, 100, T128)])
def test_pieces_cut_by_the_diagonal_hold_nothing_from_before_the_triangle(dtype, m, k, batch, kernel):
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True) == kernel
    store, stride, distinct = O.NP_STORAGE[dtype], k + m * (m - 1) // 2, 2
    x, up = _small_integers(41 + m, distinct * m * k, dtype), _small_integers(42 + m, distinct * stride, dtype)
    _, want = O.dlrm_bwd(dtype, x, up, m, k, distinct)
    poisoned = up.reshape(distinct, stride).copy()
    poisoned[:, :k] = O.f32_to_storage(np.full(1, np.nan, np.float32), dtype)[0]
    turn = np.arange(batch) % distinct
    dmlp, dgrad = device_filled(batch * k, store, 0xEE), device_filled(batch * m * k, store, 0xEE)
    R.dlrm_bwd(dtype, to_device(x.reshape(distinct, m * k)[turn]), to_device(poisoned[turn]), dmlp, dgrad, m, k, batch)
    got = O.storage_to_f32(to_host(dgrad, store), dtype).reshape(batch, m * k)
    assert np.array_equal(got, O.storage_to_f32(want.ravel(), dtype).reshape(distinct, m * k)[turn])
    assert np.array_equal(to_host(dmlp, store).reshape(batch, k).view(np.uint8), poisoned[turn][:, :k].copy().view(np.uint8))
