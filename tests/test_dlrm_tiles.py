"""GPU parity of the DLRM dot interaction on macro tiles (more than 16 features, or an embedding width without a specialised
kernel) against the CPU oracle.  Integer-valued features: every f32 sum is exact in any order, so results are equal bit for bit
after the one rounding to the result type."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host

pytestmark = pytest.mark.gpu


def _small_integers(seed, n, dtype):
    x = np.round(O.uniform_pm1(seed, n) * 2.0).astype(np.float32)
    return x if dtype == O.F32 else O.f32_to_storage(x, dtype)


# (features, width, batch): partial tiles of 64 and 128, one and several tiles, K tails and stage counts around the six-stage
# loop, batches that leave XCDs unevenly loaded; the last two are large enough for the 128 x 128 tile of the 16-bit types
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(32, 176, 5), (48, 272, 3), (64, 16, 1500), (80, 336, 9), (128, 384, 2), (144, 448, 17), (272, 96, 33), (272, 512, 86),
                                       (144, 1040, 81)])
def test_forward_on_macro_tiles(dtype, m, k, batch):
    store, stride = O.NP_STORAGE[dtype], k + m * (m - 1) // 2
    x = _small_integers(11 + m, batch * m * k, dtype)
    dout = device_filled(batch * stride + 8, store, 0xEE)
    R.dlrm_fwd(dtype, to_device(x), dout, m, k, batch)
    out = to_host(dout, store)
    assert np.all(out[batch * stride:].view(np.uint8) == 0xEE)  # nothing behind the last row
    assert np.array_equal(out[:batch * stride].view(np.uint8), O.dlrm_fwd(dtype, x, m, k, batch).ravel().view(np.uint8))
