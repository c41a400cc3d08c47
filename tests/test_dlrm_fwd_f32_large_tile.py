"""GPU parity of the DLRM forward's f32 kernel on 128 x 128 tiles, which the entry point runs for 370704 features and more only (results of 256 GiB)
and which is called here by itself.  Integer-valued features, equal bit for bit."""
import ctypes

import pytest

import oraclelib as O
import rocwmma_amd as R
from test_dlrm_fwd_rows import LIMIT, _forward

pytestmark = pytest.mark.gpu


# a tile cut by the last feature, one and several; stage counts around the six-stage loop and a partial last stage; 3 samples (ordinary stores) and
# enough for nontemporal ones
@pytest.mark.parametrize("over", [False, True])
@pytest.mark.parametrize("m,k", [(16, 16), (96, 48), (128, 208), (144, 32), (272, 240), (400, 464)])
def test_f32_on_the_large_tile(m, k, over):
    batch = 1 + LIMIT // ((m * k + k + m * (m - 1) // 2) * 4) if over else 3
    tiled = R.lib()["_ZN4r35512dlrmFwdTiledEiPKvPvjjjjP12ihipStream_t"]  # r355::dlrmFwdTiled(dtype, in, out, m, k, batch, tile, stream)
    u32, ptr = ctypes.c_uint32, ctypes.c_void_p
    tiled.argtypes, tiled.restype = [ctypes.c_int32, ptr, ptr, u32, u32, u32, u32, ptr], ctypes.c_int

    def launch(x, out):
        assert tiled(R.F32, R._ptr(x), R._ptr(out), m, k, batch, 128, None) == 0

    _forward(O.F32, m, k, batch, launch)
