"""GPU parity of the 64 x 64 macro tile (R355_KERNEL_TILED_64, and what R355_KERNEL_AUTO runs for few tiles) against the CPU
oracle: every type and orientation at tile edges, remainders of the six-stage loop and K tails.  Inputs are the reference's
integer pattern (test/device/common.hpp:203-220), for which any summation order gives the same bits, and random int8."""
import itertools

import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host
from test_gemm import _check, _inputs, _run
from test_gemm_splitk import _check_against_exact

pytestmark = pytest.mark.gpu

TYPE_PAIRS = [(O.F16, O.F16), (O.F16, O.F32), (O.BF16, O.BF16), (O.E4M3, O.F32), (O.I8, O.I32), (O.I8, O.I8), (O.F32, O.F32), (O.F64, O.F64)]
# (m, n, K stages of 128 bytes, 16-byte chunks of a last partial stage)
SHAPES = [(16, 16, 0, 1), (64, 64, 1, 0), (80, 48, 2, 3), (208, 144, 6, 0), (112, 272, 13, 7)]


@pytest.mark.parametrize("in_t,out_t", TYPE_PAIRS)
@pytest.mark.parametrize("la,lb", list(itertools.product([O.ROW, O.COL], repeat=2)))
@pytest.mark.parametrize("m,n,stages,chunks", SHAPES)
def test_tile_64_exact_inputs(in_t, out_t, la, lb, m, n, stages, chunks):
    k = (stages * 128 + chunks * 16) // np.dtype(O.NP_STORAGE[in_t]).itemsize
    ld = O.COL if m == 80 else O.ROW
    if in_t == O.I8:
        a, b, c = O.uniform_int8(1, m * k), O.uniform_int8(2, k * n), O.uniform_int8(3, m * n).astype(O.NP_STORAGE[out_t])
    else:
        a, b, c = O.fill_ref(in_t, m, k, la), O.fill_ref(in_t, k, n, lb), O.fill_ref(out_t, m, n, ld)
    for alpha, beta in ((1.0, 0.0), (2.0, -1.0)):
        cc = c if beta else None
        want = O.gemm(in_t, out_t, la, lb, ld, ld, m, n, k, a, b, cc, alpha, beta)
        got = _run(in_t, out_t, la, lb, ld, ld, m, n, k, a, b, cc, alpha, beta, R.KERNEL_TILED_64)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("in_t,out_t", [(O.F16, O.F32), (O.BF16, O.BF16), (O.E4M3, O.F32), (O.F32, O.F32)])
@pytest.mark.parametrize("la,lb", [(O.ROW, O.COL), (O.COL, O.ROW)])
def test_tile_64_random_inputs(in_t, out_t, la, lb):
    m, n, k = 144, 208, 336
    a, b, c = _inputs(in_t, out_t, m, n, k, seed=64)
    if in_t == O.F32:  # long sums in the operand type: the forward error bound of any summation order around the exact result
        got = _run(in_t, out_t, la, lb, O.ROW, O.ROW, m, n, k, a, b, c, 2.0, -1.0, R.KERNEL_TILED_64)
        _check_against_exact(in_t, m, n, k, la, lb, O.ROW, a, b, c, 2.0, -1.0, got)
        return
    want = O.gemm(in_t, out_t, la, lb, O.ROW, O.ROW, m, n, k, a, b, c, 2.0, -1.0)
    w32 = O.gemm(in_t, O.F32, la, lb, O.ROW, O.ROW, m, n, k, a, b, O.storage_to_f32(c, out_t), 2.0, -1.0) if out_t == O.BF16 else None
    _check(in_t, out_t, _run(in_t, out_t, la, lb, O.ROW, O.ROW, m, n, k, a, b, c, 2.0, -1.0, R.KERNEL_TILED_64), want, w32)


# ... and the tile's edge and the number of K splits that it runs on 256 CUs
@pytest.mark.parametrize("in_t,out_t,m,n,kbytes,edge,splits", [(O.F64, O.F64, 192, 160, 3200, 64, 3), (O.F32, O.F32, 720, 832, 3136, 64, 1),
                                                               (O.F16, O.F16, 64, 1024, 16384, 64, 16), (O.E4M3, O.F32, 96, 4912, 4400, 128, 4),
                                                               (O.I8, O.I32, 48, 2048, 5104, 64, 5)])
@pytest.mark.parametrize("la,lb", [(O.ROW, O.COL), (O.COL, O.ROW)])
def test_auto_with_a_workspace_whatever_tile_and_split_it_takes(in_t, out_t, m, n, kbytes, edge, splits, la, lb):
    k = kbytes // np.dtype(O.NP_STORAGE[in_t]).itemsize
    if in_t == O.I8:
        a, b, c = O.uniform_int8(4, m * k), O.uniform_int8(5, k * n), O.uniform_int8(6, m * n).astype(np.int32)
    else:
        a, b, c = O.fill_ref(in_t, m, k, la), O.fill_ref(in_t, k, n, lb), O.fill_ref(out_t, m, n, O.ROW)
    want = O.gemm(in_t, out_t, la, lb, O.ROW, O.ROW, m, n, k, a, b, c, 1.0, 1.0)
    da, db, dc, dd = to_device(a), to_device(b), to_device(c), device_filled(m * n, O.NP_STORAGE[out_t], 0xFF)
    args = (in_t, out_t, m, n, k, da, db, dc, dd, 1.0, 1.0, la, lb, O.ROW, O.ROW)
    need = int(R.gemm_query(R.gemm_args(*args, workspace_bytes=2 ** 62)).workspace_bytes)
    assert need > 0
    ws = device_filled(need + 4096, np.uint8, 0xFF)
    g = R.gemm_args(*args, workspace=ws, workspace_bytes=need)
    plan = R.gemm_launch_plan(g)
    assert (plan.macro_tile_m, plan.macro_tile_n, plan.split_k) == (edge, edge, splits)
    R._check(R.lib().r355_gemm(R.ctypes.byref(g), None))
    assert np.array_equal(to_host(dd, O.NP_STORAGE[out_t]), want)
    assert np.all(to_host(ws, np.uint8)[need:] == 0xFF)  # nothing behind the bytes that the plan reports
