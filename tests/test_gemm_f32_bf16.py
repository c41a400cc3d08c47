"""f32 GEMM on the bf16 matrix instructions (gemm_f32.hip): launches of more workgroups of 64 x 64 tiles than CUs, with K shares of 512
elements and more.  Partial tiles and K tails, operands from the smallest f32 to the largest, infinities, and the error against float64."""
import numpy as np
import pytest

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host

pytestmark = pytest.mark.gpu
LAYOUTS = [(O.ROW, O.COL), (O.COL, O.ROW), (O.ROW, O.ROW), (O.COL, O.COL)]


def _flat(x, layout):
    return np.ascontiguousarray(x if layout == O.ROW else x.T).ravel()


def _run(A, B, la, lb, C=None, alpha=1.0, beta=0.0, ldl=O.ROW, workspace=0, splits=1):
    (m, k), n = A.shape, B.shape[1]
    d = device_filled(m * n, np.float32, 0xFF)
    c = None if C is None else to_device(_flat(C, ldl))
    ws = device_filled(workspace, np.uint8, 0xFF) if workspace else None
    g = R.gemm_args(R.F32, R.F32, m, n, k, to_device(_flat(A, la)), to_device(_flat(B, lb)), c, d, alpha, beta, la, lb, ldl, ldl, workspace=ws,
                    workspace_bytes=workspace)
    plan = R.gemm_launch_plan(g)
    assert (plan.macro_tile_m, plan.split_k) == (64, splits) and plan.grid_x * splits > R.device_info().compute_units
    R._check(R.lib().r355_gemm(R.ctypes.byref(g), None))
    got = to_host(d, np.float32)
    return got.reshape(m, n) if ldl == O.ROW else got.reshape(n, m).T


def _uniform(seed, *shape):
    return np.random.default_rng(seed).uniform(-1, 1, shape).astype(np.float32)


# (k + 4) u (|alpha| |A| |B| + |beta| |C|): the forward bound of any order of f32 sums; the norm: half of what such sums of 512 and more products
# show on uniform operands (4.0e-7), three times what these kernels do (0.8e-7)
@pytest.mark.parametrize("la,lb", LAYOUTS)
@pytest.mark.parametrize("ldl", [O.ROW, O.COL])
@pytest.mark.parametrize("m,n,k", [(1040, 1072, 516), (1104, 1008, 636), (1024, 1088, 544)])
def test_orientations_partial_tiles_and_k_tails(la, lb, ldl, m, n, k):
    A, B, C = _uniform(1, m, k), _uniform(2, k, n), _uniform(3, m, n)
    got = _run(A, B, la, lb, C, 2.0, -0.5, ldl).astype(np.float64)
    exact = 2.0 * (A.astype(np.float64) @ B) - 0.5 * C
    bound = (k + 4) * 2.0 ** -24 * (2.0 * (np.abs(A).astype(np.float64) @ np.abs(B)) + 0.5 * np.abs(C))
    assert np.all(np.abs(got - exact) <= bound)
    assert np.linalg.norm(got - exact) <= 2e-7 * np.linalg.norm(exact)


@pytest.mark.parametrize("la,lb", LAYOUTS)
def test_every_bit_of_an_operand(la, lb):
    # one product a row: every bit of the other operand, from the largest exponents to the smallest (every tile meets some of 2^112 and more,
    # so that all of it is the second pass, on the f32 instructions)
    m, n, k = 1056, 1056, 1056
    rng = np.random.default_rng(4)
    bits = rng.integers(0, 2 ** 32, (k, n), dtype=np.uint32)
    bits = np.where((bits >> 23 & 0xFF) == 0xFF, bits & 0x807FFFFF, bits)  # finite
    values = bits.view(np.float32)
    pick = np.zeros((m, k), np.float32)
    pick[np.arange(m), rng.permutation(k)[:m]] = 1.0
    want = values[pick.argmax(axis=1)]
    assert np.array_equal(_run(pick, values, la, lb), want)
    assert np.array_equal(_run(np.ascontiguousarray(values.T), np.ascontiguousarray(pick.T), la, lb), want.T)


@pytest.mark.parametrize("la,lb", LAYOUTS)
def test_every_bit_of_the_pieces(la, lb):
    # the same for all f32 below 2^95, the denormal ones among them: no piece and no sum (2^32 times the result) overflows, so that no tile is
    # multiplied again
    m, n, k = 1056, 1056, 1056
    rng = np.random.default_rng(14)
    values = (rng.integers(0, 222 << 23, (k, n), dtype=np.uint32) | rng.integers(0, 2, (k, n), dtype=np.uint32) << 31).view(np.float32)
    pick = np.zeros((m, k), np.float32)
    pick[np.arange(m), rng.permutation(k)[:m]] = 1.0
    want = values[pick.argmax(axis=1)]
    assert np.array_equal(_run(pick, values, la, lb), want)
    assert np.array_equal(_run(np.ascontiguousarray(values.T), np.ascontiguousarray(pick.T), la, lb), want.T)


@pytest.mark.parametrize("la,lb", LAYOUTS)
def test_tiny_values_take_no_second_pass(la, lb):
    # values below 2^-110 in every row and column, and operands of nothing else: the error is that of the bf16 instructions (0.7e-7 of the norm), not of a
    # second pass with the f32 ones (2.1e-7)
    m, n, k = 1040, 1056, 528
    A, B = _uniform(15, m, k), _uniform(16, k, n)
    A[np.arange(m), np.arange(m) % k] *= np.float32(2.0 ** -120)
    B[np.arange(n) % k, np.arange(n)] *= np.float32(2.0 ** -125)
    for scale in (0, -110):
        got = _run(np.ldexp(A, scale), np.ldexp(B, -scale - 20), la, lb).astype(np.float64)
        exact = np.ldexp(A, scale).astype(np.float64) @ np.ldexp(B, -scale - 20).astype(np.float64)
        assert np.linalg.norm(got - exact) <= 1.2e-7 * np.linalg.norm(exact)


@pytest.mark.parametrize("la,lb", [(O.ROW, O.COL), (O.COL, O.ROW)])
@pytest.mark.parametrize("count", [1, 2, 3, 4])
def test_few_products(la, lb, count):
    # 2^-24 of each product is left out at most, and the leading sums of all waves are rounded to the rest once.  One product: 2^-24 for that rounding and
    # 2^-29 for those of the rest, itself 2^-7 of the whole.  More: three additions of leading sums and one of the rest, and in the norm less than the
    # f32 instructions' sums of two products and more show on such operands (3.1e-8; these 2.6e-8 to 2.7e-8, 3.5e-8 with a rounding in every wave)
    m, n, k = 1056, 1072, 1052
    rng = np.random.default_rng(19)
    A, B = np.zeros((m, k), np.float32), rng.standard_normal((k, n)).astype(np.float32)
    for _ in range(count):
        A[np.arange(m), rng.integers(0, k, m)] = rng.standard_normal(m)
    got = _run(A, B, la, lb).astype(np.float64)
    exact, size = A.astype(np.float64) @ B, np.abs(A).astype(np.float64) @ np.abs(B)
    assert np.all(np.abs(got - exact) <= (2.0 ** -23 + 2.0 ** -29 if count == 1 else 5 * 2.0 ** -24) * size)
    assert np.linalg.norm(got - exact) <= 2.9e-8 * np.linalg.norm(exact)


def test_one_product_below_the_normal_numbers():
    # rounded to 2^-149 once: products of the pieces are not rounded there one by one
    m, n, k = 1040, 1040, 528
    A, B = np.zeros((m, k), np.float32), np.ldexp(_uniform(17, k, n), -70)
    A[np.arange(m), np.arange(m) % k] = np.ldexp(_uniform(18, m), -60)
    got = _run(A, B, O.ROW, O.COL).astype(np.float64)
    assert np.all(np.abs(got - A.astype(np.float64) @ B) <= 0.6 * 2.0 ** -149)


@pytest.mark.parametrize("ea,eb", [(-125, 100), (100, -125), (-60, -70), (55, 60)])
def test_operands_of_extreme_size(ea, eb):
    # results keep their precision where the operands' last pieces would lie below the range of bf16
    m, n, k = 1040, 1040, 528
    A, B = np.ldexp(_uniform(5, m, k), ea), np.ldexp(_uniform(6, k, n), eb)
    got = _run(A, B, O.ROW, O.COL).astype(np.float64)
    exact = A.astype(np.float64) @ B
    # (operands and results below 2^-126 are rounded to multiples of 2^-149)
    bound = (k + 4) * (2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B)) + 2.0 ** -149)
    assert np.all(np.abs(got - exact) <= bound)


@pytest.mark.parametrize("la,lb", [(O.ROW, O.COL), (O.COL, O.ROW)])
def test_infinities_and_nan(la, lb):
    m, n, k = 1040, 1072, 520
    A, B = _uniform(7, m, k), _uniform(8, k, n)
    A[3, 17], A[130, 519], B[200, 70], A[1039, 0] = np.inf, -np.inf, np.nan, 3e38
    B[17, 1000] = 0.0  # infinity times zero
    B[0, 5] = 3e38  # an overflow
    got = _run(A, B, la, lb)
    with np.errstate(all="ignore"):
        want = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(got[np.isinf(got)], want[np.isinf(want)])
    fin = np.isfinite(want)
    scale = np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64) @ np.abs(np.where(np.isfinite(B), B, 0))
    assert np.all(np.abs(got[fin].astype(np.float64) - want[fin]) <= ((k + 4) * 2.0 ** -24 * scale)[fin] + np.abs(want[fin]) * 2.0 ** -24)


def test_shares_of_k():
    # 16 x 17 tiles, three shares of 22 stages, the last of 21 and one 16-byte chunk
    m, n, k = 1024, 1040, 2084
    A, B, C = _uniform(9, m, k), _uniform(10, k, n), _uniform(11, m, n)
    need = int(R.gemm_query(R.gemm_args(R.F32, R.F32, m, n, k, 0x1000, 0x2000, 0x3000, 0x4000, 1.5, 1.0, O.ROW, O.COL, O.ROW, O.ROW,
                                        workspace_bytes=2 ** 62)).workspace_bytes)
    got = _run(A, B, O.ROW, O.COL, C, 1.5, 1.0, workspace=need, splits=3)
    exact = 1.5 * (A.astype(np.float64) @ B) + C
    assert np.linalg.norm(got - exact) <= 2e-7 * np.linalg.norm(exact)


@pytest.mark.parametrize("k", [484, 512])
def test_the_shortest_k(k):
    # sixteen stages of 128 bytes, the last of one 16-byte chunk or whole: four slices a wave
    m, n = 1040, 1072
    A, B = _uniform(20, m, k), _uniform(21, k, n)
    got = _run(A, B, O.ROW, O.ROW)
    exact = A.astype(np.float64) @ B
    assert np.linalg.norm(got - exact) <= 1.2e-7 * np.linalg.norm(exact)


def test_second_pass_in_one_share_of_k():
    # an overflow and an infinity that only the second of three shares meets: its tiles of that row and column are multiplied again, the other shares' are not
    m, n, k = 1024, 1040, 2084
    A, B, C = _uniform(22, m, k), _uniform(23, k, n), _uniform(24, m, n)
    A[100, 1000], B[900, 700] = np.float32(1e34), np.inf
    need = int(R.gemm_query(R.gemm_args(R.F32, R.F32, m, n, k, 0x1000, 0x2000, 0x3000, 0x4000, 1.5, 1.0, O.ROW, O.COL, O.ROW, O.ROW,
                                        workspace_bytes=2 ** 62)).workspace_bytes)
    got = _run(A, B, O.ROW, O.COL, C, 1.5, 1.0, workspace=need, splits=3).astype(np.float64)
    with np.errstate(all="ignore"):
        exact = 1.5 * (A.astype(np.float64) @ B.astype(np.float64)) + C
    assert np.array_equal(np.isinf(got), np.isinf(exact)) and np.array_equal(got[np.isinf(got)], exact[np.isinf(exact)]) and not np.isnan(got).any()
    fin = np.isfinite(exact)
    scale = 1.5 * np.abs(A).astype(np.float64) @ np.abs(np.where(np.isfinite(B), B, 0)) + np.abs(C)
    assert np.all(np.abs(got - exact)[fin] <= ((k + 8) * 2.0 ** -24 * scale)[fin])


@pytest.mark.parametrize("la,lb", [(O.ROW, O.COL), (O.COL, O.ROW)])
@pytest.mark.parametrize("ldl", [O.ROW, O.COL])
def test_result_in_the_place_of_c(la, lb, ldl):
    m, n, k = 1072, 1040, 636
    A, B, C = _uniform(25, m, k), _uniform(26, k, n), _uniform(27, m, n)
    A[77, 300] = np.inf  # (a row of tiles that is multiplied again adds C once as well)
    B[300, :] = np.abs(B[300, :]) + np.float32(0.5)
    d = to_device(_flat(C, ldl))
    R.gemm(R.F32, R.F32, m, n, k, to_device(_flat(A, la)), to_device(_flat(B, lb)), d, d, 2.0, -0.5, la, lb, ldl, ldl)
    got = to_host(d, np.float32)
    got = (got.reshape(m, n) if ldl == O.ROW else got.reshape(n, m).T).astype(np.float64)
    assert np.all(got[77] == np.inf)
    rows = np.arange(m) != 77
    exact = 2.0 * (A[rows].astype(np.float64) @ B) - 0.5 * C[rows]
    bound = (k + 4) * 2.0 ** -24 * (2.0 * (np.abs(A[rows]).astype(np.float64) @ np.abs(B)) + 0.5 * np.abs(C[rows]))
    assert np.all(np.abs(got[rows] - exact) <= bound)
