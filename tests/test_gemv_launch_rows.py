"""How a GEMV's rows are dealt out (gemv_rows.hpp): no launch of 2^32 threads, which would run what is left modulo 2^32 and report success.  On the
host, and on the device at a row count that takes two launches."""
import ctypes
import os
import subprocess

import pytest
import torch

import rocwmma_amd as R

CSRC = os.path.join(os.path.dirname(os.path.abspath(R.__file__)), "csrc")
SOURCE = """
#include "gemv_rows.hpp"
extern "C" uint32_t launch_rows(int col, uint32_t m, uint64_t row, uint32_t es) { return r355::gemvLaunchRows(col, m, row, es); }
extern "C" void group(uint32_t m, uint64_t row, uint32_t es, uint32_t* out) { const auto g = r355::rowGroup(m, row, es); out[0] = g.waves, out[1] = g.rows; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("gemv_rows")
    (d / "rows.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "rows.so"), str(d / "rows.cpp")])
    so = ctypes.CDLL(str(d / "rows.so"))
    so.group.argtypes = [ctypes.c_uint32, ctypes.c_uint64, ctypes.c_uint32, ctypes.c_void_p]
    so.launch_rows.argtypes = [ctypes.c_int, ctypes.c_uint32, ctypes.c_uint64, ctypes.c_uint32]
    so.launch_rows.restype = ctypes.c_uint32
    return so


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("row", [16, 240, 256, 2048, 2064, 5632, 5648, 9344, 9360, 17168, 40000, 131056, 131072])
@pytest.mark.parametrize("m", [64, 8192, 2 ** 24 - 4, 2 ** 24, 2 ** 24 + 64, 2 ** 25, 2 ** 26 - 4096, 2 ** 26 + 64, 2 ** 28, 2 ** 29 + 4, 2 ** 32 - 4])
def test_threads_of_a_launch(lib, es, row, m):
    most = lib.launch_rows(0, m, row, es)
    assert 0 < most <= m and (most == m or most % 4096 == 0)
    for rows in {most, m - (m - 1) // most * most}:  # every launch but the last, and the last
        form = (ctypes.c_uint32 * 2)()
        lib.group(rows, row, es, form)
        waves, of = (4, 4) if row >= 131072 or form[0] == 0 else form  # (those of 128 KiB and more: a wave per row or sixteen for four)
        waves = 16 if row >= 131072 else waves
        assert -(-rows // of) * waves * 64 < 2 ** 32
    cols = lib.launch_rows(1, m, 16, es)
    assert 0 < cols <= m and (cols == m or cols % 4096 == 0) and -(-cols // (256 // es)) * 1024 < 2 ** 32
    # one launch where one suffices
    assert m > 2 ** 24 - 4096 or (most == m and cols == m)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [R.ROW_MAJOR, R.COL_MAJOR])
def test_more_rows_than_a_launch(layout):
    # f64 rows of 16 bytes: a wave each, so 2^26 rows are 2^32 threads; columns of 1 GiB: 2^27 rows of 32 threads
    m, k = (2 ** 26 + 64, 2) if layout == R.ROW_MAJOR else (2 ** 27 + 4160, 2)
    gen = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randint(-3, 4, (m, k) if layout == R.ROW_MAJOR else (k, m), device="cuda", generator=gen, dtype=torch.int8).to(torch.float64)
    x = torch.tensor([2.0, -1.0], dtype=torch.float64, device="cuda")
    y = torch.randint(-50, 51, (m,), device="cuda", generator=gen, dtype=torch.int8).to(torch.float64)
    out = torch.full((m + 16,), 7.0, dtype=torch.float64, device="cuda")
    R.dgemv(layout, m, k, a, x, y, out, 2.0, -1.0)
    cols = (a[:, 0], a[:, 1]) if layout == R.ROW_MAJOR else (a[0], a[1])
    assert torch.equal(out[:m], 2.0 * (2.0 * cols[0] - cols[1]) - y)
    assert bool((out[m:] == 7.0).all())
