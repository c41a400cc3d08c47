"""Problems at the edge of 32-bit counts: a K of 2^32 bytes and more, more tiles than a launch's threads can be counted for."""
import os
import subprocess
import sys

import pytest
import torch

import oraclelib as O
import rocwmma_amd as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TORCH = {O.F16: torch.float16, O.BF16: torch.bfloat16, O.E4M3: torch.float8_e4m3fn, O.I8: torch.int8, O.I32: torch.int32,
         O.F32: torch.float32, O.F64: torch.float64}


def _query(in_t, out_t, m, n, k, **kw):
    return R.gemm_query(R.gemm_args(in_t, out_t, m, n, k, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.COL_MAJOR, R.ROW_MAJOR, R.ROW_MAJOR,
                                    R.ROW_MAJOR, **kw))


# k times the element size: 2^32, a little more, and (8-bit) 2^32 only once rounded up to whole stages
LONG_K = [(O.F16, O.F32, 2 ** 31 + 64), (O.F16, O.F16, 2 ** 31), (O.F32, O.F32, 2 ** 30), (O.F64, O.F64, 2 ** 29), (O.E4M3, O.F32, 2 ** 32 - 16),
          (O.I8, O.I32, 2 ** 32 - 16)]


@pytest.mark.parametrize("in_t,out_t,k", LONG_K)
def test_a_k_beyond_32_bits_of_bytes_is_planned_by_its_length(in_t, out_t, k):
    assert _query(in_t, out_t, 16, 16, k, workspace_bytes=2 ** 64 - 1).split_k == 32  # the most shares there are


@pytest.mark.parametrize("in_t,out_t,k", LONG_K)
def test_a_k_beyond_32_bits_of_bytes_reaches_the_launch(in_t, out_t, k):
    """On a host without a device the call comes back; it used to divide by a number of stages of zero."""
    child = """
import sys; sys.path.insert(0, %r)
import rocwmma_amd as R
try:
    R.device_info()
except R.R355Error:
    g = R.gemm_args(%d, %d, 16, 16, %d, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.COL_MAJOR, R.ROW_MAJOR, R.ROW_MAJOR, R.ROW_MAJOR)
    print("status", R.lib().r355_gemm(R.ctypes.byref(g), None))
""" % (ROOT, in_t, out_t, k)
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")  # (no device: nothing is launched on these addresses)
    r = subprocess.run([sys.executable, "-c", child], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "status" in r.stdout, (r.returncode, r.stdout, r.stderr)


@pytest.mark.gpu
@pytest.mark.parametrize("in_t,out_t,k", LONG_K)
def test_a_k_beyond_32_bits_of_bytes_is_summed_to_its_end(in_t, out_t, k):
    """A and B are zero but for a few k-rows of small integers, before and behind where 32-bit byte counts wrap (two operands of 64 GiB)."""
    es = torch.empty(0, dtype=TORCH[in_t]).element_size()
    rows = [0, 1, 128 // es - 1, 128 // es, k // 2 + 5, k - 128 // es - 1, k - 1]
    torch.cuda.empty_cache()
    raw = {1: torch.int8, 2: torch.int16, 4: torch.int32, 8: torch.int64}[es]
    a, b = (torch.zeros((k, 16), dtype=raw, device="cuda") for _ in range(2))
    gen = torch.Generator(device="cuda").manual_seed(3)
    want = torch.zeros((16, 16), dtype=torch.float64, device="cuda")
    for r in rows:
        va, vb = (torch.randint(-3, 4, (16,), device="cuda", generator=gen).float() for _ in range(2))
        a[r], b[r] = va.to(TORCH[in_t]).view(raw), vb.to(TORCH[in_t]).view(raw)
        want += torch.outer(va, vb).double()
    d = torch.full((16, 16), 77, dtype=TORCH[out_t], device="cuda")
    need = _query(in_t, out_t, 16, 16, k, workspace_bytes=2 ** 64 - 1).workspace_bytes
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    R.gemm(in_t, out_t, 16, 16, k, a, b, None, d, layout_a=R.COL_MAJOR, layout_b=R.ROW_MAJOR, workspace=ws)
    assert torch.equal(d.double(), want)
    del a, b
    torch.cuda.empty_cache()


# one tile more than 2^24: with 256 threads each, 256 threads more than 32 bits count
MANY_TILES = [(R.KERNEL_TILED_64, 64), (R.KERNEL_AUTO, 64), (R.KERNEL_TILED_128, 128), (R.KERNEL_AUTO, 128)]


@pytest.mark.parametrize("kernel,edge", MANY_TILES)
def test_a_launch_holds_threads_that_32_bits_count(kernel, edge):
    plan = R.gemm_query(R.gemm_args(R.F16, R.F16, 16, edge * (2 ** 24 + 1), 8, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.ROW_MAJOR,
                                    R.COL_MAJOR, R.COL_MAJOR, R.COL_MAJOR, kernel=kernel))
    assert plan.kernel == R.KERNEL_TILED and 0 < plan.grid_x * plan.block_x < 2 ** 32
    # the widest problem there is: its tiles are not counted from a rounded-up n that wraps to zero
    plan = R.gemm_query(R.gemm_args(R.F16, R.F16, 16, 2 ** 32 - 16, 8, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.ROW_MAJOR,
                                    R.COL_MAJOR, R.COL_MAJOR, R.COL_MAJOR, kernel=kernel))
    assert 0 < plan.grid_x * plan.block_x < 2 ** 32


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,edge", MANY_TILES)
def test_more_tiles_than_a_launch_holds(kernel, edge):
    """The columns of B repeat 24929 tiles' worth, so each of the 673 repetitions has to give the same bits (edge 64: 17 and 34 GB)."""
    part, copies = edge * 97 * 257, 673  # 97 * 257 * 673 = 2^24 + 1
    torch.cuda.empty_cache()
    gen = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randint(-3, 4, (16, 8), device="cuda", generator=gen).half()
    b = torch.randint(-3, 4, (part, 8), device="cuda", generator=gen).half()  # col-major 8 x part
    want = (b.float() @ a.float().t().contiguous()).half()  # col-major 16 x part; sums of 8 products of up to 9: exact
    b = b.repeat(copies, 1)
    d = torch.full((copies, part, 16), 77, dtype=torch.float16, device="cuda")
    R.gemm(R.F16, R.F16, 16, part * copies, 8, a, b, None, d, layout_a=R.ROW_MAJOR, layout_b=R.COL_MAJOR, layout_c=R.COL_MAJOR,
           layout_d=R.COL_MAJOR, kernel=kernel)
    assert all(torch.equal(d[i], want) for i in range(copies))
    del b, d
    torch.cuda.empty_cache()
