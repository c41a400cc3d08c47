"""GPU parity of the macro tiles of 224 and 192 rows, which R355_KERNEL_AUTO takes where they share the work out better, against
the 256 x 256 tile kernels that the other tests hold against the oracle: every element is the same sum in the same order, so the
bits are the same.  Shapes with partial tiles in both directions, K tails, every orientation and C."""
import itertools

import pytest
import torch

import oraclelib as O
import rocwmma_amd as R

TORCH = {O.F16: torch.float16, O.BF16: torch.bfloat16, O.F32: torch.float32, O.I8: torch.int8, O.I32: torch.int32}
# (m, n, K in bytes) in the kernel's view, and the rows of the tiles that it runs on 256 CUs.  The last stage of K is whole, one, three,
# four or seven chunks; 9 to 14 stages, every remainder of the six-stage loop; in the last four the last tile has 16 rows, in three of
# them 16 columns too
CASES = [(2832, 4624, 1200, 224), (2496, 4176, 1408, 192), (2464, 4880, 1776, 224), (4880, 4624, 1296, 192), (2704, 4512, 1040, 224),
         (4944, 2576, 1216, 224), (4240, 2576, 1136, 192), (2704, 3344, 1600, 192)]
PAIRS = [(O.F16, O.F16), (O.F16, O.F32), (O.BF16, O.BF16), (O.I8, O.I32), (O.I8, O.I8)]


@pytest.mark.gpu
@pytest.mark.parametrize("in_t,out_t", PAIRS)
@pytest.mark.parametrize("la,lb", list(itertools.product([O.ROW, O.COL], repeat=2)))
@pytest.mark.parametrize("m,n,kbytes,rows", CASES)
def test_same_bits_as_the_256_row_tile(in_t, out_t, la, lb, m, n, kbytes, rows):
    k, ld = kbytes // (1 if in_t == O.I8 else 2), O.COL if m == 2464 else O.ROW
    if ld == O.COL:
        m, n = n, m
    gen = torch.Generator(device="cuda").manual_seed(m + n)

    def make(count, dtype, t):
        if t in (O.I8, O.I32):
            return torch.randint(-128, 128, (count,), device="cuda", generator=gen, dtype=torch.int32).to(dtype)
        return (torch.rand(count, device="cuda", generator=gen) * 2 - 1).to(dtype)

    a, b = make(m * k, TORCH[in_t], in_t), make(k * n, TORCH[in_t], in_t)
    c = make(m * n, TORCH[out_t], out_t)
    for alpha, beta in ((1.0, 0.0), (2.0, -1.0)):
        got = [torch.full((m * n + 64,), 77, device="cuda", dtype=TORCH[out_t]) for _ in range(2)]
        for d, kernel, tile in zip(got, (R.KERNEL_AUTO, R.KERNEL_TILED), (rows, 256)):
            plan = R.gemm_launch_plan(R.gemm_args(in_t, out_t, m, n, k, a, b, c if beta else None, d, alpha, beta, la, lb, ld, ld, kernel=kernel))
            assert (plan.macro_tile_m, plan.macro_tile_n) == ((tile, 256) if ld == O.ROW else (256, tile))
            R.gemm(in_t, out_t, m, n, k, a, b, c if beta else None, d, alpha, beta, layout_a=la, layout_b=lb, layout_c=ld, layout_d=ld,
                   kernel=kernel)
        assert torch.equal(*got) and bool((got[0][m * n:] == 77).all())
