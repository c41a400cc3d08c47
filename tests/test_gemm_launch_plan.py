"""r355_gemm_launch_plan: the tile, the grid and the K splits that a call runs, beside the nominal plan of r355_gemm_query.  On the
host (256 CUs where no device answers)."""
import pytest

import rocwmma_amd as R


def _args(in_t, out_t, m, n, k, ld=R.ROW_MAJOR, need=0, **kw):
    return R.gemm_args(in_t, out_t, m, n, k, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.ROW_MAJOR, R.COL_MAJOR, ld, ld,
                       workspace=0x4000 if need else None, workspace_bytes=need, **kw)


# (types, m, n, k) -> rows and columns of the tile, workgroups, shares of K with the workspace that the nominal plan asks for
@pytest.mark.parametrize("in_t,out_t,m,n,k,tile,grid,splits", [
    (R.F16, R.F16, 8192, 8192, 8192, (256, 256), 1024, 1),
    (R.BF16, R.BF16, 2832, 4624, 3080, (224, 256), 248, 1),
    (R.I8, R.I32, 5120, 5120, 5120, (224, 256), 464, 1),
    (R.F16, R.F32, 256, 256, 256, (64, 64), 16, 1),
    (R.E4M3, R.F32, 64, 8192, 8192, (128, 128), 64, 4),
    (R.F32, R.F32, 2560, 2560, 2560, (64, 64), 1600, 1),
    (R.F64, R.F64, 192, 160, 400, (64, 64), 16, 3),
    (R.F16, R.F16, 64, 1024, 8192, (64, 64), 16, 16),
])
def test_what_a_call_launches(in_t, out_t, m, n, k, tile, grid, splits):
    nominal = R.gemm_query(_args(in_t, out_t, m, n, k, need=2 ** 64 - 1))
    plan = R.gemm_launch_plan(_args(in_t, out_t, m, n, k, need=nominal.workspace_bytes))
    assert plan.kernel == nominal.kernel == R.KERNEL_TILED
    assert ((plan.macro_tile_m, plan.macro_tile_n), plan.grid_x, plan.grid_y, plan.split_k) == (tile, grid, splits, splits)
    assert plan.macro_tile_k == nominal.macro_tile_k and plan.lds_bytes <= 163840
    assert plan.split_k <= nominal.split_k and plan.workspace_bytes <= nominal.workspace_bytes
    assert (plan.workspace_bytes == 0) == (plan.split_k == 1)
    # without a workspace nothing is split; with a byte too little neither
    for need in (0, nominal.workspace_bytes - 1 if nominal.workspace_bytes else 0):
        plain = R.gemm_launch_plan(_args(in_t, out_t, m, n, k, need=need))
        assert plain.split_k == plain.grid_y == 1 and plain.workspace_bytes == 0
    # the transposed problem with a col-major D: rows and columns change places
    other = R.gemm_launch_plan(_args(in_t, out_t, n, m, k, ld=R.COL_MAJOR, need=nominal.workspace_bytes))
    assert ((other.macro_tile_n, other.macro_tile_m), other.grid_x, other.split_k) == (tile, grid, splits)


@pytest.mark.parametrize("kernel,tile,lds", [(R.KERNEL_TILED_64, 64, 40960), (R.KERNEL_TILED_128, 128, 81920), (R.KERNEL_TILED, 256, 131072),
                                             (R.KERNEL_TILED_DEEP, 256, 163840)])
def test_a_selector_is_what_runs(kernel, tile, lds):
    for query in (R.gemm_query, R.gemm_launch_plan):
        plan = query(_args(R.F16, R.F16, 2832, 4624, 3080, kernel=kernel))
        assert (plan.macro_tile_m, plan.macro_tile_n, plan.lds_bytes, plan.split_k) == (tile, tile, lds, 1)


def test_other_kernel_families():
    for query in (R.gemm_query, R.gemm_launch_plan):
        plan = query(_args(R.F64, R.F64, 64, 48, 80, lda=81, ldb=81))
        assert plan.kernel == R.KERNEL_SIMPLE and plan.split_k == 1
    sparse = R.gemm_args(R.I8, R.I32, 4096, 4096, 8192, 0x1000, 0x2000, None, 0x3000, 1.0, 0.0, R.ROW_MAJOR, R.COL_MAJOR, R.ROW_MAJOR,
                         R.ROW_MAJOR, a_meta=0x4000)
    nominal, plan = R.gemm_query(sparse), R.gemm_launch_plan(sparse)
    assert all(getattr(plan, f) == getattr(nominal, f) for f, _ in R.GemmPlan._fields_)
    with pytest.raises(R.R355Error):
        R.gemm_launch_plan(_args(R.F16, R.F16, 256, 256, 250))  # what r355_gemm refuses


# measured slower on the smaller tile (or with other splits) although the timing model prices that as a little faster
@pytest.mark.parametrize("in_t,out_t,m,n,k,tile,splits", [
    (R.BF16, R.BF16, 704, 976, 2176, (128, 128), 4),
    (R.F16, R.F16, 1120, 1856, 256, (128, 128), 1),
    (R.BF16, R.BF16, 1744, 1696, 256, (128, 128), 1),
    (R.F32, R.F32, 1792, 176, 2240, (64, 64), 5),
])
def test_a_lead_within_the_models_error_does_not_move_a_call(in_t, out_t, m, n, k, tile, splits):
    plan = R.gemm_launch_plan(_args(in_t, out_t, m, n, k, need=R.gemm_query(_args(in_t, out_t, m, n, k, need=2 ** 64 - 1)).workspace_bytes))
    assert ((plan.macro_tile_m, plan.macro_tile_n), plan.split_k) == (tile, splits)


# f32 on 64 x 64 tiles: four waves with 16 KiB each on the bf16 instructions (more workgroups than CUs, K of 16 stages of 128 bytes, shares of 22), five
# buffers of 8 KiB on the f32 ones
@pytest.mark.parametrize("m,n,k,splits,lds", [(2560, 2560, 2560, 1, 65536), (1040, 1072, 484, 1, 65536), (1040, 1072, 480, 1, 40960), (1024, 1024, 2560, 1, 40960),
                                              (1024, 1040, 2084, 3, 65536), (560, 160, 7924, 8, 40960)])
def test_lds_of_f32_tiles(m, n, k, splits, lds):
    need = R.gemm_query(_args(R.F32, R.F32, m, n, k, need=2 ** 64 - 1)).workspace_bytes if splits > 1 else 0
    plan = R.gemm_launch_plan(_args(R.F32, R.F32, m, n, k, need=need))
    assert (plan.macro_tile_m, plan.split_k, plan.lds_bytes) == (64, splits, lds)
    if splits == 1:
        for query in (R.gemm_query, R.gemm_launch_plan):
            assert query(_args(R.F32, R.F32, m, n, k, kernel=R.KERNEL_TILED_64)).lds_bytes == lds
