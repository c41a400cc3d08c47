"""Which kernel the DLRM entry points run for a shape (r355_dlrm_kernel), on the host (256 CUs where no device answers): what was measured
to be the faster one, and what is refused."""
import pytest

import rocwmma_amd as R

WAVE, BLOCKED, T64, T128 = R.DLRM_KERNEL_BLOCK_PER_WAVE, R.DLRM_KERNEL_REGISTER_BLOCKED, R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


# few features or a short K, where a macro tile is mostly padding: 1.3 to 7 times as long on tiles
@pytest.mark.parametrize("dtype,m,k,batch", [(R.BF16, 32, 48, 4704), (R.F16, 32, 16, 7000), (R.F16, 48, 16, 6200), (R.BF16, 32, 208, 4), (R.F16, 80, 16, 1800),
                                             (R.BF16, 80, 32, 4300), (R.F16, 112, 16, 900), (R.F32, 32, 16, 2400), (R.F16, 64, 96, 20)])
def test_forward_with_a_block_per_wave(dtype, m, k, batch):
    assert R.dlrm_kernel(dtype, m, k, batch) == WAVE


# a tile of 128 for samples of up to 64 features is three quarters padding and more: twice as long
@pytest.mark.parametrize("dtype", [R.F16, R.BF16, R.F32])
@pytest.mark.parametrize("m,k,batch", [(64, 112, 5000), (64, 64, 5742), (64, 288, 2602), (48, 96, 2969), (48, 1024, 1763), (176, 576, 428), (320, 192, 96)])
def test_forward_on_small_tiles(dtype, m, k, batch):
    assert R.dlrm_kernel(dtype, m, k, batch) == T64


@pytest.mark.parametrize("dtype", [R.F16, R.BF16])
@pytest.mark.parametrize("m,k,batch", [(1024, 1024, 64), (272, 1024, 128), (256, 112, 756), (96, 576, 1116), (128, 128, 2000)])
def test_forward_on_large_tiles(dtype, m, k, batch):
    assert R.dlrm_kernel(dtype, m, k, batch) == T128


# rows that a tile of 64 mostly pads, in launches of many blocks: 1.2 to 2.4 times as long on tiles
@pytest.mark.parametrize("dtype,m,k,batch", [(R.F16, 32, 208, 4021), (R.F16, 32, 656, 1963), (R.BF16, 32, 240, 4006), (R.F32, 32, 160, 3593), (R.F16, 80, 208, 1410),
                                             (R.F16, 48, 576, 2298), (R.F16, 96, 704, 585), (R.F32, 80, 208, 1012), (R.BF16, 48, 752, 783)])
def test_backward_register_blocked(dtype, m, k, batch):
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True) == BLOCKED


@pytest.mark.parametrize("dtype", [R.F16, R.BF16, R.F32])
@pytest.mark.parametrize("m,k,batch,kernel", [(112, 48, 847, T64), (320, 192, 96, T64), (1024, 256, 4, T64), (784, 16, 100, T64), (1024, 1024, 64, T128),
                                              (32, 16, 100, WAVE)])
def test_backward_on_tiles_and_with_a_block_per_wave(dtype, m, k, batch, kernel):
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True) == kernel


def test_alignment_specialised_shapes_and_refusals():
    assert R.dlrm_kernel(R.F16, 112, 48, 847, backward=True, aligned16=False) == BLOCKED
    assert R.dlrm_kernel(R.F16, 112, 48, 8, backward=True, aligned16=False) == WAVE
    for backward in (False, True):
        assert R.dlrm_kernel(R.F16, 27, 128, 65536, backward=backward) == R.DLRM_KERNEL_SPECIALISED
        assert R.dlrm_kernel(R.F16, 16, 80, 100, backward=backward) == WAVE
        for dtype, m, k, batch in ((R.F16, 33, 128, 4), (R.F16, 48, 40, 4), (R.F64, 48, 48, 4), (R.F16, 1, 64, 4), (R.F16, 48, 48, 0)):
            with pytest.raises(R.R355Error):
                R.dlrm_kernel(dtype, m, k, batch, backward=backward)
