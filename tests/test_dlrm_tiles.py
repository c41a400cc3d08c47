"""GPU parity of the DLRM dot interaction on macro tiles (more than 16 features, or an embedding width without a specialised
kernel) against the CPU oracle.  Integer-valued features: every f32 sum is exact in any order, so results are equal bit for bit
after the one rounding to the result type."""
import numpy as np
import pytest
import torch

import oraclelib as O
import rocwmma_amd as R
from gpuutil import device_filled, to_device, to_host

pytestmark = pytest.mark.gpu


def _small_integers(seed, n, dtype):
    x = np.round(O.uniform_pm1(seed, n) * 2.0).astype(np.float32)
    return x if dtype == O.F32 else O.f32_to_storage(x, dtype)


# The kernels of 256 CUs (tests/test_dlrm_kernel_choice.py holds the choice itself)
WAVE, BLOCKED, T64, T128 = R.DLRM_KERNEL_BLOCK_PER_WAVE, R.DLRM_KERNEL_REGISTER_BLOCKED, R.DLRM_KERNEL_TILED_64, R.DLRM_KERNEL_TILED_128


# (features, width, batch): partial tiles of 64, one and several tiles, K tails and stage counts around the six-stage loop, batches that leave
# XCDs unevenly loaded.  f32 runs 64 x 64 tiles throughout, the 16-bit types a block per wave in three of them and 64 x 64 tiles else
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(32, 176, 5), (48, 272, 3), (64, 16, 1500), (80, 336, 9), (128, 384, 2), (144, 448, 17), (272, 96, 33), (272, 512, 86),
                                       (144, 1040, 81)])
def test_forward_on_macro_tiles(dtype, m, k, batch):
    waves = dtype != O.F32 and (m, k) in ((32, 176), (48, 272), (64, 16))
    assert R.dlrm_kernel(dtype, m, k, batch) == (WAVE if waves else T64)
    _forward(dtype, m, k, batch)


def _forward(dtype, m, k, batch):
    store, stride = O.NP_STORAGE[dtype], k + m * (m - 1) // 2
    x = _small_integers(11 + m, batch * m * k, dtype)
    dout = device_filled(batch * stride + 8, store, 0xEE)
    R.dlrm_fwd(dtype, to_device(x), dout, m, k, batch)
    out = to_host(dout, store)
    assert np.all(out[batch * stride:].view(np.uint8) == 0xEE)  # nothing behind the last row
    assert np.array_equal(out[:batch * stride].view(np.uint8), O.dlrm_fwd(dtype, x, m, k, batch).ravel().view(np.uint8))


# the 128 x 128 tile of the 16-bit types: whole and partial last tiles, a single tile a sample, one K stage and several
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("m,k,batch", [(256, 80, 110), (80, 96, 410), (208, 80, 95), (352, 208, 36), (336, 16, 45), (496, 64, 30), (1008, 32, 8)])
def test_forward_on_the_large_tile(dtype, m, k, batch):
    assert R.dlrm_kernel(dtype, m, k, batch) == T128
    _forward(dtype, m, k, batch)


# small launches, and those around the shapes above, on whatever they run
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(256, 80, 52), (256, 80, 51), (352, 208, 26), (496, 64, 16), (1008, 32, 5), (48, 400, 6), (64, 64, 300), (48, 64, 100)])
def test_forward_on_other_shapes(dtype, m, k, batch):
    _forward(dtype, m, k, batch)


# backward: one tile and several, so that stages left of, in and right of the diagonal tile all occur, partial tiles and K stages,
# widths off the tile's edge, samples spread unevenly over the XCDs; the first three (f32: two) run a block per wave, the others 64 x 64 tiles
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(16, 80, 9), (32, 176, 5), (48, 272, 3), (64, 16, 700), (80, 80, 41), (128, 384, 2), (144, 448, 17), (272, 96, 33),
                                       (336, 272, 40), (400, 144, 3), (528, 272, 24), (48, 400, 60), (112, 48, 600)])
def test_backward_on_macro_tiles(dtype, m, k, batch):
    waves = (m, k) in ((16, 80), (32, 176)) or (dtype != O.F32 and (m, k) == (48, 272))
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True) == (WAVE if waves else T64)
    store, stride = O.NP_STORAGE[dtype], k + m * (m - 1) // 2
    x, up = _small_integers(21 + m, batch * m * k, dtype), _small_integers(22 + m, batch * stride, dtype)
    dmlp, dgrad = device_filled(batch * k + 8, store, 0xEE), device_filled(batch * m * k + 8, store, 0xEE)
    R.dlrm_bwd(dtype, to_device(x), to_device(up), dmlp, dgrad, m, k, batch)
    mlp, grad = to_host(dmlp, store), to_host(dgrad, store)
    assert np.all(mlp[batch * k:].view(np.uint8) == 0xEE) and np.all(grad[batch * m * k:].view(np.uint8) == 0xEE)
    want_mlp, want_grad = O.dlrm_bwd(dtype, x, up, m, k, batch)
    assert np.array_equal(mlp[:batch * k].view(np.uint8), want_mlp.ravel().view(np.uint8))
    g, w = grad[:batch * m * k], want_grad.ravel()  # (values: -0.0 and +0.0 are the same gradient)
    if dtype != O.F32:
        g, w = O.storage_to_f32(g, dtype), O.storage_to_f32(w, dtype)
    assert np.array_equal(g, w)


def _backward_of_repeated_samples(dtype, m, k, batch, kernel, off=0, distinct=3):
    """A batch that goes round `distinct` samples, so that the oracle has only those to do; every sample of the batch against its own.
    off: upstream and mlp_grad start that many elements behind a 16-byte boundary."""
    assert R.dlrm_kernel(dtype, m, k, batch, backward=True, aligned16=off == 0) == kernel
    store, stride = O.NP_STORAGE[dtype], k + m * (m - 1) // 2
    es = np.dtype(store).itemsize
    x, up = _small_integers(31 + m, distinct * m * k, dtype), _small_integers(32 + m, distinct * stride, dtype)
    want_mlp, want_grad = O.dlrm_bwd(dtype, x, up, m, k, distinct)
    turn = np.arange(batch) % distinct
    held = to_device(np.concatenate([np.zeros(off, store), up.reshape(distinct, stride)[turn].ravel()]))
    dmlp, dgrad = device_filled(off + batch * k + 8, store, 0xEE), device_filled(batch * m * k + 8, store, 0xEE)
    R.dlrm_bwd(dtype, to_device(x.reshape(distinct, m * k)[turn]), held.data_ptr() + off * es, dmlp.data_ptr() + off * es, dgrad, m, k, batch)
    mlp, grad = to_host(dmlp, store), to_host(dgrad, store)
    assert np.all(mlp[:off].view(np.uint8) == 0xEE) and np.all(mlp[off + batch * k:].view(np.uint8) == 0xEE)
    assert np.all(grad[batch * m * k:].view(np.uint8) == 0xEE)
    assert np.array_equal(mlp[off:off + batch * k].reshape(batch, k).view(np.uint8), want_mlp.reshape(distinct, k)[turn].view(np.uint8))
    g, w = grad[:batch * m * k], want_grad.ravel()  # (values: -0.0 and +0.0 are the same gradient)
    if dtype != O.F32:
        g, w = O.storage_to_f32(g, dtype), O.storage_to_f32(w, dtype)
    assert np.array_equal(g.reshape(batch, m * k), w.reshape(distinct, m * k)[turn])


# the 128 x 128 tile of the backward: stages left of, in and right of the diagonal tile; a partial last row tile, column tile and K stage; whole tiles
@pytest.mark.parametrize("dtype,m,k,batch", [(O.F16, 784, 400, 100), (O.F16, 992, 464, 30), (O.F16, 1040, 1040, 15), (O.BF16, 784, 400, 100),
                                             (O.BF16, 896, 384, 66), (O.F32, 896, 384, 75), (O.F32, 976, 560, 165)])
def test_backward_on_the_large_tile(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T128, distinct=2)


# the same shapes with fewer samples, and narrow ones, run 64 x 64 tiles
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch", [(784, 144, 37), (768, 128, 86), (784, 16, 74), (912, 272, 22)])
def test_backward_of_many_features_on_the_small_tile(dtype, m, k, batch):
    _backward_of_repeated_samples(dtype, m, k, batch, T64)


# the register-blocked fragment-API kernel, launches of 2048 of its waves or more: few features, rows that a tile of 64 mostly pads, and
# upstream and mlp_grad off 16-byte boundaries.  Whole and partial blocks of 2 x 4; (16, 80, 65576) is also more than one launch's grid holds
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.F32])
@pytest.mark.parametrize("m,k,batch,off", [(16, 80, 1100, 0), (16, 272, 500, 0), (16, 80, 65576, 0), (80, 96, 700, 1), (112, 48, 600, 1), (256, 256, 64, 1),
                                           (32, 208, 1200, 0), (80, 208, 1000, 0), (96, 704, 600, 0)])
def test_backward_on_the_register_blocked_kernel(dtype, m, k, batch, off):
    _backward_of_repeated_samples(dtype, m, k, batch, BLOCKED, off)


def test_forward_of_16_features_beyond_one_grid_dimension():
    """A block per wave, the batch a grid dimension of at most 65535: two launches."""
    m, k, batch, distinct = 16, 80, 65576, 3
    assert R.dlrm_kernel(O.F16, m, k, batch) == WAVE
    stride = k + m * (m - 1) // 2
    x, turn = _small_integers(41, distinct * m * k, O.F16), np.arange(batch) % distinct
    dout = device_filled(batch * stride + 8, np.uint16, 0xEE)
    R.dlrm_fwd(O.F16, to_device(x.reshape(distinct, m * k)[turn]), dout, m, k, batch)
    out = to_host(dout, np.uint16)
    assert np.all(out[batch * stride:] == 0xEEEE)
    want = O.dlrm_fwd(O.F16, x, m, k, distinct).reshape(distinct, stride)
    assert np.array_equal(out[:batch * stride].reshape(batch, stride), want[turn])


def test_backward_with_an_upstream_off_16_bytes():
    """upstream at 2 bytes past a 16-byte boundary: taken by the kernels that read single elements, as ever."""
    m, k, batch, dtype = 80, 80, 3, O.F16
    store, stride = O.NP_STORAGE[dtype], k + m * (m - 1) // 2
    x, up = _small_integers(1, batch * m * k, dtype), _small_integers(2, batch * stride, dtype)
    held = to_device(np.concatenate([np.zeros(1, store), up]))
    dmlp, dgrad = device_filled(batch * k, store, 0xEE), device_filled(batch * m * k, store, 0xEE)
    R.dlrm_bwd(dtype, to_device(x), held.data_ptr() + 2, dmlp, dgrad, m, k, batch)
    want_mlp, want_grad = O.dlrm_bwd(dtype, x, up, m, k, batch)
    assert np.array_equal(to_host(dmlp, store).view(np.uint8), want_mlp.ravel().view(np.uint8))
    assert np.array_equal(O.storage_to_f32(to_host(dgrad, store), dtype), O.storage_to_f32(want_grad.ravel(), dtype))


# (32 features run a block per wave, 257 launches of up to 65535 samples; the two tests below it run macro tiles)
def test_more_samples_than_a_launch_holds():
    """2^24 + 4096 samples of one tile each: a launch's 256-thread workgroups are counted in 32 bits of threads, so the batch goes
    out in two launches.  The batch repeats 4096 samples; each repetition has to give the same bits (18 GB, 18 GB and 18 GB)."""
    m, k, part, copies = 32, 16, 4096, 4097
    stride = k + m * (m - 1) // 2
    x = torch.randn(part, m * k, device="cuda").half().repeat(copies, 1)
    out = torch.zeros(copies, part * stride, device="cuda", dtype=torch.float16)
    R.dlrm_fwd(O.F16, x, out, m, k, part * copies)
    want = torch.zeros(part * stride, device="cuda", dtype=torch.float16)
    R.dlrm_fwd(O.F16, x, want, m, k, part)
    assert bool(want.any()) and all(torch.equal(row, want) for row in out)
    grad, mlp = x.clone().view(copies, -1), torch.zeros(copies, part * k, device="cuda", dtype=torch.float16)
    R.dlrm_bwd(O.F16, x, out, mlp, grad, m, k, part * copies)
    assert not torch.equal(grad[0], x[:part].view(-1))
    assert all(torch.equal(row, grad[0]) for row in grad) and all(torch.equal(row, mlp[0]) for row in mlp)


def test_more_samples_than_a_forward_launch_holds():
    """2^24 + 4096 samples of one tile each: a launch's 256-thread workgroups are counted in 32 bits of threads, so the batch goes
    out in two launches.  The batch repeats 4096 samples; each repetition has to give the same bits (52 and 77 GB)."""
    m, k, part, copies = 48, 16, 4096, 4097
    stride = k + m * (m - 1) // 2
    assert R.dlrm_kernel(O.F32, m, k, part) == R.dlrm_kernel(O.F32, m, k, part * copies) == T64
    torch.cuda.empty_cache()
    x = torch.randn(part, m * k, device="cuda").repeat(copies, 1)
    out = torch.zeros(copies, part * stride, device="cuda")
    R.dlrm_fwd(O.F32, x, out, m, k, part * copies)
    want = torch.zeros(part * stride, device="cuda")
    R.dlrm_fwd(O.F32, x, want, m, k, part)
    assert bool(want.any()) and all(torch.equal(row, want) for row in out)
    del x, out
    torch.cuda.empty_cache()


def test_more_samples_than_a_backward_launch_holds():
    """The same of the backward (34, 68 and 34 GB)."""
    m, k, part, copies = 64, 16, 4096, 4097
    stride = k + m * (m - 1) // 2
    assert R.dlrm_kernel(O.F16, m, k, part, backward=True) == R.dlrm_kernel(O.F16, m, k, part * copies, backward=True) == T64
    torch.cuda.empty_cache()
    x, up = (torch.randn(part, width, device="cuda").half().repeat(copies, 1) for width in (m * k, stride))
    grad, mlp = torch.zeros(copies, part * m * k, device="cuda", dtype=torch.float16), torch.zeros(copies, part * k, device="cuda", dtype=torch.float16)
    R.dlrm_bwd(O.F16, x, up, mlp, grad, m, k, part * copies)
    want_grad, want_mlp = torch.zeros(part * m * k, device="cuda", dtype=torch.float16), torch.zeros(part * k, device="cuda", dtype=torch.float16)
    R.dlrm_bwd(O.F16, x, up, want_mlp, want_grad, m, k, part)
    assert bool(want_grad.any()) and all(torch.equal(row, want_grad) for row in grad) and all(torch.equal(row, want_mlp) for row in mlp)
    del x, up, grad, mlp
    torch.cuda.empty_cache()
