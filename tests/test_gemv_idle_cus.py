"""Col-major GEMV of aligned matrices around the rules that give those with idle CUs the plan of unaligned ones (gemv.hip, leavesCusIdle), with and
without splits of K, whole and partial last blocks.  Small integers, so that every sum is exact in any order."""
import pytest
import torch

from test_gemv_askew import test_columns_off_cache_lines as _exact

pytestmark = pytest.mark.gpu


# three quarters of the CUs (256) in blocks of 32 rows (f64: 16) and one block more; 64 and 200 MB; a block; columns of a padded leading dimension
@pytest.mark.parametrize("dtype,m,k,pad", [(torch.float32, 32, 64, 0), (torch.float32, 1024, 1024, 0), (torch.float32, 2240, 2504, 0), (torch.float32, 6144, 2604, 0),
                                           (torch.float32, 6176, 2000, 0), (torch.float32, 6144, 2608, 0), (torch.float32, 2300, 2504, 4), (torch.float32, 4096, 12204, 0),
                                           (torch.float32, 4096, 12212, 0), (torch.float64, 16, 4, 0), (torch.float64, 1840, 2868, 0), (torch.float64, 3072, 2600, 0),
                                           (torch.float64, 3088, 2500, 0), (torch.float64, 1100, 2916, 4), (torch.float64, 272, 8336, 0)]
                         # runs of 64 bytes over many columns: in one piece, and in shares, which stay with the splits of aligned columns
                         + [(torch.float32, 2016, 2708, 0), (torch.float32, 2752, 4352, 0), (torch.float32, 864, 13476, 0), (torch.float64, 1216, 2792, 0),
                            (torch.float64, 352, 14812, 0)]
                         # beyond 256 MiB with K split: one round of the plan's workgroups, several, and a padded leading dimension
                         + [(torch.float32, 8256, 8192, 0), (torch.float32, 22432, 4888, 0), (torch.float32, 8380, 8324, 4), (torch.float64, 4592, 8044, 0)])
def test_aligned_columns(dtype, m, k, pad):
    assert (m + pad) * dtype.itemsize % 128 == 0
    _exact(dtype, m, k, pad, 0)
