"""The DLRM dot interaction at the edge of 32-bit counts: samples of more macro tiles than a launch holds."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import oraclelib as O
import rocwmma_amd as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_sample_of_more_64_tiles_than_a_launch_holds_is_taken():
    """f32, 370704 features: 2^24 + 5105 tiles of 64 x 64.  On a host without a device the call gets to the launch; it used to be refused."""
    child = """
import sys; sys.path.insert(0, %r)
import rocwmma_amd as R
try:
    R.device_info()
except R.R355Error:
    print("status", R.lib().r355_dlrm_fwd(R.F32, 0x10000, 0x20000, 370704, 16, 1, None))
""" % ROOT
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")  # (no device: nothing is launched on these addresses)
    r = subprocess.run([sys.executable, "-c", child], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "status" in r.stdout and "status -3" not in r.stdout, (r.returncode, r.stdout, r.stderr)  # R355_ERR_BAD_SIZE


@pytest.mark.gpu
def test_rows_of_a_sample_of_more_64_tiles_than_a_launch_holds():
    """The result takes 256 GiB: rows of it at both ends, on tile boundaries and at random, against the products themselves."""
    m, k = 370704, 16
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < (k + m * (m - 1) // 2) * 4 + (2 << 30):
        pytest.skip("not enough free device memory")
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randint(-3, 4, (m, k), device="cuda", generator=gen).float()
    out = torch.empty(k + m * (m - 1) // 2, dtype=torch.float32, device="cuda")
    R.dlrm_fwd(O.F32, x, out, m, k, 1)
    assert torch.equal(out[:k], x[0])
    rows = [1, 2, 63, 64, 65, 127, 128, 129, m - 129, m - 17, m - 16, m - 1] + np.random.default_rng(1).integers(1, m, 40).tolist()
    for row in rows:
        at = k + row * (row - 1) // 2
        assert torch.equal(out[at:at + row], (x[:row] * x[row]).sum(dim=1)), row
    del out
    torch.cuda.empty_cache()
