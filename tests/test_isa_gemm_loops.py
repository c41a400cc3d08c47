"""Static check of the generated gfx950 code (no GPU needed): the K loops of the macro-tile GEMM kernels, one wave per SIMD and bound by the
matrix instructions they issue, keep their scalars in scalar registers.  One that does not fit is written to a lane of a vector
register and read back by v_readlane_b32, an issue slot beside the matrix instructions each time."""
import os
import re

import pytest

from rocwmma_amd import build as B
from test_isa_hazards import _texts


def _loop_scalars_read_back(text):
    """Kernel -> v_readlane_b32 in its blocks of at least half as many matrix instructions as its largest one, the K loop's."""
    blocks, current = {}, None
    for line in (l.strip() for l in text.splitlines()):
        label = re.match(r"(_Z\w*gemmTiled\w*):", line)
        if label:
            current = [0, 0]
            blocks[label.group(1)] = [current]
            name = label.group(1)
        elif current is not None and line.startswith(".Lfunc_end"):
            current = None
        elif current is not None and (line.startswith((".LBB", "s_branch", "s_cbranch"))):
            current = [0, 0]
            blocks[name].append(current)
        elif current is not None:
            current[0] += line.startswith("v_mfma")
            current[1] += line.startswith("v_readlane_b32")
    return {n: sum(reads for matrix, reads in b if 2 * matrix >= max(m for m, _ in b)) for n, b in blocks.items() if max(m for m, _ in b) >= 64}


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="hipcc not installed")
def test_no_gemm_loop_reads_scalars_back_from_vector_registers():
    reads = {}
    for text in _texts()[:4]:  # the parts of gemm_tiled.hip
        reads.update(_loop_scalars_read_back(text))
    assert len(reads) > 100
    assert not {n: r for n, r in reads.items() if r}
