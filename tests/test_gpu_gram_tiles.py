"""The Gram around the line between its two kernels (1024 sub-chunks a step), at
one, two and four waves a chunk, bit for bit against the oracle."""
import pytest

import gpujachx_amd as g
from test_gpu_step import both

pytestmark = pytest.mark.gpu


# 544, 1024 and 1056 sub-chunks of two waves a chunk, 1024 and 1088 of four, 1024 of
# one; the first step's Gram and the next one's
@pytest.mark.parametrize("m,n,fam", [(2048, 544, "mmstep"), (2048, 1024, "cycwor"), (2048, 1056, "mmstep"),
                                     (4096, 512, "mmstep"), (4096, 544, "mmstep"), (3072, 2048, "cycwor")])
def test_both_sides(m, n, fam):
    g.configureGPU(0)
    both(9, m, n, n // 2, fam, 2)
