"""Motion compensation four samples at a time against the oracle, bit exact:
vectors that leave the picture on every side (the clamped taps), blocks at
its edges, one and two references, unscaled and superres-scaled rows, each bit
depth, pictures narrower than a filter's reach, with and without queued
blocks that wait on the cells inter blocks mark."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload,over", [
    ("c1_mini", dict(width=16, height=16, mv_range=400)),
    ("c1_mini", dict(width=74, height=50, mv_range=1200, bit_depth=12)),
    ("c2_mini", dict(width=96, height=80, coded_width=0, mv_sigma=400.0)),
    ("c2_mini", dict(width=200, height=72, coded_width=102, mv_sigma=300.0)),  # nearly 2:1
    ("c2_mini", dict(width=131, height=77, coded_width=120, mv_sigma=30.0, bit_depth=12, compound_frac=1.0)),
    ("c2_mini", dict(width=328, height=136, coded_width=246, bit_depth=8, compound_frac=0.0, intra_frac=0.0)),
    ("tools_mini", dict(mv_sigma=300.0)),
    # every inter tool on odd sizes and at both ends of the depths: inter halves ahead of the queue
    ("tools_mini", dict(width=333, height=157, inter_tools=0.9, bit_depth=8)),
    ("tools_mini", dict(width=142, height=230, inter_tools=0.9, bit_depth=12, intrabc=0.5)),
])
@pytest.mark.parametrize("seed", [21, 22])
def test_motion(workload, over, seed):
    clip = pkg.Clip(workload, seed, frames=4, **over)
    ora = list(pkg.decode_clip(OracleDecoder(), clip))
    for (f, _, ph), (_, _, po) in zip(pkg.decode_clip(pkg.HipDecoder(), clip), ora):
        for p in range(3):
            assert np.array_equal(ph[p], po[p]), (f, p, np.argwhere(ph[p] != po[p])[:3].tolist())
