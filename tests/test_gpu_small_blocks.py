"""The queue's small intra blocks (at most 64 samples, one per lane) against
the oracle, bit exact: every intra mode on 4x4 .. 8x8 and the rectangular
sizes beside the larger blocks' path, edges taken from packed words, from the
frame (inter neighbours) and absent, at picture edges that cut a block's above
right and below left, at each bit depth, with and without the edge filter.
"""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload,over", [
    # key frames: every block queued; sizes that end inside a block
    ("c2_mini", dict(frames=1, max_tx=4, rect_tx=0)),
    ("c2_mini", dict(frames=1, max_tx=8, width=173, height=99, coded_width=0)),
    ("c2_mini", dict(frames=1, max_tx=16, width=66, height=58, coded_width=0, bit_depth=8)),
    ("c2_mini", dict(frames=1, bit_depth=12, width=120, height=200, coded_width=90)),
    # large blocks: 32x32 to 64x64 and 2:1, one stripe of them and many; edges of both kinds
    ("c2_mini", dict(frames=1, coef_zero=0.98, width=640, height=72, coded_width=0)),
    ("c2_mini", dict(frames=3, width=392, height=328, coded_width=0, intra_frac=0.4, bit_depth=8)),
    # the smallest picture of one block column
    ("c1_mini", dict(frames=1, width=16, height=16, bit_depth=10)),
    # half the blocks intra among inter ones: edges mixed from words and frame
    ("c2_mini", dict(frames=4, intra_frac=0.5, max_tx=8)),
    ("c1_mini", dict(frames=3, intra_frac=0.3, width=250, height=138, avail_auto=0.5)),
    # edge filter off for some frames, cells marked for CFL and palette readers
    ("contract_mini", dict(frames=3, intra_frac=0.6, bit_depth=10)),
    # raw residual samples and blocks without a transform of their own
    ("c2_mini", dict(frames=2, residual_frac=0.4, tx_skip=0.7, intra_frac=0.4)),
])
@pytest.mark.parametrize("seed", [11, 12])
def test_small_blocks(workload, over, seed):
    clip = pkg.Clip(workload, seed, **over)
    ora = list(pkg.decode_clip(OracleDecoder(), clip))
    for (f, _, ph), (_, _, po) in zip(pkg.decode_clip(pkg.HipDecoder(), clip), ora):
        for p in range(3):
            assert np.array_equal(ph[p], po[p]), (f, p, np.argwhere(ph[p] != po[p])[:3].tolist())


@pytest.mark.parametrize("workload,over", [
    ("c2_mini", dict(frames=2, width=328, height=200, coded_width=0)),
    ("c2_mini", dict(frames=2, width=200, height=136, coded_width=0, bit_depth=12, intra_frac=0.5, ss_x=0, ss_y=0)),
    ("c1_mini", dict(frames=2, width=173, height=99, intra_frac=0.4, tx_skip=0.6)),
    ("tools_mini", dict(frames=3, intra_frac=0.4, levels=1)),
    ("contract_mini", dict(frames=2, intra_frac=0.5, ss_y=0)),
])
@pytest.mark.parametrize("seed", [13, 14, 15])
def test_four_to_one_blocks(workload, over, seed):
    """Intra blocks and transforms of 4x16, 16x4, 8x32, 32x8, 16x64 and 64x16."""
    test_small_blocks(workload, dict(over, rect4=1), seed)
