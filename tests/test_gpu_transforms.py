"""Inverse transforms against the oracle, bit exact, on both sides of the
rule that picks the 24-bit form: coefficients far below its bound, around it
(waves whose lanes disagree) and far above it (clamps act), every size and
type, each bit depth (the clamps' widths), 16-bit coefficients (wider ones are in
test_gpu_odd_syntax.py), coded levels and lossless blocks."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [8, 10, 12])
@pytest.mark.parametrize("scale,zero", [(40.0, 0.85), (400.0, 0.6), (1500.0, 0.3), (4000.0, 0.7), (12000.0, 0.0)])
def test_transforms(depth, scale, zero):
    for workload, over in (("c2_mini", dict(width=272, height=200, coded_width=0, intra_frac=0.3)),
                           ("contract_mini", {}), ("tools_mini", dict(levels=1))):
        clip = pkg.Clip(workload, 31, frames=2, bit_depth=depth, coef_scale=scale, coef_zero=zero, tx_skip=0.05, **over)
        ora = list(pkg.decode_clip(OracleDecoder(), clip))
        for (f, _, ph), (_, _, po) in zip(pkg.decode_clip(pkg.HipDecoder(), clip), ora):
            for p in range(3):
                assert np.array_equal(ph[p], po[p]), (workload, f, p, np.argwhere(ph[p] != po[p])[:3].tolist())
