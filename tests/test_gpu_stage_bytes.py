"""The compulsory bytes reported for a frame's prediction and transform stage,
which holds every block's transforms and the blocks of every inter tool, and
for its queue, from the frame's syntax."""
import numpy as np
import pytest

import av1ongpu_amd as pkg

pytestmark = pytest.mark.gpu
W, H, INTRA, IBC, COMPOUND, INTERINTRA, TX, NTX = 2, 3, 6, 7, 40, 45, 65, 66  # of av1h_block, in words


def _expected(wire):
    pos = (16 + 4 * 231 + 7) // 8 * 8
    n, ntx = np.frombuffer(wire, np.int64, 2, pos)
    b = np.frombuffer(wire, np.int32, n * 69, pos + 104).reshape(n, 69)
    tx = np.frombuffer(wire, np.int32, ntx * 13, pos + 104 + (n * 276 + 7) // 8 * 8).reshape(ntx, 13)
    inter = queue = 0
    for k in b:
        area, queued = k[W] * k[H], k[INTRA] or k[IBC] or k[INTERINTRA]
        if queued:
            queue += 4 * area
        if not k[INTRA] and not k[IBC]:
            inter += area * (6 if k[COMPOUND] else 4)
        for t in tx[k[TX]:k[TX] + k[NTX]]:
            inter += t[2] * t[3] * (4 if queued else 2) if t[5] > 0 else 0
    return inter, queue


@pytest.mark.parametrize("workload", ["c1_mini", "c2_mini", "tools_mini"])
def test_stage_bytes(workload):
    clip = pkg.Clip(workload, 91)
    dec, slots = pkg.HipDecoder(), {}
    for f in range(clip.frames):
        wire = pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]])
        dec.set_stage_timing(True)
        slots[f], _ = dec.decode_wire(wire, read_back=False)
        t = dec.stage_times()
        dec.set_stage_timing(False)
        assert (t["inter"][2], t["queue"][2]) == _expected(wire), f
