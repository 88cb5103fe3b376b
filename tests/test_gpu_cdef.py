"""CDEF against the oracle, bit exact, where four samples per lane in packed
16-bit words can go wrong: blocks at every plane edge (pictures of one block and
of many), every coded direction and the searched one, strengths of zero, of the
coded range, at the edge of and beyond what 16 bits hold, at 8 to 12 bits."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu

COUNTS = (16 + 4 * 231 + 7) // 8 * 8
ROW = np.dtype([("plane", "<i4"), ("x", "<i4"), ("y", "<i4"), ("pri", "<i4"), ("sec", "<i4"), ("damping", "<i4"), ("dir", "<i4")])


def _with_blocks(wire, kind, rng):
    """The frame with CDEF of random strengths on every block of its grid."""
    b = np.frombuffer(wire, np.uint8)
    counts = b[COUNTS:COUNTS + 104].view(np.int64).copy()
    h = b[16:16 + 24].view(np.int32)
    w, height = int(h[1]) or int(h[0]), int(h[2])
    pad = lambda n: (int(n) + 7) // 8 * 8
    end = len(b) - sum(pad(n * 40) for n in counts[10:])
    start = end - pad(counts[9] * ROW.itemsize)
    rows = [(p, x, y) for p in range(3) for y in range(0, pad(height) >> (p > 0), 8 >> (p > 0))
            for x in range(0, pad(w) >> (p > 0), 8 >> (p > 0))]
    u = np.zeros(len(rows), ROW)
    u["plane"], u["x"], u["y"] = np.array(rows).T
    n = len(u)
    top = {"coded": (16, 5), "large": (256, 256), "edge": (86, 86)}[kind]
    u["pri"], u["sec"] = rng.integers(0, top[0], n), rng.integers(0, top[1], n)
    u["damping"] = rng.integers(3, 7, n) if kind == "coded" else rng.integers(0, 16, n)
    u["dir"] = rng.integers(-1, 8, n)
    counts[9] = n
    data = u.tobytes()
    out = bytearray(b[:start].tobytes())
    out[COUNTS:COUNTS + 104] = counts.tobytes()
    return bytes(out) + data + bytes(-len(data) % 8) + b[end:].tobytes()


@pytest.mark.parametrize("kind", ["coded", "edge", "large"])
def test_blocks(kind):
    rng = np.random.default_rng(len(kind))
    for depth in (8, 10, 12):
        for w, h in ((8, 8), (34, 18), (71, 67), (130, 90)):
            clip = pkg.Clip("c2_mini", 47, frames=2, bit_depth=depth, width=w, height=h, coded_width=0)
            hip, ora, slots = pkg.HipDecoder(), OracleDecoder(), {}
            for f in range(clip.frames):
                wire = pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]])
                wire = _with_blocks(wire, kind, rng)
                s, got = hip.decode_wire(wire)
                so, want = ora.decode_wire(wire)
                assert s == so
                slots[f] = s
                for p in range(3):
                    assert np.array_equal(got[p], want[p]), (depth, w, h, f, p, np.argwhere(got[p] != want[p])[:3].tolist())
