"""Loop restoration against the oracle, bit exact, where tiles of four samples
per lane can go wrong: every unit size down to one sample (units that do not
start on a multiple of four), odd and ragged pictures, Wiener taps of the coded
range, at the edge of and beyond what products of 16 bits take, and every
self-guided parameter set, at 8 to 12 bits."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu

HEADER, TYPE, LOG2, COLS, WORDS = 16, 34, 37, 40, 231  # of av1h_frame_header, in words
WIENER, SGR = 2, 3
ROW = np.dtype([("type", "<i4"), ("wiener", "<i4", (2, 3)), ("set", "<i4"), ("xqd", "<i4", 2)])


def _with_units(wire, kind, log2, rng):
    """The frame with its restoration units replaced (they are the last arrays)."""
    b = np.frombuffer(wire, np.uint8)
    h = b[HEADER:HEADER + 4 * WORDS].view(np.int32).copy()
    at = (HEADER + 4 * WORDS + 7) // 8 * 8
    counts = b[at:at + 104].view(np.int64).copy()
    tail = sum((int(n) * ROW.itemsize + 7) // 8 * 8 for n in counts[10:])
    w, height, ssx, ssy = int(h[0]), int(h[2]), int(h[4]), int(h[5])
    arrays = []
    for p in range(3):
        pw, ph = (w + ssx >> ssx, height + ssy >> ssy) if p else (w, height)
        size = 1 << log2
        cols, rows = max((pw + size // 2) // size, 1), max((ph + size // 2) // size, 1)
        u = np.zeros(cols * rows, ROW)
        u["type"] = rng.choice([0, WIENER, SGR, SGR], len(u)) if kind == "mixed" else SGR if kind == "sgr" else WIENER
        u["wiener"] = rng.integers([-5, -23, -17], [11, 9, 47], (len(u), 2, 3))
        if kind == "edge":
            u["wiener"][:, :, 0] = rng.choice([-4031, 4095, 0], (len(u), 2))
        if kind == "beyond":
            u["wiener"][:, :, 0] = rng.choice([-8193, 8192, 9000], (len(u), 2))
        u["set"] = rng.integers(0, 16, len(u))
        u["xqd"] = rng.integers([-96, -32], [32, 96], (len(u), 2))
        h[TYPE + p], h[LOG2 + p], h[COLS + p], counts[10 + p] = 1, log2, cols, len(u)
        data = u.tobytes()
        arrays.append(data + bytes(-len(data) % 8))
    out = bytearray(b[:len(b) - tail].tobytes())
    out[HEADER:HEADER + 4 * WORDS] = h.tobytes()
    out[at:at + 104] = counts.tobytes()
    return bytes(out) + b"".join(arrays)


@pytest.mark.parametrize("kind,log2", [("wiener", 6), ("edge", 5), ("beyond", 4), ("sgr", 6), ("sgr", 4), ("mixed", 3),
                                       ("mixed", 2), ("mixed", 1), ("mixed", 0)])
def test_units(kind, log2):
    rng = np.random.default_rng(log2 + 16 * len(kind))
    shapes = ((34, 18), (71, 67)) if log2 < 2 else ((71, 67), (130, 90), (198, 134))
    for depth in (8, 10, 12):
        for w, h in shapes:
            clip = pkg.Clip("c2_mini", 43, frames=2, bit_depth=depth, width=w, height=h, coded_width=0)
            hip, ora, slots = pkg.HipDecoder(), OracleDecoder(), {}
            for f in range(clip.frames):
                wire = pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]])
                wire = _with_units(wire, kind, log2, rng)
                s, got = hip.decode_wire(wire)
                so, want = ora.decode_wire(wire)
                assert s == so
                slots[f] = s
                for p in range(3):
                    assert np.array_equal(got[p], want[p]), (depth, w, h, f, p, np.argwhere(got[p] != want[p])[:3].tolist())
