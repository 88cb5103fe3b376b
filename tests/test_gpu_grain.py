"""Film grain templates against the oracle, bit exact, where the wavefront of
one wave can go wrong: every filter lag, shift and noise scale, luma noise
off, chroma from luma, chroma planes with and without points, 8 to 12 bits, at
pictures of one and of many noise stripes; and its application four samples
per lane, with and without overlap and the restricted range."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu

GRAIN = 16 + 4 * 43  # byte of av1h_grain in a wire frame
NUM_Y, CFL, NUM_CB, NUM_CR, LAG, SHIFT, SCALE, OVERLAP, RESTRICTED = 2, 35, 36, 69, 103, 178, 179, 186, 187


def _patched(wire, values):
    b = bytearray(wire)
    g = np.frombuffer(b, np.int32, 188, GRAIN)
    assert g[0] == 1 and g[LAG] == 3  # apply, ar_coeff_lag as generated
    for k, v in values.items():
        g[k] = v
    return bytes(b)


@pytest.mark.parametrize("values", [
    {LAG: 0}, {LAG: 1}, {LAG: 2}, {LAG: 3},
    {LAG: 3, SHIFT: 0, SCALE: 3}, {LAG: 2, SHIFT: 3, SCALE: 0},
    {LAG: 3, NUM_Y: 0}, {LAG: 1, NUM_Y: 0, CFL: 1},
    {LAG: 3, CFL: 0, NUM_CB: 0}, {LAG: 3, CFL: 0, NUM_CR: 0}, {LAG: 2, CFL: 0, NUM_CB: 0, NUM_CR: 0},
], ids=str)
def test_templates(values):
    for depth, w, h in ((8, 64, 40), (10, 200, 168), (12, 90, 330)):
        clip = pkg.Clip("c2_mini", 41, frames=2, bit_depth=depth, width=w, height=h, coded_width=0)
        hip, ora, slots = pkg.HipDecoder(), OracleDecoder(), {}
        for f in range(clip.frames):
            wire = _patched(pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]]), values)
            s, ph = hip.decode_wire(wire)
            so, po = ora.decode_wire(wire)
            assert s == so
            slots[f] = s
            for p in range(3):
                assert np.array_equal(ph[p], po[p]), (depth, f, p, np.argwhere(ph[p] != po[p])[:3].tolist())


@pytest.mark.parametrize("values", [{}, {OVERLAP: 0}, {OVERLAP: 1, RESTRICTED: 1}, {OVERLAP: 1, CFL: 1}, {OVERLAP: 1, NUM_Y: 0},
                                    {OVERLAP: 1, CFL: 0, NUM_CR: 0}], ids=str)
def test_ragged_pictures(values):
    """Four samples per lane at right and bottom edges of every remainder."""
    for depth in (8, 10, 12):
        for w, h in ((33, 17), (66, 34), (71, 67), (97, 33), (132, 66)):
            clip = pkg.Clip("c2_mini", 53, frames=1, bit_depth=depth, width=w, height=h, coded_width=0)
            wire = _patched(clip.wire(0), values)
            _, got = pkg.HipDecoder().decode_wire(wire)
            _, want = OracleDecoder().decode_wire(wire)
            for p in range(3):
                assert np.array_equal(got[p], want[p]), (depth, w, h, p, np.argwhere(got[p] != want[p])[:3].tolist())


def _equal(wire, *where):
    _, got = pkg.HipDecoder().decode_wire(wire)
    _, want = OracleDecoder().decode_wire(wire)
    for p in range(3):
        assert np.array_equal(got[p], want[p]), (*where, p, np.argwhere(got[p] != want[p])[:3].tolist())


@pytest.mark.parametrize("ss", [(1, 0), (0, 0)], ids=["422", "444"])
@pytest.mark.parametrize("values", [{}, {LAG: 1}, {CFL: 1}, {CFL: 0, NUM_CB: 0}, {NUM_Y: 0}, {OVERLAP: 0}], ids=str)
def test_other_formats(values, ss):
    """Chroma templates of 73 rows, whose last row lies under the last luma
    row; the overlap of two stripes reads it where a block's vertical offset
    is the largest, one block in sixteen."""
    for depth, w, h in ((8, 200, 330), (10, 331, 203), (12, 90, 330)):
        for seed in (67, 68):
            clip = pkg.Clip("c2_mini", seed, frames=1, bit_depth=depth, width=w, height=h, coded_width=0, ss_x=ss[0], ss_y=ss[1])
            _equal(_patched(clip.wire(0), {OVERLAP: 1, **values}), depth, seed)


@pytest.mark.parametrize("values", [{SHIFT: -6}, {SHIFT: -9, LAG: 1}, {SCALE: -4}, {SCALE: -9, SHIFT: -7, LAG: 2}], ids=str)
def test_shifts_of_nothing(values):
    """Shifts of zero and below leave a value as it is."""
    for depth in (8, 10, 12):
        clip = pkg.Clip("c2_mini", 71, frames=1, bit_depth=depth, width=120, height=72, coded_width=0)
        _equal(_patched(clip.wire(0), {OVERLAP: 1, **values}), depth)
