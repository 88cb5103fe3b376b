"""Syntax the generator does not write, against the oracle, bit exact: intra
blocks inside the picture without a left or above neighbour, with any mode and
angle beside any other's; coefficients beyond 16 bits (32-bit pools, the
transforms' 64-bit products and clamps); inter/intra on every block size, beside
overlapped motion compensation and warps, valid and not; filters and distance
weights at random."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

pytestmark = pytest.mark.gpu
# words of av1h_block
W, H, PLANE, INTRA, IBC, MODE, LEFT, BL, ANGLE, FILTER_TYPE, MV, FILT, COMPOUND, BLEND, WEDGE, II, II_WEDGE, WARP, PARAMS = \
    2, 3, 4, 6, 7, 8, 9, 12, 13, 14, 33, 37, 40, 41, 43, 45, 47, 48, 50


def _arrays(wire):
    """A mutable copy of a wire frame, its blocks and its coefficients."""
    b, pos, at = bytearray(wire), (16 + 4 * 231 + 7) // 8 * 8, []
    counts = np.frombuffer(wire, np.int64, 13, pos)
    pos += 104
    for n, size in zip(counts[:4], (276, 52, 40, 4)):
        at.append(pos)
        pos += (int(n) * size + 7) & ~7
    return b, np.frombuffer(b, np.int32, counts[0] * 69, at[0]).reshape(-1, 69), np.frombuffer(b, np.int32, counts[3], at[3])


def _intra(wire, rng):
    b, k, _ = _arrays(wire)
    intra, n = k[:, INTRA] == 1, len(k)
    for c in range(LEFT, BL + 1):
        k[intra & (rng.random(n) < 0.25), c] = 0
    some, mode = intra & (k[:, MODE] < 13) & (rng.random(n) < 0.7), rng.integers(0, 13, n)
    k[some, MODE], k[some, ANGLE], k[some, FILTER_TYPE] = mode[some], 0, rng.integers(0, 2, some.sum())
    turned = some & (mode >= 1) & (mode <= 8)
    k[turned, ANGLE] = rng.integers(-3, 4, turned.sum())
    return bytes(b)


def _coefficients(wire, rng):
    b, _, c = _arrays(wire)
    at = np.flatnonzero(c)
    at = rng.choice(at, max(1, len(at) // int(rng.choice([3, 30, 300]))), replace=False)
    top = 1 << int(rng.choice([15, 16, 17, 18, 20, 23]))
    c[at] = rng.integers(-top, top + 1, len(at))
    return bytes(b)


def _inter(wire, rng):
    b, k, _ = _arrays(wire)
    h, n = np.frombuffer(wire, np.int32, 6, 16), len(k)
    inter = (k[:, INTRA] == 0) & (k[:, IBC] == 0)
    lw, lh = (k[:, a] << np.where(k[:, PLANE] > 0, s, 0) for a, s in ((W, h[4]), (H, h[5])))
    wedge = (lw >= 8) & (lh >= 8) & (lw <= 32) & (lh <= 32)
    ii = np.flatnonzero(inter & (k[:, COMPOUND] == 0) & (rng.random(n) < 0.4))
    k[ii, II], k[ii, II + 1], k[ii, WEDGE] = 1, rng.integers(0, 4, len(ii)), rng.integers(0, 16, len(ii))
    k[ii, II_WEDGE] = wedge[ii] & (rng.random(len(ii)) < 0.5)
    wp = np.flatnonzero(inter & (rng.random(n) < 0.2))
    k[wp, WARP] = 1
    k[wp, PARAMS:PARAMS + 6] = np.array([0, 0, 65536, 0, 0, 65536]) + rng.integers(-6000, 6001, (len(wp), 6)) * [100, 100, 1, 1, 1, 1]
    mv = np.flatnonzero(inter & (rng.random(n) < 0.3))
    k[mv, MV:MV + 4], k[mv, FILT:FILT + 2] = rng.integers(-20000, 20001, (len(mv), 4)), rng.integers(0, 4, (len(mv), 2))
    dist = inter & (k[:, COMPOUND] == 2)
    k[dist, BLEND:BLEND + 2] = rng.integers(0, 17, (dist.sum(), 2))
    return bytes(b)


@pytest.mark.parametrize("alter,workloads", [(_intra, ("c1_mini", "c2_mini", "contract_mini")),
                                             (_coefficients, ("c2_mini", "contract_mini")),
                                             (_inter, ("tools_mini", "c2_mini"))], ids=["intra", "coefficients", "inter"])
@pytest.mark.parametrize("ss", [(1, 1), (1, 0), (0, 0)], ids=["420", "422", "444"])
def test_odd_syntax(alter, workloads, ss):
    for case in range(12):
        rng = np.random.default_rng(case)
        clip = pkg.Clip(workloads[case % len(workloads)], 97 + case, frames=3, width=int(rng.integers(40, 280)),
                        height=int(rng.integers(40, 180)), coded_width=0, bit_depth=int(rng.choice([8, 10, 12])),
                        intra_frac=0.3, rect4=case % 2, ss_x=ss[0], ss_y=ss[1])
        hip, ora, slots = pkg.HipDecoder(), OracleDecoder(), {}
        for f in range(clip.frames):
            wire = alter(pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]]), rng)
            slots[f], want = ora.decode_wire(wire)
            s, got = hip.decode_wire(wire)
            assert s == slots[f]
            for p in range(3):
                assert np.array_equal(got[p], want[p]), (case, f, p, np.argwhere(got[p] != want[p])[:3].tolist())
