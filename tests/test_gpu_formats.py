"""4:2:2 and 4:4:4 pictures against the oracle, bit exact: every tool of the
generated clips at odd sizes, with superres and restoration of small units,
and CDEF blocks of every strength and direction, coded and searched, on the
chroma grids these formats have (8 and 16 lanes a block, the direction tables
of axes scaled apart, dependency cells of four samples)."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder
from test_gpu_cdef import COUNTS, ROW
from test_gpu_restoration import _with_units

pytestmark = pytest.mark.gpu
FORMATS = pytest.mark.parametrize("ss", [(1, 0), (0, 0)], ids=["422", "444"])


def _check(clip, alter=lambda wire: wire):
    hip, ora, slots = pkg.HipDecoder(), OracleDecoder(), {}
    for f in range(clip.frames):
        wire = alter(pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]]))
        s, got = hip.decode_wire(wire)
        so, want = ora.decode_wire(wire)
        assert s == so
        slots[f] = s
        for p in range(3):
            assert np.array_equal(got[p], want[p]), (f, p, np.argwhere(got[p] != want[p])[:3].tolist())


@FORMATS
@pytest.mark.parametrize("workload,over", [
    ("c1_mini", dict(width=131, height=77, intra_frac=0.4)),
    ("c2_mini", dict(width=200, height=72, coded_width=0, intra_frac=0.3)),
    ("c2_mini", dict(width=331, height=139, coded_width=190, mv_sigma=300.0)),  # superres
    ("c2_mini", dict(width=130, height=90, coded_width=0, max_tx=8, bit_depth=12, avail_auto=0.5)),
    ("contract_mini", dict(intra_frac=0.6, bit_depth=10)),
    ("tools_mini", dict(width=333, height=157, inter_tools=0.9, levels=1)),
    ("tools_mini", dict(width=142, height=230, inter_tools=0.9, bit_depth=12, intrabc=0.5, residual_frac=0.2)),
])
def test_clips(workload, over, ss):
    for seed in (73, 74):
        _check(pkg.Clip(workload, seed, frames=3, ss_x=ss[0], ss_y=ss[1], **over))


def _with_blocks(wire, kind, ss, rng):
    """The frame with CDEF of random strengths on every block of its grid."""
    b = np.frombuffer(wire, np.uint8)
    counts = b[COUNTS:COUNTS + 104].view(np.int64).copy()
    h = b[16:16 + 24].view(np.int32)
    w, height = int(h[1]) or int(h[0]), int(h[2])
    pad = lambda n: (int(n) + 7) // 8 * 8
    end = len(b) - sum(pad(n * 40) for n in counts[10:])
    start = end - pad(counts[9] * ROW.itemsize)
    rows = []
    for p in range(3):
        sx, sy = ss if p else (0, 0)
        rows += [(p, x, y) for y in range(0, pad(height) >> sy, 8 >> sy) for x in range(0, pad(w) >> sx, 8 >> sx)]
    u = np.zeros(len(rows), ROW)
    u["plane"], u["x"], u["y"] = np.array(rows).T
    n, top = len(u), {"coded": (16, 5), "edge": (86, 86), "large": (256, 256)}[kind]
    u["pri"], u["sec"] = rng.integers(0, top[0], n), rng.integers(0, top[1], n)
    u["damping"] = rng.integers(3, 7, n) if kind == "coded" else rng.integers(0, 16, n)
    u["dir"] = rng.integers(-1, 8, n) if kind != "coded" else rng.choice([-1, -1, 0, 1, 2, 3, 4, 5, 6, 7], n)
    counts[9] = n
    data = u.tobytes()
    out = bytearray(b[:start].tobytes())
    out[COUNTS:COUNTS + 104] = counts.tobytes()
    return bytes(out) + data + bytes(-len(data) % 8) + b[end:].tobytes()


@FORMATS
@pytest.mark.parametrize("kind", ["coded", "edge", "large"])
def test_cdef_blocks(kind, ss):
    rng = np.random.default_rng(len(kind) + ss[0])
    for depth in (8, 10, 12):
        for w, h in ((8, 8), (34, 18), (71, 67), (130, 90)):
            clip = pkg.Clip("c2_mini", 79, frames=2, bit_depth=depth, width=w, height=h, coded_width=0, ss_x=ss[0], ss_y=ss[1])
            _check(clip, lambda wire: _with_blocks(wire, kind, ss, rng))


@FORMATS
@pytest.mark.parametrize("kind,log2", [("wiener", 6), ("beyond", 4), ("sgr", 5), ("mixed", 2), ("mixed", 0)])
def test_restoration_units(kind, log2, ss):
    rng = np.random.default_rng(log2 + 2 * ss[0])
    for depth in (8, 10, 12):
        for w, h in ((34, 18), (71, 67)) if log2 < 2 else ((71, 67), (198, 134)):
            clip = pkg.Clip("c2_mini", 83, frames=2, bit_depth=depth, width=w, height=h, coded_width=0, ss_x=ss[0], ss_y=ss[1])
            _check(clip, lambda wire: _with_units(wire, kind, log2, rng))
