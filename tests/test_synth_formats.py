"""Clips of the other chroma formats: 4:2:2 and 4:4:4 pictures whose blocks
cover every plane once, whose wire frames round-trip and which the oracle
decodes."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from oracle_lib import OracleDecoder

HEADER, WORDS, BLOCK_INTS = 16, 231, 69  # bytes, words of av1h_frame_header and av1h_block
X, Y, W, H, PLANE = range(5)


def _blocks(wire):
    pos = (HEADER + 4 * WORDS + 7) & ~7
    n = int(np.frombuffer(wire, np.int64, 1, pos)[0])
    return np.frombuffer(wire, np.int32, n * BLOCK_INTS, pos + 13 * 8).reshape(n, BLOCK_INTS)


@pytest.mark.parametrize("ss", [(1, 1), (1, 0), (0, 0)], ids=["420", "422", "444"])
@pytest.mark.parametrize("workload", ["c1_mini", "c2_mini", "tools_mini", "contract_mini"])
def test_clip(workload, ss):
    clip = pkg.Clip(workload, 61, frames=2, width=150, height=90, coded_width=0, ss_x=ss[0], ss_y=ss[1])
    for f, _slot, planes in pkg.decode_clip(OracleDecoder(), clip):
        wire = clip.wire(f)
        assert pkg.wire_header(wire)[4:6] == ss
        assert pkg.syn_lib().av1s_wire_roundtrip(wire, len(wire)) == 1
        blocks = _blocks(wire)
        for p in range(3):
            sx, sy = ss if p else (0, 0)
            seen = np.zeros((96 >> sy, 152 >> sx), np.int32)
            for x, y, w, h in blocks[blocks[:, PLANE] == p][:, [X, Y, W, H]]:
                seen[y:y + h, x:x + w] += 1
            assert (seen == 1).all(), (f, p)
            assert planes[p].shape == ((90 + sy) >> sy, (150 + sx) >> sx)
