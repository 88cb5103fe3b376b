"""The launch-shape autotuner on a stand-in decoder: parameters of kernels that
ride in another's launch are left alone, the others measured."""
import av1ongpu_amd as pkg
from av1ongpu_amd import autotune


class _Lead:
    def __init__(self):
        lib = pkg.hip_lib()
        self.cur = {lib.av1h_tune_name(i).decode(): 8 for i in range(lib.av1h_tune_params())}
        self.tried = set()

    def tuning(self):
        return dict(self.cur)

    def set_tuning(self, values):
        self.cur.update(values)
        self.tried |= set(values)


def test_riding_kernels_are_not_tuned(monkeypatch):
    lead = _Lead()
    # the fewer workgroups the faster: noise would pick a value for any parameter measured
    monkeypatch.setattr(autotune, "_time_batches", lambda *_: 1.0 + sum(lead.cur.values()))
    riders = {"cdef_chroma", "itx_intra", "itx_intra_large"}
    assert riders <= set(lead.cur)
    chosen, base, best = autotune.tune([lead], [])
    assert lead.tried == set(lead.cur) - riders
    assert all(chosen[n] == 8 for n in riders) and chosen["mc"] == 2 and best < base
    autotune.tune([lead], [], params=["itx_intra"])
    assert "itx_intra" not in lead.tried
