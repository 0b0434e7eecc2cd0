"""What the autotuner times: no two candidates that run the same kernels.  The
FP32 and FP64 two-phase walk has leaves of its own and no tree, so neither the
leaf size nor the records fetched per round trip change it; the mixed form's
walks the LBVH."""
import pytest


class _Ctx:
    def synchronize(self):
        pass

    def timer_start(self):
        pass

    def timer_stop(self):
        return self.ms


class _Batch:
    """Stands for a packed run: what would be timed, and made-up times."""
    fast = 0

    def __init__(self, reps, spec, ctx=None):
        self.ctx = _Ctx()
        self.ctx.ms = 1.0 if spec.list_walk == self.fast else 2.0

    def set_state(self):
        pass

    def run(self, nsteps):
        pass

    def prepare(self):
        pass

    def close(self):
        pass


def _what_runs(pkg, precision, row):
    """The list and step kernels' parameters behind a row of the table."""
    leaf, walk, front, batch, lanes, _ = row
    over_tree = walk == 1 or (walk == 0 and precision == "mixed")
    return (walk, leaf if over_tree else 0, (front or 8) if walk == 0 and precision == "mixed" else 0, batch or 4,
            lanes or 1)


@pytest.mark.parametrize("precision", ["fp32", "mixed", "fp64"])
@pytest.mark.parametrize("fast", [0, 1, 3])
def test_every_candidate_runs_other_kernels(pkg, monkeypatch, precision, fast):
    monkeypatch.setattr(pkg.batched, "BatchedSimulation", _Batch)
    monkeypatch.setattr(_Batch, "fast", fast)
    best, table = pkg.autotune([], pkg.SimSpec(duration=0, precision=precision))
    assert best.list_walk == fast
    ran = [_what_runs(pkg, precision, row) for row in table]
    assert len(set(ran)) == len(ran)
    # every walk, every tree leaf size and every step shape is tried
    assert {r[0] for r in ran} == {0, 1, 3}
    assert {r[1] for r in ran if r[0] == 1} == {8, 16, 32}
    assert {r[1] for r in ran if r[0] == 0} == ({8, 16, 32} if precision == "mixed" else {0})
    assert {r[2] for r in ran if r[0] == 0} == ({8, 16} if precision == "mixed" and fast == 0 else {ran[0][2]})
    assert {r[3] for r in ran} == ({2, 4, 8} if precision == "fp32" else {4}) and {r[4] for r in ran} == {1, 2}
