"""The autotuner's assembly tiles: candidates that are different schedules, none timed twice.

Assembly tiles hold at most 64 columns, so every larger assemble_tile is the same schedule as 64.
"""
import pytest

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, csc_arrays

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tile", [16, 64, 128, 1024])
def test_no_schedule_is_timed_twice(tile):
    A = P.laplace3d(14, 14, 14, 0.5)
    s = SymLDLT()
    s.setOrdering(OrderingType.Metis)
    s.analyzePattern(A)
    s.setTuning(64, tile)
    d_vals = torch.from_numpy(csc_arrays(A)[3].copy()).to("cuda:0")
    torch.cuda.synchronize()
    _, trials, _ = s.autotune(d_vals.data_ptr(), nrhs=1, reps=1)
    schedules = [(t[0], min(t[1], 64), *t[2:]) for t, _ in trials]
    assert len(schedules) == len(set(schedules))
    assert {t[1] for t in schedules} == {16, 32, 64}
