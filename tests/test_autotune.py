"""The volume-form tuner on a stand-in batch (no GPU): the choice by element
count is a candidate like every form, wins among equals, and is what holds
without a record; a recorded choice is read back."""
import pytest

from vcp3d_open_amd import autotune
from vcp3d_open_amd.solver import volume_tiles


class StandInBatch:
    def __init__(self, ms):
        self.ms, self.nt = ms, {}

    def groups(self):
        return [dict(K=k, M=m) for k, m in self.ms]

    def set_tile(self, K, M, nt):
        self.nt[(K, M)] = nt

    def profile(self, reps):
        return [(1.0, self.ms[g].get(self.nt.get(g, 0), 9.0)) for g in self.ms]


def test_size_0_is_a_candidate():
    column = volume_tiles(5, 7)[0]
    batch = StandInBatch({(3, 4): {0: 1.0}, (5, 7): {0: 2.0, column: 1.5}, (6, 8): {0: 9.0}})
    result = autotune.tune(batch, reps=1)
    assert [result[k]["nt"] for k in ((3, 4), (5, 7), (6, 8))] == [0, column, 0]
    assert batch.nt == {(3, 4): 0, (5, 7): column, (6, 8): 0}
    for (K, M), r in result.items():
        assert list(r["ms"]) == [0] + volume_tiles(K, M)


def test_record_round_trip(tmp_path, monkeypatch):
    monkeypatch.setattr(autotune, "HERE", str(tmp_path))
    assert autotune.load_tiles() == {}
    autotune.save({(5, 7): {"nt": 0, "ms": {0: 1.0, 64: 2.0}}, (3, 4): {"nt": 16, "ms": {0: 1.0}}})
    assert autotune.load_tiles() == {(5, 7): 0, (3, 4): 16}


@pytest.mark.parametrize("shape", [(3, 4), (4, 5), (4, 6), (5, 7), (6, 8), (7, 9)])
def test_no_shape_is_pinned_to_a_workgroup_size(shape):
    """Batches and the served form read the recorded table: it names no form
    that keeps the column kernel from the cases that are faster with it."""
    assert autotune.load_tiles().get(shape, 0) in (0, volume_tiles(*shape)[0])
