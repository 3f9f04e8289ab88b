"""The committed launch parameters and the tuner's candidates, without a GPU."""
import json

from diso_amd import autotune


def _tile(run):  # include/diso_hip.h, DISO_PARAM_RUN
    t = 1
    while 2 * t <= run // 4 and 2 * t <= 8:
        t *= 2
    return t


def test_candidates_differ():
    """Each run length tried is a gather tile of its own, and all tiles are tried."""
    assert sorted(_tile(r) for r in autotune.RUNS) == [1, 2, 4, 8]


def test_committed_table_is_of_these_candidates():
    with open(autotune.TUNING_FILE) as f:
        saved = json.load(f)
    for entry in saved.values():
        assert set(entry["buckets"]) == {str(n) for n in autotune.BUCKET_SIZES} == set(entry["measured"])
        for key, p in entry["buckets"].items():
            m = entry["measured"][key]
            assert set(m["emit_backward_ms"]) == {str(r) for r in autotune.RUNS}
            assert p["run"] in autotune.RUNS and p["count_blocks_per_cu"] in autotune.COUNT_BLOCKS_PER_CU
            # the choice is (within the rounding of the saved times) one of the fastest
            assert m["emit_backward_ms"][str(p["run"])] <= 1.011 * min(m["emit_backward_ms"].values()) + 1e-4


def test_ties_go_to_the_smaller_value():
    assert autotune._choose({4: 1.009, 8: 1.0, 16: 1.2}) == 4
    assert autotune._choose({4: 1.02, 8: 1.0, 16: 0.999}) == 8
