"""The autotuner over settings that choose no kernel: one setting is timed, the
handle keeps it, and what it returns can be set on another handle."""
import pytest

from cpp_projects_amd.tune import tune_search


class Handle:
    def __init__(self, schedule):
        self.schedule, self.timing, self.was_set = schedule, False, False

    def get_schedule(self):
        return list(self.schedule)

    def enable_timing(self, on):
        self.timing = on

    def stage_times_ms(self):
        return [1.0, 0.5]

    def set_schedule(self, s):
        self.was_set = True

    set_staged = set_group_shape = set_schedule


@pytest.mark.parametrize("schedule,mode", [([3, 3, 3, 3], 0), ([4, 4, 4], 1), ([1], 0), ([], 0)])
def test_no_candidates_are_run(schedule, mode):
    h, runs = Handle(schedule), []
    best, results = tune_search(h, lambda: runs.append(h.timing), reps=2)
    assert runs == [True] * 3 and not h.timing and not h.was_set
    assert best == {"staged": mode, "shape": None, "schedule": schedule}
    assert results == [(1.5, mode, None, tuple(schedule))]
