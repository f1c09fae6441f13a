"""Sizes at which the device lists fill or their layout changes, through the C ABI:
everything is compared bit for bit with the oracle, so no tolerance is involved."""
import numpy as np
import pytest

import pyoracle
import sqd

pytestmark = pytest.mark.gpu


def _rows(lb, ub):
    """Boxes as rows of bit patterns (lb_0, ub_0, lb_1, ub_1, ...), sorted."""
    m = np.empty((lb.shape[1], 2 * lb.shape[0]), dtype=np.uint64)
    m[:, 0::2] = np.ascontiguousarray(lb).view(np.uint64).T
    m[:, 1::2] = np.ascontiguousarray(ub).view(np.uint64).T
    return m[np.lexsort(m.T[::-1])]


class Collect:
    def __init__(self):
        self.lb, self.ub = [], []

    def __call__(self, lb, ub):
        self.lb.append(lb)
        self.ub.append(ub)


@pytest.mark.parametrize("level_bytes", [1 << 16, 1 << 24])   # dense and segmented lists between the levels
@pytest.mark.parametrize("capacity", [128, 1000])
def test_sink_in_parts_after_two_static_levels(program_text, level_bytes, capacity):
    # the criticals do not fit the critical list: the last level is repeated over
    # parts of the list between the two levels, segment by segment
    o_counts, o_crit = pyoracle.Oracle(program_text("ec3")).run(generations=3, threads=8, max_criticals=1 << 19)
    assert o_counts["num_critical_cuboids"] > 4 * capacity
    ref = np.ascontiguousarray(o_crit.reshape(len(o_crit), -1)).view(np.uint64)
    s = sqd.default_settings(generation_count=3, critical_capacity=capacity, level_bytes=level_bytes)
    with sqd.Core(sqd.Program.from_lemma("ec3"), settings=s) as core:
        for _ in range(2):
            sink = Collect()
            core.set_critical_sink(sink)
            r = core.prove()
            assert r["counts"] == o_counts and r["n_critical"] == len(o_crit)
            assert np.array_equal(_rows(np.hstack(sink.lb), np.hstack(sink.ub)), ref[np.lexsort(ref.T[::-1])])
