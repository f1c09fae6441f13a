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


def _pieces(program_text, m):
    """ec3's initial cuboids, each cut into m along the first variable: every child of
    the first static level survives on them."""
    qlb, qub, _ = pyoracle.Oracle(program_text("ec3")).initial_queue()
    lb, ub = np.repeat(qlb, m, axis=1), np.repeat(qub, m, axis=1)
    j = np.tile(np.arange(m), qlb.shape[1])
    w = (ub[0] - lb[0]) / m
    lb[0], ub[0] = lb[0] + w * j, lb[0] + w * (j + 1)
    return lb, ub


# ec3: an entry of a level list has 60 bytes, and the first static level 8 children
@pytest.mark.parametrize("limit", [200, 256, 1200])           # dense lists, and segmented ones from 256 on
def test_host_calls_take_as_many_boxes_as_level_bytes_allow(program_text, limit):
    lb, ub = _pieces(program_text, limit // 4)
    o = pyoracle.Oracle(program_text("ec3"))
    s = sqd.default_settings(level_bytes=60 * 8 * limit, critical_capacity=1 << 20)
    with sqd.Core(sqd.Program.from_lemma("ec3"), settings=s) as core:
        ol, ou, oc = o.final(lb, ub)
        gl, gu, gc = core.final(lb, ub)
        assert gc == oc and np.array_equal(_rows(gl, gu), _rows(ol, ou))
        ol, ou, oc = o.split(lb, ub)
        gl, gu, gc = core.split(lb, ub)
        assert gc == oc and np.array_equal(_rows(gl, gu), _rows(ol, ou))
        one_more = np.hstack([lb, lb[:, :1]]), np.hstack([ub, ub[:, :1]])
        for call in (core.final, core.split):
            with pytest.raises(sqd.SqdError) as e:
                call(*one_more)
            assert e.value.code == -4


@pytest.mark.parametrize("n,kw", [(256, {}), (1200, {}), (9216, dict(group_levels=0xFFFFFFFF, prefilter_group=8)),
                                  (9216, dict(group_levels=0xFFFFFFFF, prefilter_group=8, grid_blocks=3)),
                                  (2304, dict(group_levels=0xFFFFFFFF, prefilter_group=2, grid_blocks=1))])
def test_segments_filled_to_their_bound(program_text, n, kw):
    # the largest round of lists kept in segments, the smallest ones among them (2,048
    # entries; 18,432 where the first level has a group test), all children of the
    # first level surviving
    lb, ub = _pieces(program_text, n // 4)
    ohl, ohu, ohas, oc = pyoracle.Oracle(program_text("ec3")).nonfinal(lb, ub)
    assert oc["num_cuboids"] == n * (8 + 1024)
    s = sqd.default_settings(level_bytes=60 * 8 * n, dequeue_buffer_size=n, **kw)
    with sqd.Core(sqd.Program.from_lemma("ec3"), settings=s) as core:
        ghl, ghu, ghas, gc = core.nonfinal(lb, ub)
    assert gc["num_cuboids"] == oc["num_cuboids"] and gc["num_leaf_cuboids"] == oc["num_leaf_cuboids"]
    assert np.array_equal(ghas, ohas)
    keep = ohas.astype(bool)
    assert np.array_equal(ghl[:, keep].view(np.uint64), ohl[:, keep].view(np.uint64))
    assert np.array_equal(ghu[:, keep].view(np.uint64), ohu[:, keep].view(np.uint64))


def _noalloc_counts(prog, settings):
    c, k = sqd.Counts(), sqd._SZ()
    rc = sqd.lib().sqd_prove_range_noalloc(0, prog._h, sqd.ctypes.byref(settings), 0, 128, sqd.ctypes.byref(c), None, None,
                                           0, sqd.ctypes.byref(k))
    if rc != 0:
        raise sqd.SqdError(rc, sqd.lib().sqd_last_error().decode())
    return c.as_dict()


def test_noalloc_falls_back_to_dense_lists():
    # the longest frontier that fits the 64 MiB array: with it, lists in segments do
    # not, and the proof runs on dense ones
    prog = sqd.Program.from_lemma("one")

    def settings(frontier):
        return sqd.default_settings(level_bytes=8 << 20, critical_capacity=4096, frontier_capacity=frontier)

    lo, hi = 1 << 16, 1 << 20                                  # 52 bytes a cuboid
    want = _noalloc_counts(prog, settings(lo))
    with pytest.raises(sqd.SqdError):
        _noalloc_counts(prog, settings(hi))
    while hi - lo > 16:
        mid = (lo + hi) // 2
        try:
            assert _noalloc_counts(prog, settings(mid)) == want
            lo = mid
        except sqd.SqdError as e:
            assert e.code == -4
            hi = mid
    with sqd.Core(prog, settings=settings(lo)) as core:
        size = sqd.ctypes.c_uint64()
        sqd._check(sqd.lib().sqd_core_memory(core._h, sqd.ctypes.byref(size)))
        assert size.value > 64 << 20                           # as a core of its own lays it out
        assert core.prove()["counts"] == want
