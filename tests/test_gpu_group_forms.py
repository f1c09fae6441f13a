"""The group tests where groups really form: with one or three blocks per launch the
children of a level take many trips, so that the first test runs, its groups are
split, listed and decided in ragged waves.  Decisions, hulls and criticals are the
oracle's bit for bit (it decides every child by itself), so no tolerance is involved."""
import numpy as np
import pytest

import pyoracle
import sqd

pytestmark = pytest.mark.gpu

ALL = 0xFFFFFFFF


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def _rows(lb, ub):
    m = np.empty((lb.shape[1], 2 * lb.shape[0]), dtype=np.uint64)
    m[:, 0::2], m[:, 1::2] = _bits(lb).T, _bits(ub).T
    return m[np.lexsort(m.T[::-1])]


def _core(key, **kw):
    return sqd.Core(sqd.Program.from_lemma(key), settings=sqd.default_settings(level_bytes=64 << 20, frontier_capacity=1 << 16, **kw))


def _queue(program_text, key, count):
    o = pyoracle.Oracle(program_text(key))
    lb, ub, _ = o.initial_queue()
    at = np.linspace(0, lb.shape[1] - 1, min(count, lb.shape[1])).astype(int)
    return o, lb[:, at], ub[:, at]


def _same_nonfinal(want, got):
    ohl, ohu, ohas, oc = want
    ghl, ghu, ghas, gc = got
    assert gc["num_cuboids"] == oc["num_cuboids"] and gc["num_leaf_cuboids"] == oc["num_leaf_cuboids"]
    assert np.array_equal(ghas, ohas)
    keep = ohas.astype(bool)
    assert np.array_equal(_bits(ghl[:, keep]), _bits(ohl[:, keep]))
    assert np.array_equal(_bits(ghu[:, keep]), _bits(ohu[:, keep]))


def _same_final(want, got):
    assert got[2] == want[2]
    assert np.array_equal(_rows(got[0], got[1]), _rows(want[0], want[1]))


@pytest.mark.parametrize("key,count", [("one", 7), ("two", 13), ("three", 33), ("four", 3), ("more1", 3), ("more2", 3),
                                       ("ec2", 15), ("ec3", 3)])
def test_plain_nonfinal(program_text, key, count):
    o, lb, ub = _queue(program_text, key, count)
    want = o.nonfinal(lb, ub)
    for blocks in (1, 3):
        with _core(key, grid_blocks=blocks) as core:
            _same_nonfinal(want, core.nonfinal(lb, ub))


@pytest.mark.parametrize("key,count", [("two", 13), ("four", 3), ("ec2", 15), ("ec3", 3)])
@pytest.mark.parametrize("group", [0, 1, 2, 8, 16, 32, 64])
def test_every_level_grouped(program_text, key, count, group):
    o, lb, ub = _queue(program_text, key, count)
    with _core(key, grid_blocks=1, group_levels=ALL, prefilter_group=group) as core:
        _same_nonfinal(o.nonfinal(lb, ub), core.nonfinal(lb, ub))


def _pieces(lb, ub, m):
    """Each box cut into m along the first variable."""
    lb, ub = np.repeat(lb, m, axis=1), np.repeat(ub, m, axis=1)
    j = np.tile(np.arange(m), lb.shape[1] // m)
    w = (ub[0] - lb[0]) / m
    lb[0], ub[0] = lb[0] + w * j, lb[0] + w * (j + 1)
    return lb, ub


# ec2's last level has 64 children of a box, ec3's 128 (8 of the first level's each):
# groups that fail as a whole, in part and not at all, and real criticals
@pytest.mark.parametrize("key,pieces", [("ec2", 5), ("ec2", 37), ("ec3", 1), ("ec3", 9)])
@pytest.mark.parametrize("kw", [{}, {"prefilter_group": 2}, {"prefilter_group": 8}, {"prefilter_group": 16},
                                {"prefilter_group": 32}, {"prefilter_group": 64}], ids=lambda k: str(list(k.values())))
def test_final_criticals(program_text, key, pieces, kw):
    o, lb, ub = _queue(program_text, key, 16)
    lb, ub = _pieces(lb, ub, pieces)
    want = o.final(lb, ub)
    assert 0 < want[2]["num_critical_cuboids"] < want[2]["num_leaf_cuboids"] or key == "ec2"
    if kw:
        kw = dict(kw, group_levels=ALL)
    for blocks in (1, 2):
        with _core(key, grid_blocks=blocks, **kw) as core:
            _same_final(want, core.final(lb, ub))


# More2's fifth variable 6 below its domain (moved there, or widened): a group's
# interval can then miss values of its children, so that the group tests would prune
# children that are not to be pruned
@pytest.mark.parametrize("widen", [False, True])
@pytest.mark.parametrize("kw", [{}, {"group_levels": ALL, "prefilter_group": 16},
                                {"fp32_prefilter": ALL, "prefilter_group": 16}], ids=["plain", "group", "fp32"])
def test_boxes_outside_the_domain(program_text, widen, kw):
    o, lb, ub = _queue(program_text, "more2", 24)
    lb[4] -= 6.0
    if not widen:
        ub[4] -= 6.0
    with _core("more2", grid_blocks=1, **kw) as core:
        _same_nonfinal(o.nonfinal(lb, ub), core.nonfinal(lb, ub))
        _same_final(o.final(lb, ub), core.final(lb, ub))
        # a call with boxes of the domain has its group tests again
        _, lb, ub = _queue(program_text, "more2", 5)
        if "fp32_prefilter" not in kw:
            _same_nonfinal(o.nonfinal(lb, ub), core.nonfinal(lb, ub))


@pytest.mark.parametrize("key,var", [("three", 0), ("three", 4), ("more1", 0), ("more1", 2)])
@pytest.mark.parametrize("how", ["inverted", "infinite"])
def test_inverted_and_infinite_boxes(program_text, key, var, how):
    o, lb, ub = _queue(program_text, key, 6)
    if how == "inverted":
        lb[var], ub[var] = ub[var].copy(), lb[var].copy()
    else:
        ub[var] = np.inf
    with _core(key, grid_blocks=1) as core:
        _same_nonfinal(o.nonfinal(lb, ub), core.nonfinal(lb, ub))
        _same_final(o.final(lb, ub), core.final(lb, ub))
        _same_final(o.split(lb, ub), core.split(lb, ub))
