"""The group test of a plain proof's last static level decides exactly as the
per-child evaluation (the oracle's), through the C ABI: at launches of one trip
(every child by itself) and of several, at counts that leave ragged waves, and
on boxes outside the program's compile-time box, for which it is switched off.
Everything is compared bit for bit, so no tolerance is involved."""
import numpy as np
import pytest

import pyoracle
import sqd

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def _same_nonfinal(program_text, key, lb, ub, **settings):
    o = pyoracle.Oracle(program_text(key))
    ohl, ohu, ohas, oc = o.nonfinal(lb, ub)
    with sqd.Core(sqd.Program.from_lemma(key), settings=sqd.default_settings(**settings)) as core:
        ghl, ghu, ghas, gc = core.nonfinal(lb, ub)
    assert gc["num_cuboids"] == oc["num_cuboids"] and gc["num_leaf_cuboids"] == oc["num_leaf_cuboids"]
    assert np.array_equal(ghas, ohas)
    keep = ohas.astype(bool)
    assert np.array_equal(_bits(ghl[:, keep]), _bits(ohl[:, keep]))
    assert np.array_equal(_bits(ghu[:, keep]), _bits(ohu[:, keep]))


@pytest.mark.parametrize("key,count", [("one", 1), ("one", 67), ("three", 1), ("three", 331), ("four", 1), ("four", 65),
                                       ("more1", 1), ("more1", 129), ("more2", 33), ("ec2", 16), ("ec3", 4)])
def test_plain_nonfinal_equals_oracle(program_text, key, count):
    qlb, qub, _ = pyoracle.Oracle(program_text(key)).initial_queue()
    idx = np.linspace(0, qlb.shape[1] - 1, min(count, qlb.shape[1])).astype(int)
    _same_nonfinal(program_text, key, qlb[:, idx], qub[:, idx])


@pytest.mark.parametrize("key,group", [("ec2", 0), ("ec3", 0), ("three", 0), ("three", 8)])
def test_boxes_outside_the_domain(program_text, key, group):
    # one box beyond the compile-time box's upper end: the call evaluates child by child
    qlb, qub, _ = pyoracle.Oracle(program_text(key)).initial_queue()
    lb, ub = qlb[:, :40].copy(), qub[:, :40].copy()
    ub[0, 0] += 2.0
    _same_nonfinal(program_text, key, lb, ub, prefilter_group=group, group_levels=0xFFFFFFFF if group else 0)
