"""Performance cases of the prover core: the calls that a user's program makes.

A user lowers a lemma statement, makes a core (or a service) for it and proves
ranges of the statement's first variable on it, or, behind the reference's proof
driver, hands the core arrays of cuboids.  Each case is one such call:

  prove     a job on a core of one row, or a batch of jobs on a core of several,
            over ranges of the first variable's initial subdivisions; in plain
            binary64 (the default), with the binary32 prefilter on the last static
            level or with the binary64 group test there (the two choices the
            autotuner makes)
  nonfinal  one non-final pass over an array of cuboids in host memory
  stream    jobs of several statements through the proof service

Outputs are the counts (whole numbers) and the hulls.
"""
import random
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "squares-in-disk_amd"))
import sqd  # noqa: E402

# Per statement: variables, static levels, initial subdivisions of the first
# variable, how many of them at its low and at its high end have next to no work
# (a job over "nearly all" of the statement starts and ends there), cuboids of
# the whole proof, and binary64 operations per cuboid when every cuboid is
# evaluated by itself (the op-counting CPU restatement).
STATEMENTS = {
    "top2": (1, 0, 128, 16, 16, 168, 74),
    "one": (3, 2, 128, 45, 2, 2869888, 99),
    "two": (4, 2, 128, 26, 24, 7181696, 220),
    "three": (5, 2, 64, 7, 21, 3549856, 324),
    "four": (6, 3, 64, 3, 15, 37245328, 396),
    "five": (7, 4, 128, 0, 108, 3392, 700),
    "six": (8, 4, 128, 0, 116, 14848, 724),
    "seven": (9, 5, 128, 0, 124, 1808, 700),
    "more2": (6, 3, 128, 0, 104, 123127968, 247),
    "more1": (5, 2, 128, 0, 23, 1056154896, 505),
}
# cuboids that one initial cuboid costs in a non-final pass (mean over the
# initial queue), and operations per cuboid
NONFINAL = {"one": (34500, 99), "three": (1200, 324), "four": (6000, 396), "more1": (8000, 505)}
LARGEST = 1.0e9      # cuboids of a drawn case, at most

# statements of the stream: the ones whose proofs take about a millisecond
STREAM = ("one", "two", "three", "four", "six", "top2")


def listed():
    return [
        # the smallest proof: one variable, no static grid; all launches and latency
        {"name": "top2_plain", "kind": "prove", "statement": "top2", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # eight variables, four levels of initial queue, few cuboids: latency of short levels
        {"name": "six_plain", "kind": "prove", "statement": "six", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # the headline workload: one whole proof, one round, a 256 x 256 static grid
        {"name": "one_plain", "kind": "prove", "statement": "one", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # an ordinary proof: five variables, 64 x 32 grid under three dynamic variables
        {"name": "three_plain", "kind": "prove", "statement": "three", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # the largest statement with a fixed number of subcontainers, three static levels
        {"name": "four_plain", "kind": "prove", "statement": "four", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # a long proof whose middle levels keep many cuboids
        {"name": "more2_plain", "kind": "prove", "statement": "more2", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # the longest proof: arc cosines, dynamic splits, some 160 rounds
        {"name": "more1_plain", "kind": "prove", "statement": "more1", "mode": "plain", "group": 0, "jobs": 1, "share": 1},
        # throughput of many proofs at once with the binary32 prefilter, as the service batches them
        {"name": "one_fp32_batch", "kind": "prove", "statement": "one", "mode": "fp32", "group": 16, "jobs": 32, "share": 1},
        {"name": "four_fp32_batch", "kind": "prove", "statement": "four", "mode": "fp32", "group": 16, "jobs": 7, "share": 1},
        # the reference's proof driver handing over a batch of cuboids (its default queue pops about a thousand)
        {"name": "more1_nonfinal", "kind": "nonfinal", "statement": "more1", "count": 1003},
        # one proof with the binary64 group test, the autotuner's choice where no binary32 is wanted
        {"name": "two_group", "kind": "prove", "statement": "two", "mode": "group", "group": 0, "jobs": 1, "share": 1},
        # jobs of several statements, whole ones and slices down to a 64th, through the service
        {"name": "stream", "kind": "stream", "count": 24},
    ]


def draw(rng):
    kind = rng.choice(["prove", "prove", "prove", "prove", "nonfinal", "nonfinal", "stream"])
    if kind == "prove":
        statement = rng.choice(sorted(STATEMENTS))
        share = round(2 ** -rng.uniform(0, 4), 3)
        cost = STATEMENTS[statement][5] * min(1, share * 2)   # a slice may lie where the work is dense
        most = max(1, min(32, int(LARGEST / cost)))
        mode = rng.choice(["plain", "fp32", "group"]) if STATEMENTS[statement][1] else "plain"
        group = 0 if mode == "plain" else rng.choice([0, 8, 16, 32])
        jobs = rng.randint(2, most) if most > 1 and rng.random() < 0.4 else 1
        return {"kind": kind, "statement": statement, "mode": mode, "group": group, "jobs": jobs, "share": share}
    if kind == "nonfinal":
        return {"kind": kind, "statement": rng.choice(sorted(NONFINAL)), "count": int(2 ** rng.uniform(0, 13))}
    return {"kind": kind, "count": rng.randint(6, 40)}


class State:
    """What the user's program holds: the program, a core or a service, and the inputs."""

    def __init__(self, kind):
        self.kind = kind
        self.core = self.service = None

    def __del__(self):
        for h in (self.core, self.service):
            if h is not None:
                h.close()


def _range(rng, statement, share):
    """A job's range: nearly all of the statement, or a slice of up to that share of it where there is work."""
    _, _, n, low, high, _, _ = STATEMENTS[statement]
    if share == 1:
        return rng.randint(0, low), n - rng.randint(0, high)
    most = max(1, int(n * share))
    width = rng.randint(max(1, most * 3 // 4), most)
    first = rng.randint(min(low, n - width), max(min(low, n - width), n - high - width))
    return first, first + width


def _settings(case):
    last = 1 << max(0, STATEMENTS[case["statement"]][1] - 1)
    kw = {"fp32": {"fp32_prefilter": last}, "group": {"group_levels": last}}.get(case["mode"], {})
    if case["jobs"] > 1:   # the sizes that the service gives each row of a batch
        kw.update(jobs=case["jobs"], level_bytes=256 << 20, frontier_capacity=1 << 22)
    return sqd.default_settings(prefilter_group=case["group"], **kw)


def prepare(case, seed):
    rng = random.Random(seed * 7919 + 17)
    s = State(case["kind"])
    if s.kind == "prove":
        s.core = sqd.Core(sqd.Program.from_lemma(case["statement"]), 0, _settings(case))
        s.ranges = [_range(rng, case["statement"], case["share"]) for _ in range(case["jobs"])]
    elif s.kind == "nonfinal":
        # cuboids of the statement's initial queue, picked at random (the queue comes in no fixed order)
        s.core = sqd.Core(sqd.Program.from_lemma(case["statement"]), 0)
        lb, ub, _ = s.core.initial_queue()
        order = np.lexsort(lb)
        lb, ub = lb[:, order], ub[:, order]
        at = np.array([rng.randrange(lb.shape[1]) for _ in range(case["count"])])
        s.lb, s.ub = np.ascontiguousarray(lb[:, at]), np.ascontiguousarray(ub[:, at])
    else:
        s.programs = {k: sqd.Program.from_lemma(k) for k in STREAM}
        s.service = sqd.Service(0, workers=4, batch_jobs=4, fp32_prefilter=0, level_bytes=64 << 20,
                                frontier_capacity=1 << 20, core_bytes_estimate=1 << 29)
        s.jobs = []
        for i in range(case["count"]):
            k = STREAM[i % len(STREAM)]
            s.jobs.append((s.programs[k],) + _range(rng, k, 1 / 2 ** (i * 5 % 7)))
    return s


def run(s):
    if s.kind == "prove":
        if len(s.ranges) == 1:
            r = s.core.prove_range(*s.ranges[0])
            return [r["counts"], r["n_critical"]]
        done = s.core.prove_batch(s.ranges)
        return np.array([list(r["counts"].values()) + [r["n_critical"]] + list(r["fp32_stats"]) for r in done])
    if s.kind == "nonfinal":
        return list(s.core.nonfinal(s.lb, s.ub))
    ids = [s.service.submit(*job) for job in s.jobs]
    done = [s.service.wait(i) for i in ids]
    return np.array([list(r["counts"].values()) + [r["n_critical"], r["status"]] for r in done])


def work(case):
    """The cuboids a call decides times the binary64 operations of one, when each is
    evaluated by itself, and the boxes that go in and come out."""
    kind = case["kind"]
    if kind == "prove":
        nargs, _, n, _, _, cuboids, ops = STATEMENTS[case["statement"]]
        total = cuboids * case["share"] * case["jobs"]
        return {"bytes": 16.0 * nargs + 8 * 8 * case["jobs"], "flops": total * ops}
    if kind == "nonfinal":
        nargs = STATEMENTS[case["statement"]][0]
        cuboids, ops = NONFINAL[case["statement"]]
        return {"bytes": case["count"] * (32.0 * nargs + 1), "flops": float(case["count"]) * cuboids * ops}
    total = 0.0
    for i in range(case["count"]):
        k = STREAM[i % len(STREAM)]
        total += STATEMENTS[k][5] / 2 ** (i * 5 % 7) * STATEMENTS[k][6]
    return {"bytes": case["count"] * 64.0, "flops": total}
