"""Order of the stores that a polling host reads.

A host-driven call polls a ticket in pinned memory and then reads what the kernels
stored to pinned memory before it.  A barrier orders memory inside a block only, so
every wave has to wait for its own stores (vmcnt(0)) before the barrier in front of
the ticket.  That is read off the gfx950 code of the kernels, without a GPU.
"""
import re
import shutil
import subprocess

import pytest

from sqd import build

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None, reason="needs hipcc")


def _kernel(source, name, tmp_path):
    """The instructions of a kernel (labels among them), from the build's own flags."""
    out = tmp_path / "k.s"
    cmd = [build.HIPCC] + build.HIPFLAGS + build._inc() + ["--offload-device-only", "-S", str(source), "-o", str(out)]
    r = subprocess.run([str(c) for c in cmd], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    lines = []
    for line in out.read_text().splitlines():
        if lines or re.match(r"_Z\w*%s\w*:" % name, line):
            line = line.split(";")[0].strip()
            if line:
                lines.append(line)
            if line == "s_endpgm":
                return lines
    raise AssertionError("no kernel " + name)


def _waits(line):
    return line.startswith("s_waitcnt") and "vmcnt(0)" in line


def test_state_before_ticket(tmp_path):
    code = _kernel(build.PKG / "csrc" / "runtime.hip", "k_round_end", tmp_path)
    host = [i for i, l in enumerate(code) if "store" in l and "sc0 sc1" in l]
    barrier = max(i for i, l in enumerate(code) if l == "s_barrier")
    assert len(host) >= 2 and host[-2] < barrier < host[-1]       # state, barrier, ticket
    # every wave passes the wait: it stands in the barrier's own basic block
    block = max(i for i, l in enumerate(code[:barrier]) if l.endswith(":") or l.startswith("s_cbranch"))
    assert any(_waits(l) for l in code[max(block, host[-2]):barrier])


def test_hulls_before_the_kernel_ends(tmp_path):
    # the hulls are announced by the ticket of a later kernel: they have to be out
    # (past the caches, and acknowledged) when this one ends
    code = _kernel(build.GEN / "ec2.hip", "k_hull_decode", tmp_path)
    stores = [i for i, l in enumerate(code) if l.startswith(("global_store", "flat_store"))]
    host = [i for i in stores if "sc0 sc1" in code[i]]
    assert len(host) == 2 * 4 + 1                                  # two bounds of four variables, and `has`
    end = code.index("s_endpgm")
    # the wait follows the stores in their own basic block: no lane that stored skips it
    block = [l for l in code[host[-1]:end]]
    wait = next(i for i, l in enumerate(block) if _waits(l))
    assert not any(l.endswith(":") or l.startswith("s_cbranch") for l in block[:wait])
