"""Where the generated code may take an arc cosine's cheap enclosure instead of the
exact interval.  An operation that drops sign cases or domain checks because of
compile-time bounds (product, quotient, square root, arc cosine) gives an interval
that need not contain the exact result once an operand crosses its bounds, so what
it reads has to be exact; sums and comparisons hold for any interval."""
import re
import shutil
import subprocess

import pytest

from sqd import build

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def generate(tmp_path_factory):
    exe = tmp_path_factory.mktemp("codegen") / "codegen"
    cmd = ["g++", "-std=c++17", "-O1"] + build._inc()
    cmd += [str(build.ROOT / "tests/codegen_driver.cpp"), str(build.PKG / "host/ivarp/codegen.cpp")]
    cmd += [str(s) for s in build.HOST_SOURCES] + ["-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]

    def run(text):
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return r.stdout
    return run


def _acos(source):
    """The last template argument of every arc cosine in the constraints' functions."""
    out = re.findall(r"iv_acos<\w+, \w+, (\w+)>", source)
    assert out
    return set(out)


def _second_checks(source):
    return re.findall(r"!c\d+<true>\(lb, ub, C\)\.poss", source)


@pytest.mark.parametrize("key", ["more1", "more2"])
def test_sums_take_the_enclosure(program_text, generate, key):
    src = generate(program_text(key))
    assert _acos(src) == {"EXACT"} and _second_checks(src)


@pytest.mark.parametrize("key", ["more1", "more2"])
@pytest.mark.parametrize("op,kids", [("mul", 2), ("div", 2), ("sqrt", 1)])
def test_operations_with_signs_read_exact_values(program_text, generate, key, op, kids):
    # the difference that reads the arc cosine becomes a product, a quotient or a root of it
    lines = program_text(key).splitlines()
    acos = [l.split()[1] for l in lines if l.startswith("node ") and l.split()[2] == "acos"]
    assert len(acos) == 1
    for i, l in enumerate(lines):
        f = l.split()
        if f[0] == "node" and f[2] == "sub" and acos[0] in f[5:5 + int(f[4])]:
            lines[i] = " ".join(f[:2] + [op, f[3], str(kids), acos[0]] + f[6:5 + kids] + f[5 + int(f[4]):])
    src = generate("\n".join(lines) + "\n")
    assert _acos(src) == {"true"} and not _second_checks(src)
