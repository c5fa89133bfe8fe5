"""The kernels that an exec launches, through tests/host/route.cpp (no GPU)."""
import collections
import functools
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "host", "route")
HEURISTIC, UNNAMED = -1, -2
Route = collections.namedtuple("Route", "launches lds threads grid kernels")


def _short(name):
    """'void mi355::(anonymous namespace)::k<1, 2>(...)' -> 'k<1, 2>'"""
    return re.match(r"(?:void )?(?:\w+::)*(\w+(?:<[^()]*>)?)\(", name.replace("(anonymous namespace)::", "")).group(1)


@functools.lru_cache(None)
def _build():
    subprocess.check_call(["make", "-C", os.path.dirname(EXE), "-s", EXE])


def routes(execs):
    """execs: descriptors, or (descriptor, algorithm, tile, workspace) -> a Route for each"""
    _build()
    lines = ["%s %d %d %d\n" % ((bytes(e[0]).hex(),) + tuple(int(v) for v in e[1:])) for e in
             (e if isinstance(e, tuple) else (e, HEURISTIC, -1, True) for e in execs)]
    r = subprocess.run([EXE], input="".join(lines), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    out = []
    for line in r.stdout.splitlines():
        numbers, *names = line.split("\t")
        out.append(Route(*(int(v) for v in numbers.split()), tuple(_short(n) for n in names)))
    assert len(out) == len(lines)
    return out
