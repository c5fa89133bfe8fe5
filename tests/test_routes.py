"""Which kernels an exec of the heuristic's choice launches (tests/host/route.cpp, no GPU), for layers where two ways were timed as graph
replays: the faster one, to 5 %, which a rule over sizes may miss where both are close."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "host", "route")
NCHW, NCHW4 = 0, 3


def _routes(layers):
    """layers: (format, n, ic, ih, iw, oc, f, stride, group, residual) -> (launches, dynamic LDS and threads of the last) each"""
    if not os.path.exists(EXE):
        subprocess.check_call(["make", "-C", os.path.dirname(EXE), "-s", EXE])
    r = subprocess.run([EXE], input="".join(" ".join(str(int(v)) for v in l) + "\n" for l in layers), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    out = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
    assert len(out) == len(layers)
    return out


# n, ic, ih, iw, oc, f, stride, residual; us packed (two launches) and in one launch
PLAIN_NCHW = [
    (44, 206, 29, 90, 254, 1, 2, 0, 28.8, 35.2),
    (40, 5, 75, 49, 185, 3, 2, 0, 18.5, 20.6),
    (51, 7, 89, 27, 197, 1, 2, 0, 13.9, 19.6),
    (17, 15, 103, 91, 237, 1, 2, 0, 16.1, 19.2),
    (55, 134, 105, 35, 200, 3, 2, 0, 54.8, 77.9),
    (50, 4, 57, 93, 204, 3, 2, 0, 28.0, 34.5),
    (57, 6, 59, 107, 194, 3, 2, 0, 28.1, 51.4),
    (56, 17, 84, 85, 236, 1, 2, 0, 29.0, 44.4),
    (25, 200, 41, 85, 182, 3, 2, 0, 38.9, 38.7),    # fewer workgroups
    (57, 61, 90, 69, 243, 1, 2, 1, 51.0, 53.5),     # a residual
    (51, 11, 75, 104, 234, 5, 2, 1, 65.9, 54.2),    # 25 taps
    (52, 49, 63, 104, 163, 1, 2, 0, 34.0, 22.1),    # rows of whole quads
    (6, 75, 61, 45, 150, 3, 1, 1, 16.4, 11.6),      # stride 1
]


def test_plain_nchw_strides():
    got = _routes([(NCHW, n, ic, ih, iw, oc, f, s, 1, z) for n, ic, ih, iw, oc, f, s, z, _, _ in PLAIN_NCHW])
    for (launches, _, _), layer in zip(got, PLAIN_NCHW):
        packed, one = layer[-2:]
        assert launches in (1, 2)
        assert (packed if launches == 2 else one) <= 1.05 * min(packed, one), layer
