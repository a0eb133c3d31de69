"""Which path the solvers of test_gpu_bounded_fused.py take: where its two runs
were the same path, its comparison says nothing.  And that comparison, with the
path asserted, for the block shapes that its boxes leave out.

A solver asks for the plan of its own precision.  FP64 blocks of 513-point lines
with three coefficient tables (free-slip ends), or two and the metrics of a
stretched mesh, do not fit in 64 KB of LDS, nor do 257 points in x with their
tile; FP32 ones do.  Uniform no-slip walls of 513 points fit in both, with 65
segments of 8 points on 8 lines (FP32: 31 of 17 on 32).  Lines of 17 points have
two segments in FP64 only.  The tolerances are that file's: 1e-11 of the velocity
after 4 steps in FP64; in FP32 bulk at most 1.5 times the per-operator path's
error, plus 1e-7."""
import math
import os

import pytest

from test_gpu_bounded_fused import CASES, FREE, WALL, _run

pytestmark = pytest.mark.gpu

X = pytest.importorskip("incompact3d_amd")

# (box, precision) that no fused sweep covers
PER_OPERATOR = {("free-y-513", 0), ("wall-s2-513", 0)}

# box, and whether FP64 and FP32 solvers run it fused
BLOCKS = {
    "wall-513": (dict(nx=64, ny=513, nz=16, itimescheme=5, **{**WALL, "dt": 5e-4}), (True, True)),
    "wall-s1-513": (dict(nx=64, ny=513, nz=16, itimescheme=5, istret=1, **{**WALL, "dt": 5e-4}), (False, True)),
    "free-y1-wall-yn-513": (dict(nx=64, ny=513, nz=16, itimescheme=5, **{**WALL, "dt": 5e-4, "ncly1": 1}),
                            (False, True)),
    "free-y-257": (dict(nx=64, ny=257, nz=16, ncly1=1, nclyn=1, yly=math.pi, itimescheme=5), (True, True)),
    "wall-s2-257": (dict(nx=64, ny=257, nz=16, itimescheme=5, istret=2, **{**WALL, "dt": 5e-4}), (True, True)),
    "free-x-257": (dict(nx=257, ny=32, nz=16, nclx1=1, nclxn=1, xlx=math.pi, itimescheme=5), (False, True)),
    "free-x-513": (dict(nx=513, ny=16, nz=32, nclx1=1, nclxn=1, xlx=math.pi, itimescheme=3), (False, True)),
    "free-z-513": (dict(nx=33, ny=33, nz=513, itimescheme=5, **FREE), (False, True)),
    "free-17": (dict(nx=17, ny=17, nz=17, itimescheme=5, **FREE), (True, False)),
    "wall-s2-17": (dict(nx=64, ny=17, nz=16, itimescheme=5, istret=2, **WALL), (True, False)),
}


def _paths(kw, precision):
    """(path of a solver, path of one created with X3D_UNFUSED_MOMENTUM) on the context of kw."""
    out = []
    for unfused in (False, True):
        if unfused:
            os.environ["X3D_UNFUSED_MOMENTUM"] = "1"
        try:
            s = X.Solver(X.make_params(**kw), precision)
        finally:
            os.environ.pop("X3D_UNFUSED_MOMENTUM", None)
        out.append(s.fused)
        s.close()
    return tuple(out)


@pytest.mark.parametrize("name", list(CASES))
def test_path_of_compared_boxes(torch_cuda, name):
    kw = {"re": 1600.0, "dt": 0.004, **CASES[name]}
    X.init(X.make_params(**kw))
    try:
        for precision in (0, 1):
            assert _paths(kw, precision) == ((name, precision) not in PER_OPERATOR, False), precision
    finally:
        X.finalize()


@pytest.mark.parametrize("name", list(BLOCKS))
def test_block_shapes_match_per_operator(torch_cuda, name):
    box, fused = BLOCKS[name]
    kw = {"re": 1600.0, "dt": 0.004, **box}
    p = X.make_params(**kw)
    X.init(p)
    try:
        out = {}
        for precision in (0, 1):
            assert _paths(kw, precision) == (fused[precision], False)
            for unfused in (False, True):
                print(f"{name}, precision {precision}, unfused={unfused}", flush=True)
                out[precision, unfused] = _run(p, kw, precision, unfused, False)
        scale = max(float(a.abs().max()) for a in out[0, True][0])

        def err(a, b):
            return max(float((x - y).abs().max()) for x, y in zip(a[0], b[0])) / scale

        assert err(out[0, False], out[0, True]) <= 1e-11
        for a, b in zip(out[0, False][1], out[0, True][1]):
            assert math.isclose(a, b, rel_tol=1e-9, abs_tol=1e-9)
        e_f, e_u = err(out[1, False], out[0, True]), err(out[1, True], out[0, True])
        assert e_f <= 1.5 * e_u + 1e-7, (e_f, e_u)
    finally:
        X.finalize()


def test_lines_of_more_than_1024_points_stay_refused(torch_cuda):
    kw = dict(nx=64, ny=1025, nz=16, itimescheme=5, **WALL)
    X.init(X.make_params(**kw))
    try:
        for precision in (0, 1):
            assert _paths(kw, precision) == (False, False)
            s = X.Solver(X.make_params(**kw), precision)
            s.init_channel(0.1, 3)
            with pytest.raises(X.X3DError, match="line length > 1024"):
                s.step(1)
            s.close()
    finally:
        X.finalize()
