"""Which path the solvers of test_gpu_bounded_fused.py take: where its two runs
were the same path, its comparison says nothing.  And that comparison, with the
path asserted, for the block shapes that its boxes leave out.

FP64 blocks of 513-point lines with three coefficient tables (free-slip ends),
or two and the metrics of a stretched mesh, do not fit in 64 KB of LDS, and
those boxes run one launch per derivative; uniform no-slip walls fit, with 65
segments of 8 points on 8 lines (FP32: 31 of 17 on 32).  The tolerances are that
file's: 1e-11 of the velocity after 4 steps in FP64; in FP32 bulk at most 1.5
times the per-operator path's error, plus 1e-7."""
import math
import os

import pytest

from test_gpu_bounded_fused import CASES, WALL, _run

pytestmark = pytest.mark.gpu

X = pytest.importorskip("incompact3d_amd")

# (box, precision) that no fused sweep covers
PER_OPERATOR = {("free-y-513", 0), ("free-y-513", 1), ("wall-s2-513", 0), ("wall-s2-513", 1)}

BLOCKS = {
    "wall-513": dict(nx=64, ny=513, nz=16, itimescheme=5, **{**WALL, "dt": 5e-4}),
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
    kw = {"re": 1600.0, "dt": 0.004, **BLOCKS[name]}
    p = X.make_params(**kw)
    X.init(p)
    try:
        out = {}
        for precision in (0, 1):
            assert _paths(kw, precision) == (True, False)
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
