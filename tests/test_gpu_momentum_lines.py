"""GPU parity of the x momentum sweep where a wavefront takes the three
components of a line (more than 8192 lines) with the per-operator path
(X3D_UNFUSED_MOMENTUM at solver creation), for every number of points a lane
holds, plain AB3 and the general update, line counts that leave the last
wavefronts fewer lines, and the last count that keeps a wavefront a component.

FP64: the same operations in another order, 1e-11 of the velocity after 3
steps.  FP32 bulk: both against the FP64 run; the sweep's error is at most 1.5
times the other's, plus 1e-7."""
import math
import os

import pytest

pytestmark = pytest.mark.gpu

WALL = dict(xlx=4 * math.pi, yly=2.0, zlz=4 * math.pi / 3, ncly1=2, nclyn=2, re=500.0, dt=0.002, istret=2,
            beta=0.259, isecondder=5)
CASES = {
    "8192": dict(nx=64, ny=64, nz=128),
    "64": dict(nx=64, ny=128, nz=128),
    "128": dict(nx=128, ny=128, nz=128),
    "256-rk3": dict(nx=256, ny=64, nz=256, itimescheme=5),
    "512": dict(nx=512, ny=128, nz=128),
    "wall-64": dict(nx=64, ny=65, nz=128, itimescheme=5, **WALL),
    "wall-256": dict(nx=256, ny=129, nz=128, itimescheme=3, **WALL),
}


def _run(X, p, kw, precision, unfused):
    if unfused:
        os.environ["X3D_UNFUSED_MOMENTUM"] = "1"
    try:
        s = X.Solver(p, precision)
    finally:
        os.environ.pop("X3D_UNFUSED_MOMENTUM", None)
    if "ncly1" in kw:
        s.init_channel(0.1, 3)
        s.set_forcing(1, 2.0 / 3.0)
        s.set_rotation(0.12, 2)
    else:
        s.init_tgv()
    s.step(3)
    u = [t.clone() for t in s.velocity()]
    s.close()
    return u


@pytest.mark.parametrize("name", list(CASES))
def test_matches_per_operator(torch_cuda, name):
    import incompact3d_amd as X
    kw = {"re": 1600.0, "dt": 0.004, **CASES[name]}
    p = X.make_params(**kw)
    X.init(p)
    try:
        out = {(precision, unfused): _run(X, p, kw, precision, unfused)
               for precision in (0, 1) for unfused in (False, True)}
    finally:
        X.finalize()
    ref = out[0, True]
    scale = max(float(a.abs().max()) for a in ref)

    def err(a):
        return max(float((x - y).abs().max()) for x, y in zip(a, ref)) / scale

    assert err(out[0, False]) <= 1e-11
    assert err(out[1, False]) <= 1.5 * err(out[1, True]) + 1e-7
