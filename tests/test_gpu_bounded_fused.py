"""GPU parity of the fused sweeps along bounded directions and of RK3 on them
(bounded.hip, and the general velocity update of momentum.hip and
projection.hip) against the per-operator path, which every one of these boxes
can also take (X3D_UNFUSED_MOMENTUM at solver creation) and which the other
tests hold against the oracle.

Boxes: every kind of end and pairing the solver accepts in each direction,
stretched walls, AB3 and RK3, forcing and rotation, LES; line lengths at the
edges of the segments (33 points: one row left between the end segments of 8
or 16, and the 32-point pressure lines: two FP32 segments and nothing
between; 65, 129) beside periodic lines of other lengths.

FP64: the two paths do the same operations in another order; 1e-11 of the
velocity after 4 steps.  FP32 bulk: both are measured against the FP64 run;
the fused path's error is at most 1.5 times the other's, plus 1e-7."""
import math
import os

import pytest

pytestmark = pytest.mark.gpu

X = pytest.importorskip("incompact3d_amd")

FREE = dict(nclx1=1, nclxn=1, ncly1=1, nclyn=1, nclz1=1, nclzn=1, xlx=math.pi, yly=math.pi, zlz=math.pi)
WALL = dict(xlx=4 * math.pi, yly=2.0, zlz=4 * math.pi / 3, ncly1=2, nclyn=2, re=500.0, dt=0.002)
CASES = {
    "free-33-rk3": dict(nx=33, ny=33, nz=33, itimescheme=5, **FREE),
    "free-65x33x129-ab3": dict(nx=65, ny=33, nz=129, itimescheme=3, **FREE),
    "free-x": dict(nx=33, ny=64, nz=16, nclx1=1, nclxn=1, xlx=math.pi, itimescheme=5),
    "free-y": dict(nx=64, ny=65, nz=32, ncly1=1, nclyn=1, yly=math.pi, itimescheme=5),
    "free-xy": dict(nx=65, ny=33, nz=32, nclx1=1, nclxn=1, ncly1=1, nclyn=1, xlx=math.pi, yly=math.pi,
                    itimescheme=3),
    "periodic-rk3": dict(nx=128, ny=32, nz=16, itimescheme=5),
    "wall-rk3": dict(nx=64, ny=33, nz=32, itimescheme=5, **WALL),
    "wall-s2-rk3": dict(nx=64, ny=65, nz=16, itimescheme=5, isecondder=5, istret=2, **WALL),
    "wall-s1-ab3": dict(nx=128, ny=33, nz=16, itimescheme=3, isecondder=5, istret=1, **WALL),
    "wall-s3-256": dict(nx=256, ny=129, nz=16, itimescheme=5, istret=3, **WALL),
    "wall-free-x": dict(nx=33, ny=33, nz=32, itimescheme=5, **{**WALL, "nclx1": 1, "nclxn": 1}),
    "wall-free-yn": dict(nx=64, ny=33, nz=16, itimescheme=5, **{**WALL, "nclyn": 1}),
    # segments one row longer in x; blocks over 512 threads
    "free-x-129": dict(nx=129, ny=32, nz=16, nclx1=1, nclxn=1, xlx=math.pi, itimescheme=5),
    "free-y-513": dict(nx=64, ny=513, nz=16, ncly1=1, nclyn=1, yly=math.pi, itimescheme=5),
    "wall-s2-513": dict(nx=64, ny=513, nz=16, itimescheme=3, istret=2, isecondder=5, **{**WALL, "dt": 5e-4}),
    "free-y1-wall-yn": dict(nx=64, ny=65, nz=16, itimescheme=3, **{**WALL, "ncly1": 1}),
}


def _run(p, kw, precision, unfused, les):
    if unfused:
        os.environ["X3D_UNFUSED_MOMENTUM"] = "1"
    try:
        s = X.Solver(p, precision)
    finally:
        os.environ.pop("X3D_UNFUSED_MOMENTUM", None)
    walls = 2 in (kw.get("ncly1"), kw.get("nclyn"))
    if walls:
        s.init_channel(0.1, 3)
        if kw["itimescheme"] == 5:
            s.set_forcing(1, 2.0 / 3.0)
        else:
            s.set_forcing(2, 0.01)
        s.set_rotation(0.12, 3)
    else:
        s.init_tgv()
    if les:
        s.set_les(1, cs=0.17, iconserv=1)
    s.step(4)
    u = [t.clone() for t in s.velocity()]
    d = s.divu_stats()
    s.close()
    return u, d


@pytest.mark.parametrize("name", list(CASES))
def test_fused_matches_per_operator(torch_cuda, name):
    kw = {"re": 1600.0, "dt": 0.004, **CASES[name]}
    p = X.make_params(**kw)
    les = name in ("free-33-rk3", "free-x", "periodic-rk3")
    X.init(p)
    try:
        out = {}
        for precision in (0, 1):
            for unfused in (False, True):
                print(f"{name}, precision {precision}, unfused={unfused}", flush=True)
                out[precision, unfused] = _run(p, kw, precision, unfused, les)
        scale = max(float(a.abs().max()) for a in out[0, True][0])

        def err(a, b):
            return max(float((x - y).abs().max()) for x, y in zip(a[0], b[0])) / scale

        assert err(out[0, False], out[0, True]) <= 1e-11
        for a, b in zip(out[0, False][1], out[0, True][1]):
            assert abs(a - b) <= 1e-9 * max(1.0, abs(b))
        e_f, e_u = err(out[1, False], out[0, True]), err(out[1, True], out[0, True])
        assert e_f <= 1.5 * e_u + 1e-7, (e_f, e_u)
    finally:
        X.finalize()
