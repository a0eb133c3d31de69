"""GPU parity of the single-operator kernels on anchored segments (free-slip
and no-slip ends, and periodic lines that are no whole number of segments):
every operator and direction at the line lengths where the segments change
shape, against the oracle.

Lengths, for segments of 8 FP64 and 16 FP32 rows: 16 and 17 (two FP64
segments, and the shortest with rows between), 31, 32 and 33 (the same in
FP32, and one row either side), 40, 47, 100, 130; for y also the longest
full-row block of each precision and one more, where the segments grow by a
row (512, 513).  The other two extents are odd, so that no tile of lines is
full.  Shorter and foreign-coefficient lines stay on the other kernels and are
covered by the tests of the derivative entries.

Tolerances as for those entries: FP64 1e-12 relative to the largest value,
FP32 2e-5."""
import numpy as np
import pytest

from oracle import x3d_oracle as O
from tests.helpers import seeded_field

pytestmark = pytest.mark.gpu

X = pytest.importorskip("incompact3d_amd")

TOL = {"f64": 1e-12, "f32": 2e-5}
OPS = ("der1", "der2", "dervp", "intervp", "derpv", "interpv")
LENGTHS = [(ax, n, bc) for ax in "xyz" for n in (16, 17, 31, 32, 33, 40, 47, 100, 130)
           for bc in ((0, 0), (1, 1), (2, 2))]
LENGTHS += [("y", n, bc) for n in (33, 47) for bc in ((1, 2), (2, 1))]
LENGTHS += [("y", n, bc) for n in (512, 513) for bc in ((1, 1), (2, 2))]


def _grid(axis, n):
    g = {"x": 9, "y": 11, "z": 13}
    g[axis] = n
    return g


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("axis,n,bc", LENGTHS, ids=lambda v: str(v).replace(" ", ""))
def test_operators(torch_cuda, axis, n, bc, dtype):
    import torch
    dt = torch.float64 if dtype == "f64" else torch.float32
    g = _grid(axis, n)
    kw = dict(nx=g["x"], ny=g["y"], nz=g["z"])
    kw.update({f"ncl{axis}1": bc[0], f"ncl{axis}n": bc[1]})
    p = X.make_params(**kw)
    X.init(p)
    try:
        S = O.Schemes(O.Params(**kw))
        d = "xyz".index(axis)
        nm = n if bc[0] == 0 else n - 1
        fns = dict(der1=O.der1, der2=O.der2, dervp=O.dervp, intervp=O.intervp, derpv=O.derpv, interpv=O.interpv)
        for op in OPS:
            for par in (0, 1):
                if bc[0] != 0 and par == 0 and op in ("intervp", "derpv", "interpv"):
                    continue
                shape = [g["z"], g["y"], g["x"]]
                if op.endswith("pv"):
                    shape[2 - d] = nm
                out = list(shape)
                if op.endswith("vp"):
                    out[2 - d] = nm
                elif op.endswith("pv"):
                    out[2 - d] = n
                f = seeded_field(tuple(shape), 7 * n + par)
                u = torch.tensor(f, dtype=dt, device="cuda")
                t = torch.full(out, float("nan"), dtype=dt, device="cuda")
                print(f"{op} {axis} {n} {bc} parity {par} {dtype}", flush=True)
                X.line_op_async(d, op, par, u, t)
                X.synchronize()
                ref = fns[op](S, u.double().cpu().numpy(), axis, par)
                got = t.double().cpu().numpy()
                assert np.isfinite(got).all(), (op, par)
                err = np.abs(got - ref).max() / np.abs(ref).max()
                assert err <= TOL[dtype], (op, par, err)
    finally:
        X.finalize()


@pytest.mark.parametrize("precision", [0, 1])
def test_fused_operand_and_epilogue(torch_cuda, precision):
    """The product input, factor and accumulator of the per-operator step
    (EPI forms) on free-slip y lines, through two steps of it against the
    oracle's."""
    import os
    kw = dict(nx=64, ny=33, nz=16, re=1600.0, dt=0.004, itimescheme=3, ncly1=1, nclyn=1, yly=np.pi)
    p = X.make_params(**kw)
    X.init(p)
    try:
        po = O.Params(**kw)
        S = O.Schemes(po)
        st = O.tgv_state(po)
        for _ in range(2):
            O.step(S, st)
        os.environ["X3D_UNFUSED_MOMENTUM"] = "1"
        try:
            s = X.Solver(p, precision)
        finally:
            os.environ.pop("X3D_UNFUSED_MOMENTUM", None)
        s.init_tgv()
        s.step(2)
        tol = 1e-11 if precision == 0 else 2e-5
        for a, b in zip(s.velocity(), (st.ux, st.uy, st.uz)):
            assert np.abs(a.cpu().numpy() - b).max() <= tol * max(1.0, np.abs(b).max())
        s.close()
    finally:
        X.finalize()
