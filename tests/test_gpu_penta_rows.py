"""GPU parity of the pentadiagonal solves of the stretched Poisson equation
against the oracle at the sizes where their launch changes: lines whose
eliminated values fit in LDS and lines that do not (FP64: 62 rows are the
most, FP32: 124), tiles of lines that end inside a factor plane, few kz
planes, both numbers of systems per line.

Bar: 1e-12 relative in FP64 and 1e-5 in FP32, as for every stretched solve.
"""
import pytest

from oracle import x3d_oracle as O
from tests.helpers import rel_err, seeded_field

pytestmark = pytest.mark.gpu

CASES = [
    dict(nx=16, ny=17, nz=8, ncly1=2, nclyn=2, istret=2, beta=0.3),
    dict(nx=64, ny=17, nz=16, ncly1=2, nclyn=1, istret=3, beta=0.4),
    dict(nx=16, ny=129, nz=8, ncly1=2, nclyn=1, istret=3, beta=0.4),
    dict(nx=32, ny=257, nz=16, ncly1=1, nclyn=1, istret=1, beta=0.7),
    dict(nx=16, ny=257, nz=8, ncly1=2, nclyn=1, istret=3, beta=0.4),
]


@pytest.mark.parametrize("kw", CASES, ids=lambda k: f"s{k['istret']}_{k['nx']}x{k['ny']}x{k['nz']}")
def test_rows(torch_cuda, kw):
    import torch
    import incompact3d_amd as X
    p = O.Params(**kw)
    X.init(X.make_params(**kw))
    try:
        S = O.Schemes(p)
        f = seeded_field((p.nz, p.nym, p.nx), seed=5, lengths=(p.xlx, p.yly, p.zlz))
        f -= f.mean()
        ref = O.poisson(S, f)
        for tdt, bar in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
            d = torch.tensor(f, dtype=tdt, device="cuda")
            X.poisson(d)
            err = rel_err(d.double().cpu().numpy(), ref)
            assert err <= bar, f"{kw} {tdt}: {err:.3e}"
    finally:
        X.finalize()
