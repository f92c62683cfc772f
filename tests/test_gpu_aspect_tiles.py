"""The per-point aspect kernel at the edges of its 4 x 4 tiles, for every
half-width from 2: F and F^T against the FP64 oracle. The (2H+1)^2 weights of an
output of F are non-negative with unit sum, those of F^T have a sum below 4
(at most 4 mirror images of a tap); an FP32 sum of up to 441 terms of unit
total weight, rounded at random, stays well within 32 x 2^-24 = 1.9e-6 of the
largest input, 4 times that for F^T."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_oracle import aspect_field

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

DEV = torch.device("cuda:0")


def _context(n, m, lm, h):
    cfg = M.Config.for_grid(n, m, lm, gm=2, h=h, hz=1)
    P = O.OracleParams(nx=n, ny=m, K=lm, lm=lm, nvcol=1, hx=h, hy=h, hz=1, p=2, gm=2, ampl01=cfg.mg_ampl01,
                       ampl02=cfg.mg_ampl02)
    asp = aspect_field(n, m, (h + 1) ** 2 / 8.0 / 1.55, seed=n + m + h)
    return cfg, P, asp


@pytest.mark.parametrize("n,m,lm,h", [(10, 8, 65, 2), (14, 10, 5, 3), (22, 18, 64, 4), (16, 12, 3, 5),
                                      (12, 14, 66, 6), (18, 14, 9, 7), (30, 16, 4, 8), (18, 22, 6, 9),
                                      (20, 42, 63, 10)])
def test_aspect_tiles_match_oracle(n, m, lm, h):
    cfg, P, asp = _context(n, m, lm, h)
    with M.MGBF(cfg) as op:
        op.set_aspect(1, asp)
        x = np.random.default_rng(h).standard_normal(op.dims.gen_shape(1)).astype(np.float32)
        xd = torch.from_numpy(x).to(DEV)
        for stage, adj in ((M.STAGE_F, False), (M.STAGE_FT, True)):
            y = op.stage(stage, 1, xd).cpu().double().numpy()
            ref = O.radial_aspect(P, asp, x.astype(np.float64), adjoint=adj)
            assert np.max(np.abs(y - ref)) <= (7.7e-6 if adj else 1.9e-6) * np.max(np.abs(x)), (stage, h)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_stay_inside_the_ellipses(bad):
    # an output without a weight on the bad point is what it is without it
    n, m, lm, h = 40, 36, 6, 6
    cfg, P, asp = _context(n, m, lm, h)
    with M.MGBF(cfg) as op:
        op.set_aspect(1, asp)
        x = torch.randn(op.field_shape(), generator=torch.Generator().manual_seed(1)).to(DEV)
        xb = x.clone()
        xb[17, 19, 3] = bad
        e = np.zeros((m, n, lm))
        e[17, 19, 3] = 1.0
        for stage, adj in ((M.STAGE_F, False), (M.STAGE_FT, True)):
            y, yb = op.stage(stage, 1, x).cpu(), op.stage(stage, 1, xb).cpu()
            hit = torch.from_numpy(O.radial_aspect(P, asp, e, adjoint=adj) != 0.0)
            assert not torch.isfinite(yb[hit]).any() and 20 < int(hit.sum()) < 169
            assert torch.isfinite(yb[~hit]).all()
            assert (yb - y)[~hit].abs().max() <= 2e-6
