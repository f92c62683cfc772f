"""Tiles of 2 columns a lane on every pass kind that takes them (plain, with
either prolongation, with the vertical band), for disc, product and box taps, on
column counts that leave the last tile partial: against the FP64 oracle,
normwise relative error 1e-5 for operators as in test_gpu_parity.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, field, oparams, relerr, to_dev

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

FAST6 = dict(mgbf_proc=8, mg_ampl02=0.4)


@pytest.mark.parametrize("nx,ny,lm,n_ens,h,hz,kw", [
    (42, 30, 32, 2, 6, 3, dict()),                    # band of half-width 6
    (42, 30, 32, 2, 6, 2, dict(lquart=True)),         # 4, quadratic transfer
    (38, 26, 16, 4, 3, 4, dict()),                    # 8
    (46, 34, 64, 1, 8, 3, dict(lquart=True)),
    (42, 38, 8, 8, 6, 3, FAST6),
    (42, 38, 8, 8, 6, 4, dict(FAST6, lquart=True)),
    (40, 28, 33, 1, 5, 3, dict(lquart=True)),         # laid end to end, band of its own
    (44, 28, 65, 1, 4, 3, dict()),
])
def test_two_columns_match_oracle(nx, ny, lm, n_ens, h, hz, kw):
    cfg = M.Config.for_grid(nx, ny, lm, n_ens=n_ens, gm=2, h=h, hz=hz, weights=[1.0, 0.6], **kw)
    with M.MGBF(cfg) as op:
        d = op.dims
        x = field(d.gen_shape(1), 3)
        ref = O.wawt(oparams(cfg, d), x.astype(np.float64))
        for tj in (3, 10):
            op.set_tiles({(g, kind): (2, tj) for g in (1, 2) for kind in (0, 1, 2)})
            assert all(op.tiles()[(g, kind)] == (2, tj) for g in (1, 2) for kind in (0, 1, 2))
            assert relerr(op.filtering_procedure(to_dev(x)), ref) <= TOL_OP, tj


@pytest.mark.parametrize("lquart", [False, True])
def test_two_columns_of_a_box_match_oracle(lquart):
    cfg = M.Config.for_grid(42, 30, 32, gm=2, h=4, hz=3, lquart=lquart)
    cfg.hx, cfg.hy = 4, 6
    with M.MGBF(cfg) as op:
        d = op.dims
        x = field(d.gen_shape(1), 4)
        ref = O.wawt(oparams(cfg, d), x.astype(np.float64))
        op.set_tiles({(g, kind): (2, 7) for g in (1, 2) for kind in (0, 1)})
        assert relerr(op.filtering_procedure(to_dev(x)), ref) <= TOL_OP
