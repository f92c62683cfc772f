"""Vertical bands over columns that fit no power of two (whole columns in LDS
to 128 levels that 4 does not divide; a value a thread else) against the
FP64 oracle: Vf and Vf^T at each half-width, on aligned and unaligned fields,
and their product, of twice the half-width, at the end of W A W^T with constant
weights. Normwise relative errors as in test_gpu_parity.py: 2e-6 for stages,
1e-5 for operators."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, TOL_STAGE, field, oparams, relerr, to_dev

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


@pytest.mark.parametrize("lm,hz", [(5, 2), (11, 4), (13, 1), (14, 5), (17, 8), (33, 2), (65, 3), (66, 4), (65, 7),
                                   (90, 6), (126, 8), (127, 4), (127, 9), (129, 3), (130, 8)])
def test_bands_match_oracle(lm, hz):
    cfg = M.Config.for_grid(24, 20, lm, n_ens=2, gm=1, h=3, hz=hz)
    with M.MGBF(cfg) as op:
        d = op.dims
        P = oparams(cfg, d)
        x = field(d.gen_shape(1), lm + hz)
        x64 = x.astype(np.float64)
        xd = to_dev(x)
        off = torch.empty(xd.numel() + 1, device="cuda")[1:].view(xd.shape)   # 4 bytes past a 16-byte boundary
        off.copy_(xd)
        for stage, adj in ((M.STAGE_VF, False), (M.STAGE_VFT, True)):
            ref = O.vertical(P, x64, adjoint=adj)
            assert relerr(op.stage(stage, 1, xd), ref) <= TOL_STAGE, stage
            assert relerr(op.stage(stage, 1, off, out=torch.empty_like(off)), ref) <= TOL_STAGE, stage
        # a unit value reaches hz levels and no further
        for L in (0, lm // 2, lm - 1):
            e = torch.zeros(d.gen_shape(1))
            e.view(-1, lm)[:, L] = 1.0
            for stage in (M.STAGE_VF, M.STAGE_VFT):
                y = op.stage(stage, 1, e.cuda()).cpu().view(-1, lm)
                assert y[:, L].abs().min() > 0.0
                assert not y[:, : max(0, L - hz)].any() and not y[:, L + hz + 1:].any()


@pytest.mark.parametrize("lm,hz", [(13, 3), (65, 4), (66, 4), (127, 4), (65, 5), (33, 3)])
def test_product_band_matches_oracle(lm, hz):
    cfg = M.Config.for_grid(28, 24, lm, n_ens=1, gm=2, h=4, hz=hz, weights=[1.0, 0.6])
    with M.MGBF(cfg) as op:
        d = op.dims
        x = field(d.gen_shape(1), lm)
        assert relerr(op.filtering_procedure(to_dev(x)), O.wawt(oparams(cfg, d), x.astype(np.float64))) <= TOL_OP
