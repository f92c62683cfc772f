"""Half-widths 9 and 10 with the vertical band fused into the last pass: whole
columns in a wave, bands of half-width 4, 6 and 8, either transfer stencil, disc
and product taps, 4 and 2 columns a lane, against the FP64 oracle (normwise
relative error 1e-5 for operators, as in test_gpu_parity.py). No vertical pass
runs beside it."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, field, oparams, relerr, sync, to_dev

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


@pytest.mark.parametrize("h", [9, 10])
@pytest.mark.parametrize("lm,n_ens,hz,kw", [(32, 2, 3, dict()), (16, 4, 2, dict(lquart=True)), (64, 1, 4, dict()),
                                            (8, 8, 3, dict(mgbf_proc=8, p=1)),
                                            (32, 2, 4, dict(mgbf_proc=8, p=1, lquart=True))])
def test_band_fuses_at_wide_filters(h, lm, n_ens, hz, kw):
    kw = dict(kw)
    if kw.get("mgbf_proc") == 8:   # the factors whose product filter reaches h
        kw["mg_ampl02"] = {9: 0.235, 10: 0.215}[h]
    cfg = M.Config.for_grid(54, 46, lm, n_ens=n_ens, gm=2, h=h, hz=hz, weights=[1.0, 0.6], **kw)
    with M.MGBF(cfg) as op:
        d = op.dims
        if kw.get("mgbf_proc") == 8:
            assert d.ntaps2 == (2 * h + 1) ** 2
        x = field(d.gen_shape(1), h)
        ref = O.wawt(oparams(cfg, d), x.astype(np.float64))
        for ti in (4, 2):
            for tj in (5, 23):
                op.set_tiles({(1, 2): (ti, tj)})
                op.timers(True)
                y = op.filtering_procedure(to_dev(x))
                sync()
                t = op.read_timers()
                op.timers(False)
                assert t["vfilt"][1] == 0 and t["vfiltT"][1] == 0
                assert relerr(y, ref) <= TOL_OP, (ti, tj)
