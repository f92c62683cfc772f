"""The square roots of constant weights where they ride in passes with the
prolongation, the fused vertical band and the restriction: B^(1/2) v = W A^(1/2) v
and B^(T/2) x = A^(1/2) W^T x on a stack of whole 64-k chunks and 16-column
tiles, with the vector kernel's default tiles and with the matrix cores pinned on
every pass kind, against the FP64 oracle's W and W^T (normwise relative error
1e-5 for operators, as in test_gpu_parity.py)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, field, oparams, relerr, to_dev

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


@pytest.mark.parametrize("engine", ["vector", "matrix cores"])
@pytest.mark.parametrize("h,hz,kw", [(6, 3, dict()), (6, 4, dict(lquart=True)), (3, 3, dict()),
                                     (6, 3, dict(mgbf_proc=8, mg_ampl02=0.4))])
def test_square_root_matches_oracle(engine, h, hz, kw):
    w = [0.7, 2.5]
    cfg = M.Config.for_grid(64, 48, 32, n_ens=2, gm=2, h=h, hz=hz, weights=w, **kw)
    with M.MGBF(cfg) as op:
        d = op.dims
        assert d.km_all % 64 == 0
        if engine != "vector":
            op.set_tiles({(g, k): (16, 16) for g in (1, 2) for k in range(4) if g < 2 or k == 0})
            assert all(op.tiles()[k][0] == 16 for k in ((1, 0), (1, 1), (1, 2), (1, 3), (2, 0)))
        P = oparams(cfg, d)
        sizes = [int(np.prod(d.gen_shape(g))) for g in (1, 2)]
        root = np.concatenate([np.full(n, np.sqrt(v)) for n, v in zip(sizes, w)])
        v = np.random.default_rng(8).standard_normal(d.mg_size).astype(np.float32)
        x = field(d.gen_shape(1), 9)
        assert relerr(op.apply(M.OP_BSQRT, to_dev(v)), O.w(P, root * v.astype(np.float64))) <= TOL_OP
        ref = root * O.wt(P, x.astype(np.float64)).ravel()
        assert relerr(op.apply(M.OP_BSQRTT, to_dev(x)).reshape(-1), ref) <= TOL_OP
