"""The rows of the transposed aspect matrix where they are more than one launch
of a weight a thread takes (its threads stride over them). F^T on 400 x 300
points of half-width 6, 20.3 million weights, against the FP64 oracle: weights
below 4 in sum a row, an FP32 sum of at most 4 x 169 terms, 7.7e-6 of the
largest input, as on the small grids of test_gpu_aspect_tiles.py. And beyond
2^32 weights, where a launch of a thread each loses all but the remainder: F
and F^T as transposes of one another in FP64 inner products, whose FP32 terms'
errors (2e-6 each, of random sign) average out over 10^7 points to well below
1e-7 of |Fx| |v|."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_oracle import aspect_field

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


def test_transposed_rows_of_a_large_grid():
    n, m, lm, h = 400, 300, 2, 6
    cfg = M.Config.for_grid(n, m, lm, gm=2, h=h, hz=1)
    P = O.OracleParams(nx=n, ny=m, K=lm, lm=lm, nvcol=1, hx=h, hy=h, hz=1, p=2, gm=2, ampl01=cfg.mg_ampl01,
                       ampl02=cfg.mg_ampl02)
    asp = aspect_field(n, m, (h + 1) ** 2 / 8.0 / 1.55, seed=4)
    with M.MGBF(cfg) as op:
        op.set_aspect(1, asp)
        x = np.random.default_rng(2).standard_normal(op.dims.gen_shape(1)).astype(np.float32)
        y = op.stage(M.STAGE_FT, 1, torch.from_numpy(x).cuda()).cpu().double().numpy()
        ref = O.radial_aspect(P, asp, x.astype(np.float64), adjoint=True)
        assert np.max(np.abs(y - ref)) <= 7.7e-6 * np.max(np.abs(x))


def test_transposed_rows_beyond_two_to_the_32_weights():
    n, m, h = 3136, 3120, 10
    cfg = M.Config.for_grid(n, m, 2, gm=1, h=h, hz=1)
    asp = np.zeros((m, n, 3))
    asp[..., 0], asp[..., 1], asp[..., 2] = 0.9 * cfg.mg_ampl02, 0.8 * cfg.mg_ampl02, 0.3
    assert n * m * (2 * h + 1) ** 2 > 2 ** 32
    with M.MGBF(cfg) as op:
        op.set_aspect(1, asp)
        g = torch.Generator(device="cuda").manual_seed(3)
        x = torch.randn(op.field_shape(), generator=g, device="cuda")
        v = torch.randn(op.field_shape(), generator=g, device="cuda")
        fx = op.stage(M.STAGE_F, 1, x).double()
        ftv = op.stage(M.STAGE_FT, 1, v).double()
        a, b = (fx * v.double()).sum().item(), (x.double() * ftv).sum().item()
        assert abs(a - b) <= 1e-7 * fx.norm().item() * v.double().norm().item()
