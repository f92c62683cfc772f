"""Per-point aspects without the rows of the transposed matrix
(MGBF_ASPECT_SCATTER=1, and where the device has no room for them): F^T from the
taps of F, with constant and per-point weights, against the FP64 oracle at the
tolerances of test_gpu_aspect_tiles.py, and the device memory of one set of
weights instead of two."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, relerr
from test_oracle import aspect_field

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

DEV = torch.device("cuda:0")


def _context(n, m, lm, h, gm=2):
    cfg = M.Config.for_grid(n, m, lm, gm=gm, h=h, hz=1)
    P = O.OracleParams(nx=n, ny=m, K=lm, lm=lm, nvcol=1, hx=h, hy=h, hz=1, p=2, gm=gm, ampl01=cfg.mg_ampl01,
                       ampl02=cfg.mg_ampl02)
    return cfg, P, aspect_field(n, m, (h + 1) ** 2 / 8.0 / 1.55, seed=n + m + h)


@pytest.mark.parametrize("n,m,lm,h", [(10, 8, 65, 2), (22, 18, 64, 4), (12, 14, 66, 6), (30, 16, 4, 8),
                                      (20, 42, 63, 10)])
def test_transpose_from_the_taps_matches_oracle(n, m, lm, h, monkeypatch):
    monkeypatch.setenv("MGBF_ASPECT_SCATTER", "1")
    cfg, P, asp = _context(n, m, lm, h)
    with M.MGBF(cfg) as op:
        op.set_aspect(1, asp)
        x = np.random.default_rng(h).standard_normal(op.dims.gen_shape(1)).astype(np.float32)
        xd = torch.from_numpy(x).to(DEV)
        for stage, adj in ((M.STAGE_F, False), (M.STAGE_FT, True)):
            ref = O.radial_aspect(P, asp, x.astype(np.float64), adjoint=adj)
            y = op.stage(stage, 1, xd).cpu().double().numpy()
            assert np.max(np.abs(y - ref)) <= (7.7e-6 if adj else 1.9e-6) * np.max(np.abs(x)), stage


@pytest.mark.parametrize("field", [False, True])
def test_operator_is_the_same_with_and_without_the_rows(field, monkeypatch):
    cfg, _, asp = _context(40, 36, 33, 5)
    out = []
    for scatter in ("0", "1"):
        monkeypatch.setenv("MGBF_ASPECT_SCATTER", scatter)
        with M.MGBF(cfg) as op:
            g = torch.Generator(device="cuda").manual_seed(6)
            x = torch.randn(op.field_shape(), generator=g, device="cuda")
            keep = [0.5 + torch.rand(op.dims.gen_shape(i), generator=g, device="cuda") for i in (1, 2)]
            if field:
                for i, f in enumerate(keep, start=1):
                    op.set_weights(i, field=f)
            op.set_aspect(1, asp)
            out.append(op.filtering_procedure(x).cpu().double().numpy())
            torch.cuda.synchronize()
    assert relerr(out[1], out[0]) <= TOL_OP


def test_half_the_memory_without_the_rows(monkeypatch):
    n, m, h = 1024, 1024, 6
    taps = 4 * n * m * (2 * h + 1) ** 2   # 709 MB
    cfg = M.Config.for_grid(n, m, 2, gm=1, h=h, hz=1)
    asp = np.zeros((m, n, 3))
    asp[..., :2] = 0.8 * cfg.mg_ampl02
    used = []
    for scatter in ("0", "1"):
        monkeypatch.setenv("MGBF_ASPECT_SCATTER", scatter)
        with M.MGBF(cfg) as op:
            free = torch.cuda.mem_get_info()[0]
            op.set_aspect(1, asp)
            used.append(free - torch.cuda.mem_get_info()[0])
            op.set_aspect(1, None)
            assert abs(free - torch.cuda.mem_get_info()[0]) < 0.1 * taps
    assert abs(used[0] - 2 * taps) < 0.1 * taps and abs(used[1] - taps) < 0.1 * taps
