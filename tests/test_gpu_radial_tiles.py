"""The vector radial kernel at the edges of its layouts: stacks that are no
multiple of 64 k (laid end to end over the column tiles, or 64-k chunks with
idle lanes at the end), column tiles that are not full, tiles of 1, 2, 3 and
all rows, every half-width and kind of taps, with each epilogue, against the
FP64 oracle. Tolerance as in test_gpu_parity.py: normwise relative error 1e-5
for operators."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M
from test_gpu_parity import TOL_OP, field, oparams, relerr, sync, to_dev

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

FAST = dict(mgbf_proc=8, p=1, mg_ampl02=2.0)      # product taps of half-width 1
FAST6 = dict(mgbf_proc=8, mg_ampl02=0.4)          # half-width 6

CASES = [
    # nx, ny, lm, n_ens, gm, h, hz, options
    (32, 24, 1, 1, 2, 6, 0, dict(l_vertical_filter=False)),     # 64 tiles a wave
    (26, 20, 2, 1, 2, 4, 1, dict()),                            # 32
    (44, 28, 7, 3, 3, 3, 2, dict()),                            # 21 k: 3 tiles and a bit
    (48, 40, 32, 1, 3, 6, 3, dict()),                           # 2 tiles a wave
    (40, 32, 8, 3, 2, 6, 3, dict()),                            # 2 tiles and two thirds
    (48, 40, 16, 4, 2, 8, 4, dict()),                           # the band (8) fused: 4 columns a wave
    (36, 28, 8, 8, 2, 4, 3, dict()),                            # the band (6), 8 columns a wave
    (36, 52, 33, 1, 2, 5, 3, dict()),                           # more than half a wave
    (52, 36, 65, 1, 3, 6, 3, dict()),                           # one more than a wave
    (40, 32, 127, 1, 2, 4, 3, dict()),                          # chunks with one idle lane
    (40, 40, 65, 2, 2, 7, 3, dict()),                           # 130: end to end
    (72, 56, 12, 2, 3, 9, 3, dict()),
    (80, 96, 5, 5, 3, 10, 2, dict()),
    (48, 40, 32, 1, 3, 6, 3, dict(lquart=True)),
    (52, 36, 65, 1, 3, 3, 3, dict(lquart=True)),
    (44, 40, 65, 1, 3, 6, 3, FAST),                             # restriction beside half-width 1
    (44, 40, 33, 1, 3, 6, 2, dict(FAST, lquart=True)),
    (40, 48, 16, 3, 3, 6, 3, FAST6),
    (40, 48, 16, 3, 3, 6, 3, dict(FAST6, lquart=True)),
]


def _heights(op, tj):
    """Every pass at tj rows a wave (even with the restriction)."""
    tiles = {}
    for g in range(1, op.dims.gm + 1):
        h = min(tj, op.dims.gen_shape(g)[0])
        for kind, ti in ((0, 2), (1, 4), (2, 4), (3, 4)):
            tiles[(g, kind)] = (ti, max(2, h + (h & 1)) if kind == 3 else h)
    op.set_tiles(tiles)


@pytest.mark.parametrize("nx,ny,lm,n_ens,gm,h,hz,kw", CASES)
def test_layouts_match_oracle(nx, ny, lm, n_ens, gm, h, hz, kw):
    cfg = M.Config.for_grid(nx, ny, lm, n_ens=n_ens, gm=gm, h=h, hz=hz, weights=[1.0, 0.6, 0.3], **kw)
    with M.MGBF(cfg) as op:
        d = op.dims
        P = oparams(cfg, d)
        x = field(d.gen_shape(1), 11)
        v = np.random.default_rng(12).standard_normal(d.mg_size).astype(np.float32)
        ref = O.wawt(P, x.astype(np.float64)), O.wt(P, x.astype(np.float64)), O.w(P, v.astype(np.float64))
        for tj in (None, 1, 3, ny):
            if tj is not None:
                _heights(op, tj)
            for code, arg, r in ((M.OP_WAWT, x, ref[0]), (M.OP_WT, x, ref[1]), (M.OP_W, v, ref[2])):
                assert relerr(op.apply(code, to_dev(arg)), r) <= TOL_OP, (code, tj)


@pytest.mark.parametrize("lm,n_ens", [(33, 1), (32, 1), (127, 1), (64, 1)])
def test_weight_fields_in_every_layout(lm, n_ens):
    cfg = M.Config.for_grid(52, 36, lm, n_ens=n_ens, gm=3, h=6, hz=3)
    with M.MGBF(cfg) as op:
        d = op.dims
        rng = np.random.default_rng(5)
        wf = [(0.5 + rng.random(d.gen_shape(g))).astype(np.float32) for g in (1, 2, 3)]
        keep = [to_dev(w) for w in wf]
        for g, w in enumerate(keep, start=1):
            op.set_weights(g, field=w)
        x = field(d.gen_shape(1), 21)
        ref = O.wawt(oparams(cfg, d), x.astype(np.float64), wfield=[w.astype(np.float64) for w in wf])
        for tj in (None, 1, 36):
            if tj is not None:
                _heights(op, tj)
            assert relerr(op.filtering_procedure(to_dev(x)), ref) <= TOL_OP, tj
        sync()


@pytest.mark.parametrize("hx,hy,lquart", [(4, 6, False), (7, 3, True)])
def test_box_taps_match_oracle(hx, hy, lquart):
    # unequal halos: the taps run as a box of the larger half-width
    cfg = M.Config.for_grid(44, 60, 33, gm=3, h=min(hx, hy), hz=3, lquart=lquart)
    cfg.hx, cfg.hy = hx, hy
    with M.MGBF(cfg) as op:
        d = op.dims
        x = field(d.gen_shape(1), 31)
        ref = O.wawt(oparams(cfg, d), x.astype(np.float64))
        for tj in (None, 1, 60):
            if tj is not None:
                _heights(op, tj)
            assert relerr(op.filtering_procedure(to_dev(x)), ref) <= TOL_OP, tj


@pytest.mark.parametrize("km2,h", [(1, 6), (2, 4), (3, 6), (70, 3)])
def test_two_dimensional_variables_behind_three_dimensional_ones(km2, h):
    cfg = M.Config.for_grid(52, 36, 16, gm=3, h=h, hz=2, mgbf_proc=4, km3=2, km2=km2)
    with M.MGBF(cfg) as op:
        d = op.dims
        x = field(d.gen_shape(1), 41)
        y = op.filtering_procedure(to_dev(x))
        assert relerr(y, O.wawt(oparams(cfg, d), x.astype(np.float64))) <= TOL_OP


def test_default_tiles_fill_the_chip_in_whole_rounds():
    # 384 x 384 x 320: 480 waves a row of tiles, 96 rows give 1920 of the 2048
    # that fit; 24 x 24 x 32 has too few waves for 4 columns a lane
    with M.MGBF(M.Config.for_grid(384, 384, 32, n_ens=10, gm=4, h=6, hz=3)) as op:
        assert op.tiles()[(1, 0)] == (4, 96) and op.tiles()[(1, 3)] == (4, 96)
    with M.MGBF(M.Config.for_grid(192, 192, 32, gm=4, h=6, hz=3)) as op:
        assert op.tiles()[(4, 0)][0] == 2 and op.tiles()[(4, 3)][0] == 4
