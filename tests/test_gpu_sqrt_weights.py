"""B^(1/2) = W A^(1/2) and its transpose with constant generation weights,
whose square roots ride in the filter passes, against the same weights given
as fields, whose square roots are scale passes of their own. The two differ
by where one product by sqrt(w) is rounded: 2 roundings of 2^-24 per value,
through sums of weights whose magnitudes add up to less than 4 per axis."""
import pytest

torch = pytest.importorskip("torch")

from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


@pytest.mark.parametrize("kw", [dict(), dict(l_filt_g1=False), dict(lquart=True, lm=13, h=3),
                                dict(mgbf_proc=8, p=1, mg_ampl02=2.0), dict(l_vertical_filter=False)])
def test_constant_weights_match_constant_fields(kw):
    kw = dict(kw)
    w = [0.7, 0.3, 2.5]
    cfg = M.Config.for_grid(48, 40, kw.pop("lm", 16), gm=3, h=kw.pop("h", 6), hz=2, n_ens=2, weights=w, **kw)
    g = torch.Generator(device="cuda").manual_seed(3)
    with M.MGBF(cfg) as op, M.MGBF(cfg) as opf:
        fields = [torch.full(op.dims.gen_shape(i), v, device="cuda") for i, v in enumerate(w, start=1)]
        for i, f in enumerate(fields, start=1):
            opf.set_weights(i, field=f)
        v = torch.randn(op.mg_numel(), generator=g, device="cuda")
        x = torch.randn(op.field_shape(), generator=g, device="cuda")
        for code, arg in ((M.OP_BSQRT, v), (M.OP_BSQRTT, x)):
            a, b = op.apply(code, arg), opf.apply(code, arg)
            assert (a - b).abs().max() <= 2e-6 * arg.abs().max()
