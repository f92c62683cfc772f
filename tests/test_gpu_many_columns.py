"""The vertical band over more columns than a launch of 4 threads a column can
number (2^30 of 3 levels, 12.9 GB a field): the first and the last columns
against the band's own weights on a small field, which the FP64 oracle checks
elsewhere. Equal kernels on equal columns: the values are the same to the bit."""
import pytest

torch = pytest.importorskip("torch")

from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


def test_columns_beyond_two_to_the_30():
    n, lm = 32768, 3
    with M.MGBF(M.Config.for_grid(n, n, lm, gm=1, h=2, hz=1)) as op:
        x = torch.randn(op.field_shape(), device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
        assert x.numel() // lm >= 2 ** 30
        y = op.stage(M.STAGE_VF, 1, x, out=torch.full_like(x, float("nan")))
        ends = [x[:64, :64].clone(), x[-64:, -64:].clone(), x[16384:16448, 7:71].clone()]
        got = [y[:64, :64].clone(), y[-64:, -64:].clone(), y[16384:16448, 7:71].clone()]
        assert not torch.isnan(y[::97, ::101]).any()
        del x, y
    torch.cuda.empty_cache()
    with M.MGBF(M.Config.for_grid(64, 64, lm, gm=1, h=2, hz=1)) as op:
        for a, b in zip(ends, got):
            assert torch.equal(op.stage(M.STAGE_VF, 1, a.contiguous()), b)
