"""A launch takes about as long whether or not its blocks divide by the 8 XCDs:
the plain pass of a narrow filter on a stack laid end to end, whose tiles share
cache lines with their neighbours, at 16 rows (801 blocks) and at 25 (512). The
two differ by up to 15 % in the rows that they load; blocks dealt round-robin to
the XCDs took 1.5 times."""
import pytest

torch = pytest.importorskip("torch")

from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


def _time(op, x, y, tj):
    op.set_tiles({(1, 0): (4, tj)})
    best = 1e9
    for _ in range(6):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(30):
            op.stage(M.STAGE_F, 1, x, out=y)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def test_block_counts_off_a_multiple_of_8():
    with M.MGBF(M.Config.for_grid(154, 566, 48, gm=2, h=3, hz=2, km3=3, km2=2, mgbf_proc=1)) as op:
        assert op.dims.km_all == 146
        x = torch.randn(op.dims.gen_shape(1), device="cuda")
        y = torch.empty_like(x)
        assert _time(op, x, y, 16) <= 1.25 * _time(op, x, y, 25)
