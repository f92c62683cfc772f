"""The host's part of a call of the 3-D procedures: what it works out from the
context alone is worked out when the context is made. A field 96 times as tall
takes the same launches; only the check of the fused restriction's windows
still walks its rows (a few ns a row), so that the call may cost the host 2.5
times as much (a search over all heights in every call made it 4 times and
more)."""
import time

import pytest

torch = pytest.importorskip("torch")

from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


def _host_us(ny):
    with M.MGBF(M.Config.for_grid(32, ny, 16, gm=3, h=6, hz=2, mgbf_proc=4, km3=1, km2=2)) as op:
        x = torch.randn(op.dims.gen_shape(1), device="cuda")
        y = torch.empty_like(x)
        best = 1e9
        for _ in range(12):
            t0 = time.perf_counter()
            for _ in range(5):
                op.filtering_procedure(x, out=y)
            best = min(best, time.perf_counter() - t0)
            torch.cuda.synchronize()
        return best / 5 * 1e6


def test_host_time_of_a_call_does_not_grow_with_the_rows():
    short, tall = _host_us(64), _host_us(6144)
    assert tall <= 2.5 * short, (short, tall)
