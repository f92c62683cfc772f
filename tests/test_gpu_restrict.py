"""The restriction kernel at the edges of its tiles (4 coarse columns by 2 to
16 coarse rows a wave, a table of its own next to a domain edge) against the
FP64 oracle. Both stencils have weights of sum of magnitudes below 2 per axis
and a window of at most 8 x 8 values, so an FP32 result is within
4 x 16 x 2^-24 = 3.8e-6 of the largest input; 4e-6 is allowed."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)


# coarse sides of 3 and 4 (every column within the edges), 5, 7, 9 (a last
# tile of 1 or 3 columns), one long side (strips of 16, 8, .. rows)
@pytest.mark.parametrize("quad", [False, True])
@pytest.mark.parametrize("nx,ny,lm", [(6, 8, 4), (8, 6, 33), (10, 14, 65), (18, 10, 64), (34, 262, 7), (1032, 24, 65)])
def test_restriction_tiles_match_oracle(nx, ny, lm, quad):
    cfg = M.Config.for_grid(nx, ny, lm, gm=2, h=3, hz=1, lquart=quad)
    with M.MGBF(cfg) as op:
        x = np.random.default_rng(nx + ny).standard_normal(op.dims.gen_shape(1)).astype(np.float32)
        y = op.stage(M.STAGE_R, 1, torch.from_numpy(x).to("cuda:0"))
        ref = O.restrict(x.astype(np.float64), quad)
        err = np.max(np.abs(y.cpu().double().numpy() - ref))
        assert err <= 4e-6 * np.max(np.abs(x))
