"""Vertical band over whole columns whose length does not fit the wave, on the
GPU against a float64 sum over each column's band matrix."""
import numpy as np
import pytest
import torch

from standalone_mgbf_loc_amd import mgbf as M

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


# column lengths that are odd and 2 mod 4, shorter than the window, about the
# wave and the longest staged one (the next is too long); 1, part and several
# waves of columns; each half-width of the band
@pytest.mark.parametrize("lm,hz,n_ens,nx,ny", [
    (5, 2, 1, 8, 8),
    (7, 3, 3, 8, 16),
    (13, 1, 1, 24, 8),
    (33, 2, 1, 8, 40),
    (65, 3, 2, 24, 16),
    (66, 4, 1, 16, 16),
    (127, 4, 1, 8, 24),
    (255, 3, 1, 16, 24),
    (258, 3, 1, 16, 24),
])
def test_columns_match_band_matrix(lm, hz, n_ens, nx, ny):
    cfg = M.Config.for_grid(nx, ny, lm, n_ens=n_ens, gm=2, h=2, hz=hz)
    g = torch.Generator().manual_seed(lm)
    with M.MGBF(cfg) as op:
        d = op.dims
        x = torch.randn(d.gen_shape(1), generator=g)
        xg = x.cuda()
        for stage in (M.STAGE_VF, M.STAGE_VFT):
            # the band matrix of one column, from unit columns
            e = torch.zeros(d.gen_shape(1))
            ev = e.view(-1, lm)
            assert ev.shape[0] >= lm
            ev[:lm] = torch.eye(lm)
            mat = op.stage(stage, 1, e.cuda()).cpu().view(-1, lm)[:lm].double().numpy()
            got = op.stage(stage, 1, xg).cpu().view(-1, lm).double().numpy()
            cols = x.view(-1, lm).double().numpy()
            want = cols @ mat
            # 2 hb + 1 products, each rounded once on its way into the sum
            bound = (2 * 8 + 1) * EPS * (np.abs(cols) @ np.abs(mat)) + 1e-30
            assert (np.abs(got - want) <= bound).all()
            # banded, symmetric in the levels under the transpose
            assert not np.tril(mat, -2 * hz - 1).any() and not np.triu(mat, 2 * hz + 1).any()
            if stage == M.STAGE_VF:
                fwd = mat
            else:
                assert np.abs(fwd - mat.T).max() <= 4 * EPS * np.abs(fwd).max()


def test_columns_at_an_odd_address():
    """Pointers that are no multiple of 16 bytes take the narrow loads."""
    cfg = M.Config.for_grid(16, 8, 65, gm=2, h=2, hz=3)
    with M.MGBF(cfg) as op:
        shape = op.dims.gen_shape(1)
        n = int(np.prod(shape))
        buf = torch.randn(n + 1, device="cuda")
        a = op.stage(M.STAGE_VF, 1, buf[1:].view(shape))
        b = op.stage(M.STAGE_VF, 1, buf[1:].clone().view(shape))
        assert torch.equal(a, b)
