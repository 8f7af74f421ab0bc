"""The bubbles inject from packed coefficients (inject.hip) over the lmax
it is compiled for and the cell sizes it has code for, with a grid point
exactly on a centre and points outside the radial grids, against the oracle.

At a point both sides sum, per bubble, (lmax+1)^2 harmonics times cell
polynomials.  The chains have at most (lmax+1)^2 + 4 lmax + 4 nlip roundings
of terms that sum to at most A = sum_k |c|^k sum_j |lip_jk| * max sum_lm |f_lm|
(|c| <= the cell's half width, |Y_lm| <= 1), so the sides differ by at most
twice that many 2^-53 A.
"""
import numpy as np
import pytest

import dage_amd
import oracle as O
from _helpers import slater_bubbles
from test_gpu_bubbles import lib_bubbles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,nlip,lmin", [(0, 7, 0), (1, 5, 0), (2, 3, 0), (3, 7, 1), (5, 5, 0),
                                            (6, 4, 2), (7, 7, 0), (8, 7, 0), (8, 5, 3), (10, 6, 0),
                                            (12, 7, 0), (12, 2, 5)])
def test_packed_inject(ctx, lmax, nlip, lmin):
    rng = np.random.default_rng(100 * lmax + nlip)
    bub, _ = slater_bubbles(rng, 3, lmax=lmax, nlip=nlip, r_max=5.0)
    ax = O.Axis.ncell_fixed(-6.0, 6.0, 5, 4)  # 17 points
    bub.centers[0] = [ax.points[5], ax.points[8], ax.points[11]]
    g = dage_amd.Grid3D(ctx, [ax.qmin] * 3, [ax.steps] * 3, ax.nlip)
    cube = dage_amd.DeviceCube(ctx, (ax.n,) * 3)
    cube.set_to_zero()
    lib_bubbles(ctx, bub).inject(g, cube, lmin=lmin, multiplier=1.0)
    got = cube.download()
    ref = O.bubbles_eval_grid(bub, ax.points, ax.points, ax.points, lmin=lmin)
    half = abs(O.lip_first_last(nlip)[0])
    powers = half ** np.arange(nlip - 1, -1, -1)
    amp = (np.abs(O.lip_coeffs(nlip)) * powers).sum()
    A = amp * sum(np.abs(b).sum(axis=1).max() for b in bub.bf)
    bound = 2 * ((lmax + 1) ** 2 + 4 * lmax + 4 * nlip) * 2.0 ** -53 * A
    print(f"lmax {lmax}, nlip {nlip}: {np.abs(got - ref).max() / bound:.4f} of the bound")
    assert np.abs(ref).max() > 0  # (and zero outside the radial grids)
    assert np.all(got[ref == 0.0] == 0.0) or lmin > 0
    assert np.abs(got - ref).max() <= bound
