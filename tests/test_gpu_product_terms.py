"""Products of bubbles' radial functions by output harmonic (bubbles_ops.hip)
against the oracle, for orders and radial lengths that are no multiple of the
64-point blocks."""
import numpy as np
import pytest

import oracle as O
from _helpers import slater_bubbles
from test_gpu_bubbles import lib_bubbles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l1,l2,ncell", [(0, 0, 3), (1, 3, 11), (4, 4, 33), (6, 2, 22)])
def test_product_by_output(ctx, l1, l2, ncell):
    """Each output (l,m) sums at most (l1+1)^2 (l2+1)^2 terms c f1 f2."""
    rng = np.random.default_rng(l1 + 10 * l2)
    b1, _ = slater_bubbles(rng, 2, lmax=l1, ncell=ncell)
    b2 = O.BubbleSet(b1.centers, b1.steps,
                     [np.asfortranarray(rng.standard_normal((len(b), (l2 + 1) ** 2))) for b in b1.bf],
                     l2, 0, 7)
    out = lib_bubbles(ctx, b1).multiply(lib_bubbles(ctx, b2))
    # |c| <= 2 (l1 + l2) + 1
    terms = ((l1 + 1) * (l2 + 1)) ** 2 + 4
    for i in range(2):
        got = out.get(i)[3]
        ref = O.bubble_product(l1, b1.bf[i], l2, b2.bf[i])
        mag = np.abs(b1.bf[i]).sum(axis=1) * np.abs(b2.bf[i]).sum(axis=1)
        bound = 2 * terms * (2 * (l1 + l2) + 1) * 2.0 ** -53 * mag
        print(f"{l1} x {l2}: {np.abs(got - ref).max():.2e} of {np.abs(ref).max():.2e}")
        assert np.all(np.abs(got - ref) <= bound[:, None])
