"""The streamed x/y and z passes (stream.hip) against the separate passes
(DAGE_APPLY_STREAM=0) and the oracle, at sizes around the 16-point tiles,
rectangular grids, and axes where the banded ring and the full kernel meet.

Both paths sum the same products (the flushed matrices' zeros are skipped by
either), in another order: at every point they differ by at most
2 (nx + ny + nz + T + 3) 2^-53 times the sum of the products' magnitudes.
"""
import ctypes

import numpy as np
import pytest

import dage_amd
import oracle as O
from _helpers import rel_maxdiff
from dage_amd._lib import call

pytestmark = pytest.mark.gpu

CASES = [
    # cells per input axis, per output axis (None: same grid), nlip, cell length
    ((1, 2, 4), None, 2, 0.4),
    ((14, 15, 16), None, 2, 0.4),                 # 15, 16, 17 points
    ((30, 31, 32), None, 2, 0.3),
    ((47, 16, 33), None, 2, 0.3),
    ((8, 10, 12), (3, 5, 2), 5, 0.5),             # rectangular: always the full kernel
    ((24, 4, 10), (4, 24, 11), 4, 0.5),
    ((16, 16, 16), None, 5, 0.6),                 # 65 points: five tiles, one launch
    ((52, 22, 4), None, 5, 0.6),                  # 209 points: the full kernels are too small
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_streamed_passes(ctx, monkeypatch, case):
    cin, cout, nlip, h = CASES[case]
    lo = [-0.5 * h * n + 0.05 * k for k, n in enumerate(cin)]
    ain = [O.Axis(a, np.full(n, h), nlip) for a, n in zip(lo, cin)]
    aout = ain if cout is None else [O.Axis(a + 0.3 * h, np.full(n, 0.8 * h), nlip)
                                     for a, n in zip(lo, cout)]
    rng = np.random.default_rng(60 + case)
    x = np.asfortranarray(rng.standard_normal([a.n for a in ain]))
    q = dage_amd.GaussQuad(nlin=12, nlog=12, tlin=2.0, tlog=300.0)
    w = O.coulomb_weights(q.tw)
    F = [O.exponentials(i, o, q.tp, False) for i, o in zip(ain, aout)]  # (out, in, t)
    S = np.zeros([a.n for a in aout])
    for t in range(len(q.tp)):
        v = np.abs(x)
        for axis in range(3):
            v = np.moveaxis(np.tensordot(np.abs(F[axis][:, :, t]), v, axes=(1, axis)), 0, axis)
        S += abs(w[t]) * v

    def grid(axes):
        return dage_amd.Grid3D(ctx, [a.qmin for a in axes], [a.steps for a in axes], nlip)

    gin = grid(ain)
    gout = gin if cout is None else grid(aout)
    op = dage_amd.Coulomb3D(ctx, gin, gout, q, coda=False)
    a = dage_amd.DeviceCube(ctx, x.shape, x)
    b = dage_amd.DeviceCube(ctx, S.shape)
    got = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("DAGE_APPLY_STREAM", mode)
        ctx.profile(True)
        op.transform_cuda_cube(a, b)
        streamed = ctx.profile_query("gemm_f64_xymode")[1]
        ctx.profile(False)
        assert (streamed > 0) == (mode == "1")
        got[mode] = b.download().copy()
    n = sum(i.n for i in ain) + len(q.tp) + 3
    diff = np.abs(got["1"] - got["0"])
    print(f"case {case}: {x.shape} -> {S.shape}, {(diff / (2 * n * 2.0 ** -53 * S)).max():.3f} of the "
          f"bound, {diff.max() / np.abs(got['0']).max():.2e} of max|out|")
    assert np.all(diff <= 2 * n * 2.0 ** -53 * S)
    ref = O.transform_cube(F[0], F[1].transpose(1, 0, 2).copy("F"), F[2].transpose(1, 0, 2).copy("F"),
                           w, 0.0, x, add_coda=False)
    assert rel_maxdiff(got["1"], ref) < 1e-10


@pytest.mark.parametrize("n,band", [(5, 5), (17, 17), (31, 31), (33, 33), (95, 95), (97, 12), (209, 20)])
def test_infinity_on_odd_axes(ctx, monkeypatch, n, band):
    """Positive matrices and inputs, one infinity near the end of the x axis:
    every output it reaches is +inf, not NaN (an odd axis ends in the middle
    of the x product's pairs of points)."""
    ax, short = O.Axis(0.0, np.full(n - 1, 0.2), 2), O.Axis(0.0, np.full(4, 0.2), 2)
    q = dage_amd.GaussQuad(nlin=3, nlog=0, tlin=2.0, tlog=2.0)
    T = q.get_npoints()
    rng = np.random.default_rng(n)

    def matrix(m):
        i = np.arange(m)
        return np.where(np.abs(i[:, None] - i) <= band, 1.0, 0.0)[:, :, None] * rng.uniform(0.5, 1.0, (m, m, T))

    Fx, Fy, Fz = matrix(n), matrix(n), matrix(5)
    g = dage_amd.Grid3D(ctx, [0.0] * 3, [ax.steps, ax.steps, short.steps], 2)
    op = dage_amd.Coulomb3D(ctx, g, g, q, coda=False)
    op.set_matrices(np.asfortranarray(Fx), np.asfortranarray(Fy), np.asfortranarray(Fz))
    monkeypatch.setenv("DAGE_APPLY_STREAM", "1")
    for x, y, z in ((n - 2, 0, 1), (n - 1, n // 2, 2), (n - 3, n - 1, 0), (0, n - 2, 4)):
        cube = rng.uniform(0.5, 1.0, (n, n, 5))
        cube[x, y, z] = np.inf
        a, b = dage_amd.DeviceCube(ctx, cube.shape, cube), dage_amd.DeviceCube(ctx, cube.shape)
        ctx.profile(True)
        op.transform_cuda_cube(a, b)
        assert ctx.profile_query("gemm_f64_xymode")[1] > 0
        ctx.profile(False)
        out = b.download()
        reach = (Fx[:, x, 0] > 0)[:, None, None] & (Fy[y, :, 0] > 0)[None, :, None] & np.ones(5, bool)
        assert np.all(np.isposinf(out[reach])), (x, y, z)
    op.close()


def test_separate_z_pass_keeps_its_split_rule(ctx, monkeypatch):
    """Different grids with an axis above 208 points run the separate passes,
    whose z pass splits its sum for about 1024 blocks: the workspace holds
    that many partials, not the streamed pass's."""
    monkeypatch.setenv("DAGE_APPLY_TCHUNK", "24")
    nin, nout = (241, 241, 65), (121, 121, 33)
    gin, gout = (dage_amd.Grid3D(ctx, [0.0] * 3, [np.full((n - 1) // 4, s) for n in shape], 5)
                 for shape, s in ((nin, 0.4), (nout, 0.8)))
    q = dage_amd.GaussQuad(nlin=12, nlog=12, tlin=2.0, tlog=300.0)
    op = dage_amd.Coulomb3D(ctx, gin, gout, q, coda=False)
    size = ctypes.c_size_t()
    call("dage_operator_workspace_bytes", op.handle, ctypes.byref(size))
    per_t = nout[0] * (nin[1] + nout[1]) * nin[2]
    tiles = (nout[0] * nout[1] + 63) // 64  # one 48-column tile in z
    splits = (1024 + tiles - 1) // tiles
    assert splits == 5 and size.value == 8 * (24 * per_t + splits * nout[0] * nout[1] * nout[2])
    op.close()


@pytest.mark.parametrize("shape,streams", [((65, 65, 65), True), ((45, 57, 61), True),
                                           ((9, 213, 145), False), ((41, 401, 41), False),
                                           ((5, 173, 85), False)])
def test_thin_boxes_keep_the_separate_passes(ctx, monkeypatch, shape, streams):
    """The default route by shape; the same result as on the other route (the
    bound of this file's header, with every |entry| at most its row's sum)."""
    monkeypatch.delenv("DAGE_APPLY_STREAM", raising=False)
    g = dage_amd.Grid3D(ctx, [0.0] * 3, [np.full((n - 1) // 4, 0.8) for n in shape], 5)
    op = dage_amd.Coulomb3D(ctx, g, g, dage_amd.GaussQuad(nlin=20, nlog=20, tlin=2.0, tlog=500.0))
    x = np.random.default_rng(7).uniform(0.0, 1.0, shape)
    a, b = dage_amd.DeviceCube(ctx, shape, x), dage_amd.DeviceCube(ctx, shape)
    ctx.profile(True)
    op.transform_cuda_cube(a, b)
    count = ctx.profile_query("gemm_f64_xymode")[1], ctx.profile_query("gemm_f64_xmode")[1]
    ctx.profile(False)
    assert (count[0] > 0) == streams and (count[1] > 0) == (not streams)
    got = b.download().copy()
    monkeypatch.setenv("DAGE_APPLY_STREAM", "0" if streams else "1")
    op.transform_cuda_cube(a, b)
    assert rel_maxdiff(got, b.download()) < 1e-13
    op.close()


def tile_kernels(ctx):
    """The x/y kernels that the profiled applies launched."""
    names = [f"stream_xy_{k}{n}" for k in ("full", "ring") for n in range(2, 14)]
    ran = {k for k in names if ctx.profile_query(k)[1] > 0}
    ctx.profile(False)
    return ran


# points per axis, band half-width in x and y (None: dense), t-points, the x/y
# kernels
KERNELS = [
    ((17, 31, 5), None, 2, {"full2"}), ((33, 48, 5), None, 2, {"full3"}),
    ((49, 64, 5), None, 2, {"full5"}), ((65, 80, 5), None, 2, {"full5"}),
    ((96, 81, 5), None, 2, {"full6"}), ((97, 112, 5), None, 2, {"full7"}),
    ((113, 17, 5), None, 2, {"full8"}), ((144, 129, 5), None, 2, {"full9"}),
    ((145, 160, 5), None, 2, {"full10"}), ((161, 33, 5), None, 2, {"full11"}),
    ((49, 177, 5), None, 2, {"full12"}), ((208, 193, 5), None, 2, {"full13"}),
    ((81, 65, 5), 12, 2, {"ring3"}), ((129, 145, 5), 30, 2, {"ring5"}),
    ((145, 143, 5), 48, 2, {"ring7"}), ((177, 161, 5), 64, 2, {"ring9"}),
    ((193, 209, 5), 80, 2, {"ring11"}), ((225, 241, 5), 96, 2, {"ring13"}),
    ((399, 33, 3), 96, 2, {"ring13"}), ((33, 399, 3), 96, 2, {"ring13"}),
    # wide bands first, in launches of their own when each fills the card
    ((225, 225, 65), (96,) * 3 + (12,) * 7, 10, {"ring13", "ring3"}),
    # more than 13 z tiles (two groups), and more than 64 steps in a split
    ((17, 17, 209), None, 3, {"full2"}), ((65, 65, 225), None, 40, {"full5"}),
]


@pytest.mark.parametrize("case", range(len(KERNELS)))
def test_every_kernel(ctx, monkeypatch, case):
    n, band, T, kernels = KERNELS[case]
    q = dage_amd.GaussQuad(nlin=T, nlog=0, tlin=2.0, tlog=2.0)
    rng = np.random.default_rng(case)

    def matrix(axis):
        m = n[axis]
        F = rng.standard_normal((m, m, T))  # (out, in, t)
        i = np.arange(m)
        for t in range(T):
            b = m if band is None or axis == 2 else band if np.isscalar(band) else band[t]
            F[np.abs(i[:, None] - i) > b, t] = 0.0
        return F

    F = [matrix(a) for a in range(3)]
    monkeypatch.setenv("DAGE_APPLY_STREAM", "1")
    monkeypatch.setenv("DAGE_APPLY_BAND", "0")
    g = dage_amd.Grid3D(ctx, [0.0] * 3, [np.full(m - 1, 0.2) for m in n], 2)
    op = dage_amd.Coulomb3D(ctx, g, g, q, coda=False)
    op.set_matrices(np.asfortranarray(F[0]), *(np.asfortranarray(F[a].transpose(1, 0, 2)) for a in (1, 2)))
    x = rng.standard_normal(n)
    w = O.coulomb_weights(q.tw)
    ref, S = np.zeros(n), np.zeros(n)
    for t in range(T):
        v, s = x, np.abs(x)
        for axis in range(3):
            v = np.moveaxis(np.tensordot(F[axis][:, :, t], v, axes=(1, axis)), 0, axis)
            s = np.moveaxis(np.tensordot(np.abs(F[axis][:, :, t]), s, axes=(1, axis)), 0, axis)
        ref += w[t] * v
        S += abs(w[t]) * s
    a, b = dage_amd.DeviceCube(ctx, n, x), dage_amd.DeviceCube(ctx, n)
    ctx.profile(True)
    op.transform_cuda_cube(a, b)
    assert tile_kernels(ctx) == {"stream_xy_" + k for k in kernels}
    # the reference's own rounding has the same bound
    err = np.abs(b.download() - ref) / (2 * (sum(n) + T + 3) * 2.0 ** -53 * S)
    print(f"{n}: {err.max():.3f} of the bound")
    assert np.all(err <= 1.0)
    op.close()


@pytest.mark.parametrize("n,energies", [(65, [-0.3, -1.1, -2.0]), (145, [-0.2, -0.9]), (33, [-0.5] * 7)])
def test_batches(ctx, monkeypatch, n, energies):
    """Right-hand sides with weights of their own, streamed and separate."""
    g = dage_amd.Grid3D(ctx, [-0.05 * (n - 1)] * 3, [np.full((n - 1) // 4, 0.4)] * 3, 5)
    q = dage_amd.GaussQuad(nlin=10, nlog=10, tlin=2.0, tlog=300.0)
    rng = np.random.default_rng(n)
    rhs = [rng.standard_normal((n, n, n)) for _ in energies]
    got = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("DAGE_APPLY_STREAM", mode)
        batch = dage_amd.HelmholtzBatch(ctx, [g] * len(rhs), energies, q)
        for i, r in enumerate(rhs):
            batch.upload(i, r)
        ctx.profile(True)
        batch.apply_eager()
        assert bool(tile_kernels(ctx)) == (mode == "1")
        got[mode] = [batch.download(i).copy() for i in range(len(rhs))]
        # the other route in the workspace that was reserved for this one
        monkeypatch.setenv("DAGE_APPLY_STREAM", "1" if mode == "0" else "0")
        batch.apply_eager()
        for i in range(len(rhs)):
            assert rel_maxdiff(batch.download(i), got[mode][i]) < 1e-13
        batch.close()
    for a, b in zip(got["0"], got["1"]):
        assert rel_maxdiff(a, b) < 1e-13
