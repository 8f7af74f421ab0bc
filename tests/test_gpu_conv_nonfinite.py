"""Infinities in the filter gradient's operands reach the sums they belong to
and no others: the zero padding of the kernels' tiles (columns past the last
one or past an x chunk, rows and planes outside the volume) must not meet one
(0 * inf is NaN)."""
import ctypes

import numpy as np
import pytest

import dage_amd
import dage_amd.learned as L
import oracle as O

pytestmark = pytest.mark.gpu

SIZES = {"wide": [(1, 1, 1), (5, 3, 2), (16, 2, 2), (17, 3, 2), (63, 2, 2), (129, 3, 3), (145, 2, 2)],
         "few": [(1, 1, 1), (5, 3, 2), (16, 2, 2), (17, 3, 2), (129, 3, 3), (145, 2, 2), (291, 2, 2)]}


def gradient(ctx, x, g):
    (cin, nz, ny, nx), cout = x.shape, g.shape[0]
    bufs = [L._Buf(ctx, n) for n in (x.nbytes, g.nbytes, 4 * cout * cin * 27, 4 * cout)]
    bufs[0].upload(x)
    bufs[1].upload(g)
    dage_amd._lib.call("dage_conv3d_backward_filter", ctx.handle, nx, ny, nz, cin, cout,
                       *[ctypes.c_void_p(b.ptr) for b in bufs])
    out = bufs[2].download(np.float32, cout * cin * 27), bufs[3].download(np.float32, cout)
    for b in bufs:
        b.close()
    return out[0].reshape(cout, cin, 27), out[1]


def edges(n):
    """First and last points, and those around the x chunks' ends."""
    chunks = (n + 143) // 144
    w = (n + chunks - 1) // chunks
    return sorted({i for c in range(chunks + 1) for b in (c * w, c * 144) for i in (b - 2, b - 1, b, b + 1)
                   if 0 <= i < n} | {n - 1})


def check(ctx, nx, ny, nz, cin, cout):
    rng = np.random.default_rng(nx + cin)
    x0 = rng.uniform(0.5, 1.0, (cin, nz, ny, nx)).astype(np.float32)
    g = rng.uniform(0.5, 1.0, (cout, nz, ny, nx)).astype(np.float32)  # no inf - inf
    w = np.zeros((cout, cin, 27))
    for i in edges(nx):
        for k, j in ((0, 0), (nz - 1, ny - 1)):
            c, o = i % cin, i % cout
            x = x0.copy()
            x[c, k, j, i] = np.inf
            gw, gb = gradient(ctx, x, g)
            _, rw, rb = O.conv3d_backward(x.astype(np.float64), w, g.astype(np.float64))
            assert np.array_equal(np.isposinf(gw), np.isposinf(rw)), ("in", i, j, k)
            assert np.array_equal(np.isfinite(gw), np.isfinite(rw)), ("in", i, j, k)
            ok = np.isfinite(rw)
            assert np.allclose(gw[ok], rw[ok], rtol=1e-4) and np.allclose(gb, rb, rtol=1e-4)
            h = g.copy()
            h[o, k, j, i] = np.inf
            gw, gb = gradient(ctx, x0, h)
            _, rw, rb = O.conv3d_backward(x0.astype(np.float64), w, g.astype(np.float64))
            assert np.isposinf(gb[o]) and np.all(np.isfinite(np.delete(gb, o)))
            assert not np.any(np.isfinite(gw[o, :, 13]))
            assert np.allclose(np.delete(gw, o, 0), np.delete(rw, o, 0), rtol=1e-4), ("gout", i, j, k)


@pytest.mark.parametrize("size", SIZES["wide"])
@pytest.mark.parametrize("cin,cout", [(16, 16), (3, 5)])
def test_infinity_stays_with_its_taps(ctx, size, cin, cout):
    check(ctx, *size, cin, cout)


@pytest.mark.parametrize("size", SIZES["few"])
@pytest.mark.parametrize("cin,cout", [(2, 16), (1, 16), (16, 1), (16, 2), (7, 2), (1, 1)])
def test_infinity_few_channels(ctx, size, cin, cout):
    check(ctx, *size, cin, cout)
