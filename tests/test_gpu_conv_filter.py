"""The filter gradient on FP32 MFMA (conv3d.hip) at the edges of its tiles:
x segments and chunks (144 columns), blocks of many rows whose ranges cross
planes, every kind of channel count, against the FP64 oracle.

A gradient is an FP32 sum of at most P = nx ny nz exact-product terms, added
along chains of at most D terms (a lane group's 9 points of each of its
block's rows, 4 per matrix product, then 4 wavefronts and the blocks), so
|error| <= D 2^-23 sum |g| |in|.
"""
import ctypes

import numpy as np
import pytest

import dage_amd
import dage_amd.learned as L
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # nx, ny, nz, cin, cout
    (1, 1, 1, 16, 16), (2, 3, 5, 16, 16), (15, 4, 3, 16, 16), (17, 9, 31, 16, 16),
    (129, 5, 3, 16, 16), (144, 2, 2, 16, 16), (145, 3, 2, 16, 16), (200, 2, 3, 16, 16),
    (33, 7, 5, 3, 5), (64, 3, 3, 9, 16), (128, 2, 2, 16, 7),
    (1, 1, 1, 2, 16), (17, 9, 31, 2, 16), (129, 5, 3, 1, 16), (289, 2, 2, 2, 16),
    (17, 9, 31, 16, 1), (143, 3, 2, 16, 2), (145, 2, 2, 7, 1), (5, 4, 3, 1, 1), (600, 1, 2, 1, 1),
    # several rows per block (1024 blocks with few channels, 256 with 16 x 16),
    # the planes' rows no multiple of them: 5, 7, 9 and 5 rows, then 6 and 8
    (5, 61, 83, 2, 16), (7, 83, 79, 1, 16), (6, 71, 127, 16, 1), (9, 67, 71, 16, 2),
    (5, 37, 41, 16, 16), (18, 43, 47, 9, 16),
]


@pytest.mark.parametrize("nx,ny,nz,cin,cout", CASES)
def test_filter_gradient(ctx, nx, ny, nz, cin, cout):
    rng = np.random.default_rng(nx + 7 * ny + cin + 100 * cout)
    x = rng.standard_normal((cin, nz, ny, nx)).astype(np.float32)
    g = rng.standard_normal((cout, nz, ny, nx)).astype(np.float32)
    w = np.zeros((cout, cin, 27))
    bufs = [L._Buf(ctx, n) for n in (x.nbytes, g.nbytes, 4 * cout * cin * 27, 4 * cout)]
    bufs[0].upload(x)
    bufs[1].upload(g)
    ptrs = [ctypes.c_void_p(b.ptr) for b in bufs]
    got = []
    for _ in range(2):
        dage_amd._lib.call("dage_conv3d_backward_filter", ctx.handle, nx, ny, nz, cin, cout,
                           *ptrs)
        got.append((bufs[2].download(np.float32, cout * cin * 27),
                    bufs[3].download(np.float32, cout)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    _, rw, rb = O.conv3d_backward(x.astype(np.float64), w, g.astype(np.float64))
    _, sw, sb = O.conv3d_backward(np.abs(x).astype(np.float64), w, np.abs(g).astype(np.float64))
    D = 36 * ((ny * nz + 255) // 256) + 4 + 1024
    for name, a, r, s in (("gw", got[0][0], rw, sw), ("gb", got[0][1], rb, sb)):
        err = np.abs(a.astype(np.float64) - r.ravel())
        print(f"{name}: error {(err / np.maximum(D * 2.0 ** -23 * s.ravel(), 1e-300)).max():.4f} of the bound")
        assert np.all(err <= D * 2.0 ** -23 * s.ravel())
    for b in bufs:
        b.close()
