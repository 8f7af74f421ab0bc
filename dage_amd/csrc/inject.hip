// Bubbles inject: cube(x,y,z) += multiplier * sum_bubbles sum_{l>=lmin,m}
//                 interp(r^k f_lm)(r) * S_lm(x-c)/r^l
// (Bubbles_eval_3dgrid, src/bubbles/bubbles.F90:2148-2211, and the CUDA
// Bubbles::inject it dispatches to, src/bubbles/bubbles_cuda.cu:3090-3340).
//
// One fused launch for all bubbles and all (l,m): one thread per cube point,
// a wavefront per 4 x 4 x 4 patch of points.  Per bubble the thread finds
// the radial cell (grid.F90:1212-1246, from a lookup table), evaluates the
// nlip cell polynomials once by Horner (lip.F90:551-566), reuses them for every
// (l,m); the Racah solid harmonics come from the recursion of
// harmonics.F90:586-659, fully unrolled for the compile-time lmax.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "dage_internal.hpp"

namespace dage {
namespace {

// Global-address-space views of the bubble tables: the pointers come out of
// device memory (the descriptors), where the compiler may otherwise treat
// them as generic and emit flat loads, or vector loads for uniform addresses.
typedef const double __attribute__((address_space(1))) *gdptr;
typedef const int __attribute__((address_space(1))) *giptr;
// Constant address space: loads at wavefront-uniform addresses are scalar
// whatever else the kernel does to memory.
typedef const double __attribute__((address_space(4))) *cdptr;
typedef double d8 __attribute__((ext_vector_type(8)));
typedef const d8 __attribute__((address_space(4))) *cd8ptr;

struct InjectArgs {
    const double *gx, *gy, *gz;  // cube grid points
    int nx, ny, nz;
    const BubbleDev *bubs;
    int nbub;
    int lmin;
    int nlip;
    double first;
    double multiplier;
    double *cube;
    const double *head;  // constants (PackArgs::head)
};

// The radial coefficients as the inject kernel reads them: kPackW per (cell,
// (l,m)), at pack + ((cell - 1)*nlm + lm)*kPackW.  The nlip values of a cell
// sit in the table of an (l,m) at multiples of nlip - 1, mostly not aligned:
// three scalar loads each; here they are one aligned 64-byte load, and a
// cell's (l,m) are neighbours.
constexpr int kPackW = 8;
static_assert(kMaxNlip <= kPackW, "cells wider than a packed row");

// The kernel's constants, in front of the packed coefficients: the cell
// polynomials (polynomial j, decreasing powers from j*kPackW on) and the
// factors of the harmonics' recursion: from kHarm + l^2 on the one of m = +-l,
// then the two of |m| = 0..l-1.  As literals or kernel arguments the compiler
// keeps them in registers across the bubbles, 218 of them at lmax 8, and
// spills.
constexpr int kHarm = kPackW * kMaxNlip;
constexpr int kHead = (kHarm + (kMaxBubbleLmax + 1) * (kMaxBubbleLmax + 1) + kPackW - 1) / kPackW * kPackW;

struct PackArgs {
    const BubbleDev *bubs;
    int nlm, nlip;
    double *head_dev;
    double head[kHead];
};

__global__ void __launch_bounds__(256) pack_radial_kernel(PackArgs A) {
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int e = threadIdx.x; e < kHead; e += 256) A.head_dev[e] = A.head[e];
    const BubbleDev B = A.bubs[blockIdx.y];
    const long n = (long)B.ncell * A.nlm * kPackW;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += gridDim.x * 256L) {
        const int j = (int)(e % kPackW);
        const long r = e / kPackW;
        const int lm = (int)(r % A.nlm);
        const long c = r / A.nlm;
        B.pack[e] = j < A.nlip ? B.f[(long)lm * B.npts + c * (A.nlip - 1) + j] : 0.0;
    }
}

// x*x - y*y with both squares rounded, as where they are shared with r^2
__device__ inline double square_diff(double x, double y) {
#pragma clang fp contract(off)
    return x * x - y * y;
}

// a*b + c with c straight from a scalar register (the compiler would move it
// to vector registers for a two-operand fmac, two moves per multiply-add)
__device__ inline double fma_s(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
}

// Grid1D_get_icell (grid.F90:1212-1246): the 1-based cell c with
// celld[c-1] <= r < celld[c] (the last cell from its start up to qmax), 0
// outside [0, qmax].  The reference bisects; here the lookup-table entry one
// bin below r (a margin for the rounding of r*tscale) is at or below r's
// cell, and upward steps stop at the first cell start above r: the same
// cell, in one or two dependent loads instead of about log2(ncell).
__device__ inline int radial_icell_tab(const BubbleDev &B, double r) {
    if (!(r >= 0.0 && r <= B.qmax)) return 0;  // also rejects NaN
    const gdptr celld = (gdptr)B.celld;
    if (celld[B.ncell - 1] <= r) return B.ncell;
    const int k = min(max((int)(r * B.tscale) - 1, 0), kCellTab - 1);
    int ic = ((giptr)B.ctab)[k];
    while (celld[ic] <= r) ++ic;
    return ic;
}

// NLIP > 0: compile-time cell size (unrolled Horner and dot products);
// NLIP == 0: A.nlip at run time.
//
// The reference divides every S_lm by r^l (RealSphericalHarmonics_eval,
// harmonics.F90:1360-1370); here each l's sum over m is scaled once by
// (1/r)^l, which moves the result by rounding only (1e-16 relative per term).
// Each l's 2l + 1 harmonics are generated from the previous two l's by the
// recursion of harmonics.F90:586-659 right before they are consumed, so two
// levels live at a time and one kernel serves every lmax.
//
// A wavefront covers a 4 x 4 x 4 patch of points (lane l: x = l & 3,
// y = (l >> 2) & 3, z = l >> 4), a block four patches along x.  The points
// of one patch almost always fall in one or two radial cells of a bubble,
// so the wavefront loops over the distinct cells present (ballot, lowest
// lane first): the cell index is wavefront-uniform inside the loop and the
// coefficients of the cell are read once per wavefront through scalar loads
// instead of once per lane.
//
// Bound by FP64 issue and, behind it, the latency of the scalar loads: at
// lmax 4 and nlip 7 some 390 FP64 instructions per point and bubble.  With
// packed coefficients and the constants in memory, before -> after: 241^3, four
// bubbles of lmax 4, 955 -> 840 us; 129^3, ten bubbles, lmax 4 twice and lmax 8
// once, 3.78 -> 2.31 ms.  Moving the sum over (l,m) before the polynomials and
// the harmonics' factors into the coefficients took 600 us and 1.77 ms, with
// errors of the same size, but other roundings: where a product of two
// functions nearly cancels, they showed at 1e-13 of the result.
template <int LMAX, int NLIP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LMAX <= 8 ? 4 : 3)))
bubbles_inject_kernel(InjectArgs A) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ix = blockIdx.x * 16 + wave * 4 + (lane & 3);
    const int iy = blockIdx.y * 4 + ((lane >> 2) & 3);
    const int iz = blockIdx.z * 4 + (lane >> 4);
    // no early exit: every lane takes part in the wavefront-uniform cell loop
    const bool inside = ix < A.nx && iy < A.ny && iz < A.nz;
    constexpr int NMAX = NLIP > 0 ? NLIP : kMaxNlip;
    constexpr int NLM = (LMAX + 1) * (LMAX + 1);
    const int nlip = NLIP > 0 ? NLIP : A.nlip;
    const double px = A.gx[inside ? ix : 0], py = A.gy[inside ? iy : 0],
                 pz = A.gz[inside ? iz : 0];
    constexpr double kEps = 2.220446049250313e-16;  // epsilon(0.d0)
    double total = 0.0;
    for (int b = 0; b < A.nbub; ++b) {
        const BubbleDev B = A.bubs[b];
        const double dx = px - B.cx, dy = py - B.cy, dz = pz - B.cz;
        const double r = sqrt(dx * dx + dy * dy + dz * dz);
        const int ic = inside ? radial_icell_tab(B, r) : 0;
        unsigned long long todo = __ballot(ic != 0);
        if (todo == 0ull) continue;
        const int icl = ic > 0 ? ic - 1 : 0;
        const double crd = (r - ((gdptr)B.celld)[icl]) / ((gdptr)B.steps)[icl] + A.first;
        double polys[NMAX];
        {
            cdptr lip = (cdptr)A.head;
            asm volatile("" : "+s"(lip));  // opaque: not kept across the bubbles
#pragma unroll
            for (int j = 0; j < NMAX; ++j) {
                if (j >= nlip) break;
                const d8 c = *(cd8ptr)(lip + j * kPackW);
                double v = c[0];
#pragma unroll
                for (int q = 1; q < NMAX; ++q) {
                    if (q >= nlip) break;
                    v = fma_s(v, crd, c[q]);
                }
                polys[j] = v;
            }
        }
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double inv = (r > kEps) ? 1.0 / r : 1.0;  // r <= eps: r^l taken as 1
        while (todo != 0ull) {
            const int leader = __builtin_ctzll(todo);
            const int c = __builtin_amdgcn_readlane(ic, leader);  // uniform cell
            const bool mine = ic == c;
            todo &= ~__ballot(mine);
            if (!mine) continue;
            // re-read from the first active lane so the address stays scalar
            // (inside the branch the compiler may otherwise substitute the
            // per-lane ic for c)
            const int cs = __builtin_amdgcn_readfirstlane(c);
            const cd8ptr f = (cd8ptr)(B.pack + (long)(cs - 1) * (kPackW * NLM));
            // opaque, so that neither the harmonics nor the constants are kept
            // across the cells
            double x = dx, y = dy, z = dz;
            cdptr head = (cdptr)A.head;
            asm volatile("" : "+v"(x), "+v"(y), "+v"(z), "+s"(head));
            double S[2][2 * LMAX + 1];  // levels l - 1 and l, entry m + LMAX
            double res = 0.0, ipow = 1.0;
#pragma unroll
            for (int l = 0; l <= LMAX; ++l) {
                double *t = S[l & 1] + LMAX;              // level l - 2, replaced by l
                const double *p = S[(l & 1) ^ 1] + LMAX;  // level l - 1
                if (l == 0) {
                    t[0] = 1.0;
                } else if (l == 1) {
                    t[-1] = y;
                    t[0] = z;
                    t[1] = x;
                } else {
                    const cdptr h = head + kHarm + l * l;
#pragma unroll
                    for (int m = -(l - 1); m <= l - 1; ++m) {
                        const int am = m < 0 ? -m : m;
                        double v = h[1 + 2 * am] * (z * p[m]);
                        if (l - am > 1) v = v - h[2 + 2 * am] * (r2 * t[m]);
                        t[m] = v;
                    }
                    t[-l] = h[0] * (y * p[l - 1] + x * p[-(l - 1)]);
                    t[l] = h[0] * (l == 2 ? square_diff(x, y) : x * p[l - 1] - y * p[-(l - 1)]);
                }
                if (l >= A.lmin) {
                    double sl = 0.0;
#pragma unroll
                    for (int m = -l; m <= l; ++m) {
                        const d8 fl = f[l * l + l + m];
                        double fv = 0.0;
#pragma unroll
                        for (int j = 0; j < NMAX; ++j) {
                            if (j >= nlip) break;
                            fv += fl[j] * polys[j];
                        }
                        sl += fv * t[m];
                    }
                    res += sl * ipow;
                }
                ipow *= inv;
            }
            total += res;
        }
    }
    if (inside) {
        const long id = ix + (long)A.nx * (iy + (long)A.ny * iz);
        A.cube[id] = A.cube[id] + A.multiplier * total;
    }
}

template <int LMAX>
void launch_inject(const InjectArgs &A, dim3 g, dim3 block, hipStream_t s) {
    if (A.nlip == 7)
        hipLaunchKernelGGL((bubbles_inject_kernel<LMAX, 7>), g, block, 0, s, A);
    else if (A.nlip == 5)
        hipLaunchKernelGGL((bubbles_inject_kernel<LMAX, 5>), g, block, 0, s, A);
    else
        hipLaunchKernelGGL((bubbles_inject_kernel<LMAX, 0>), g, block, 0, s, A);
}

}  // namespace

int bubbles_sync_device(dage_bubbles bub) {
    if (!bub->dirty) return DAGE_OK;
    std::vector<BubbleDev> desc(bub->nbub);
    size_t cells = 0;
    for (const BubbleHost &h : bub->host) cells += h.ncell;
    const size_t pack = kHead + cells * bub->nlm() * kPackW;
    if (pack > bub->pack_size) {
        DAGE_HIP_CHECK(hipStreamSynchronize(bub->ctx->stream));
        if (bub->d_pack) DAGE_HIP_CHECK(hipFree(bub->d_pack));
        bub->d_pack = nullptr;
        bub->pack_size = 0;
        DAGE_HIP_CHECK(hipMalloc((void **)&bub->d_pack, sizeof(double) * pack));
        bub->pack_size = pack;
    }
    cells = 0;
    for (int b = 0; b < bub->nbub; ++b) {
        const BubbleHost &h = bub->host[b];
        BubbleDev &d = desc[b];
        d.cx = h.center[0];
        d.cy = h.center[1];
        d.cz = h.center[2];
        d.qmax = h.qmax;
        d.ncell = h.ncell;
        d.npts = h.ncell * (bub->nlip - 1) + 1;
        d.celld = h.d_buf;
        d.steps = h.d_buf + h.ncell;
        d.f = h.d_buf + 2 * h.ncell;
        d.pack = bub->d_pack + kHead + cells * bub->nlm() * kPackW;
        cells += h.ncell;
        d.ctab = h.d_tab;
        d.tscale = kCellTab / h.qmax;
    }
    DAGE_HIP_CHECK(hipMemcpy(bub->d_desc, desc.data(), sizeof(BubbleDev) * bub->nbub,
                             hipMemcpyHostToDevice));
    bub->dirty = false;
    return DAGE_OK;
}

int bubbles_inject(dage_bubbles bub, dage_grid3d grid, int lmin, double multiplier,
                   double *cube) {
    dage_ctx ctx = bub->ctx;
    if (bub->lmax > kMaxBubbleLmax) {
        set_error("bubbles lmax %d outside 0..%d", bub->lmax, kMaxBubbleLmax);
        return DAGE_ERR_UNSUPPORTED;
    }
    DAGE_TRY(bubbles_sync_device(bub));
    InjectArgs A{};
    A.gx = grid->d_points[0];
    A.gy = grid->d_points[1];
    A.gz = grid->d_points[2];
    A.nx = grid->shape(0);
    A.ny = grid->shape(1);
    A.nz = grid->shape(2);
    A.bubs = bub->d_desc;
    A.nbub = bub->nbub;
    A.lmin = lmin;
    A.nlip = bub->nlip;
    double last;
    lip_first_last(bub->nlip, &A.first, &last);
    PackArgs P{};
    A.head = bub->d_pack;
    A.multiplier = multiplier;
    A.cube = cube;
    const dim3 block(256, 1, 1);  // four 4x4x4 patches along x
    const dim3 g((A.nx + 15) / 16, (A.ny + 3) / 4, (A.nz + 3) / 4);
    hipEvent_t ev;
    prof_begin(ctx, "bubbles_inject_kernel", &ev);
    // on every call: the tables change on the device
    int ncell = 1;
    for (const BubbleHost &h : bub->host) ncell = std::max(ncell, h.ncell);
    P.bubs = A.bubs;
    P.head_dev = bub->d_pack;
    P.nlm = bub->nlm();
    P.nlip = A.nlip;
    double lip[kMaxNlip * kMaxNlip];  // lip[j + nlip*q], decreasing powers
    DAGE_REQUIRE(lip_coeffs(bub->nlip, 1, lip) == 0, DAGE_ERR_ARG, "unsupported bubble nlip");
    for (int j = 0; j < A.nlip; ++j)
        for (int q = 0; q < A.nlip; ++q) P.head[j * kPackW + q] = lip[j + A.nlip * q];
    for (int l = 2; l <= bub->lmax; ++l) {
        double *h = P.head + kHarm + l * l;
        h[0] = std::sqrt((2 * l - 1.0) / (2.0 * l));
        for (int m = 0; m < l; ++m) {
            h[1 + 2 * m] = (2 * l - 1.0) / std::sqrt(1.0 * (l + m) * (l - m));
            h[2 + 2 * m] = std::sqrt((l + m - 1.0) * (l - m - 1.0) / ((l + m) * (l - m)));
        }
    }
    const long pn = ((long)ncell * P.nlm * kPackW + 255) / 256;
    hipLaunchKernelGGL(pack_radial_kernel, dim3((unsigned)std::min<long>(pn, 1024), A.nbub), dim3(256),
                       0, ctx->stream, P);
    DAGE_HIP_CHECK(hipGetLastError());
    switch (bub->lmax) {
    case 0: launch_inject<0>(A, g, block, ctx->stream); break;
    case 1: launch_inject<1>(A, g, block, ctx->stream); break;
    case 2: launch_inject<2>(A, g, block, ctx->stream); break;
    case 3: launch_inject<3>(A, g, block, ctx->stream); break;
    case 4: launch_inject<4>(A, g, block, ctx->stream); break;
    case 5: launch_inject<5>(A, g, block, ctx->stream); break;
    case 6: launch_inject<6>(A, g, block, ctx->stream); break;
    case 7: launch_inject<7>(A, g, block, ctx->stream); break;
    case 8: launch_inject<8>(A, g, block, ctx->stream); break;
    case 9: launch_inject<9>(A, g, block, ctx->stream); break;
    case 10: launch_inject<10>(A, g, block, ctx->stream); break;
    case 11: launch_inject<11>(A, g, block, ctx->stream); break;
    default: launch_inject<12>(A, g, block, ctx->stream); break;
    }
    DAGE_HIP_CHECK(hipGetLastError());
    prof_end(ctx, "bubbles_inject_kernel", ev);
    return DAGE_OK;
}

}  // namespace dage
