// Streaming FP64 passes of the tensor-quadrature apply: the x and y mode
// products in one kernel (no x-pass intermediate in memory) and the z mode
// product with the t-sum in its accumulators.
//
//   stream_xy:  U_t(xo,yo,zi) = w_t sum_yi [sum_xi Fx_t(xo,xi) in(xi,yi,zi)] Fy_t(yi,yo)
//   stream_z:   C(xy,zo) (+)= sum_t sum_zi U_t(xy,zi) Fz_t(zi,zo)
//
// Both run on v_mfma_f64_16x16x4f64 (lane l holds A(l%16, l/16) and
// B(l/16, l%16); result register r of lane l is D(4r + l/16, l%16)).
//
// stream_xy.  A wavefront owns 16 output x points of one (right-hand side, t,
// z-plane).  Its Fx_t columns stay in registers as B fragments for the whole
// plane; the plane streams by in panels of 16 input rows, read from global
// memory straight into A fragments (16 rows of 64 bytes per load), up to three
// blocks ahead.  Per panel
// the x product V(16 yi, 16 xo) leaves the MFMA in exactly the B layout of
// the y product (register r: yi = 4r + l/16, xo = l%16), which multiplies it
// with the panel's Fy_t rows (A fragments from LDS, shared by the block's
// wavefronts) into the accumulators of the output y tiles.  V never leaves
// the registers, the input is read once per tile and U written once, 128
// contiguous bytes at a time.
//   FULL (axes up to 13 tiles of 16): every tile has its accumulator.
//   RING (matrices banded within HB tiles of the diagonal): only the 2HB+1
//   tiles a panel reaches; after panel p the tile p-HB is complete, is stored
//   and the accumulators move up one slot.
//
// stream_z.  A wavefront owns 16 contiguous (xo,yo) columns and up to 13 tiles
// of 16 output z points; U fragments come straight from global memory (four
// rows of 128 bytes per load), Fz_t panels from LDS.
//
// The k-steps (4 input points; pairs of them in the x product) that are zero
// on a whole tile are skipped by wavefront-uniform bit tests, so the passes
// execute the bands of the matrices to 4 or 8 points by 16.
//
// Issue slots, not the MFMAs, bound a first version that tested every address
// and read the matrices in their own layouts (16 other instructions per
// MFMA), so the operands are prepared for the loops: the matrices are packed
// once per operator into 16 x 16 blocks of MFMA fragments, padded with zeros
// (pack_blocks_kernel), and the cubes are accessed through buffer descriptors
// whose range check drops what lies outside.
//
// Measured per call, us (x + y passes -> x/y pass; z pass before -> after):
//   97^3, T = 40, one right-hand side     535 -> 331,   256 -> 139
//   129^3, t 8..27, 12 right-hand sides  6655 -> 3746, 2791 -> 1504
//   385^3, t 10..28, one                15850 -> 9905, 7530 -> 5660
// The executed MFMAs alone take 144, 2138, 5624 (x/y) and 63, 959, 2707 (z).
// The rest is waits for the panel loads at the panel barriers (half the wave
// cycles of the z pass at 97^3) and, at 385^3, the 8.2 GB of U that the
// x/y pass writes and the z pass reads.
#include "dage_internal.hpp"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

namespace dage {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kMaxTiles = 13;  // accumulator tiles of one wavefront

__device__ inline unsigned xcd_tile(unsigned L, unsigned total) {
    const unsigned q = total >> 3, r = total & 7u, x = L & 7u;
    return x * q + min(x, r) + (L >> 3);
}

typedef double d2 __attribute__((ext_vector_type(2)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned long long u64;

// Raw buffer access: loads beyond `bytes` return zero, stores there are
// dropped.  An offset with the top bit set is always outside.
constexpr unsigned kOutside = 0x80000000u;

__device__ inline __amdgpu_buffer_rsrc_t buffer(const double *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, (int)bytes, 0x00027000);
}
__device__ inline double buf_ld(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
__device__ inline d2 buf_ld2(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
__device__ inline void buf_st(__amdgpu_buffer_rsrc_t r, unsigned off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)off, 0, 0);
}

// A packed matrix: block (t, a, b) of 16 x 16 at ((t*na + a)*nb + b)*256,
// where lane l, k-step k (0..3) is element ((k/2)*64 + l)*2 + k%2 of it.
constexpr int kBlk = 256;

// PAIRS (Fx: a = output tile, b = input block): lane l, k-step k is input
// point 8*(k/2) + 2*(l/16) + k%2 of the block, so that a lane's two k-steps
// are neighbours in memory.  Else (Fy, Fz: a = input panel, b = output tile)
// it is input point 4k + l/16.  The output point is l%16 of the tile.
// Element (input i, output o) of t at f[i*si + o*so + t*st].
template <bool PAIRS>
__global__ void __launch_bounds__(256) pack_blocks_kernel(const double *f, long si, long so,
                                                          long st, int ni, int no, int na, int nb,
                                                          long total, double *out) {
    for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += gridDim.x * 256L) {
        const int q = (int)(e & 255);
        long r = e >> 8;
        const int b = (int)(r % nb);
        r /= nb;
        const int a = (int)(r % na);
        const long t = r / na;
        const int l = (q >> 1) & 63, k = 2 * (q >> 7) + (q & 1);
        int i, o = 16 * (PAIRS ? a : b) + (l & 15);
        if (PAIRS) {
            // the pair of the last point of an odd axis is loaded one point
            // early (tail_delta): the point is its second element
            i = 16 * b + 8 * (k >> 1) + 2 * (l >> 4);
            i = i + 1 == ni ? ((k & 1) ? i : ni) : i + (k & 1);
        } else {
            i = 16 * a + 4 * k + (l >> 4);
        }
        out[e] = (i < ni && o < no) ? f[i * si + o * so + t * st] : 0.0;
    }
}

// Wavefronts per SIMD of stream_xy_kernel<N> and stream_z_kernel<N>: as many
// as the accumulators, Fx and the loads in flight leave registers for.
constexpr int xy_waves(int n, int w) {  // blocks of w wavefronts
    return n <= 2 ? 4 : (n <= 5 ? 3 : (n <= 9 || (n == 10 && w == 4) ? 2 : 1));
}
constexpr int z_waves(int n) { return n <= 6 ? 4 : (n <= 9 ? 3 : 2); }

struct StreamXY {
    const double *in;       // in_b(xi, yi, zi) at in + b*nin + xi + nxi*(yi + nyi*zi)
    const double *fxp, *fyp;  // packed Fx (nxt x nxb blocks) and Fy (nyb x nyt)
    double *U;              // U_{b,t} at U + b*Ub + (t - tu)*Ut + xo + nxo*(yo + nyo*zi)
    const double *w;        // weight of (b, t): w[b*wS + t]
    long wS, nin, Ut, Ub;
    int nxi, nyi, nzi, nxo, nyo;
    int t0, tcount, tu;     // this launch's t-points; t of U's first slot
    const int2 *xr, *yr;    // xr[t*nxt + x tile], yr[t*nyt + y tile]: their k-step ranges
    int nxt, nxb, nyt, nyb; // 16-point blocks of the axes (t: output, b: input)
    int groups;             // groups of W output x tiles
};

template <int N, int W, bool RING>
__global__ void __launch_bounds__(64 * W)
    __attribute__((amdgpu_waves_per_eu(xy_waves(N, W))))
    stream_xy_kernel(StreamXY a) {
    constexpr int HB = (N - 1) / 2;
    constexpr int FT = 128 * N;                       // 16-byte pieces of an Fy panel
    constexpr int FW = (FT + 64 * W - 1) / (64 * W);  // per thread
    __shared__ d2 FYs[2][FT];                         // N packed blocks

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15, lk = lane >> 4;
    unsigned L = xcd_tile(blockIdx.x, gridDim.x);
    const int g = (int)(L % (unsigned)a.groups);
    L /= (unsigned)a.groups;
    const int tl = (int)(L % (unsigned)a.tcount);
    L /= (unsigned)a.tcount;
    const int z0 = (int)(L % (unsigned)a.nzi);
    const int b = (int)(L / (unsigned)a.nzi);
    const int t = a.t0 + tl;
    // the idle wavefronts of a short last group fall on another SIMD in
    // every block
    const int slot = (int)((unsigned)(wave + blockIdx.x / (unsigned)a.groups) % (unsigned)W);
    const int it = g * W + slot;
    const bool active = it < a.nxt;
    // first 16-point x block of the window; the full one ends with the axis, so
    // that the block of the axis end is known at compile time
    const int xs = RING ? (active ? it - HB : 0) : a.nxb - N;
    const __amdgpu_buffer_rsrc_t rin =
        buffer(a.in + (long)b * a.nin + (long)z0 * a.nxi * a.nyi,
               8u * (unsigned)a.nxi * (unsigned)a.nyi);
    const d2 *fyp = reinterpret_cast<const d2 *>(a.fyp) + (long)t * a.nyb * a.nyt * (kBlk / 2) -
                    (RING ? HB * (kBlk / 2) : 0) + tid;

    // bit c: 8-point group c of the window holds nonzeros
    unsigned xneed = 0;
    if (active) {
        const int2 r = a.xr[(long)t * a.nxt + it];
        const int lo = __builtin_amdgcn_readfirstlane(r.x) / 2 - 2 * xs;
        const int hi = (__builtin_amdgcn_readfirstlane(r.y) + 1) / 2 - 2 * xs;
        if (lo < hi) xneed = ((1u << hi) - 1u) & ~((1u << lo) - 1u);
    }
    // Fx fragments of the window (blocks outside the axis are not used)
    d2 fx[2 * N];
    {
        const d2 *p = reinterpret_cast<const d2 *>(a.fxp) +
                      (((long)t * a.nxt + (active ? it : 0)) * a.nxb + xs) * (kBlk / 2) + lane;
#pragma unroll
        for (int s = 0; s < 2 * N; ++s) fx[s] = p[64 * s];
    }
    // lane j: the k-steps output y tile j needs.  Held in registers: masks
    // read per panel through scalar loads cost one cache-missing load
    // latency per panel (15 % of the pass at 385^3).
    int ylo = 0, yhi = 0;
    if (active && lane < a.nyt) {
        const int2 r = a.yr[(long)t * a.nyt + lane];
        ylo = r.x;
        yhi = r.y;
    }

    // A fragments of the input panel: this lane's row lrow, points 2*lk and
    // 2*lk + 1 of every group.  Every load of the panel loop is issued on
    // every pass, those without use to an address outside the buffer: the
    // number of loads in flight is then known at compile time and a wait
    // leaves the younger ones in flight (loads behind a branch made every
    // wait drain all of them).
    // Block q of a panel sits in slot q % D and the load of the D-th block
    // after it is issued as soon as it has been used.
    constexpr int D = N <= 3 ? N : 3, NQ = (N + D - 1) / D * D;
    d2 x[2 * D];
    const unsigned prow = 128u * (unsigned)a.nxi;  // bytes per panel
    unsigned xoff = 8u * (unsigned)(a.nxi * lrow + 2 * lk + 16 * xs);
    // the block that holds the axis end: a pair that starts at the last point
    // is loaded one point early (the packed Fx has its factors in the second
    // place), pairs past the end from outside
    const int qend = (a.nxi & 15) ? (a.nxi >> 4) - xs : -1;
    auto tail_delta = [&](int c) {
        const int left = (a.nxi & 15) - 8 * c - 2 * lk;  // points from the pair's first on
        return left >= 2 ? 0u : (left == 1 ? 0u - 8u : kOutside);
    };
    const bool tail = !RING && qend >= 0;
    const unsigned tail0 = RING || tail ? tail_delta(0) : 0u, tail1 = RING || tail ? tail_delta(1) : 0u;
    auto at_end = [&](int q) { return RING ? q == qend : q == N - 1; };
    const bool odd0 = tail0 == 0u - 8u, odd1 = tail1 == 0u - 8u;
    auto load_x = [&](int q, unsigned xm) {
        const unsigned skip = (xm >> (2 * q)) & 3u ? 0u : kOutside;
        const int d = 2 * (q % D);
        x[d] = buf_ld2(rin, (xoff + 128 * q + (at_end(q) ? tail0 : 0u)) | skip);
        x[d + 1] = buf_ld2(rin, (xoff + 128 * q + 64 + (at_end(q) ? tail1 : 0u)) | skip);
    };
    d2 rf[FW];
    // the panel's Fy blocks: all nyt of them, or the window from p - HB (the
    // packed matrix is padded by a window on both sides)
    auto load_fy = [&](int p) {
        const d2 *src = fyp + ((long)p * a.nyt + (RING ? p : 0)) * (kBlk / 2);
#pragma unroll
        for (int r = 0; r < FW; ++r)
            rf[r] = src[64 * W * (r + 1) <= FT ? 64 * W * r : min(64 * W * r, FT - 1 - tid)];
    };
    auto store_fy = [&](int buf) {
#pragma unroll
        for (int r = 0; r < FW; ++r)
            if (64 * W * (r + 1) <= FT || tid + 64 * W * r < FT) FYs[buf][tid + 64 * W * r] = rf[r];
    };

    d4 acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
    const double alpha = a.w[(long)b * a.wS + t];
    const long uplane = (long)a.nxo * a.nyo;
    const __amdgpu_buffer_rsrc_t ru =
        buffer(a.U + (long)b * a.Ub + (long)(t - a.tu) * a.Ut + z0 * uplane,
               8u * (unsigned)a.nxo * (unsigned)a.nyo);
    // this lane's U offset in output row lk (columns past the axis: outside)
    const unsigned ucol = 16 * it + lrow < a.nxo
                              ? 8u * (unsigned)(16 * it + lrow + a.nxo * lk) : kOutside;
    auto store_tile = [&](const d4 &v, int j) {
        const unsigned skip = active && j >= 0 && j < a.nyt ? 0u : kOutside;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            buf_st(ru, (ucol + 8u * (unsigned)a.nxo * (unsigned)(16 * j + 4 * r)) | skip,
                   alpha * v[r]);
    };

    const int np = a.nyb;
    load_fy(0);
#pragma unroll
    for (int q = 0; q < D; ++q)
        if (q < N) load_x(q, xneed);
    store_fy(0);
    __syncthreads();
    for (int p = 0; p < np; ++p) {
        // past the last panel the loads are repeated or lie outside
        load_fy(min(p + 1, np - 1));
        d4 v = d4{0.0, 0.0, 0.0, 0.0};
        // opaque per panel: otherwise every test is hoisted out of the panel
        // loop into (spilled) scalar registers
        unsigned xm = xneed;
        asm volatile("" : "+s"(xm));
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (q < N) {
                const int d = 2 * (q % D);
                if (RING ? __builtin_expect(q == qend, 0) : q == N - 1 && tail) {
                    // the point before the last counts in its own pair; here
                    // it would turn an infinity into a NaN
                    x[d][0] = odd0 ? 0.0 : x[d][0];
                    x[d + 1][0] = odd1 ? 0.0 : x[d + 1][0];
                }
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    if (__builtin_expect((xm >> (2 * q + c)) & 1u, 1)) {
                        v = __builtin_amdgcn_mfma_f64_16x16x4f64(x[d + c][0], fx[2 * q + c][0], v, 0, 0, 0);
                        v = __builtin_amdgcn_mfma_f64_16x16x4f64(x[d + c][1], fx[2 * q + c][1], v, 0, 0, 0);
                    }
            }
            if (q + D == NQ) xoff += prow;  // from here on the next panel
            if (q + D < N) load_x(q + D, xm);
            else if (q + D >= NQ && q + D - NQ < N) load_x(q + D - NQ, xm);
        }
        // bit j of m[k]: accumulator j needs k-step 4p + k
        unsigned m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u64 w = __ballot(4 * p + k >= ylo && 4 * p + k < yhi);
            m[k] = RING ? (unsigned)(p >= HB ? w >> (p - HB) : w << (HB - p)) : (unsigned)w;
        }
        const d2 *fy = FYs[p & 1] + lane;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if ((((m[0] | m[1] | m[2] | m[3]) >> j) & 1u) == 0) continue;
            const d2 f01 = fy[128 * j], f23 = fy[128 * j + 64];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (__builtin_expect((m[k] >> j) & 1u, 1))
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(k < 2 ? f01[k & 1] : f23[k & 1],
                                                                  v[k], acc[j], 0, 0, 0);
        }
        if (RING) {
            store_tile(acc[0], p - HB);
#pragma unroll
            for (int j = 0; j + 1 < N; ++j) acc[j] = acc[j + 1];
            acc[N - 1] = d4{0.0, 0.0, 0.0, 0.0};
        }
        // the other buffer was last read before the previous barrier
        store_fy((p + 1) & 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < (RING ? N - 1 : N); ++j) store_tile(acc[j], RING ? np - HB + j : j);
}

constexpr int kMaxSplits = 16, kMaxGroups = 5;  // of one z launch

struct StreamZ {
    const double *U;    // U_{b,t}(n, zi) at U + b*Ub + (t - tu)*Ut + n + M3*zi
    const double *fzp;  // packed Fz (nzb x nzt blocks)
    double *C;          // partial s of b at C + b*cB + s*cS + n + M3*zo
    long Ut, Ub, cB, cS;
    int M3, nzi, nzo;
    int tu;
    const int4 *steps;  // {t, panel, masks of k-steps 0 and 1, of 2 and 3}
    int nzt, nzb;
    int ngroups, mgroups, splits;
    int ninit;          // partials below this: C += instead of C =
    int2 cut[kMaxGroups][kMaxSplits];  // steps [x, y) of each group and split
};

template <int N>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(z_waves(N))))
    stream_z_kernel(StreamZ a) {
    constexpr int FT = 128 * N, FW = (FT + 255) / 256;
    __shared__ d2 FZs[2][FT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15, lk = lane >> 4;
    unsigned L = xcd_tile(blockIdx.x, gridDim.x);
    const int mg = (int)(L % (unsigned)a.mgroups);
    L /= (unsigned)a.mgroups;
    const int ng = (int)(L % (unsigned)a.ngroups);
    L /= (unsigned)a.ngroups;
    const int sp = (int)(L % (unsigned)a.splits);
    const int b = (int)(L / (unsigned)a.splits);
    const int j0 = mg * N;
    const long n0 = ((long)ng * 4 + wave) * 16 + lrow;
    const int i0 = a.cut[mg][sp].x, i1 = a.cut[mg][sp].y;

    d4 acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};

    if (i0 < i1) {
        // Lane l holds step base + l of the list, and of the next 64: a step
        // costs register reads only (masks read per panel through scalar
        // loads cost a load latency per panel).
        int base = i0;
        auto chunk = [&](int c) { return a.steps[min(c + lane, i1 - 1)]; };
        int4 st = chunk(base), sn = chunk(base + 64);
        auto rd = [&](int v, int i) { return __builtin_amdgcn_readlane(v, i - base); };
        // rows of the panel past the axis end lie outside its buffer
        const unsigned uo = n0 < a.M3 ? 8u * (unsigned)(n0 + (long)a.M3 * lk) : kOutside;
        const unsigned urow = 32u * (unsigned)a.M3;
        const double *Ub = a.U + (long)b * a.Ub;
        const d2 *fz = reinterpret_cast<const d2 *>(a.fzp) + (long)j0 * (kBlk / 2) + tid;
        d2 rf[FW];
        double u[2][4];
        auto load_fz = [&](int t, int p) {  // every load is unconditional (see stream_xy_kernel)
            const d2 *src = fz + ((long)t * a.nzb + p) * a.nzt * (kBlk / 2);
#pragma unroll
            for (int r = 0; r < FW; ++r)
                rf[r] = src[256 * (r + 1) <= FT ? 256 * r : min(256 * r, FT - 1 - tid)];
        };
        auto load_u = [&](double (&d)[4], int t, int p) {
            const __amdgpu_buffer_rsrc_t r =
                buffer(Ub + (long)(t - a.tu) * a.Ut + (long)a.M3 * (16 * p),
                       8u * (unsigned)a.M3 * (unsigned)min(16, a.nzi - 16 * p));
#pragma unroll
            for (int k = 0; k < 4; ++k) d[k] = buf_ld(r, uo + urow * (unsigned)k);
        };
        auto store = [&](int buf) {
#pragma unroll
            for (int r = 0; r < FW; ++r)
                if (256 * (r + 1) <= FT || tid + 256 * r < FT) FZs[buf][tid + 256 * r] = rf[r];
        };
        // U is loaded two steps ahead (it comes from memory), Fz one step
        // ahead (from the L2); past the end the last step's loads repeat.
        int t1, p1, m01 = rd(st.z, i0), m23 = rd(st.w, i0), n01, n23;
        load_fz(rd(st.x, i0), rd(st.y, i0));
        load_u(u[0], rd(st.x, i0), rd(st.y, i0));
        {
            const int i = min(i0 + 1, i1 - 1);
            t1 = rd(st.x, i), p1 = rd(st.y, i), n01 = rd(st.z, i), n23 = rd(st.w, i);
        }
        load_u(u[1], t1, p1);
        store(0);
        __syncthreads();
        int i = i0;
        auto step = [&](int slot) {
            double cu[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) cu[k] = u[slot][k];
            load_fz(t1, p1);
            const int in = min(i + 2, i1 - 1);
            if (in - base >= 64) {
                base += 64;
                st = sn;
                sn = chunk(base + 64);
            }
            t1 = rd(st.x, in), p1 = rd(st.y, in);
            const unsigned a01 = (unsigned)m01, a23 = (unsigned)m23;
            m01 = n01, m23 = n23, n01 = rd(st.z, in), n23 = rd(st.w, in);
            load_u(u[slot], t1, p1);
            const unsigned any = a01 | (a01 >> 16) | a23 | (a23 >> 16);
            const d2 *f = FZs[slot] + lane;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (((any >> j) & 1u) == 0) continue;
                const d2 f01 = f[128 * j], f23 = f[128 * j + 64];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (__builtin_expect(((k < 2 ? a01 : a23) >> (j + 16 * (k & 1))) & 1u, 1))
                        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            k < 2 ? f01[k & 1] : f23[k & 1], cu[k], acc[j], 0, 0, 0);
            }
            store(slot ^ 1);
            __syncthreads();
            ++i;
        };
        while (true) {
            step(0);
            if (i >= i1) break;
            step(1);
            if (i >= i1) break;
        }
    }
    double *C = a.C + (long)b * a.cB + (long)sp * a.cS;
    const bool add = sp < a.ninit;
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int zo = 16 * (j0 + j) + 4 * r + lk;
            if (zo < a.nzo && n0 < a.M3) {
                double *d = C + n0 + (long)a.M3 * zo;
                *d = add ? *d + acc[j][r] : acc[j][r];
            }
        }
}

template <int N, int W, bool RING>
int launch_xy_w(const StreamXY &a0, int B, hipStream_t s) {
    StreamXY a = a0;
    a.groups = (a.nxt + W - 1) / W;
    const long blocks = (long)a.groups * a.tcount * a.nzi * B;
    DAGE_REQUIRE(blocks > 0 && blocks < (1L << 31), DAGE_ERR_ARG,
                 "x/y pass of %ld blocks does not fit one launch", blocks);
    hipLaunchKernelGGL((stream_xy_kernel<N, W, RING>), dim3((unsigned)blocks), dim3(64 * W), 0, s, a);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

// Wavefronts per block of stream_xy_kernel<N> for nxt x tiles: the group size
// that leaves the fewest idle, of those that fill the SIMDs (3 per block only
// with 3 per SIMD: with 2, two of a CU's eight slots stay empty; 385^3, 25 x
// tiles, N = 7 and 9: 12.0 -> 10.0 ms with 2 instead of 3)
int group_size(int N, int nxt) {
    auto idle = [&](int w) { return (nxt + w - 1) / w * w - nxt; };
    const int w = N >= 3 && N <= 5 ? 3 : 2;
    return idle(w) < idle(4) ? w : 4;
}

template <int N, bool RING>
int launch_xy_n(const StreamXY &a, int B, hipStream_t s) {
    constexpr int w = N >= 3 && N <= 5 ? 3 : 2;
    if (group_size(N, a.nxt) == w) return launch_xy_w<N, w, RING>(a, B, s);
    return launch_xy_w<N, 4, RING>(a, B, s);
}

template <int N>
int launch_z(const StreamZ &a, int B, hipStream_t s) {
    const long blocks = (long)a.mgroups * a.ngroups * a.splits * B;
    DAGE_REQUIRE(blocks > 0 && blocks < (1L << 31), DAGE_ERR_ARG,
                 "z pass of %ld blocks does not fit one launch", blocks);
    hipLaunchKernelGGL(stream_z_kernel<N>, dim3((unsigned)blocks), dim3(256), 0, s, a);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

// Groups of output z tiles and the tiles of each.
void z_groups(long nzo, int *groups, int *tiles) {
    const int nt = (int)((nzo + 15) / 16);
    *groups = (nt + kMaxTiles - 1) / kMaxTiles;
    *tiles = (nt + *groups - 1) / *groups;
}

}  // namespace

// The tile ranges of one axis: rows of t (n of them, span lo/hi per row,
// first at row0, stride rs per point) -> [first, last+1) k-step per output
// tile, and the smallest half-width in tiles that covers them.
int tile_ranges(const int *span, long row0, long n, long no, int2 *out) {
    const int nt = (int)((no + 15) / 16);
    int hb = 0;
    for (int j = 0; j < nt; ++j) {
        const int a = 16 * j, b = (int)std::min<long>(a + 16, no);
        long lo = -1, hi = -1;
        for (long i = 0; i < n; ++i) {
            const long r = row0 + i;
            if (span[2 * r] < b && span[2 * r + 1] >= a) {
                if (lo < 0) lo = i;
                hi = i;
            }
        }
        out[j] = lo < 0 ? make_int2(0, 0) : make_int2((int)(lo / 4), (int)(hi / 4 + 1));
        if (lo >= 0)
            hb = std::max(hb, std::max(j - (int)(lo / 16), (int)(hi / 16) - j));
    }
    return hb;
}

// Ranges, packed matrices and tables of the streamed passes (axes up to 1024
// points: the ranges only beyond); span: the row spans of
// build_masks (x rows t*nxi.., then y, then z).
int build_stream(dage_operator op, const std::vector<int> &span) {
    const long T = op->ntp;
    long nt[3], nb[3], row[3], ranges = 0, r0 = 0;
    size_t pk = 0, off[3];
    for (int a = 0; a < 3; ++a) {
        nt[a] = (op->dout[a] + 15) / 16;
        nb[a] = (op->din[a] + 15) / 16;
        row[a] = r0;
        r0 += T * op->din[a];
        ranges += T * nt[a];
        // a window of kMaxTiles blocks before and after each matrix
        off[a] = pk + kMaxTiles * (size_t)kBlk;
        pk += ((size_t)T * nt[a] * nb[a] + 2 * kMaxTiles) * kBlk;
    }
    std::vector<int2> rg(ranges);
    op->tile_hb.assign(T, 0);
    op->tile_blocks.assign(T, make_int2(0, 0));
    int2 *rp = rg.data();
    for (int a = 0; a < 3; ++a) {
        for (long t = 0; t < T; ++t) {
            int2 *r = rp + t * nt[a];
            const int hb = tile_ranges(span.data(), row[a] + t * op->din[a], op->din[a],
                                       op->dout[a], r);
            if (a == 2) continue;
            op->tile_hb[t] = std::max(op->tile_hb[t], hb);
            int n = 0;  // 16 x 16 blocks
            for (long j = 0; j < nt[a]; ++j) n += r[j].x < r[j].y ? (r[j].y + 3) / 4 - r[j].x / 4 : 0;
            (a == 0 ? op->tile_blocks[t].x : op->tile_blocks[t].y) = n;
        }
        rp += T * nt[a];
    }
    hipStream_t s = op->ctx->stream;
    const size_t rb = sizeof(int2) * rg.size();
    if (!op->d_ranges) DAGE_HIP_CHECK(hipMalloc((void **)&op->d_ranges, rb));
    DAGE_HIP_CHECK(hipMemcpyAsync(op->d_ranges, rg.data(), rb, hipMemcpyHostToDevice, s));
    for (int a = 0; a < 3; ++a)
        if (op->din[a] > 1024 || op->dout[a] > 1024) {  // 64 tiles per mask
            DAGE_HIP_CHECK(hipStreamSynchronize(s));
            return DAGE_OK;
        }
    // z steps: the panels of every t that some tile of the group needs, split
    // s of S taking the panels p of t with (t*nb + p) % S = s.  One list per
    // S: the split of the sum does not depend on which panels are skipped.
    std::vector<int4> st;
    op->z_off.clear();
    {
        const int2 *zr = rg.data() + T * (nt[0] + nt[1]);
        int G, N;
        z_groups(op->dout[2], &G, &N);
        std::vector<int4> all;
        for (int g = 0; g < G; ++g) {
            all.clear();
            for (long t = 0; t < T; ++t)
                for (int p = 0; p < nb[2]; ++p) {
                    unsigned m[4] = {0, 0, 0, 0};
                    for (int j = 0; j < N && g * N + j < nt[2]; ++j) {
                        const int2 r = zr[t * nt[2] + g * N + j];
                        for (int k = 0; k < 4; ++k)
                            if (4 * p + k >= r.x && 4 * p + k < r.y) m[k] |= 1u << j;
                    }
                    if (m[0] | m[1] | m[2] | m[3])
                        all.push_back(make_int4((int)t, p, (int)(m[0] | m[1] << 16),
                                                (int)(m[2] | m[3] << 16)));
                }
            for (int S = 1; S <= kMaxSplits; ++S)
                for (int k = 0; k < S; ++k) {
                    op->z_off.push_back((int)st.size());
                    for (const int4 &e : all)
                        if ((e.x * nb[2] + e.y) % S == k) st.push_back(e);
                }
        }
        op->z_off.push_back((int)st.size());
        op->z_t.resize(st.size());
        for (size_t i = 0; i < st.size(); ++i) op->z_t[i] = st[i].x;
    }
    if (!op->d_steps)  // every panel of every t, whatever the matrices hold
        DAGE_HIP_CHECK(hipMalloc((void **)&op->d_steps,
                                 sizeof(int4) * (size_t)(kMaxGroups * kMaxSplits * T * nb[2])));
    DAGE_HIP_CHECK(hipMemcpyAsync(op->d_steps, st.data(), sizeof(int4) * st.size(),
                                  hipMemcpyHostToDevice, s));
    if (!op->d_pack) {
        DAGE_HIP_CHECK(hipMalloc((void **)&op->d_pack, 8 * pk));
        DAGE_TRY(fill_zero(op->ctx, op->d_pack, pk));
    }
    // Fx (nxo, nxi, T): element (i, o) at i*nxo + o; Fy, Fz (ni, no, T): i + o*ni
    const double *src[3] = {op->d_fx, op->d_fy, op->d_fz};
    for (int a = 0; a < 3; ++a) {
        const long total = T * nt[a] * nb[a] * kBlk;
        const long ni = op->din[a], no = op->dout[a];
        const dim3 grid((unsigned)std::min<long>((total + 255) / 256, 65536));
        if (a == 0)
            hipLaunchKernelGGL(pack_blocks_kernel<true>, grid, dim3(256), 0, s, src[a], no, 1L,
                               ni * no, (int)ni, (int)no, (int)nt[a], (int)nb[a], total,
                               op->d_pack + off[a]);
        else
            hipLaunchKernelGGL(pack_blocks_kernel<false>, grid, dim3(256), 0, s, src[a], 1L, ni,
                               ni * no, (int)ni, (int)no, (int)nb[a], (int)nt[a], total,
                               op->d_pack + off[a]);
        DAGE_HIP_CHECK(hipGetLastError());
        op->pack_off[a] = off[a];
    }
    DAGE_HIP_CHECK(hipStreamSynchronize(s));  // the host tables go out of scope
    return DAGE_OK;
}

void stream_mats(dage_operator op, ApplyMats *m) {
    if (!op->d_ranges) return;
    m->xr = op->d_ranges;
    m->yr = m->xr + (long)op->ntp * ((op->dout[0] + 15) / 16);
    if (!op->d_pack) return;
    m->fxp = op->d_pack + op->pack_off[0];
    m->fyp = op->d_pack + op->pack_off[1];
    m->fzp = op->d_pack + op->pack_off[2];
    m->hb = op->tile_hb.data();
    m->blocks = op->tile_blocks.data();
    m->zsteps = op->d_steps;
    m->z_off = op->z_off.data();
    m->z_t = op->z_t.data();
}

// Accumulator tiles of t's x/y pass: the ring that covers its band, or every
// tile of the axes when those are fewer (negative); 0: neither fits.
static int xy_tiles(const ApplyMats &m, int t) {
    auto tiles = [](int n) { return (n + 15) / 16; };
    const int full = std::max(std::max(tiles(m.din[0]), tiles(m.dout[0])),
                              std::max(tiles(m.din[1]), tiles(m.dout[1])));
    const bool square = m.din[0] == m.dout[0] && m.din[1] == m.dout[1] && m.dout[1] <= 1024;
    const int ring = square ? 2 * std::max(1, m.hb[t]) + 1 : kMaxTiles + 1;
    if (ring <= kMaxTiles && ring < full) return ring;
    // four tiles run on five: a kernel of four spilled at three wavefronts per
    // SIMD and is slower at two (57^3: 101 and 86 us, 74 on five)
    return full <= kMaxTiles ? -std::max(full == 4 ? 5 : full, 2) : 0;
}

// DAGE_APPLY_STREAM (read at every call): 0 never streams, 1 wherever it can
// (comparison runs, tests), else where it is faster (stream_pays).
static char stream_mode() {
    const char *e = std::getenv("DAGE_APPLY_STREAM");
    return e ? e[0] : 0;
}

// Whether the streamed passes take this operator's sizes at all.
static bool streams(const ApplyMats &m) {
    if (!m.fxp) return false;
    // byte offsets within a plane of the cubes and 16 planes of U below 2^31
    if ((long)m.din[0] * (m.din[1] + 32) >= (1L << 28)) return false;
    if ((long)m.dout[0] * (m.dout[1] + 16) >= (1L << 24)) return false;
    return stream_mode() != '0';
}

int stream_count(const ApplyMats &m, int t0, int t1) {
    int n = 0;
    if (streams(m))
        for (int t = t0; t < t1; ++t) n += xy_tiles(m, t) != 0;
    return n;
}

// Rounds of the card's wavefront slots below which a launch is not worth its
// narrower ring: its blocks start and end together, and the tail costs more
// than the registers saved.  Fewest launches (one kernel for all) / this line
// / a launch per ring width: 65^3 110 / 110 / 123 us, 97^3 349 / 331 / 348,
// 193^3 3395 / 2913 / 2914, 385^3 11888 / 9905 / 9902.
constexpr double kMinRounds = 2.0;

// Number of leading t-points of [t0, t1) that one stream_xy launch of B
// right-hand sides takes (0: the first one cannot run streamed), and its
// accumulator tiles.
int stream_run(const ApplyMats &m, int t0, int t1, int B, int *tiles) {
    if (t0 >= t1 || !streams(m)) return 0;
    int end = t0;
    while (end < t1 && xy_tiles(m, end) != 0) ++end;
    // rounds of the card's wavefront slots that n t-points fill
    const double waves = (double)((m.dout[0] + 15) / 16) * m.din[2] * B;
    auto rounds = [&](int n, int c) { return n * waves / (1024.0 * xy_waves(std::abs(c), 2)); };
    auto wider = [](int a, int b) { return a < 0 || b < 0 ? std::min(a, b) : std::max(a, b); };
    int e = t0, code = 0;
    while (e < end) {
        int n = xy_tiles(m, e), f = e + 1;
        while (f < end && xy_tiles(m, f) == n) ++f;
        if (e > t0 && rounds(e - t0, code) >= kMinRounds) {
            // the run is long enough; so must be what it leaves
            int w = 0;
            for (int t = e; t < end; ++t) w = wider(w, xy_tiles(m, t));
            if (rounds(end - e, w) >= kMinRounds) break;
        }
        code = e > t0 ? wider(code, n) : n;
        e = f;
    }
    *tiles = code;
    return e - t0;
}

// Estimated us of the x and y products of [t0, t1) on the streamed and on the
// separate passes.  Both grow with the 16 x 16 blocks that the matrices need,
// but the streamed kernel pads the x axis to whole tiles and groups of
// wavefronts and loads its whole window for every wavefront and panel, while
// the separate passes pad only the flattened rows: thin boxes are slower
// streamed (9 x 213 x 145 points: 579 against 172 us, 41 x 401 x 41: 651
// against 394).  The coefficients are least-squares fits to the measured times
// of 1380 boxes, pairs of grids and batches with axes of 5 to 421 points
// (standard deviation 14 % streamed, 17 % separate).  Streaming needs a margin of
// 5 %: with it the call is slower than without in under 1 % of them by more
// than 5 %, and of the boxes with sides within 1.6 of each other all but one of
// 236 stream (they gain 1.1 to 1.8).
constexpr double kLaunch = 5.2;   // a launch
constexpr double kStart = 2.1;    // a wavefront's Fx window and first loads
constexpr double kPanel = 0.81;   // a panel
constexpr double kLoad = 0.116;   // a block of a wavefront's window, per panel
constexpr double kBlock = 0.111;  // a block's products
constexpr double kBesides = 10.0; // the separate passes' launches beside
constexpr double kSepLaunch = 11.3;       // the two passes
constexpr double kSepStep = 1.06;         // a panel of either sum
constexpr double kSepBlock = 1.41e-3;     // a block's products of 64 rows
constexpr double kSepPanel = 3.8e-4;      // the rows' panels
constexpr double kMargin = 1.05;

static void xy_costs(const ApplyMats &m, int t0, int t1, int B, double *stream, double *separate) {
    const int nxt = (m.dout[0] + 15) / 16, nxb = (m.din[0] + 15) / 16;
    const int nyb = (m.din[1] + 15) / 16;
    const double rx = (m.din[1] * (long)m.din[2] + 63) / 64 * (double)B;
    const double ry = (m.dout[0] * (long)m.din[2] + 63) / 64 * (double)B;
    bool rest = false;  // t-points that run separately in any case
    *stream = *separate = 0.0;
    for (int t = t0, r, code = 0; t < t1; t += r) {
        r = stream_run(m, t, t1, B, &code);
        if (r == 0) {
            rest = true;
            r = 1;
            continue;
        }
        double x = 0.0, y = 0.0;
        for (int e = t; e < t + r; ++e) x += m.blocks[e].x, y += m.blocks[e].y;
        *separate += kSepBlock * (rx * x + ry * y) + kSepPanel * (rx * x / nxb + ry * y / nyb);
        // wavefronts per SIMD, those of them with work, rounds of the card
        const int N = std::abs(code), W = group_size(N, nxt), groups = (nxt + W - 1) / W;
        const double w = xy_waves(N, W), act = w * nxt / (groups * W);
        const double rounds = (double)groups * W * r * m.din[2] * B / (1024.0 * w);
        const double blk = kBlock * (x / nxt + y / nyb) / r;  // of a wavefront's panel
        const double one = kPanel + kLoad * N + blk;
        const double round = kStart + nyb * std::max(one, kLoad * N * w + blk * act);
        *stream += kLaunch + std::max(0.5 * kStart + nyb * one, rounds * round);
    }
    if (rest) *stream += kBesides;
    else *separate += kSepLaunch + kSepStep * (nxb + nyb);
}

// Whether the t-points of [t0, t1) that can run streamed do.
bool stream_pays(const ApplyMats &m, int t0, int t1, int B) {
    if (stream_count(m, t0, t1) == 0) return false;
    if (stream_mode() == '1') return true;
    double stream, separate;
    xy_costs(m, t0, t1, B, &stream, &separate);
    return kMargin * stream <= separate;
}

int stream_xy(dage_ctx ctx, const ApplyMats &m, int tiles, const double *in, double *U, long Ut,
              long Ub, int tu, const double *w, long wS, int t0, int tc, int B, const char *name) {
    StreamXY a{};
    a.in = in; a.fxp = m.fxp; a.fyp = m.fyp; a.U = U; a.w = w;
    a.wS = wS; a.Ut = Ut; a.Ub = Ub;
    a.nxi = m.din[0]; a.nyi = m.din[1]; a.nzi = m.din[2];
    a.nxo = m.dout[0]; a.nyo = m.dout[1];
    a.nin = (long)a.nxi * a.nyi * a.nzi;
    a.t0 = t0; a.tcount = tc; a.tu = tu;
    a.xr = m.xr; a.yr = m.yr;
    a.nxt = (a.nxo + 15) / 16; a.nyt = (a.nyo + 15) / 16;
    a.nxb = (a.nxi + 15) / 16; a.nyb = (a.nyi + 15) / 16;
    if (ctx->profiling) {
        char kernel[32];
        std::snprintf(kernel, sizeof kernel, "stream_xy_%s%d", tiles < 0 ? "full" : "ring", std::abs(tiles));
        prof_count(ctx, kernel);
    }
    hipEvent_t ev;
    prof_begin(ctx, name, &ev);
    int rc = DAGE_OK;
    hipStream_t s = ctx->stream;
    switch (tiles) {
    case 3: rc = launch_xy_n<3, true>(a, B, s); break;
    case 5: rc = launch_xy_n<5, true>(a, B, s); break;
    case 7: rc = launch_xy_n<7, true>(a, B, s); break;
    case 9: rc = launch_xy_n<9, true>(a, B, s); break;
    case 11: rc = launch_xy_n<11, true>(a, B, s); break;
    case 13: rc = launch_xy_n<13, true>(a, B, s); break;
    case -2: rc = launch_xy_n<2, false>(a, B, s); break;
    case -3: rc = launch_xy_n<3, false>(a, B, s); break;
    case -5: rc = launch_xy_n<5, false>(a, B, s); break;
    case -6: rc = launch_xy_n<6, false>(a, B, s); break;
    case -7: rc = launch_xy_n<7, false>(a, B, s); break;
    case -8: rc = launch_xy_n<8, false>(a, B, s); break;
    case -9: rc = launch_xy_n<9, false>(a, B, s); break;
    case -10: rc = launch_xy_n<10, false>(a, B, s); break;
    case -11: rc = launch_xy_n<11, false>(a, B, s); break;
    case -12: rc = launch_xy_n<12, false>(a, B, s); break;
    case -13: rc = launch_xy_n<13, false>(a, B, s); break;
    default: DAGE_REQUIRE(false, DAGE_ERR_STATE, "t-point %d is not streamed", t0);
    }
    prof_end(ctx, name, ev);
    return rc;
}

// Splits of the z pass's steps at B right-hand sides.  A block holds one
// wavefront per SIMD, so the pass takes as long as the most blocks a CU gets
// times their length; each split adds a write and a read of C, 4 % of the
// unsplit pass.  97^3 (148 blocks unsplit): 177 / 176 / 150 / 164 / 182 us at
// 3 / 4 / 5 / 6 / 7 splits; 31^3: 41 us unsplit, 9 at 12 or more.
int z_splits(const ApplyMats &m, int B) {
    const long M3 = (long)m.dout[0] * m.dout[1];
    int G, N;
    z_groups(m.dout[2], &G, &N);
    const long blocks = (M3 + 63) / 64 * G * B;
    int best = 1;
    double cost = 1e300;
    for (int k = 1; k <= kMaxSplits; ++k) {
        const double c = (double)((blocks * k + 255) / 256) / k + 0.04 * k * blocks / 256;
        if (c < cost) cost = c, best = k;
    }
    return best;
}

int stream_z(dage_ctx ctx, const ApplyMats &m, const double *U, long Ut, long Ub, int tu, double *C,
             long cB, long cS, int splits, int ninit, int t0, int tc, int B,
             const char *name) {
    StreamZ a{};
    a.U = U; a.fzp = m.fzp; a.C = C;
    a.Ut = Ut; a.Ub = Ub; a.cB = cB; a.cS = cS;
    a.M3 = m.dout[0] * m.dout[1];
    a.nzi = m.din[2]; a.nzo = m.dout[2];
    a.tu = tu;
    a.steps = m.zsteps;
    a.nzt = (a.nzo + 15) / 16; a.nzb = (a.nzi + 15) / 16;
    a.splits = splits;
    a.ninit = ninit;
    int n;
    z_groups(a.nzo, &a.mgroups, &n);
    a.ngroups = (a.M3 + 63) / 64;
    DAGE_REQUIRE(a.mgroups <= kMaxGroups && splits >= 1 && splits <= kMaxSplits, DAGE_ERR_STATE,
                 "%d groups, %d splits of a z pass", a.mgroups, splits);
    for (int g = 0; g < a.mgroups; ++g)
        for (int k = 0; k < splits; ++k) {
            const int *off = m.z_off + (g * kMaxSplits * (kMaxSplits + 1) + splits * (splits - 1)) / 2 + k;
            auto first = [&](int t) {
                return (int)(std::lower_bound(m.z_t + off[0], m.z_t + off[1], t) - m.z_t);
            };
            a.cut[g][k] = make_int2(first(t0), first(t0 + tc));
        }
    hipEvent_t ev;
    prof_begin(ctx, name, &ev);
    int rc = DAGE_OK;
    hipStream_t s = ctx->stream;
    switch (n) {
    case 1: rc = launch_z<1>(a, B, s); break;
    case 2: rc = launch_z<2>(a, B, s); break;
    case 3: rc = launch_z<3>(a, B, s); break;
    case 4: rc = launch_z<4>(a, B, s); break;
    case 5: rc = launch_z<5>(a, B, s); break;
    case 6: rc = launch_z<6>(a, B, s); break;
    case 7: rc = launch_z<7>(a, B, s); break;
    case 8: rc = launch_z<8>(a, B, s); break;
    case 9: rc = launch_z<9>(a, B, s); break;
    case 10: rc = launch_z<10>(a, B, s); break;
    case 11: rc = launch_z<11>(a, B, s); break;
    case 12: rc = launch_z<12>(a, B, s); break;
    default: rc = launch_z<13>(a, B, s); break;
    }
    prof_end(ctx, name, ev);
    return rc;
}

}  // namespace dage
