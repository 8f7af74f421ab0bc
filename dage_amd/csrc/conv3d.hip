// 3x3x3 convolution layers for the learned orbital-update preconditioner:
// BF16 weights, FP32 activations and FP32 accumulation, zero padding,
// forward / backward-data / backward-filter, plus the Adam step, the MSE
// loss and FP64 <-> FP32 conversions between SCF cubes and activations.
//
// Layout: activations [c][z][y][x] (x fastest: the cube layout, one cube per
// channel); weights [cout][cin][27] with tap = (dx+1) + 3 (dy+1) + 9 (dz+1);
// BF16 weights are the upper 16 bits of the FP32 master weights rounded to
// nearest even.  Every reduction (filter gradient, loss) is a fixed-order
// two-stage sum, so training is deterministic.
//
// The 16 -> 16 layers (forward, and backward-data as the same convolution
// with transposed, mirrored weights) run on bf16 MFMA: every FP32 activation
// is split into three bf16 terms (24 bits, so the products are as exact as
// FP32 ones) and multiplied with the bf16 weights, FP32 accumulation.  A
// block streams along z through its (16*NS) x 4 column of the volume: one
// input plane (with a one-point halo) sits in LDS, pre-split, and feeds the
// three output planes it touches, whose accumulators stay in registers; the
// weights stay in registers as MFMA operands for the whole launch.
// Algorithmic work: 2*16*16*27 = 13824 FLOPs per voxel (dense, as FP32);
// HBM roofline 128 bytes per voxel (16 channels in and out, FP32).
//
// Forward and backward-data layers with 1 or 2 channels on a side run as FP32
// VALU kernels, the filter gradients on FP32 MFMA.
#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "dage_internal.hpp"

namespace dage {
namespace {

constexpr int kMaxC = 16;

int use_device(dage_ctx ctx) {
    DAGE_REQUIRE(ctx != nullptr, DAGE_ERR_ARG, "null context handle");
    DAGE_HIP_CHECK(hipSetDevice(ctx->device));
    return DAGE_OK;
}

int grid_of(long n) { return (int)std::min<long>((n + 255) / 256, 65536); }

__device__ inline float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline uint16_t f32_to_bf16(float f) {
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
    const uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);                    // nearest even
    return (uint16_t)(r >> 16);
}

// The VALU layers' weight table: w[(o*cin + c)*27 + t] (bf16) as FP32 at
// wf[(c*27 + t)*cout + o], so one (c, t) tap's cout weights are contiguous.
__global__ void __launch_bounds__(256) weights_f32_kernel(const uint16_t *w, int cout, int cin,
                                                          float *wf) {
    const int n = cout * cin * 27;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int o = i / (cin * 27), ct = i - o * (cin * 27);
        wf[ct * cout + o] = bf16_to_f32(w[i]);
    }
}

// The weights (FP32 copies of the bf16 values) are read at wavefront-uniform
// indices through scalar loads, so every multiply-add takes its weight from
// a scalar register; no LDS, no per-lane weight loads.
template <int COUT>
__global__ void __launch_bounds__(256) conv_fwd_kernel(const float *__restrict__ in, int cin,
                                                       const float *__restrict__ wf,
                                                       const float *__restrict__ bias, int relu,
                                                       float *__restrict__ out, int nx, int ny,
                                                       int nz) {
    typedef const float __attribute__((address_space(1))) *gfptr;
    const gfptr ws = (gfptr)wf;
    const gfptr bs = (gfptr)bias;
    const long vol = (long)nx * ny * nz;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < vol;
         p += (long)gridDim.x * blockDim.x) {
        const int x = (int)(p % nx);
        const long r = p / nx;
        const int y = (int)(r % ny);
        const int z = (int)(r / ny);
        float acc[COUT];
#pragma unroll
        for (int o = 0; o < COUT; ++o) acc[o] = bs[o];
        for (int c = 0; c < cin; ++c) {
            const float *ic = in + (long)c * vol;
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
                const int xx = x + dx, yy = y + dy, zz = z + dz;
                const bool ok = xx >= 0 && xx < nx && yy >= 0 && yy < ny && zz >= 0 && zz < nz;
                const float v = ok ? ic[xx + (long)nx * (yy + (long)ny * zz)] : 0.0f;
#pragma unroll
                for (int o = 0; o < COUT; ++o) acc[o] += ws[(c * 27 + t) * COUT + o] * v;
            }
        }
#pragma unroll
        for (int o = 0; o < COUT; ++o)
            out[(long)o * vol + p] = (relu && acc[o] < 0.0f) ? 0.0f : acc[o];
    }
}

// gin[c][p] = sum_o sum_t W[o][c][t] gout[o][p - off(t)]
__global__ void __launch_bounds__(256) conv_bwd_data_kernel(const float *gout, int cout, int cin,
                                                            const uint16_t *w, float *gin, int nx,
                                                            int ny, int nz) {
    __shared__ float ws[kMaxC * kMaxC * 27];
    const int nw = cout * cin * 27;
    for (int i = threadIdx.x; i < nw; i += 256) ws[i] = bf16_to_f32(w[i]);
    __syncthreads();
    const long vol = (long)nx * ny * nz;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < vol;
         p += (long)gridDim.x * blockDim.x) {
        const int x = (int)(p % nx);
        const long r = p / nx;
        const int y = (int)(r % ny);
        const int z = (int)(r / ny);
        float acc[kMaxC];
#pragma unroll
        for (int c = 0; c < kMaxC; ++c) acc[c] = 0.0f;
        for (int o = 0; o < cout; ++o) {
            const float *go = gout + (long)o * vol;
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
                const int xx = x - dx, yy = y - dy, zz = z - dz;
                const bool ok = xx >= 0 && xx < nx && yy >= 0 && yy < ny && zz >= 0 && zz < nz;
                const float g = ok ? go[xx + (long)nx * (yy + (long)ny * zz)] : 0.0f;
#pragma unroll
                for (int c = 0; c < kMaxC; ++c)
                    if (c < cin) acc[c] += ws[(o * cin + c) * 27 + t] * g;
            }
        }
        for (int c = 0; c < cin; ++c) gin[(long)c * vol + p] = acc[c];
    }
}

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kCY = 4;  // output y-rows per block: one per wavefront

__device__ inline __bf16 bf16_bits(uint16_t b) { return __builtin_bit_cast(__bf16, b); }

// 16 -> 16 channel 3x3x3 convolution on bf16 MFMA (v_mfma_f32_16x16x32_bf16;
// lane l holds A(l%16, 8(l/16)..+7) and B(8(l/16)..+7, l%16); result
// register r of lane l is D(4(l/16)+r, l%16)).  D rows are 16 x-points of
// one output row, columns the 16 output channels; K = 32 runs over two taps
// (dx, dy) of one dz times 16 input channels, 5 K-steps per dz (the tenth
// tap slot is zero).  Block (bx, by, bz) owns x in [16*NS*bx, +16*NS),
// y in [4*by, +4) (wavefront w: row 4*by + w) and z in [bz*zchunk, +zchunk).
// out = act(sum + bias); bias may be null (zero).
template <int NS>
__global__ void __launch_bounds__(256) conv16_mfma_kernel(const float *in, const uint16_t *w,
                                                          const float *bias, int relu, float *out,
                                                          int nx, int ny, int nz, int zchunk) {
    constexpr int PX = 16 * NS + 2;  // halo plane extent in x and y
    constexpr int PY = kCY + 2;
    constexpr int NPT = PX * PY;
    constexpr int PTS = 48;          // bf16 per plane point: 3 terms x 16 channels
    constexpr int LOADS = (NPT + 255) / 256;
    __shared__ __attribute__((aligned(16))) __bf16 plane[2][NPT * PTS];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lrow = lane & 15, kg = lane >> 4;
    const int x0 = blockIdx.x * 16 * NS, y0 = blockIdx.y * kCY, z0 = blockIdx.z * zchunk;
    const int z1 = min(nz, z0 + zchunk);
    const long pl = (long)nx * ny, vol = pl * nz;

    // B operands: bw[dzi][j] = W[o = lane%16][c = 8(kg&1)+i][tau + 9 dzi], tau = 2j + kg/2
    bf8 bw[3][5];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const int tau = 2 * j + (kg >> 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int c = 8 * (kg & 1) + i;
                bw[d][j][i] = bf16_bits(tau < 9 ? w[(lrow * 16 + c) * 27 + tau + 9 * d] : 0);
            }
        }
    const float bo = bias ? bias[lrow] : 0.0f;

    f4 acc[3][NS];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[q][s] = f4{0.f, 0.f, 0.f, 0.f};

    // plane loads: thread point e = tid + 256 r, all 16 channels
    float raw[LOADS][16];
    auto load_plane = [&](int zi) {
#pragma unroll
        for (int r = 0; r < LOADS; ++r) {
            const int e = tid + 256 * r;
            const int ly = e / PX, lx = e - (e / PX) * PX;
            const int x = x0 - 1 + lx, y = y0 - 1 + ly;
            const bool ok = e < NPT && x >= 0 && x < nx && y >= 0 && y < ny && zi >= 0 && zi < nz;
            const long base = ok ? (long)zi * pl + (long)y * nx + x : 0;
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const float v = in[base + c * vol];
                raw[r][c] = ok ? v : 0.0f;
            }
        }
    };
    auto store_plane = [&](int buf) {
#pragma unroll
        for (int r = 0; r < LOADS; ++r) {
            const int e = tid + 256 * r;
            if (e >= NPT) continue;
            bf8 t[3][2];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const float x = raw[r][c];
                const __bf16 h = (__bf16)x;
                const float r1 = x - (float)h;
                const __bf16 m = (__bf16)r1;
                const float r2 = r1 - (float)m;
                t[0][c >> 3][c & 7] = h;
                t[1][c >> 3][c & 7] = m;
                t[2][c >> 3][c & 7] = (__bf16)r2;
            }
            bf8 *dst = reinterpret_cast<bf8 *>(&plane[buf][e * PTS]);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                dst[2 * q] = t[q][0];
                dst[2 * q + 1] = t[q][1];
            }
        }
    };
    auto epilogue = [&](f4 (&a)[NS], int zo) {
        const int y = y0 + wave;
        if (y >= ny) return;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int x = x0 + 16 * s + 4 * kg + r;
                if (x >= nx) continue;
                float v = a[s][r] + bo;
                if (relu && v < 0.0f) v = 0.0f;
                out[lrow * vol + (long)zo * pl + (long)y * nx + x] = v;
            }
    };

    const int nplanes = z1 - z0 + 2;  // input planes z0-1 .. z1
    load_plane(z0 - 1);
    store_plane(0);
    __syncthreads();

    // plane q = zi - (z0 - 1) feeds outputs zi+1, zi, zi-1 in slots (R+1)%3,
    // R, (R+2)%3 with R = q % 3; output zi-1 is complete afterwards.
    auto step = [&](int q, auto rc) {
        constexpr int R = decltype(rc)::value;
        constexpr int SN = (R + 1) % 3, SC = R, SP = (R + 2) % 3;
        if (q >= nplanes) return;
        const int zi = z0 - 1 + q;
        const int buf = q & 1;
        const bool more = q + 1 < nplanes;
        if (more) load_plane(zi + 1);
        const bool dn = zi + 1 >= z0 && zi + 1 < z1;  // output zi+1 (weights dz = -1)
        const bool dc = zi >= z0 && zi < z1;          // output zi    (dz = 0)
        const bool dp = zi - 1 >= z0 && zi - 1 < z1;  // output zi-1  (dz = +1)
        if (zi >= 0 && zi < nz) {
            const __bf16 *pb = plane[buf];
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int j = 0; j < 5; ++j) {
                    const int tau = min(2 * j + (kg >> 1), 8);  // slot 9 has zero weights
                    const int ly = wave + tau / 3, lx = 16 * s + lrow + tau % 3;
                    const bf8 *src =
                        reinterpret_cast<const bf8 *>(pb + (ly * PX + lx) * PTS + 8 * (kg & 1));
                    const bf8 a0 = src[0], a1 = src[2], a2 = src[4];
                    if (dn) {
                        acc[SN][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, bw[0][j], acc[SN][s], 0, 0, 0);
                        acc[SN][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bw[0][j], acc[SN][s], 0, 0, 0);
                        acc[SN][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, bw[0][j], acc[SN][s], 0, 0, 0);
                    }
                    if (dc) {
                        acc[SC][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, bw[1][j], acc[SC][s], 0, 0, 0);
                        acc[SC][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bw[1][j], acc[SC][s], 0, 0, 0);
                        acc[SC][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, bw[1][j], acc[SC][s], 0, 0, 0);
                    }
                    if (dp) {
                        acc[SP][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, bw[2][j], acc[SP][s], 0, 0, 0);
                        acc[SP][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bw[2][j], acc[SP][s], 0, 0, 0);
                        acc[SP][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, bw[2][j], acc[SP][s], 0, 0, 0);
                    }
                }
        }
        if (dp) epilogue(acc[SP], zi - 1);
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[SP][s] = f4{0.f, 0.f, 0.f, 0.f};
        if (more) store_plane(buf ^ 1);
        __syncthreads();
    };
    for (int q = 0; q < nplanes; q += 3) {
        step(q, std::integral_constant<int, 0>{});
        step(q + 1, std::integral_constant<int, 1>{});
        step(q + 2, std::integral_constant<int, 2>{});
    }
}

// W'[c][o][26 - t] = W[o][c][t] (bf16 bits): backward-data weights
__global__ void __launch_bounds__(256) transpose_mirror_kernel(const uint16_t *w, int cout,
                                                               int cin, uint16_t *wt) {
    const int n = cout * cin * 27;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
        const int t = e % 27, c = (e / 27) % cin, o = e / (27 * cin);
        wt[(c * cout + o) * 27 + 26 - t] = w[e];
    }
}

// x-subtiles per block for an x extent: least padded width, halo included
int conv_ns(int nx) {
    int best = 1;
    double best_cost = 1e30;
    for (int ns = 1; ns <= 4; ++ns) {
        const int bw = 16 * ns;
        const double cost = (double)((nx + bw - 1) / bw) * (bw + 2);
        if (cost < best_cost - 1e-9) { best_cost = cost; best = ns; }
    }
    return best;
}

int launch_conv16(dage_ctx ctx, int nx, int ny, int nz, const float *in, const uint16_t *w,
                  const float *bias, int relu, float *out) {
    const int ns = conv_ns(nx);
    const int bx = (nx + 16 * ns - 1) / (16 * ns), by = (ny + kCY - 1) / kCY;
    const int want = std::max(1, (2048 + bx * by - 1) / (bx * by));  // z-chunks for ~2048 blocks
    const int zchunk = std::max(2, (nz + want - 1) / want);
    const dim3 grid(bx, by, (nz + zchunk - 1) / zchunk);
    hipEvent_t ev;
    prof_begin(ctx, "conv16_mfma_kernel", &ev);
    switch (ns) {
    case 1: hipLaunchKernelGGL(conv16_mfma_kernel<1>, grid, dim3(256), 0, ctx->stream, in, w, bias, relu, out, nx, ny, nz, zchunk); break;
    case 2: hipLaunchKernelGGL(conv16_mfma_kernel<2>, grid, dim3(256), 0, ctx->stream, in, w, bias, relu, out, nx, ny, nz, zchunk); break;
    case 3: hipLaunchKernelGGL(conv16_mfma_kernel<3>, grid, dim3(256), 0, ctx->stream, in, w, bias, relu, out, nx, ny, nz, zchunk); break;
    default: hipLaunchKernelGGL(conv16_mfma_kernel<4>, grid, dim3(256), 0, ctx->stream, in, w, bias, relu, out, nx, ny, nz, zchunk); break;
    }
    DAGE_HIP_CHECK(hipGetLastError());
    prof_end(ctx, "conv16_mfma_kernel", ev);
    return DAGE_OK;
}

// Filter gradient gW[o][c][t] = sum_p gout[o][p] in[c][p + off(t)] as matrix
// products over the voxels on FP32 MFMA (v_mfma_f32_16x16x4f32: lane l holds
// A(l%16, l/16) and B(l/16, l%16); result register r of lane l is
// D(4(l/16)+r, l%16)): exact FP32 products, FP32 sums.  A block takes a range
// of x-rows (y, z) of one x chunk and walks along y with the rows it needs in
// LDS: one barrier per row, the next rows on their way in registers.  A
// channel row in LDS has kRowS floats (4 times an odd number: 16 channels at
// this stride and 4 segments an odd number apart fall on different banks).
// Sums run per wavefront over its block's rows, then over the wavefronts and
// (sum_blocks_kernel) the blocks, in a fixed order.
//
// Both replace a VALU kernel whose threads owned one (o, c) pair's 27 taps:
// bound by its LDS reads (two per multiply-add of a tap) and, with few
// channels, by idle threads.  Whole calls at 129^3, 16 -> 16: 1305 -> 310 us
// (29.7 GFLOP, 195 us at the 152 TFLOP/s of a large FP32 product; the matrix
// cores are busy 67 % of the time, the rest is the row barriers and the
// segments' padding from 129 to 144 points); 2 -> 16: 630 -> 88, 16 -> 1: 1131 ->
// 62 us (31 us for the bytes at 4.7 TB/s).
constexpr int kSegL = 9;               // longest x segment of a lane group
constexpr int kRowS = 16 * kSegL + 4;  // 148
constexpr int kStage = 3;              // 64-float loads that cover a row

// A channel row of a volume as a buffer: loads outside [0, nx), or of a row
// or channel that does not exist, return zero.
__device__ inline __amdgpu_buffer_rsrc_t row_buffer(const float *p, long vol, int c, int nc, int y,
                                                    int z, int nx, int ny, int nz) {
    const bool ok = c < nc && y >= 0 && y < ny && z >= 0 && z < nz;
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p + (ok ? (long)c * vol + (long)nx * (y + (long)ny * z) : 0)), 0,
        ok ? 4 * nx : 0, 0x00027000);
}
__device__ inline float row_load(__amdgpu_buffer_rsrc_t r, int x) {
    const unsigned off = x < 0 ? 0x80000000u : 4u * (unsigned)x;
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}

// Up to 16 x 16 channels.  Wavefront (dz, w) of 12 sums the 9 taps of one dz
// over segment 4w + l/16 (L points) of each row: A = gout (16 o x 4 voxels),
// B = in (4 voxels x 16 c) of the tap's row; along the segment one LDS read
// per row feeds the three dx taps in turn.
template <int L>
__global__ void __launch_bounds__(768) conv_filter_mfma_kernel(const float *in, const float *gout,
                                                               int cin, int cout, int nx, int ny,
                                                               int nz, int rows_per_block,
                                                               float *part) {
    constexpr int ROW = 16 * kRowS;
    // input rows (dz, y & 3), then output rows y & 1; at the end the sums
    __shared__ float sm[14 * ROW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int dz = wave >> 2, w = wave & 3;
    const int n = lane & 15, k = lane >> 4;
    const int x0 = blockIdx.y * 16 * L;
    const long vol = (long)nx * ny * nz;
    const long nrows = (long)ny * nz;
    const long r0 = (long)blockIdx.x * rows_per_block;
    const long r1 = min(nrows, r0 + rows_per_block);
    const int start = (4 * w + k) * L, last = nx - x0 - start;
    const bool padded = nx - x0 < 4 * (w + 1) * L && nx - x0 >= 4 * w * L;  // holds column nx

    // A row's sums start at zero and are added to the block's after it: chains
    // of L matrix products and of the rows instead of their product (one
    // accumulator for all rows had 3 times the error).
    f4 sum[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) sum[t] = f4{0.f, 0.f, 0.f, 0.f};
    float sumb = 0.0f;

    // staging: wavefront `wave` takes channel rows wave, wave + 12, ... of the
    // 48 input rows and of the 16 output rows
    float ri[4][kStage], ro[2][kStage];
    auto load_in = [&](int y, int z) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = wave + 12 * q;
            const __amdgpu_buffer_rsrc_t r = row_buffer(in, vol, e & 15, cin, y, z + (e >> 4) - 1, nx, ny, nz);
#pragma unroll
            for (int h = 0; h < kStage; ++h) ri[q][h] = row_load(r, x0 - 1 + lane + 64 * h);
        }
    };
    auto store_in = [&](int y) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = wave + 12 * q;
            float *d = sm + (4 * (e >> 4) + (y & 3)) * ROW + (e & 15) * kRowS;
#pragma unroll
            for (int h = 0; h < kStage; ++h)
                if (lane + 64 * h < kRowS) d[lane + 64 * h] = ri[q][h];
        }
    };
    auto load_out = [&](int y, int z) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e = wave + 12 * q;
            const __amdgpu_buffer_rsrc_t r = row_buffer(gout, vol, e, cout, y, z, nx, ny, nz);
#pragma unroll
            for (int h = 0; h < kStage; ++h) {
                const int x = lane + 64 * h;
                ro[q][h] = row_load(r, x < 16 * L ? x0 + x : -1);
            }
        }
    };
    auto store_out = [&](int y) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e = wave + 12 * q;
            float *d = sm + (12 + (y & 1)) * ROW + e * kRowS;
#pragma unroll
            for (int h = 0; h < kStage; ++h)
                if (e < 16 && lane + 64 * h < kRowS) d[lane + 64 * h] = ro[q][h];
        }
    };

    // One row's products.  The left tap of the first padding column is
    // in[nx - 1], times a zero of gout: where that is not finite, MASK makes it
    // zero (in every row, 129^3 at 16 x 16: 328 us instead of 310).
    auto add_row = [&](int y, auto mask) {
        constexpr bool MASK = decltype(mask)::value;
        const float *go = sm + (12 + (y & 1)) * ROW + n * kRowS + start;
        const float *ir[3];
        float v0[3], v1[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            ir[d] = sm + (4 * dz + ((y + d - 1) & 3)) * ROW + n * kRowS + start;
            v0[d] = !MASK || 0 < last ? ir[d][0] : 0.0f;
            v1[d] = ir[d][1];
        }
        f4 acc[9];
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
        float accb = 0.0f;
#pragma unroll
        for (int x = 0; x < L; ++x) {
            const float g = go[x];
            accb += g;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const float v2 = ir[d][x + 2];
                acc[3 * d] = __builtin_amdgcn_mfma_f32_16x16x4f32(g, v0[d], acc[3 * d], 0, 0, 0);
                acc[3 * d + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g, v1[d], acc[3 * d + 1], 0, 0, 0);
                acc[3 * d + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(g, v2, acc[3 * d + 2], 0, 0, 0);
                v0[d] = !MASK || x + 1 < last ? v1[d] : 0.0f;
                v1[d] = v2;
            }
        }
#pragma unroll
        for (int t = 0; t < 9; ++t) sum[t] += acc[t];
        sumb += accb;
    };

    for (long row = r0; row < r1;) {
        const int z = (int)(row / ny), ya = (int)(row - (long)z * ny);
        const int yb = (int)min((long)ny, ya + r1 - row);  // rows [ya, yb) of plane z
        for (int y = ya - 1; y <= ya + 1; ++y) {
            load_in(y, z);
            store_in(y);
        }
        load_out(ya, z);
        store_out(ya);
        __syncthreads();
        for (int y = ya; y < yb; ++y) {
            // row y + 2 replaces y - 2, output row y + 1 replaces y - 1
            load_in(y + 2, z);
            load_out(y + 1, z);
            bool bad = false;
            if (padded)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    bad |= !__builtin_isfinite(sm[(4 * dz + ((y + d - 1) & 3)) * ROW + n * kRowS + nx - x0]);
            if (__builtin_expect(__any(bad), 0)) add_row(y, std::true_type{});
            else add_row(y, std::false_type{});
            store_in(y + 2);
            store_out(y + 1);
            __syncthreads();
        }
        row += yb - ya;
    }
    // sum over the four segments' wavefronts
    float *red = sm + (w * 3 + dz) * 36 * 64 + lane, *redb = sm + 12 * 36 * 64;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(t * 4 + r) * 64] = sum[t][r];
    if (dz == 1) redb[w * 64 + lane] = sumb;
    __syncthreads();
    const int len = cout * cin * 27 + cout;
    float *pp = part + ((long)blockIdx.y * gridDim.x + blockIdx.x) * len;
    for (int e = tid; e < 3 * 36 * 64; e += 768) {
        const int l = e & 63, q = e >> 6, t = q >> 2;
        const int o = 4 * (l >> 4) + (q & 3), c = l & 15;
        float s = 0.0f;
        for (int v = 0; v < 4; ++v) s += sm[v * 3 * 36 * 64 + e];
        if (o < cout && c < cin) pp[(o * cin + c) * 27 + t] = s;
    }
    if (tid < cout) {
        float s = 0.0f;
        for (int v = 0; v < 16; ++v) s += redb[16 * v + tid];
        pp[cout * cin * 27 + tid] = s;
    }
}

// One side with CH = 1 or 2 channels (Y), the other (X) with up to 16:
// R[m][col] = sum_p X[m][p] Y[ch][p + off(t)], col = 27 ch + t, and
// col = 27 CH the plain sum of X.  The taps are the columns of B, so a
// 4-voxel step costs 2 CH MFMAs.  X = gout: R is gW and the last
// column gb.  X = in (SWAP): gW[ch][m][26 - t] = R[m][27 ch + t], and
// gb[ch] is summed from the staged rows of Y.
template <int CH, bool SWAP>
__global__ void __launch_bounds__(256) conv_filter_few_kernel(const float *X, const float *Y,
                                                              int nm, int nx, int ny, int nz,
                                                              int width, int rows_per_block,
                                                              float *part) {
    constexpr int NT = 2 * CH, YQ = (3 * CH + 3) / 4;
    constexpr int RED = NT * 4 * 64;
    // X rows (y & 1, m), at the end the sums; Y rows (dz, y & 3, ch), a row
    // of ones and one of zeros (the columns past the taps)
    __shared__ float sx[2 * 16 * kRowS];
    __shared__ float sy[(12 * CH + 2) * kRowS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, k = lane >> 4;
    const int x0 = blockIdx.y * width;
    const long vol = (long)nx * ny * nz;
    const long nrows = (long)ny * nz;
    const long r0 = (long)blockIdx.x * rows_per_block;
    const long r1 = min(nrows, r0 + rows_per_block);

    // An infinity of Y or X meets no zero of the padding past the row, of the
    // next chunk or, where X = in, outside the volume: the columns of
    // [xlo, xhi) have all their neighbours in the row and run in whole steps
    // of 4, the others in a masked step; X = in: the first and the last column
    // without the taps outside, and a row's sums without the rows outside.
    const int xend = min(width, nx - x0), xlo = SWAP && x0 == 0;
    const int xhi = xend - (SWAP && x0 + xend == nx);
    f4 sum[NT];
    float accb[CH];
    // this lane's column: input row y + ty - 1 (ty < 0: any), offset, and its
    // place among the 9 rows (9: none) with 16 times its place in the row
    int ty[NT], to[NT], tc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        sum[j] = f4{0.f, 0.f, 0.f, 0.f};
        const int col = 16 * j + n, ch = min(col / 27, CH - 1), t = (col - 27 * ch) % 27;
        const bool tap = col < 27 * CH;
        ty[j] = tap ? t / 3 % 3 : -1;
        tc[j] = tap ? t / 3 + 16 * (t % 3) : 9 + 16;
        to[j] = (tap ? 4 * (t / 9) * CH + ch : 12 * CH + (col > 27 * CH)) * kRowS + (tap ? t % 3 : 0) + k;
    }
    if (tid < kRowS) {
        sy[12 * CH * kRowS + tid] = 1.0f;
        sy[(12 * CH + 1) * kRowS + tid] = 0.0f;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) accb[c] = 0.0f;

    float rx[4][kStage], ry[YQ][kStage];
    auto load_x = [&](int y, int z) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const __amdgpu_buffer_rsrc_t r = row_buffer(X, vol, wave + 4 * q, nm, y, z, nx, ny, nz);
#pragma unroll
            for (int h = 0; h < kStage; ++h) {
                const int x = lane + 64 * h;
                rx[q][h] = row_load(r, x < width ? x0 + x : -1);
            }
        }
    };
    auto store_x = [&](int y) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int h = 0; h < kStage; ++h)
                if (lane + 64 * h < kRowS) sx[(16 * (y & 1) + wave + 4 * q) * kRowS + lane + 64 * h] = rx[q][h];
    };
    auto load_y = [&](int y, int z) {
#pragma unroll
        for (int q = 0; q < YQ; ++q) {
            const int e = wave + 4 * q;
            const __amdgpu_buffer_rsrc_t r =
                row_buffer(Y, vol, e % CH, e < 3 * CH ? CH : 0, y, z + e / CH - 1, nx, ny, nz);
#pragma unroll
            for (int h = 0; h < kStage; ++h) ry[q][h] = row_load(r, x0 - 1 + lane + 64 * h);
        }
    };
    auto store_y = [&](int y) {
#pragma unroll
        for (int q = 0; q < YQ; ++q) {
            const int e = wave + 4 * q;
            if (e >= 3 * CH) continue;
            float *d = sy + ((4 * (e / CH) + (y & 3)) * CH + e % CH) * kRowS;
#pragma unroll
            for (int h = 0; h < kStage; ++h)
                if (lane + 64 * h < kRowS) d[lane + 64 * h] = ry[q][h];
        }
    };

    for (long row = r0; row < r1;) {
        const int z = (int)(row / ny), ya = (int)(row - (long)z * ny);
        const int yb = (int)min((long)ny, ya + r1 - row);
        for (int y = ya - 1; y <= ya + 1; ++y) {
            load_y(y, z);
            store_y(y);
        }
        load_x(ya, z);
        store_x(ya);
        __syncthreads();
        for (int y = ya; y < yb; ++y) {
            load_y(y + 2, z);
            load_x(y + 1, z);
            if (SWAP && tid < width) {
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    // (past the last column the row holds zeros)
                    accb[c] += x0 + tid < nx ? sy[((4 + (y & 3)) * CH + c) * kRowS + tid + 1] : 0.0f;
            }
            const float *xr = sx + (16 * (y & 1) + n) * kRowS + k;
            const float *yr[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j)
                yr[j] = sy + (ty[j] < 0 ? 0 : ((y + ty[j] - 1) & 3) * CH * kRowS) + to[j];
            f4 acc[NT];  // this row's sums (see conv_filter_mfma_kernel)
            // a step apart: wavefront 0 the columns 1..3, 1 those from xs on,
            // 2 the first and 3 the last column
            const int xs = xhi & ~3;
            {
                const int x = wave == 1 ? xs : (wave == 3 ? xend - 1 : 0), c = x + k;
                const bool on = wave == 0   ? xlo && xs > 0 && k > 0
                                : wave == 1 ? c >= xlo && c < xhi
                                : wave == 2 ? xlo && k == 0
                                            : xhi < xend && nx > 1 && k == 0;
                const bool first = SWAP && wave == 2, last = SWAP && (wave == 3 || (first && nx == 1));
                const float a = on ? xr[x] : 0.0f;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        a, on ? yr[j][x] : 0.0f, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    const int dx = tc[j] >> 4;
                    if ((first && dx == 0) || (last && dx == 2)) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
                }
            }
#pragma unroll 3
            for (int x = 4 * wave + (wave < xlo ? 16 : 0); x < xs; x += 16) {
                const float a = xr[x];
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, yr[j][x], acc[j], 0, 0, 0);
            }
            // bit 3 dz + dy: the row of that tap exists
            const int yok = (y > 0) + 2 + 4 * (y + 1 < ny);
            const int rows = (z > 0 ? yok : 0) + 8 * yok + (z + 1 < nz ? 64 * yok : 0) + 512;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                if (!SWAP || ((rows >> (tc[j] & 15)) & 1)) sum[j] += acc[j];
            store_y(y + 2);
            store_x(y + 1);
            __syncthreads();
        }
        row += yb - ya;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) sx[wave * RED + (j * 4 + r) * 64 + lane] = sum[j][r];
#pragma unroll
    for (int c = 0; c < CH; ++c) sy[c * 256 + tid] = accb[c];
    __syncthreads();
    const int cout = SWAP ? CH : nm, cin = SWAP ? nm : CH;
    float *pp = part + ((long)blockIdx.y * gridDim.x + blockIdx.x) * (cout * cin * 27 + cout);
    for (int e = tid; e < NT * 4 * 64; e += 256) {
        const int l = e & 63, q = e >> 6;
        const int m = 4 * (l >> 4) + (q & 3), col = 16 * (q >> 2) + (l & 15);
        const float s = ((sx[e] + sx[RED + e]) + sx[2 * RED + e]) + sx[3 * RED + e];
        if (m >= nm || col > 27 * CH) continue;
        const int ch = col / 27, t = col - 27 * ch;
        if (col == 27 * CH) {
            if (!SWAP) pp[cout * cin * 27 + m] = s;
        } else {
            pp[SWAP ? (ch * nm + m) * 27 + 26 - t : (m * CH + ch) * 27 + t] = s;
        }
    }
    if (SWAP && wave < CH) {  // a fixed tree over the columns
        float s = 0.0f;
        for (int h = 0; h < 4; ++h) s += sy[256 * wave + lane + 64 * h];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) pp[cout * cin * 27 + wave] = s;
    }
}

// Sum of the blocks' partials, 32 entries per block: 8 thread rows take every
// eighth block, then a fixed sum over the rows, in FP64 (the serial FP32 loop
// over 1024 blocks took 230 us at 6928 entries, this one 9).  The first
// nw sums go to gw, the others to gb.
__global__ void __launch_bounds__(256) sum_blocks_kernel(const float *part, int nblocks, int len,
                                                         int nw, float *gw, float *gb) {
    __shared__ double red[8][32];
    const int col = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int i = blockIdx.x * 32 + col;
    double s = 0.0;
    if (i < len)
#pragma unroll 4
        for (int b = g; b < nblocks; b += 8) s += part[(long)b * len + i];
    red[g][col] = s;
    __syncthreads();
    if (g == 0 && i < len) {
#pragma unroll
        for (int q = 1; q < 8; ++q) s += red[q][col];
        (i < nw ? gw : gb - nw)[i] = (float)s;
    }
}

__global__ void __launch_bounds__(256) relu_bwd_kernel(long n, const float *out, float *g) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        if (out[i] <= 0.0f) g[i] = 0.0f;
}

__global__ void __launch_bounds__(256) adam_kernel(int n, float *w, const float *g, float *m,
                                                   float *v, float lr, float b1, float b2,
                                                   float eps, float c1, float c2,
                                                   uint16_t *wbf) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        wbf[i] = f32_to_bf16(wi);
    }
}

__global__ void __launch_bounds__(256) to_bf16_kernel(int n, const float *w, uint16_t *wbf) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        wbf[i] = f32_to_bf16(w[i]);
}

// grad = scale*(pred - target); part[block] = sum over the block's range of (pred - target)^2
__global__ void __launch_bounds__(256) mse_kernel(long n, const float *pred, const float *target,
                                                  float scale, float *grad, double *part) {
    __shared__ double red[256];
    double s = 0.0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x) {
        const float d = pred[i] - target[i];
        grad[i] = scale * d;
        s += (double)d * d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) cvt_f64_f32_kernel(long n, const double *x, double scale,
                                                          float *y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        y[i] = (float)(scale * x[i]);
}

__global__ void __launch_bounds__(256) axpy_f32_f64_kernel(long n, double a, const float *x,
                                                           double *y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        y[i] = y[i] + a * (double)x[i];
}

int check_dims(int nx, int ny, int nz, int cin, int cout) {
    DAGE_REQUIRE(nx > 0 && ny > 0 && nz > 0, DAGE_ERR_ARG, "empty volume");
    DAGE_REQUIRE(cin >= 1 && cin <= kMaxC && cout >= 1 && cout <= kMaxC, DAGE_ERR_UNSUPPORTED,
                 "channels %d -> %d outside 1..%d", cin, cout, kMaxC);
    return DAGE_OK;
}

}  // namespace
}  // namespace dage

using namespace dage;

extern "C" {

int dage_conv3d_forward(dage_ctx ctx, int nx, int ny, int nz, int cin, int cout, const float *in,
                        const uint16_t *w, const float *bias, int relu, float *out) {
    DAGE_TRY(use_device(ctx));
    DAGE_TRY(check_dims(nx, ny, nz, cin, cout));
    DAGE_REQUIRE(in && w && bias && out && in != out, DAGE_ERR_ARG, "bad argument");
    DAGE_REQUIRE(cout == 1 || cout == kMaxC, DAGE_ERR_UNSUPPORTED,
                 "forward supports 1 or %d output channels", kMaxC);
    const long vol = (long)nx * ny * nz;
    if (cin == kMaxC && cout == kMaxC)
        return launch_conv16(ctx, nx, ny, nz, in, w, bias, relu, out);
    void *scr = nullptr;  // FP32 weight table
    const int nw = cout * cin * 27;
    DAGE_TRY(ctx_scratch(ctx, sizeof(float) * nw, &scr));
    float *wf = static_cast<float *>(scr);
    hipLaunchKernelGGL(weights_f32_kernel, dim3((nw + 255) / 256), dim3(256), 0, ctx->stream, w,
                       cout, cin, wf);
    DAGE_HIP_CHECK(hipGetLastError());
    if (cout == 1)
        hipLaunchKernelGGL(conv_fwd_kernel<1>, dim3(grid_of(vol)), dim3(256), 0, ctx->stream, in,
                           cin, wf, bias, relu, out, nx, ny, nz);
    else
        hipLaunchKernelGGL(conv_fwd_kernel<kMaxC>, dim3(grid_of(vol)), dim3(256), 0, ctx->stream,
                           in, cin, wf, bias, relu, out, nx, ny, nz);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_conv3d_backward_data(dage_ctx ctx, int nx, int ny, int nz, int cin, int cout,
                              const float *gout, const uint16_t *w, float *gin) {
    DAGE_TRY(use_device(ctx));
    DAGE_TRY(check_dims(nx, ny, nz, cin, cout));
    DAGE_REQUIRE(gout && w && gin && gout != gin, DAGE_ERR_ARG, "bad argument");
    const long vol = (long)nx * ny * nz;
    if (cin == kMaxC && cout == kMaxC) {
        void *scr = nullptr;  // transposed, mirrored weights
        DAGE_TRY(ctx_scratch(ctx, sizeof(uint16_t) * kMaxC * kMaxC * 27, &scr));
        uint16_t *wt = static_cast<uint16_t *>(scr);
        hipLaunchKernelGGL(transpose_mirror_kernel, dim3(27), dim3(256), 0, ctx->stream, w, cout,
                           cin, wt);
        DAGE_HIP_CHECK(hipGetLastError());
        return launch_conv16(ctx, nx, ny, nz, gout, wt, nullptr, 0, gin);
    }
    hipLaunchKernelGGL(conv_bwd_data_kernel, dim3(grid_of(vol)), dim3(256), 0, ctx->stream, gout,
                       cout, cin, w, gin, nx, ny, nz);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_conv3d_backward_filter(dage_ctx ctx, int nx, int ny, int nz, int cin, int cout,
                                const float *in, const float *gout, float *gw, float *gb) {
    DAGE_TRY(use_device(ctx));
    DAGE_TRY(check_dims(nx, ny, nz, cin, cout));
    DAGE_REQUIRE(in && gout && gw && gb, DAGE_ERR_ARG, "bad argument");
    // The entry point's own limit: three rows of every input and one of every
    // output channel in 64 KB (nx <= 254 at 16 x 16).  The kernels below cut x
    // into chunks and would take any extent.
    DAGE_REQUIRE(sizeof(float) * ((size_t)cin * 3 * (nx + 2) + (size_t)cout * nx) <= 64 * 1024,
                 DAGE_ERR_UNSUPPORTED, "x extent %d beyond the 64 KB of rows", nx);
    // x chunks of at most 16*kSegL columns; blocks of rows for one block per
    // CU (16 x 16 channels: 132 KB of LDS) or four (the few-channel kernel,
    // bound by its loads)
    const bool few = std::min(cin, cout) <= 2;
    const int chunks = (nx + 16 * kSegL - 1) / (16 * kSegL);
    const int width = (nx + chunks - 1) / chunks;
    int L = (width + 15) / 16;
    if (L % 4 == 0) ++L;  // segments a multiple of 4 apart share banks
    const long nrows = (long)ny * nz;
    const int want = std::max(1, (few ? 1024 : 256) / chunks);
    const int rows = (int)((nrows + want - 1) / want);
    const int rblocks = (int)((nrows + rows - 1) / rows), nblocks = rblocks * chunks;
    const int nw = cout * cin * 27, len = nw + cout;
    void *scr = nullptr;
    DAGE_TRY(ctx_scratch(ctx, sizeof(float) * (size_t)nblocks * len, &scr));
    float *part = static_cast<float *>(scr);
    const dim3 grid(rblocks, chunks);
    if (!few) {
        auto run = [&](auto l) {
            hipLaunchKernelGGL(conv_filter_mfma_kernel<decltype(l)::value>, grid, dim3(768), 0,
                               ctx->stream, in, gout, cin, cout, nx, ny, nz, rows, part);
        };
        switch (L) {
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        case 5: run(std::integral_constant<int, 5>{}); break;
        case 6: run(std::integral_constant<int, 6>{}); break;
        case 7: run(std::integral_constant<int, 7>{}); break;
        default: run(std::integral_constant<int, kSegL>{}); break;
        }
    } else {
        const bool swap = cin > 2;
        const float *X = swap ? in : gout, *Y = swap ? gout : in;
        const int nm = swap ? cin : cout;
        auto run = [&](auto ch, auto sw) {
            hipLaunchKernelGGL((conv_filter_few_kernel<decltype(ch)::value, decltype(sw)::value>),
                               grid, dim3(256), 0, ctx->stream, X, Y, nm, nx, ny, nz, width, rows,
                               part);
        };
        const std::integral_constant<int, 1> one{};
        const std::integral_constant<int, 2> two{};
        if (swap) cout == 1 ? run(one, std::true_type{}) : run(two, std::true_type{});
        else cin == 1 ? run(one, std::false_type{}) : run(two, std::false_type{});
    }
    DAGE_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(sum_blocks_kernel, dim3((len + 31) / 32), dim3(256), 0, ctx->stream, part,
                       nblocks, len, nw, gw, gb);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_relu_backward(dage_ctx ctx, long n, const float *out, float *grad) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && out && grad, DAGE_ERR_ARG, "bad argument");
    hipLaunchKernelGGL(relu_bwd_kernel, dim3(grid_of(n)), dim3(256), 0, ctx->stream, n, out, grad);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_adam_step(dage_ctx ctx, int n, float *w, const float *g, float *m, float *v, float lr,
                   float beta1, float beta2, float eps, int step, uint16_t *w_bf16) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && w && g && m && v && w_bf16 && step >= 1, DAGE_ERR_ARG, "bad argument");
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid_of(n)), dim3(256), 0, ctx->stream, n, w, g, m, v,
                       lr, beta1, beta2, eps, c1, c2, w_bf16);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_weights_to_bf16(dage_ctx ctx, int n, const float *w, uint16_t *w_bf16) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && w && w_bf16, DAGE_ERR_ARG, "bad argument");
    hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_of(n)), dim3(256), 0, ctx->stream, n, w, w_bf16);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_mse_loss(dage_ctx ctx, long n, const float *pred, const float *target, float *grad,
                  double *loss) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && pred && target && grad && loss, DAGE_ERR_ARG, "bad argument");
    const int nb = std::min<long>(1024, (n + 255) / 256);
    void *scr = nullptr;
    DAGE_TRY(ctx_scratch(ctx, sizeof(double) * nb, &scr));
    double *part = static_cast<double *>(scr);
    hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(256), 0, ctx->stream, n, pred, target,
                       (float)(2.0 / (double)n), grad, part);
    DAGE_HIP_CHECK(hipGetLastError());
    std::vector<double> h(nb);
    DAGE_HIP_CHECK(hipMemcpyAsync(h.data(), part, sizeof(double) * nb, hipMemcpyDeviceToHost,
                                  ctx->stream));
    DAGE_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    double s = 0.0;
    for (double v : h) s += v;
    *loss = s / (double)n;
    return DAGE_OK;
}

int dage_cvt_f64_f32(dage_ctx ctx, long n, const double *x, double scale, float *y) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && x && y, DAGE_ERR_ARG, "bad argument");
    hipLaunchKernelGGL(cvt_f64_f32_kernel, dim3(grid_of(n)), dim3(256), 0, ctx->stream, n, x,
                       scale, y);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_axpy_f32_f64(dage_ctx ctx, long n, double a, const float *x, double *y) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(n > 0 && x && y, DAGE_ERR_ARG, "bad argument");
    hipLaunchKernelGGL(axpy_f32_f64_kernel, dim3(grid_of(n)), dim3(256), 0, ctx->stream, n, a, x,
                       y);
    DAGE_HIP_CHECK(hipGetLastError());
    return DAGE_OK;
}

int dage_device_alloc(dage_ctx ctx, size_t bytes, void **ptr) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(ptr != nullptr && bytes > 0, DAGE_ERR_ARG, "bad argument");
    DAGE_HIP_CHECK(hipMalloc(ptr, bytes));
    return DAGE_OK;
}

int dage_device_free(dage_ctx ctx, void *ptr) {
    DAGE_TRY(use_device(ctx));
    if (ptr) DAGE_HIP_CHECK(hipFree(ptr));
    return DAGE_OK;
}

int dage_memcpy(dage_ctx ctx, void *dst, const void *src, size_t bytes, int kind) {
    DAGE_TRY(use_device(ctx));
    DAGE_REQUIRE(dst && src, DAGE_ERR_ARG, "bad argument");
    DAGE_REQUIRE(kind >= 0 && kind <= 2, DAGE_ERR_ARG, "kind 0 (h2d), 1 (d2h) or 2 (d2d)");
    const hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice
                                      : (kind == 1 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice);
    DAGE_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, k, ctx->stream));
    DAGE_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return DAGE_OK;
}

}  // extern "C"
