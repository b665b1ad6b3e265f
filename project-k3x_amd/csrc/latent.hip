// latent.hip -- the fp32 side of the backend interface: dense fp32 and
// row-major MXFP4 matrix-vector products with double accumulation, the fp32
// SiTU MLP, and the resident latent MoE layer
// (runtime/src/backend_cpu.cpp:22-122, :305-339) around the bank's grouped
// expert path.
//
// Every product here is HBM-bound (one token, or a few, per weight byte), so
// the kernels stream each weight row once with 16-byte loads per lane and
// keep the reference's arithmetic: each product formed exactly in double
// (fp32 x fp32, or fp32 x an MXFP4 value of two significant bits) and summed
// in double, one rounding to fp32 at the end.  Only the summation order
// differs from the reference's sequential loop (a lane-strided sum and a
// butterfly), which moves the double sum by a few units in its last place,
// far below the fp32 rounding that follows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "k3x_device.hpp"
#include "k3x_internal.hpp"

using namespace k3x_dev;

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr uint32_t kMaxTokens = 4;  // tokens per weight pass

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

__device__ inline float situ(float g, float u, float beta, int has_linear, float linear) {
    // runtime/src/ops.cpp:20-30 in fp32 with the library's expf / tanhf.
    const float sig = 1.0f / (1.0f + expf(-g));
    const float bg = beta * tanhf(g / beta) * sig;
    const float bu = has_linear ? linear * tanhf(u / linear) : u;
    return bg * bu;
}

// One output row per wave, T <= kMaxTokens tokens per pass (x rows
// [T][x_stride]): shapes that the vector kernel below does not take, and (VEC:
// 16-byte loads, cols % 4 == 0, rows 16-byte aligned) columns too short for it.
// OUT: 0 y = Wx; 1 y = Wx + add (fp32 add, as routed[row] += shared[row]);
// 2 y = Wx and the split copy ys = [bf16 hi | bf16 lo] rows of 2 rows_total;
// 3 y = situ(W x, W2 x) (the gate / up pair of an MLP).
struct GemvArgs {
    const float* W;
    const float* W2;      // OUT 3: the up matrix
    uint32_t rows, cols;
    const float* x;
    uint32_t x_stride;
    uint32_t T;
    float* y;
    uint32_t y_stride;
    const float* add;     // OUT 1, [T][y_stride]
    uint16_t* ys;         // OUT 2, [T][2 * y_stride]
    float beta, linear;
    int has_linear;
    const uint32_t* status;
};

template <int OUT, bool VEC>
__global__ __launch_bounds__(kThreads) void f32_gemv_kernel(GemvArgs a) {
    if (*(volatile const uint32_t*)a.status) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t r = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (r >= a.rows) return;
    constexpr int M = OUT == 3 ? 2 : 1;
    const float* wr[M];
    wr[0] = a.W + (size_t)r * a.cols;
    if constexpr (M == 2) wr[1] = a.W2 + (size_t)r * a.cols;
    for (uint32_t t0 = 0; t0 < a.T; t0 += kMaxTokens) {
        const uint32_t nt = min(a.T - t0, kMaxTokens);
        double acc[M][kMaxTokens];
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (uint32_t t = 0; t < kMaxTokens; ++t) acc[m][t] = 0.0;
        if constexpr (VEC) {
            // Four 16-byte loads per lane in flight (4 KiB per wave).
            constexpr uint32_t kStep = 64 * 4 * 4;
            for (uint32_t c0 = 0; c0 < a.cols; c0 += kStep) {
                f32x4 w[M][4];
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t c = c0 + (q * 64 + lane) * 4;
                        w[m][q] = c < a.cols ? *reinterpret_cast<const f32x4*>(wr[m] + c)
                                             : f32x4{0.f, 0.f, 0.f, 0.f};
                    }
#pragma unroll
                for (uint32_t t = 0; t < kMaxTokens; ++t) {
                    if (t >= nt) break;
                    const float* xr = a.x + (size_t)(t0 + t) * a.x_stride;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t c = c0 + (q * 64 + lane) * 4;
                        if (c >= a.cols) continue;
                        const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + c);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int m = 0; m < M; ++m)
                                acc[m][t] =
                                    __builtin_fma((double)w[m][q][i], (double)xv[i], acc[m][t]);
                    }
                }
            }
        } else {
            for (uint32_t c = lane; c < a.cols; c += 64) {
                float w[M];
#pragma unroll
                for (int m = 0; m < M; ++m) w[m] = wr[m][c];
#pragma unroll
                for (uint32_t t = 0; t < kMaxTokens; ++t) {
                    if (t >= nt) break;
                    const double xv = (double)a.x[(size_t)(t0 + t) * a.x_stride + c];
#pragma unroll
                    for (int m = 0; m < M; ++m)
                        acc[m][t] = __builtin_fma((double)w[m], xv, acc[m][t]);
                }
            }
        }
#pragma unroll
        for (uint32_t t = 0; t < kMaxTokens; ++t) {
            if (t >= nt) break;
            float v[M];
#pragma unroll
            for (int m = 0; m < M; ++m) v[m] = (float)wave_sum(acc[m][t]);
            if (lane != 0) continue;
            const size_t at = (size_t)(t0 + t) * a.y_stride + r;
            if constexpr (OUT == 0) {
                a.y[at] = v[0];
            } else if constexpr (OUT == 1) {
                a.y[at] = __fadd_rn(a.add[at], v[0]);
            } else if constexpr (OUT == 2) {
                a.y[at] = v[0];
                const uint16_t hi = f32_to_bf16(v[0]);
                uint16_t* ys = a.ys + (size_t)(t0 + t) * 2 * a.y_stride;
                ys[r] = hi;
                ys[a.y_stride + r] = act_lo_bf16(v[0], hi);
            } else {
                a.y[at] = situ(v[0], v[M - 1], a.beta, a.has_linear, a.linear);
            }
        }
    }
}

// The vector form (16-byte loads: cols and strides multiples of 4, rows
// 16-byte aligned).  A wave takes two matrix rows (a gate / up pair, or two
// output rows), so a lane's x values, staged in LDS kCols columns at a time
// by the workgroup, are read and converted to double once for both; the
// weights are non-temporal (read once a call) and eight 16-byte loads a lane
// are in flight.  Lane l sums columns 4 (64 i + l) .. + 3, i ascending.
// The tail of a row has a body of its own, so that the full steps carry no bounds
// (384 x 7168, one token 10.9 -> 9.5 us, 36 x 7168 10.6 -> 9.4; the latent layer at 8
// tokens 254 -> 246).
// Bound: HBM.  Measured (7168 columns, one token) against a row a wave with x
// read from the cache beside every weight: the gate/up of 6144 rows and a
// 3584-row matrix 3.5 and 3.2 TB/s in two launches, 6.6 in one; two down
// matrices 4.5 and 4.3 TB/s, 6.4 in one.
// A launch runs one job or two (workgroups of job 0 first): independent
// products fill the device together.
enum JobOut { kOutPlain, kOutSplit, kOutSitu, kOutSum, kOutAdd };

struct VecJob {
    JobOut out;
    uint32_t rows, cols;
    const float* W;
    const float* x;
    uint32_t x_stride;
    // kOutSitu: the up matrix (same x).  kOutSum: y = W x + W2 x2 (each
    // product rounded to fp32 first, then a float add).  kOutAdd: y = x2 + W x,
    // x2 rows of y's shape.
    const float* W2;
    uint32_t cols2;
    const float* x2;
    uint32_t x2_stride;
    float* y;
    uint32_t y_stride;
    uint16_t* ys;  // kOutSplit, [T][2 * y_stride]
    float beta, linear;
    int has_linear;
};

struct VecArgs {
    VecJob job[2];
    uint32_t blocks0;  // workgroups of job 0
    uint32_t T;
    const uint32_t* status;
};

constexpr uint32_t kCols = 1024;

// acc[r][t] += w[r] . x[t] over the columns from c0, by the whole workgroup: kCols
// of them (FULL) or the cols - c0 that are left, whose absent quarters of 256
// are neither loaded nor multiplied.
template <int NT, bool FULL>
__device__ __forceinline__ void dot_block(const float* const (&w)[2], uint32_t c0, uint32_t cols,
                                          const float* x, uint32_t x_stride, uint32_t nt,
                                          f32x4 (&s_x)[NT][kCols / 4], double (&acc)[2][NT]) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t cx = c0 + threadIdx.x * 4;
    const uint32_t quarters = FULL ? 4 : (cols - c0 + 255) / 256;  // workgroup-uniform
    f32x4 xv[NT], wv[2][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        xv[t] = (FULL || cx < cols) && (uint32_t)t < nt
                    ? *reinterpret_cast<const f32x4*>(x + (size_t)t * x_stride + cx)
                    : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t c = c0 + (q * 64 + lane) * 4;
            if constexpr (FULL)
                wv[r][q] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w[r] + c));
            else
                wv[r][q] = c < cols ? *reinterpret_cast<const f32x4*>(w[r] + c)
                                    : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    // The barriers wait for LDS only: the weights stay in flight.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < NT; ++t) s_x[t][threadIdx.x] = xv[t];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if (!FULL && (uint32_t)t >= nt) break;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!FULL && (uint32_t)q >= quarters) break;
            const f32x4 v = s_x[t][q * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    acc[r][t] = __builtin_fma((double)wv[r][q][i], (double)v[i], acc[r][t]);
        }
    }
}

template <int NT>
__device__ inline void dot_rows(const float* const (&w)[2], uint32_t cols, const float* x,
                                uint32_t x_stride, uint32_t nt, f32x4 (&s_x)[NT][kCols / 4],
                                double (&acc)[2][NT]) {
    uint32_t c0 = 0;
    for (; c0 + kCols <= cols; c0 += kCols)
        dot_block<NT, true>(w, c0, cols, x, x_stride, nt, s_x, acc);
    if (c0 < cols) dot_block<NT, false>(w, c0, cols, x, x_stride, nt, s_x, acc);
}

template <int NT>
__global__ __launch_bounds__(kThreads) void f32_gemv_vec_kernel(VecArgs a) {
    static_assert(kThreads * 4 == kCols, "a thread stages four columns a token");
    __shared__ f32x4 s_x[NT][kCols / 4];
    if (*(volatile const uint32_t*)a.status) return;
    const bool second = blockIdx.x >= a.blocks0;
    const VecJob& j = a.job[second ? 1 : 0];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (blockIdx.x - (second ? a.blocks0 : 0)) * kWaves + (threadIdx.x >> 6);
    // Rows past the matrix repeat its last one (not stored).
    const bool pair = j.out == kOutSitu;
    const uint32_t r0 = pair ? wave : 2 * wave;
    const uint32_t ra = min(r0, j.rows - 1), rb = pair ? ra : min(r0 + 1, j.rows - 1);
    for (uint32_t t0 = 0; t0 < a.T; t0 += NT) {
        const uint32_t nt = min(a.T - t0, (uint32_t)NT);
        double acc[2][NT];
        float v[2][NT], v2[2][NT];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[r][t] = 0.0;
        const float* const w[2] = {j.W + (size_t)ra * j.cols,
                                   (pair ? j.W2 : j.W) + (size_t)rb * j.cols};
        dot_rows<NT>(w, j.cols, j.x + (size_t)t0 * j.x_stride, j.x_stride, nt, s_x, acc);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t) v[r][t] = (float)wave_sum(acc[r][t]);
        if (j.out == kOutSum) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[r][t] = 0.0;
            const float* const w2[2] = {j.W2 + (size_t)ra * j.cols2, j.W2 + (size_t)rb * j.cols2};
            dot_rows<NT>(w2, j.cols2, j.x2 + (size_t)t0 * j.x2_stride, j.x2_stride, nt, s_x, acc);
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t) v2[r][t] = (float)wave_sum(acc[r][t]);
        }
        if (lane != 0) continue;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if ((uint32_t)t >= nt) break;
            float* y = j.y + (size_t)(t0 + t) * j.y_stride;
            if (pair) {
                if (r0 < j.rows) y[r0] = situ(v[0][t], v[1][t], j.beta, j.has_linear, j.linear);
                continue;
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (r0 + r >= j.rows) break;
                float sum = v[r][t];
                if (j.out == kOutSum) sum = __fadd_rn(sum, v2[r][t]);
                if (j.out == kOutAdd)
                    sum = __fadd_rn(j.x2[(size_t)(t0 + t) * j.x2_stride + r0 + r], sum);
                y[r0 + r] = sum;
                if (j.out == kOutSplit) {
                    const uint16_t hi = f32_to_bf16(v[r][t]);
                    uint16_t* ys = j.ys + (size_t)(t0 + t) * 2 * j.y_stride;
                    ys[r0 + r] = hi;
                    ys[j.y_stride + r0 + r] = act_lo_bf16(v[r][t], hi);
                }
            }
        }
    }
}

// One MXFP4 row per wave in the K3X layout (packed [rows][cols / 2], low
// nibble = even column; E8M0 scales [rows][cols / 32]); lane l takes the
// 32-element groups l, l + 64, ...  The 32 products of a group are exact in
// fp32 only up to their alignment, so each one is formed in double
// (runtime/src/ops.cpp:57-76).
__global__ __launch_bounds__(kThreads) void mxfp4_gemv_kernel(
    const uint8_t* __restrict__ packed, const uint8_t* __restrict__ scales, uint32_t rows,
    uint32_t cols, const float* __restrict__ x, uint32_t T, float* __restrict__ y,
    const uint32_t* status) {
    if (*(volatile const uint32_t*)status) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t r = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (r >= rows) return;
    const uint32_t groups = cols / 32;
    const uint4* pr = reinterpret_cast<const uint4*>(packed + (size_t)r * cols / 2);
    const uint8_t* sr = scales + (size_t)r * groups;
    for (uint32_t t0 = 0; t0 < T; t0 += kMaxTokens) {
        const uint32_t nt = min(T - t0, kMaxTokens);
        double acc[kMaxTokens];
#pragma unroll
        for (uint32_t t = 0; t < kMaxTokens; ++t) acc[t] = 0.0;
        for (uint32_t gi = lane; gi < groups; gi += 64) {
            const uint4 c = pr[gi];
            const float sc = e8m0_to_f32(sr[gi]);
            const uint32_t words[4] = {c.x, c.y, c.z, c.w};
            float wv[32];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // Eight bf16 values, element 2i in the low half of dword i.
                const uint4 d = __builtin_bit_cast(uint4, dequant8(words[j], sc));
                const uint32_t dw[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    wv[8 * j + 2 * i] = __uint_as_float(dw[i] << 16);
                    wv[8 * j + 2 * i + 1] = __uint_as_float(dw[i] & 0xffff0000u);
                }
            }
#pragma unroll
            for (uint32_t t = 0; t < kMaxTokens; ++t) {
                if (t >= nt) break;
                const float4* xr =
                    reinterpret_cast<const float4*>(x + (size_t)(t0 + t) * cols + (size_t)gi * 32);
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float4 xv = xr[q];
                    acc[t] = __builtin_fma((double)wv[4 * q + 0], (double)xv.x, acc[t]);
                    acc[t] = __builtin_fma((double)wv[4 * q + 1], (double)xv.y, acc[t]);
                    acc[t] = __builtin_fma((double)wv[4 * q + 2], (double)xv.z, acc[t]);
                    acc[t] = __builtin_fma((double)wv[4 * q + 3], (double)xv.w, acc[t]);
                }
            }
        }
#pragma unroll
        for (uint32_t t = 0; t < kMaxTokens; ++t) {
            if (t >= nt) break;
            const float v = (float)wave_sum(acc[t]);
            if (lane == 0) y[(size_t)(t0 + t) * rows + r] = v;
        }
    }
}

// RMSNorm of fp32 rows (runtime/src/ops.cpp:10-18): double sum of squares,
// inverse = 1 / sqrt(float(sum / n) + eps) in fp32, out = x * inverse * w.
constexpr int kNormWaves = 16, kNormThreads = 64 * kNormWaves;

__global__ __launch_bounds__(kNormThreads) void rmsnorm_f32_kernel(const float* __restrict__ x,
                                                               const float* __restrict__ w,
                                                               uint32_t n, uint32_t n_div,
                                                               float eps,
                                                               float* __restrict__ out,
                                                               const uint32_t* status) {
    __shared__ double part[kNormWaves];
    if (*(volatile const uint32_t*)status) return;
    const float* xr = x + (size_t)blockIdx.x * n;
    double sq = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += kNormThreads)
        sq = __builtin_fma((double)xr[i], (double)xr[i], sq);
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sq;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int i = 0; i < kNormWaves; ++i) tot += part[i];
    const float inv = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn((float)(tot / (double)n_div), eps)));
    float* orow = out + (size_t)blockIdx.x * n;
    for (uint32_t i = threadIdx.x; i < n; i += kNormThreads)
        orow[i] = __fmul_rn(__fmul_rn(xr[i], inv), w[i]);
}

int launched(k3x_hip_ctx* ctx, unsigned n) {
    ctx->kernel_launches += n;
    return hipGetLastError() == hipSuccess ? K3X_OK : K3X_ERR_BACKEND_UNAVAILABLE;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

bool vec_ok(const float* W, const float* x, uint32_t cols, uint32_t x_stride) {
    return cols % 4 == 0 && x_stride % 4 == 0 && aligned16(W) && aligned16(x);
}

int launch_vec(k3x_hip_ctx* ctx, const VecJob& a, const VecJob* b, uint32_t T) {
    VecArgs args{};
    args.T = T;
    args.status = ctx->status;
    auto blocks = [](const VecJob& j) {
        const uint32_t waves = j.out == kOutSitu ? j.rows : (j.rows + 1) / 2;
        return (waves + kWaves - 1) / kWaves;
    };
    args.job[0] = a;
    args.blocks0 = blocks(a);
    uint32_t total = args.blocks0;
    if (b) {
        args.job[1] = *b;
        total += blocks(*b);
    }
    if (T == 1)
        hipLaunchKernelGGL(f32_gemv_vec_kernel<1>, dim3(total), dim3(kThreads), 0, ctx->stream, args);
    else if (T == 2)
        hipLaunchKernelGGL(f32_gemv_vec_kernel<2>, dim3(total), dim3(kThreads), 0, ctx->stream, args);
    else if (T <= 4)
        hipLaunchKernelGGL(f32_gemv_vec_kernel<4>, dim3(total), dim3(kThreads), 0, ctx->stream, args);
    else  // passes of eight tokens
        hipLaunchKernelGGL(f32_gemv_vec_kernel<8>, dim3(total), dim3(kThreads), 0, ctx->stream, args);
    return launched(ctx, 1);
}

template <int OUT, bool VEC = false>
int launch_gemv(k3x_hip_ctx* ctx, GemvArgs a, hipStream_t stream) {
    a.status = ctx->status;
    hipLaunchKernelGGL((f32_gemv_kernel<OUT, VEC>), dim3((a.rows + kWaves - 1) / kWaves),
                       dim3(kThreads), 0, stream, a);
    return launched(ctx, 1);
}

// Whether a product alone runs a row a wave instead of the vector kernel's two,
// whose staging of 1024 columns and sums over a pass of eight tokens outweigh
// short rows' loads: up to 768 columns, but only to 512 where the passes are full and x
// is another kernel's output of this call (x_new), which every wave would fetch for
// itself from beyond its L2.  us, row a wave / vector: 7168 rows of 64 columns, 1 token
// 4.4 / 4.4, 5 8.0 / 14.9, 9 12.2 / 26.9; 4096 x 512, 5 tokens 7.7 / 9.6, 8 9.3 / 10.1;
// 4096 x 768, 9 tokens 12.1 / 15.8; 512 x 768, 8 tokens 7.4 / 8.3, 16 12.8 / 14.3, and
// as the down product of an MLP of 1024 columns, with its gate / up, 22.1 / 19.7 and
// 38.2 / 33.6; 4096 x 1024, 5 tokens 11.8 / 9.9.  (The latent layer's paired products
// keep the vector kernel: a launch less is worth more there.)
bool short_cols(uint32_t cols, uint32_t T, bool x_new) {
    return cols <= (T % 8 == 0 && x_new ? 512u : 768u);
}

VecJob plain_job(const float* W, uint32_t rows, uint32_t cols, const float* x, float* y) {
    VecJob j{};
    j.out = kOutPlain;
    j.rows = rows;
    j.cols = cols;
    j.W = W;
    j.x = x;
    j.x_stride = cols;
    j.y = y;
    j.y_stride = rows;
    return j;
}

GemvArgs plain_args(const float* W, uint32_t rows, uint32_t cols, const float* x, uint32_t T,
                    float* y) {
    GemvArgs a{};
    a.W = W;
    a.rows = rows;
    a.cols = cols;
    a.x = x;
    a.x_stride = cols;
    a.T = T;
    a.y = y;
    a.y_stride = rows;
    return a;
}

// y = W x; x_new: x is written by a kernel of the same call.
int matvec(k3x_hip_ctx* ctx, const float* W, uint32_t rows, uint32_t cols, const float* x,
           uint32_t T, float* y, bool x_new) {
    if (!vec_ok(W, x, cols, cols))
        return launch_gemv<0>(ctx, plain_args(W, rows, cols, x, T, y), ctx->stream);
    if (short_cols(cols, T, x_new))
        return launch_gemv<0, true>(ctx, plain_args(W, rows, cols, x, T, y), ctx->stream);
    return launch_vec(ctx, plain_job(W, rows, cols, x, y), nullptr, T);
}

// act = situ(gate x, up x) as a vector job.
VecJob situ_job(const float* gate, const float* up, uint32_t rows, uint32_t cols, const float* x,
                float* act, float beta, bool has_linear, float linear) {
    VecJob j = plain_job(gate, rows, cols, x, act);
    j.out = kOutSitu;
    j.W2 = up;
    j.beta = beta;
    j.has_linear = has_linear;
    j.linear = linear;
    return j;
}

bool situ_vec_ok(const float* gate, const float* up, const float* x, uint32_t cols) {
    return vec_ok(gate, x, cols, cols) && aligned16(up);
}

// act = situ(gate x, up x).
int situ_product(k3x_hip_ctx* ctx, const float* gate, const float* up, uint32_t rows,
                 uint32_t cols, const float* x, uint32_t T, float* act, float beta, bool has_linear,
                 float linear) {
    const bool vec = situ_vec_ok(gate, up, x, cols);
    if (vec && !short_cols(cols, T, false))
        return launch_vec(ctx, situ_job(gate, up, rows, cols, x, act, beta, has_linear, linear),
                          nullptr, T);
    GemvArgs g = plain_args(gate, rows, cols, x, T, act);
    g.W2 = up;
    g.beta = beta;
    g.has_linear = has_linear;
    g.linear = linear;
    return vec ? launch_gemv<3, true>(ctx, g, ctx->stream) : launch_gemv<3>(ctx, g, ctx->stream);
}

bool dims_ok(uint32_t rows, uint32_t cols, uint32_t T) {
    return rows && cols && T && rows <= (1u << 24) && cols <= (1u << 24) && T <= (1u << 16);
}

// Device scratch of the latent layer, grow-only, apart from the layer
// scratch the grouped expert call carves.
int ensure_latent(k3x_hip_ctx* ctx, size_t bytes) {
    if (bytes <= ctx->latent_bytes) return K3X_OK;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    if (ctx->latent_scratch) (void)hipFree(ctx->latent_scratch);
    ctx->latent_scratch = nullptr;
    ctx->latent_bytes = 0;
    const size_t rounded = (bytes + (1u << 20) - 1) & ~(size_t)((1u << 20) - 1);
    if (hipMalloc(&ctx->latent_scratch, rounded) != hipSuccess) {
        (void)hipGetLastError();
        return K3X_ERR_BACKEND_UNAVAILABLE;
    }
    ctx->latent_bytes = rounded;
    return K3X_OK;
}

}  // namespace

extern "C" {

int k3x_hip_dense_f32_matvec(k3x_hip_ctx* ctx, const float* W, uint32_t rows, uint32_t cols,
                             const float* x, uint32_t tokens, float* y) {
    if (!ctx || !W || !x || !y || !dims_ok(rows, cols, tokens)) return K3X_ERR_INVALID_EXTENT;
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    return matvec(ctx, W, rows, cols, x, tokens, y, false);
}

int k3x_hip_mxfp4_matvec(k3x_hip_ctx* ctx, const uint8_t* packed, const uint8_t* scales,
                         uint32_t rows, uint32_t cols, const float* x, uint32_t tokens, float* y) {
    if (!ctx || !packed || !scales || !x || !y || !dims_ok(rows, cols, tokens) || cols % 32)
        return K3X_ERR_INVALID_EXTENT;
    if (!aligned16(packed) || !aligned16(x)) return K3X_ERR_INVALID_EXTENT;  // 16-byte loads
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    hipLaunchKernelGGL(mxfp4_gemv_kernel, dim3((rows + kWaves - 1) / kWaves), dim3(kThreads), 0,
                       ctx->stream, packed, scales, rows, cols, x, tokens, y, ctx->status);
    return launched(ctx, 1);
}

int k3x_hip_dense_situ_mlp(k3x_hip_ctx* ctx, const float* gate, const float* up,
                           const float* down, uint32_t hidden, uint32_t inter, uint32_t out_rows,
                           float situ_beta, int has_situ_linear, float situ_linear_beta,
                           const float* x, uint32_t tokens, float* act, float* y) {
    if (!ctx || !gate || !up || !down || !x || !act || !y || !dims_ok(inter, hidden, tokens) ||
        !dims_ok(out_rows, inter, tokens))
        return K3X_ERR_INVALID_EXTENT;
    // The betas are used as given, as situ_glu does (no checks there).
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    const int st = situ_product(ctx, gate, up, inter, hidden, x, tokens, act, situ_beta,
                                has_situ_linear != 0, situ_linear_beta);
    return st ? st : matvec(ctx, down, out_rows, inter, act, tokens, y, true);
}

int k3x_hip_resident_moe_layer(k3x_hip_ctx* ctx, k3x_hip_bank* bank,
                               const k3x_hip_latent_weights* w, const k3x_hip_moe_params* p,
                               const float* x, const uint32_t* ids, const float* contributions,
                               const uint32_t* host_ids, const float* host_contributions,
                               float* out, float* mixed_out) {
    if (!ctx || !bank || !w || !p || !x || !ids || !contributions || !out || bank->ctx != ctx)
        return K3X_ERR_INVALID_EXTENT;
    const uint32_t H = w->hidden, L = w->latent, S = w->shared_inter, T = p->tokens;
    const uint32_t Ln = w->latent_norm ? w->latent_norm : L;  // RMSNorm divisor
    if (!w->routed_down || !w->routed_norm || !w->routed_up || !w->shared_gate ||
        !w->shared_up || !w->shared_down || !dims_ok(L, H, T) || !dims_ok(S, H, T) ||
        bank->desc.hidden != L || bank->desc.shared_inter != 0 || p->flags || Ln > L)
        return K3X_ERR_INVALID_EXTENT;
    if (p->glu != K3X_GLU_SITU || !std::isfinite(p->rms_epsilon) || !(p->rms_epsilon > 0.0f))
        return K3X_ERR_INVALID_MXFP4;
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    // Per-call buffers: latent [T][L] fp32 and its split bf16 rows [T][2 L],
    // the expert mix [T][L] fp32 (+ its bf16 cast), its RMSNorm [T][L], the
    // routed projection [T][H] and the shared activation [T][S].
    const size_t f_lat = (size_t)T * L * 4, f_hid = (size_t)T * H * 4, f_sh = (size_t)T * S * 4;
    auto up256 = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t need = up256(f_lat) * 3 + up256(f_lat) + up256((size_t)T * L * 2) +
                        up256(f_hid) + up256(f_sh);
    int st = ensure_latent(ctx, need);
    if (st) return st;
    uint8_t* base = static_cast<uint8_t*>(ctx->latent_scratch);
    size_t at = 0;
    auto take = [&](size_t b) {
        uint8_t* q = base + at;
        at += up256(b);
        return q;
    };
    float* latent = (float*)take(f_lat);
    uint16_t* latent_split = (uint16_t*)take(f_lat);  // [T][2 L] bf16
    float* mixed = mixed_out ? mixed_out : (float*)take(f_lat);
    float* normed = (float*)take(f_lat);
    uint16_t* mixed_bf16 = (uint16_t*)take((size_t)T * L * 2);
    float* routed = (float*)take(f_hid);
    float* sact = (float*)take(f_sh);
    // The shared MLP needs x only: its gate/up rides in the launch of the
    // latent projection, its down projection in the last one, where both
    // products of a launch take 16-byte loads; each product that does not is
    // a launch of its own, the others keep theirs.  (The scratch of `latent`
    // and the others starts 256-byte aligned.)
    const bool has_linear = p->has_situ_linear != 0;
    bool shared_done = false;
    // latent = routed_down . x (backend_cpu.cpp:317), with its split copy.
    if (vec_ok(w->routed_down, x, H, H)) {
        VecJob l = plain_job(w->routed_down, L, H, x, latent);
        l.out = kOutSplit;
        l.ys = latent_split;
        const VecJob g = situ_job(w->shared_gate, w->shared_up, S, H, x, sact, p->situ_beta,
                                  has_linear, p->situ_linear_beta);
        shared_done = situ_vec_ok(w->shared_gate, w->shared_up, x, H);
        if ((st = launch_vec(ctx, l, shared_done ? &g : nullptr, T))) return st;
    } else {
        GemvArgs a = plain_args(w->routed_down, L, H, x, T, latent);
        a.ys = latent_split;
        if ((st = launch_gemv<2>(ctx, a, ctx->stream))) return st;
    }
    if (!shared_done &&
        (st = situ_product(ctx, w->shared_gate, w->shared_up, S, H, x, T, sact, p->situ_beta,
                           has_linear, p->situ_linear_beta)))
        return st;
    // The experts on the latent, mixed in slot order in fp32
    // (backend_cpu.cpp:318-325): the bank's grouped path with fp32 input and
    // activations.
    k3x_hip_moe_params ep = *p;
    ep.flags = K3X_FLAG_SPLIT_INPUT | K3X_FLAG_SPLIT_ACT;
    k3x_hip_moe_taps taps{};
    taps.out_f32 = mixed;
    if ((st = k3x_hip_moe_forward_routed(ctx, bank, &ep, latent_split, ids, contributions,
                                         host_ids, host_contributions, mixed_bf16, &taps)))
        return st;
    // normalized = rms_norm(mixed, routed_norm) (backend_cpu.cpp:327-328).
    hipLaunchKernelGGL(rmsnorm_f32_kernel, dim3(T), dim3(kNormThreads), 0, ctx->stream, mixed,
                       w->routed_norm, L, Ln, p->rms_epsilon, normed, ctx->status);
    if ((st = launched(ctx, 1))) return st;
    // routed = routed_up . normalized (backend_cpu.cpp:329-330), shared =
    // shared_down . sact, out = routed + shared (:331-335) in one launch.
    const bool down_vec = vec_ok(w->shared_down, sact, S, S);
    if (down_vec && vec_ok(w->routed_up, normed, L, L)) {
        VecJob o = plain_job(w->routed_up, H, L, normed, out);
        o.out = kOutSum;
        o.W2 = w->shared_down;
        o.cols2 = S;
        o.x2 = sact;
        o.x2_stride = S;
        return launch_vec(ctx, o, nullptr, T);
    }
    if ((st = matvec(ctx, w->routed_up, H, L, normed, T, routed, true))) return st;
    if (down_vec) {
        VecJob o = plain_job(w->shared_down, H, S, sact, out);
        o.out = kOutAdd;
        o.x2 = routed;
        o.x2_stride = H;
        return launch_vec(ctx, o, nullptr, T);
    }
    GemvArgs d = plain_args(w->shared_down, H, S, sact, T, out);
    d.add = routed;
    return launch_gemv<1>(ctx, d, ctx->stream);
}

}  // extern "C"
