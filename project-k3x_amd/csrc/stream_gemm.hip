// stream_gemm.hip -- the streaming expert GEMM: experts with few rows (1 to
// 64 a record), where the MXFP4 weights' stream from HBM bounds the launch
// and the rows only ride along (which calls take it: k3x_select.hpp).
//
// Workgroup = 4 waves, one record (expert, up to kStreamRows rows; a record
// with more is walked in chunks) x kRb 16-row output blocks, each wave its
// own NT blocks (gate/up: NT pairs of 16 gate + 16 up rows) over the full K.
// Per K tile (128 K):
//   * each wave loads its weight tiles into registers and dequantises them
//     once (v_cvt_scalef32_pk_bf16_fp4) for all of the chunk's row tiles;
//   * the chunk's activation rows (gathered through pair_token for the
//     gate/up) arrive in LDS by buffer loads that write LDS directly, in a
//     ring of kStages tiles, shared by the four waves.  Only the chunk's own
//     row tiles (1, 2 or 4 of 16 rows) are fetched and multiplied.
// Two workgroups or more (by MAXT) share a CU, so one's barriers, prologue and
// epilogue run under the other's stream.  Split rows ([hi | lo] bf16 halves
// of fp32 values) multiply both halves against each weight fragment, which
// is loaded and dequantised once.
//
// Bound: HBM up to about 32 rows an expert, the products and their LDS reads
// past that.  Measured, experts' weight bytes over the launch's time
// (H=7168, I=2048 experts; the rate before is the kernel that ran the size):
//   T=16 (7 rows at most)    gate/up 6.2 -> 6.7 TB/s, down 6.7 -> 6.4
//   T=64 (24 at most)        gate/up 4.1 -> 6.5, down 4.8 -> 5.9
//   T=127 (44 at most)       gate/up 3.9 -> 6.3, down 3.6 -> 5.8
//   T=331 (97 at most)       gate/up 3.9 -> 5.3, down 3.8 -> 4.6
// and with split down rows (3584 x 3072 experts) at T=97 2.6 -> 6.1.  (Down at
// one row tile is the one that lost; the gate/up of the same calls and their
// shorter grouping gain several times that.)
// Uniform 16, 32 and 64 rows an expert: 6.3, 5.5 and 4.1 TB/s gate/up.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "k3x_gemm.hpp"

using namespace k3x_dev;
using k3x_hip::StreamGemmArgs;

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kStages = 4;  // ring tiles: one multiplied, three requested; a scale dword's tiles

// Waits until at most N of this wave's vector-memory requests are
// outstanding and all its LDS operations are done, then meets the workgroup.
template <int N>
__device__ inline void wait_and_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <bool GATEUP, bool SPLITIN, bool SPLITOUT, int MAXT, int NT>
__global__ __launch_bounds__(kThreads, MAXT == 1 && !SPLITIN ? 4 : MAXT <= 2 && !SPLITIN ? 3 : 2)
void stream_gemm(StreamGemmArgs a) {
    constexpr int S = GATEUP ? 2 : 1;             // matrices per output row block
    constexpr int TERMS = SPLITIN ? 2 : 1;        // halves of an activation row
    constexpr uint32_t kStage = TERMS * MAXT * 256;  // 16-byte words per ring stage
    constexpr uint32_t kCols = kWaves * NT * 16;     // output columns per workgroup
    constexpr uint32_t kEs = GATEUP && !SPLITOUT ? 2 : 4;  // staged element bytes
    constexpr uint32_t kPitch = kCols * kEs + 16;          // staged row bytes
    // The epilogue stages the chunk's rows in the ring's bytes, in one pass.
    constexpr uint32_t kRing = kStages * kStage;
    constexpr uint32_t kOut = MAXT * 16 * kPitch / 16;
    constexpr uint32_t kA4 = kRing > kOut ? kRing : kOut;
    // One LDS array: a second variable makes the compiler drain the ring's
    // LDS-DMA requests before reads of either.
    __shared__ u32x4 s_a4[kA4 + MAXT * 4];
    uint32_t* const s_yrow = reinterpret_cast<uint32_t*>(s_a4 + kA4);
    if (*a.status) return;
    const uint32_t nblk = (a.nrb + kWaves * NT - 1) / (kWaves * NT);
    // Consecutive workgroups go to the eight XCDs in turn: record i belongs
    // to XCD i % 8, whose L2 then serves its rows to all nblk workgroups.
    const uint32_t xcd = blockIdx.x % 8, seq = blockIdx.x / 8;
    const uint32_t item = seq / nblk * 8 + xcd, jb = seq % nblk;
    if (item >= *a.n_recs) return;
    uint32_t e, cnt, off;
    if (a.recs4) {
        const uint4 rec = a.recs4[item];
        e = rec.x;
        cnt = rec.y;
        off = rec.z;
    } else {
        const uint2 rec = a.recs[item];
        e = rec.x & 0xffffu;
        cnt = rec.x >> 16;
        off = rec.y;
    }
    e = __builtin_amdgcn_readfirstlane(e);
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    off = __builtin_amdgcn_readfirstlane(off);
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t g = lane >> 4, n = lane & 15;
    const uint32_t kt = __builtin_amdgcn_readfirstlane(a.kt);
    const uint32_t lane16 = lane * 16, lane4 = lane * 4;
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.codes + e * a.codes_per_expert), (short)0,
        a.nrb * kt * (S * 1024u), 0x00020000);
    const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(a.scales + e * a.scales_per_expert), (short)0,
        (uint32_t)(a.scales_per_expert * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a.a), (short)0, a.a_bytes, 0x00020000);
    // Row blocks past the matrix (nrb not a multiple of the workgroup's)
    // repeat the last one and are not stored.
    uint32_t rb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) rb[nt] = min((jb * kWaves + wave) * NT + nt, a.nrb - 1);
    // MFMA operand of lane (n, g), 8-column group j, in 16-byte words: row n
    // (+ 16 per row tile, 256 words) chunk 4 g + j of the row-quad layout
    // (grouped_gemm.hip).
    uint32_t apos[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        apos[j] = (n >> 2) * 64 + ((4 * g + j) ^ (n >> 2)) * 4 + (n & 3);

    auto chunk = [&](auto mt_count, uint32_t m0) {
        constexpr int MT = decltype(mt_count)::value;
        constexpr int kALoads = TERMS * MT;  // activation requests per wave and tile
        constexpr int kWLoads = NT * S;      // weight requests per wave and tile
        const uint32_t rows = min(cnt - m0, (uint32_t)(MT * 16));
        // Wave w's request q fills row quad w * MT + q; rows past the chunk's
        // end repeat its last row (never stored).
        uint32_t aoff[MT];
#pragma unroll
        for (int q = 0; q < MT; ++q) {
            const uint32_t quad = wave * MT + q;
            const uint32_t rr = off + m0 + min(4 * quad + (lane & 3), rows - 1);
            const uint32_t src = a.gather ? a.pair_token[rr] : rr;
            aoff[q] = (src * a.a_stride + ((lane >> 2) ^ (quad & 3)) * 8) * 2;
        }
        uint32_t yv = 0;
        if constexpr (!GATEUP) {
            if (tid < MT * 16) {
                const uint32_t r = off + m0 + min(tid, rows - 1);
                yv = a.scatter ? a.pair_token[r] * a.top_k + a.pair_slot[r] : r;
            }
        }
        f32x4 acc[MT][NT][S];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int w = 0; w < S; ++w) acc[mt][nt][w] = f32x4{0.f, 0.f, 0.f, 0.f};
        u32x4 bc[kStages][NT][S];
        uint32_t sc[NT][S], scn[NT][S];
        const uint32_t last = kt - 1;
#define STREAM_LOAD_A(k, buf)                                                          \
    _Pragma("unroll") for (int t = 0; t < TERMS; ++t)                                  \
        _Pragma("unroll") for (int q = 0; q < MT; ++q)                                 \
            load_lds16(arsrc, &s_a4[(buf) * kStage + (t * MT * 4 + wave * MT + q) * 64], \
                       aoff[q], (k) * 256 + t * a.a_lo * 2);
#define STREAM_LOAD_B(d, k)                                                            \
    _Pragma("unroll") for (int nt = 0; nt < NT; ++nt)                                  \
        _Pragma("unroll") for (int w = 0; w < S; ++w) bc[d][nt][w] =                   \
            __builtin_amdgcn_raw_buffer_load_b128(wrsrc, lane16,                       \
                                                  ((rb[nt] * kt + (k)) * S + w) * 1024, kNt);
#define STREAM_LOAD_SC(dst, kq)                                                        \
    _Pragma("unroll") for (int nt = 0; nt < NT; ++nt)                                  \
        _Pragma("unroll") for (int w = 0; w < S; ++w) dst[nt][w] =                     \
            __builtin_amdgcn_raw_buffer_load_b32(srsrc, lane4,                         \
                                                 ((rb[nt] * a.ks + (kq)) * S + w) * 256, kNt);
        constexpr int kNt = 2;  // non-temporal: each weight byte is read once a call
        STREAM_LOAD_SC(sc, 0u)
#pragma unroll
        for (int d = 0; d < kStages - 1; ++d) {
            STREAM_LOAD_A(min((uint32_t)d, last), d)
            STREAM_LOAD_B(d, min((uint32_t)d, last))
            asm volatile("" ::: "memory");
        }
        if constexpr (!GATEUP) {
            if (tid < MT * 16) s_yrow[tid] = yv;
        }
        wait_and_barrier<(kStages - 2) * (kALoads + kWLoads)>();

        for (uint32_t kb = 0; kb < kt; kb += kStages) {
#pragma unroll
            for (int d = 0; d < kStages; ++d) {
                const uint32_t k = kb + d;
                const u32x4* sa = s_a4 + d * kStage;
                // The operands of column group j + 1 are read from LDS before the
                // multiplies of group j (the scheduler sinks the reads to
                // their use otherwise).
                u32x4 an[TERMS * MT];
#pragma unroll
                for (int i = 0; i < TERMS * MT; ++i) an[i] = sa[i * 256 + apos[0]];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32x4 av[TERMS * MT];
#pragma unroll
                    for (int i = 0; i < TERMS * MT; ++i) {
                        av[i] = an[i];
                        if (j < 3) an[i] = sa[i * 256 + apos[(j + 1) % 4]];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    bf16x8 bw[NT][S];
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int w = 0; w < S; ++w)
                            bw[nt][w] = dequant8(bc[d][nt][w][j],
                                                 e8m0_to_f32((sc[nt][w] >> (8 * d)) & 0xffu));
#pragma unroll
                    for (int t = 0; t < TERMS; ++t)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            const bf16x8 af = as_bf16x8(av[t * MT + mt]);
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                                for (int w = 0; w < S; ++w)
                                    acc[mt][nt][w] = mfma16x16x32(af, bw[nt][w], acc[mt][nt][w]);
                        }
                }
                if (k == last) break;  // workgroup-uniform
                // Step k's requests: tile k + kStages - 1 (past the end the last
                // tile again: the loads stay unconditional, their count exact).
                STREAM_LOAD_A(min(k + kStages - 1, last), (d + kStages - 1) % kStages)
                STREAM_LOAD_B((d + kStages - 1) % kStages, min(k + kStages - 1, last))
                if (d == 0) {
                    STREAM_LOAD_SC(scn, min(kb / 4 + 1, a.ks - 1))
                }
                // Tile k + 1, requested at step k - 2, has arrived once only
                // the requests of steps k - 1 and k are outstanding (the
                // counter retires in issue order).
                constexpr int kTwo = 2 * (kALoads + kWLoads);
                if (d <= 1) wait_and_barrier<kTwo + kWLoads>();
                else wait_and_barrier<kTwo>();
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int w = 0; w < S; ++w) sc[nt][w] = scn[nt][w];
        }
        // The repeated requests land before the ring is reused.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

        // Epilogue through LDS: row-major rows of the workgroup's columns,
        // then 16-byte stores (see grouped_gemm.hip).
        uint8_t* stage = reinterpret_cast<uint8_t*>(s_a4);
        const uint32_t col0 = jb * kCols, ncols = a.nrb * 16 - min(col0, a.nrb * 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t row = 16 * mt + 4 * g + i;
                    const uint32_t col = (wave * NT + nt) * 16 + n;
                    if constexpr (GATEUP && SPLITOUT) {
                        *reinterpret_cast<float*>(stage + row * kPitch + col * 4) =
                            glu(acc[mt][nt][0][i], acc[mt][nt][S - 1][i], a.glu);
                    } else if constexpr (GATEUP) {
                        reinterpret_cast<uint16_t*>(stage + row * kPitch)[col] =
                            f32_to_bf16(glu(acc[mt][nt][0][i], acc[mt][nt][S - 1][i], a.glu));
                    } else {
                        *reinterpret_cast<float*>(stage + row * kPitch + col * 4) =
                            acc[mt][nt][0][i];
                    }
                }
        __syncthreads();
        constexpr uint32_t kChunks = kCols * kEs / 16;  // 16-byte pieces per row
        for (uint32_t c = tid; c < rows * kChunks; c += kThreads) {
            const uint32_t row = c / kChunks, ch = c % kChunks;
            if (ch * (16 / kEs) >= ncols) continue;
            const u32x4 v = *reinterpret_cast<const u32x4*>(stage + row * kPitch + ch * 16);
            if constexpr (GATEUP && SPLITOUT) {
                uint32_t h[2], l[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const float v0 = __uint_as_float(v[2 * q]), v1 = __uint_as_float(v[2 * q + 1]);
                    const uint16_t h0 = f32_to_bf16(v0), h1 = f32_to_bf16(v1);
                    h[q] = (uint32_t)h0 | (uint32_t)h1 << 16;
                    l[q] = (uint32_t)act_lo_bf16(v0, h0) | (uint32_t)act_lo_bf16(v1, h1) << 16;
                }
                uint16_t* dst = a.act + (size_t)(off + m0 + row) * a.act_stride + col0 + ch * 4;
                *reinterpret_cast<uint2*>(dst) = make_uint2(h[0], h[1]);
                *reinterpret_cast<uint2*>(dst + a.act_lo) = make_uint2(l[0], l[1]);
            } else if constexpr (GATEUP) {
                *reinterpret_cast<u32x4*>(a.act + (size_t)(off + m0 + row) * a.act_stride + col0 +
                                          ch * 8) = v;
            } else {
                *reinterpret_cast<u32x4*>(a.y + (size_t)s_yrow[row] * a.y_stride + col0 + ch * 4) =
                    v;
            }
        }
    };
    for (uint32_t m0 = 0; m0 < cnt;) {
        const uint32_t left = cnt - m0;
        if (m0) __syncthreads();  // the last chunk has been copied out
        if (MAXT >= 4 && left > 32 && left <= 48) {
            chunk(std::integral_constant<int, (MAXT >= 4 ? 3 : MAXT)>{}, m0);
            m0 += 48;
        } else if (MAXT >= 4 && left > 32) {
            chunk(std::integral_constant<int, (MAXT >= 4 ? 4 : MAXT)>{}, m0);
            m0 += 64;
        } else if (MAXT >= 2 && left > 16) {
            chunk(std::integral_constant<int, (MAXT >= 2 ? 2 : MAXT)>{}, m0);
            m0 += 32;
        } else {
            chunk(std::integral_constant<int, 1>{}, m0);
            m0 += 16;
        }
    }
}

#undef STREAM_LOAD_A
#undef STREAM_LOAD_B
#undef STREAM_LOAD_SC

// Output 16-row blocks (pairs, for gate/up) per wave, by the row tiles of the
// launch: few blocks while the rows' traffic from the L2 stays below the
// weights' (more workgroups a CU; down at one row tile and T=13 6.1 TB/s with
// two blocks, 6.4 with one), more as the rows grow or come in two halves
// (split down at T=16: 5.6 TB/s with one block, 6.4 with two; four row tiles:
// gate/up 6.5 with one or two, down 5.7 with two, 5.9 with four).
template <bool GATEUP, bool SPLITIN, int MAXT>
constexpr int blocks_per_wave() {
    if (GATEUP) return MAXT <= 2 ? 1 : 2;
    if (SPLITIN) return MAXT == 1 ? 2 : 4;
    return MAXT == 1 ? 1 : MAXT == 2 ? 2 : 4;
}
template <bool GATEUP, bool SPLITIN, bool SPLITOUT, int MAXT>
void launch(const StreamGemmArgs& a, uint32_t max_recs, hipStream_t stream) {
    constexpr int NT = blocks_per_wave<GATEUP, SPLITIN, MAXT>();
    const uint32_t per = kWaves * NT;
    hipLaunchKernelGGL((stream_gemm<GATEUP, SPLITIN, SPLITOUT, MAXT, NT>),
                       dim3((max_recs + 7) / 8 * 8 * ((a.nrb + per - 1) / per)), dim3(kThreads),
                       0, stream, a);
}

// MAXT by the most rows an expert can have, at most TMAX (records with more
// rows are walked in chunks).  Two row tiles up to 96 tokens: few of many experts
// have more than 32 rows there, and the others gain from three workgroups a CU
// instead of two.  384 experts, Top-16, layer us with two / four row tiles: T=64
// 687 / 693, 80 738 / 742, 96 754 / 766; level from there (97 730 / 733, 104 778
// / 771, 112 786 / 800), then four (120 812 / 784, 127 884 / 835).  Few busy
// experts would want four earlier (16 experts Top-8: T=48 119 / 118, 64 166 / 132,
// 96 233 / 183).
template <bool GATEUP, bool SPLITIN, bool SPLITOUT, int TMAX>
void launch_tiles(const StreamGemmArgs& a, uint32_t max_recs, uint32_t max_rows,
                  hipStream_t stream) {
    if (max_rows <= 16) launch<GATEUP, SPLITIN, SPLITOUT, 1>(a, max_recs, stream);
    else if (max_rows <= 96) launch<GATEUP, SPLITIN, SPLITOUT, 2>(a, max_recs, stream);
    else launch<GATEUP, SPLITIN, SPLITOUT, TMAX>(a, max_recs, stream);
}

}  // namespace

namespace k3x_hip {

int launch_stream_gemm(k3x_hip_ctx* ctx, bool gateup, const StreamGemmArgs& a, uint32_t max_recs,
                       uint32_t max_rows, hipStream_t stream) {
    if (!stream) stream = ctx->stream;
    if (!a.nrb || !a.kt || !max_recs || !max_rows || (!a.recs4 && !a.recs) || !a.n_recs)
        return K3X_ERR_INVALID_EXTENT;
    // One expert's tiles and scales are addressed in 32 bits (stream_addressable).
    if ((uint64_t)a.nrb * a.kt * (gateup ? 2048u : 1024u) >= (1ull << 32) ||
        (uint64_t)a.scales_per_expert * 4 >= (1ull << 32))
        return K3X_ERR_INVALID_EXTENT;
    // The epilogue stores 16-byte row pieces (8-byte ones for split rows).
    if (gateup ? ((uintptr_t)a.act % 16 || a.act_stride % 8 || a.act_lo % 8)
               : ((uintptr_t)a.y % 16 || a.y_stride % 4))
        return K3X_ERR_INVALID_EXTENT;
    if (gateup && a.a_lo && a.act_lo) launch_tiles<true, true, true, 2>(a, max_recs, max_rows, stream);
    else if (gateup && a.a_lo) launch_tiles<true, true, false, 2>(a, max_recs, max_rows, stream);
    else if (gateup && a.act_lo) launch_tiles<true, false, true, 4>(a, max_recs, max_rows, stream);
    else if (gateup) launch_tiles<true, false, false, 4>(a, max_recs, max_rows, stream);
    else if (a.a_lo) launch_tiles<false, true, false, 2>(a, max_recs, max_rows, stream);
    else launch_tiles<false, false, false, 4>(a, max_recs, max_rows, stream);
    ctx->kernel_launches += 1;
    return hipGetLastError() == hipSuccess ? K3X_OK : K3X_ERR_BACKEND_UNAVAILABLE;
}

}  // namespace k3x_hip
