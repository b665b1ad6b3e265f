// storage.hip -- CRC32C of device bytes, for K3X storage extents checked once
// they are in HBM (the value of runtime/src/crc32c.cpp:22-28).
//
// CRC32C is linear over GF(2).  Write raw(A) for the register after A from a
// zero register; then the register after A || B from r is adv(r, |B|) ^
// raw(B), where adv(r, m) advances r over m zero bytes.  So:
//   * each lane takes 64 contiguous bytes of a 4 KiB chunk and forms their
//     raw CRC four bytes at a time (slicing-by-4 tables in LDS);
//   * a wave folds its 64 lane values into the chunk's raw CRC in a binary
//     tree, adv(left, 64 * 2^k) ^ right at level k, with adv by a fixed
//     length tabulated as four 256-entry byte tables (adv is linear);
//   * the workgroup that completes an extent folds its chunk values with one
//     wave: each lane a run of 2^m of them in order, then the lane tree with
//     the advances by 2^m chunks and up, read from the tables in the L2.
// Chunks are counted from an extent's end, in workgroups of four: the first
// ones may reach before its start, where they read zeros, which leave a raw
// CRC unchanged.  The host adds the preset register's advance and, for
// k3x_hip_crc32c, a tail below 16 bytes.  One launch takes all the extents of
// an expert, and looks for 0xFF bytes in the scales on the way.
// Bound: LDS table lookups (about 1.4 per byte) on large buffers; latency on
// an expert's records, so a wave takes 16 KiB there (64 KiB from kBigBytes,
// where the fold of the values would grow long), and a workgroup counts
// itself in once (counted per 4 KiB, 1344 increments of one word took 60 us).
// Measured: an admission of four 17.5 MB experts and the token run through
// them 1747 -> 229 us; one 17.5 MB buffer 55 -> 39 us, 256 MiB 120 -> 112 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "k3x_device.hpp"
#include "k3x_internal.hpp"
#include "k3x_reader.hpp"

using namespace k3x_dev;

namespace {

constexpr uint32_t kPoly = 0x82f63b78u;  // reflected Castagnoli polynomial
constexpr size_t kChunk = 4096;          // bytes per wave
constexpr int kLevels = 6;               // wave tree: 64 B .. 2 KiB halves
constexpr int kTables = 3 + kLevels;     // LDS: slicing, the tree levels, advances by 4 KiB
                                         // and by one chunk
constexpr int kSub = 4, kBigSub = 16;    // 4 KiB sub-chunks of a wave's chunk, and of a big
                                         // buffer's
constexpr size_t kBigBytes = 32u << 20;
constexpr size_t kHostBytes = 1024;      // k3x_hip_crc32c: below, the host folds the bytes
constexpr int kAdvLevels = 40;           // advance tables: 64 * 2^k bytes
constexpr int kCrcThreads = 256;

// Host tables: T[k][256] slicing-by-4, and advance tables A_m[4][256] with
// adv(r, m) = A_m[0][r & 255] ^ A_m[1][(r >> 8) & 255] ^ ...
struct CrcTables {
    uint32_t slice[4][256];
    uint32_t adv[kAdvLevels][4][256];  // m = 64 * 2^k (4 KiB at 6, 64 KiB at 10)
};

uint32_t adv_apply(const uint32_t (&a)[4][256], uint32_t r) {
    return a[0][r & 255] ^ a[1][(r >> 8) & 255] ^ a[2][(r >> 16) & 255] ^ a[3][r >> 24];
}

const CrcTables& host_tables() {
    static const CrcTables t = [] {
        CrcTables c{};
        for (uint32_t i = 0; i < 256; ++i) {
            uint32_t r = i;
            for (int b = 0; b < 8; ++b) r = (r >> 1) ^ (kPoly & (0u - (r & 1u)));
            c.slice[0][i] = r;
        }
        for (int k = 1; k < 4; ++k)
            for (uint32_t i = 0; i < 256; ++i)
                c.slice[k][i] = (c.slice[k - 1][i] >> 8) ^ c.slice[0][c.slice[k - 1][i] & 255];
        // adv over 64 zero bytes, directly; then doubling: adv_2m = adv_m o adv_m.
        for (int b = 0; b < 4; ++b)
            for (uint32_t x = 0; x < 256; ++x) {
                uint32_t r = x << (8 * b);
                for (int m = 0; m < 64; ++m) r = c.slice[0][r & 255] ^ (r >> 8);
                c.adv[0][b][x] = r;
            }
        for (int k = 1; k < kAdvLevels; ++k)
            for (int b = 0; b < 4; ++b)
                for (uint32_t x = 0; x < 256; ++x)
                    c.adv[k][b][x] = adv_apply(c.adv[k - 1], c.adv[k - 1][b][x]);
        return c;
    }();
    return t;
}

// adv(r) by a table in LDS or global memory.
__device__ inline uint32_t adv_by(const uint32_t* a, uint32_t r) {
    return a[r & 255] ^ a[256 + ((r >> 8) & 255)] ^ a[512 + ((r >> 16) & 255)] ^
           a[768 + (r >> 24)];
}

// The extents of one launch; extent i's results go to words slot[i] of the
// state (k3x_hip::ExtentState).
struct ExtentArgs {
    const uint8_t* data[k3x_hip::kExtents];
    uint64_t bytes[k3x_hip::kExtents];   // multiples of 16, > 0
    uint32_t first[k3x_hip::kExtents + 1];  // chunks of the extents before
    uint32_t slot[k3x_hip::kExtents];
    uint32_t n;
    uint32_t find_ff;                    // bit i: look for 0xFF bytes in extent i
    const uint32_t* tables;              // slicing [4][256], advance [kAdvLevels][4][256]
    uint32_t* vals;                      // [chunks]
    k3x_hip::ExtentState* state;         // device; counts and hits zero before and after
    k3x_hip::ExtentResult* host;         // pinned copy of the results
};

// One wave per chunk of SUB 4 KiB sub-chunks, four consecutive chunks of one
// extent a workgroup, grid-stride.  Each sub-chunk's raw CRC comes out of the
// lane tree; every lane folds them in order.
template <int SUB>
__global__ __launch_bounds__(kCrcThreads) void crc32c_extents_kernel(ExtentArgs a) {
    constexpr int kSubLevel = SUB == kSub ? 8 : 10;  // advance table of one chunk
    static_assert((64 << kSubLevel) == SUB * (int)kChunk, "advance by a chunk");
    __shared__ uint32_t t[kTables][1024];
    __shared__ uint32_t s_last;
    for (uint32_t i = threadIdx.x; i < (kTables - 1) * 1024; i += kCrcThreads)
        (&t[0][0])[i] = a.tables[i];
    for (uint32_t i = threadIdx.x; i < 1024; i += kCrcThreads)
        t[kTables - 1][i] = a.tables[(1 + kSubLevel) * 1024 + i];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t total = a.first[a.n];
    for (uint32_t c0 = blockIdx.x * 4; c0 < total; c0 += gridDim.x * 4) {
        uint32_t x = 0;
        while (x + 1 < a.n && c0 >= a.first[x + 1]) ++x;  // the chunks' extent
        const uint32_t nch = a.first[x + 1] - a.first[x], c = c0 + wave;
        const int64_t at =
            (int64_t)a.bytes[x] - (int64_t)(a.first[x + 1] - c) * (SUB * kChunk) + lane * 64;
        const uint8_t* src = a.data[x];
        u32x4 v[4], nx[4];
        auto load = [&](u32x4 (&d)[4], int sc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t p = at + (int64_t)sc * kChunk + 16 * i;
                d[i] = p >= 0 ? *reinterpret_cast<const u32x4*>(src + p) : u32x4{0u, 0u, 0u, 0u};
            }
        };
        uint32_t acc = 0, hit = 0;
        load(nx, 0);
        for (int sc = 0; sc < SUB; ++sc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = nx[i];
            if (sc + 1 < SUB) load(nx, sc + 1);
            uint32_t r = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t w = ~v[i][j];  // a zero byte of it is a 0xFF byte
                    hit |= (w - 0x01010101u) & ~w & 0x80808080u;
                    r ^= v[i][j];
                    r = t[0][768 + (r & 255)] ^ t[0][512 + ((r >> 8) & 255)] ^
                        t[0][256 + ((r >> 16) & 255)] ^ t[0][r >> 24];
                }
#pragma unroll
            for (int k = 0; k < kLevels; ++k)
                r = adv_by(t[1 + k], r) ^ __shfl_down(r, 1u << k);
            acc = adv_by(t[1 + kLevels], acc) ^ r;
        }
        // Publish the chunks' values (lane 0 holds each), then count the
        // workgroup in; the one whose count completes the extent folds it.
        k3x_hip::ExtentState* st = a.state;
        const uint32_t slot = a.slot[x];
        const bool ff = (a.find_ff >> x & 1u) && __any(hit != 0);
        if (lane == 0) {
            __hip_atomic_store(a.vals + c, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (ff)
                __hip_atomic_fetch_or(&st->hits[slot], 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            s_last = __hip_atomic_fetch_add(&st->counts[slot], 1u, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) == nch / 4 - 1;
        __syncthreads();
        if (!s_last || wave) continue;  // s_last is written again past the next barrier only
        // 64 runs of 2^m values, the list padded with zeros at its front.
        uint32_t m = 0;
        while ((64u << m) < nch) ++m;
        const uint32_t pad = (64u << m) - nch, run = 1u << m;
        uint32_t r = 0;
        for (uint32_t k0 = 0; k0 < run; k0 += 8) {
            uint32_t q[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t i = lane * run + k0 + k;
                const bool in = k0 + k < run && i >= pad;
                q[k] = in ? __hip_atomic_load(a.vals + a.first[x] + (i - pad), __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT)
                          : 0u;
            }
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                if (k0 + k < run) r = adv_by(t[kTables - 1], r) ^ q[k];
        }
        for (int k = 0; k < 6; ++k)
            r = adv_by(a.tables + (size_t)(1 + kSubLevel + m + k) * 1024, r) ^
                __shfl_down(r, 1u << k);
        if (lane == 0) {
            const uint32_t h = __hip_atomic_load(&st->hits[slot], __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            st->result.raw[slot] = r;
            st->result.ff[slot] = h;
            a.host->raw[slot] = r;
            a.host->ff[slot] = h;
            __hip_atomic_store(&st->counts[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&st->hits[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

int ensure_crc(k3x_hip_ctx* ctx, size_t chunks) {
    if (!ctx->crc_tables) {
        // Tables, then the zeroed state; the pinned results beside them.
        const CrcTables& h = host_tables();
        std::vector<uint32_t> dev((1 + kAdvLevels) * 1024 + sizeof(k3x_hip::ExtentState) / 4);
        std::memcpy(dev.data(), h.slice, 4096);
        std::memcpy(dev.data() + 1024, h.adv, sizeof(h.adv));
        uint32_t* p = nullptr;
        void* pinned = nullptr;
        if (hipHostMalloc(&pinned, sizeof(k3x_hip::ExtentResult), 0) != hipSuccess ||
            hipMalloc((void**)&p, dev.size() * 4) != hipSuccess ||
            hipMemcpy(p, dev.data(), dev.size() * 4, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            if (p) (void)hipFree(p);
            if (pinned) (void)hipHostFree(pinned);
            return K3X_ERR_BACKEND_UNAVAILABLE;
        }
        ctx->crc_tables = p;
        ctx->crc_state = reinterpret_cast<k3x_hip::ExtentState*>(p + (1 + kAdvLevels) * 1024);
        ctx->crc_host = static_cast<k3x_hip::ExtentResult*>(pinned);
    }
    const size_t need = std::max<size_t>(chunks, 1);
    if (need > ctx->crc_chunk_cap) {
        // Earlier launches may still use the old buffer.
        if (ctx->crc_chunks && hipStreamSynchronize(ctx->stream) != hipSuccess)
            return K3X_ERR_BACKEND_UNAVAILABLE;
        if (ctx->crc_chunks) (void)hipFree(ctx->crc_chunks);
        ctx->crc_chunks = nullptr;
        ctx->crc_chunk_cap = 0;
        if (hipMalloc((void**)&ctx->crc_chunks, need * 4) != hipSuccess) {
            (void)hipGetLastError();
            return K3X_ERR_BACKEND_UNAVAILABLE;
        }
        ctx->crc_chunk_cap = need;
    }
    return K3X_OK;
}

}  // namespace

namespace k3x_hip {

void free_crc(k3x_hip_ctx* ctx) {
    if (ctx->crc_tables) (void)hipFree(ctx->crc_tables);
    if (ctx->crc_chunks) (void)hipFree(ctx->crc_chunks);
    if (ctx->crc_host) (void)hipHostFree(ctx->crc_host);
    ctx->crc_tables = ctx->crc_chunks = nullptr;
    ctx->crc_state = nullptr;
    ctx->crc_host = nullptr;
    ctx->crc_chunk_cap = 0;
}

int launch_extent_check(k3x_hip_ctx* ctx, const Extent* ext, uint32_t n) {
    if (!n || n > kExtents) return K3X_ERR_INVALID_EXTENT;
    ExtentArgs a{};
    uint64_t largest = 0, chunks = 0;
    for (uint32_t i = 0; i < n; ++i) {
        if (!ext[i].bytes || ext[i].bytes % 16 || ext[i].slot >= kExtents ||
            reinterpret_cast<uintptr_t>(ext[i].data) % 16)
            return K3X_ERR_INVALID_EXTENT;
        largest = std::max<uint64_t>(largest, ext[i].bytes);
    }
    const bool big = largest >= kBigBytes;
    const uint64_t per = kChunk * (big ? kBigSub : kSub);
    for (uint32_t i = 0; i < n; ++i) {
        a.data[i] = static_cast<const uint8_t*>(ext[i].data);
        a.bytes[i] = ext[i].bytes;
        a.first[i] = (uint32_t)chunks;
        a.slot[i] = ext[i].slot;
        a.find_ff |= (ext[i].find_ff ? 1u : 0u) << i;
        chunks += ((ext[i].bytes + per - 1) / per + 3) / 4 * 4;  // whole workgroups
        if (chunks >= (1ull << 26)) return K3X_ERR_INVALID_EXTENT;  // 2^26 * 64 KiB
    }
    a.first[n] = (uint32_t)chunks;
    a.n = n;
    if (int st = ensure_crc(ctx, chunks)) return st;
    a.tables = ctx->crc_tables;
    a.vals = ctx->crc_chunks;
    a.state = ctx->crc_state;
    a.host = ctx->crc_host;
    const dim3 grid((unsigned)std::min<uint64_t>(chunks / 4, (uint64_t)ctx->cu_count * 8));
    if (big)
        hipLaunchKernelGGL(crc32c_extents_kernel<kBigSub>, grid, dim3(kCrcThreads), 0, ctx->stream,
                           a);
    else
        hipLaunchKernelGGL(crc32c_extents_kernel<kSub>, grid, dim3(kCrcThreads), 0, ctx->stream, a);
    ctx->kernel_launches += 1;
    return hipGetLastError() == hipSuccess ? K3X_OK : K3X_ERR_BACKEND_UNAVAILABLE;
}

uint32_t raw_of_crc(uint32_t crc, uint64_t bytes) {
    const CrcTables& h = host_tables();
    uint32_t r = 0xffffffffu;
    for (uint64_t i = 0; i < bytes % 64; ++i) r = h.slice[0][r & 255] ^ (r >> 8);
    for (int k = 0; k < kAdvLevels; ++k)
        if (bytes / 64 >> k & 1) r = adv_apply(h.adv[k], r);
    return ~crc ^ r;
}

int crc32c_device(k3x_hip_ctx* ctx, const void* data, size_t bytes, uint32_t* crc) {
    if (!ctx || (!data && bytes) || !crc) return K3X_ERR_INVALID_EXTENT;
    if (reinterpret_cast<uintptr_t>(data) % 16) return K3X_ERR_INVALID_EXTENT;
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    // Whole 16-byte words on the device, the tail on the host; a few bytes, or a
    // tail beside a few more, wholly there: one small copy, no launch (us, host /
    // device: 100 bytes 21.6 / 32.8, 512 22.4 / 23.6, 4095 28.2 / 33.1; 2048
    // 25.0 / 23.6).
    const bool host = bytes < kHostBytes || (bytes < kChunk && bytes % 16);
    const size_t body = host ? 0 : bytes & ~(size_t)15, tail = bytes - body;
    uint8_t tail_bytes[kChunk];
    if (body) {
        const Extent e{data, body, 0, false};
        if (int st = launch_extent_check(ctx, &e, 1)) return st;
    }
    if (tail && hipMemcpyAsync(tail_bytes, static_cast<const uint8_t*>(data) + body, tail,
                               hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
        return K3X_ERR_BACKEND_UNAVAILABLE;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    // ~raw_of_crc(0, n) is the preset register advanced over n bytes.
    uint32_t r = ~raw_of_crc(0u, body) ^ (body ? ctx->crc_host->raw[0] : 0u);
    const CrcTables& h = host_tables();
    for (size_t i = 0; i < tail; ++i) r = h.slice[0][(r ^ tail_bytes[i]) & 255] ^ (r >> 8);
    *crc = ~r;
    return K3X_OK;
}

}  // namespace k3x_hip

extern "C" int k3x_hip_crc32c(k3x_hip_ctx* ctx, const void* data, size_t bytes, uint32_t* crc) {
    return k3x_hip::crc32c_device(ctx, data, bytes, crc);
}

// ---------------------------------------------------------------------------
// K3X storage objects: the reader's checked directory (k3x_reader.cpp) and
// the expert load of load_storage_expert, feeding the bank through one pinned
// staging buffer and one device staging buffer per storage object.
// ---------------------------------------------------------------------------
#include <string>

struct k3x_hip_storage {
    k3x_reader::Directory dir;   // the checked directory (k3x_reader.cpp)
    uint8_t* pinned = nullptr;   // hipHostMalloc
    size_t pinned_bytes = 0;
    uint8_t* staging = nullptr;  // device
    size_t staging_bytes = 0;
    int staging_device = -1;
};

namespace {

void close_storage(k3x_hip_storage* s) {
    k3x_reader::close(&s->dir);
    if (s->pinned) (void)hipHostFree(s->pinned);
    if (s->staging) {
        (void)hipSetDevice(s->staging_device);
        (void)hipFree(s->staging);
    }
}

}  // namespace

extern "C" {

int k3x_hip_storage_open(const char* path, k3x_hip_storage** out) {
    if (!path || !out) return K3X_ERR_INVALID_EXTENT;
    *out = nullptr;
    auto* s = new (std::nothrow) k3x_hip_storage();
    if (!s) return K3X_ERR_BACKEND_UNAVAILABLE;
    const int st = k3x_reader::open_checked(&s->dir, path);
    if (st) {
        close_storage(s);
        delete s;
        return st;
    }
    *out = s;
    return K3X_OK;
}

int k3x_hip_storage_close(k3x_hip_storage* s) {
    if (!s) return K3X_ERR_INVALID_EXTENT;
    close_storage(s);
    delete s;
    return K3X_OK;
}

int k3x_hip_storage_verify(k3x_hip_storage* s) {
    if (!s) return K3X_ERR_INVALID_EXTENT;
    return k3x_reader::verify_checksums(s->dir);
}

int k3x_hip_storage_upload_expert(k3x_hip_storage* s, k3x_hip_bank* bank, uint32_t expert,
                                  uint32_t layer_id, uint32_t expert_id, uint64_t* bytes_read,
                                  uint8_t* ordered_sha256) {
    if (!s || !bank) return K3X_ERR_INVALID_EXTENT;
    if (!(s->dir.optional_features & 1u)) return K3X_ERR_INVALID_EXTENT;  // not a storage fixture
    const auto& d = bank->desc;
    const std::string base = "model.layers." + std::to_string(layer_id) +
                             ".feed_forward.experts." + std::to_string(expert_id) + ".";
    const char* roles[3] = {"gate", "up", "down"};
    const uint64_t shape[3][2] = {{d.inter, d.hidden}, {d.inter, d.hidden}, {d.hidden, d.inter}};
    const k3x_reader::TensorRecord* rec[3];
    for (int m = 0; m < 3; ++m) {
        const uint64_t id = k3x_reader::fnv1a64(base + roles[m]);
        rec[m] = nullptr;
        for (const auto& t : s->dir.tensors)
            if (t.id == id) rec[m] = &t;
        if (!rec[m]) return K3X_ERR_TENSOR_NOT_FOUND;
        const auto& t = *rec[m];
        const uint64_t n = shape[m][0] * shape[m][1];
        // valid_native_matrix (runtime/src/storage_slice.cpp:19-33).
        if (t.dtype != 2 || t.quant != 1 || t.rank != 2 || t.layer != (int32_t)layer_id ||
            t.expert != (int32_t)expert_id || t.dims[0] != shape[m][0] ||
            t.dims[1] != shape[m][1] || t.dims[2] || t.dims[3] || t.data_length != n / 2 ||
            t.aux_length != n / 32)
            return K3X_ERR_INVALID_MXFP4;
    }
    uint64_t off[6], len[6], at[6];
    uint32_t crc[6];
    size_t total = 0;
    for (int m = 0; m < 3; ++m) {
        off[2 * m] = rec[m]->data_offset;
        len[2 * m] = rec[m]->data_length;
        crc[2 * m] = rec[m]->data_crc;
        off[2 * m + 1] = rec[m]->aux_offset;
        len[2 * m + 1] = rec[m]->aux_length;
        crc[2 * m + 1] = rec[m]->aux_crc;
    }
    for (int i = 0; i < 6; ++i) {
        at[i] = total;
        total += (len[i] + 255) & ~(uint64_t)255;
    }
    if (expert >= bank->desc.experts) return K3X_ERR_INVALID_MXFP4;
    k3x_hip_ctx* ctx = bank->ctx;
    if (hipSetDevice(ctx->device) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    if (total > s->pinned_bytes) {
        if (s->pinned) (void)hipHostFree(s->pinned);
        s->pinned = nullptr;
        s->pinned_bytes = 0;
        if (hipHostMalloc((void**)&s->pinned, total, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return K3X_ERR_BACKEND_UNAVAILABLE;
        }
        s->pinned_bytes = total;
    }
    if (total > s->staging_bytes || s->staging_device != ctx->device) {
        if (s->staging) {
            (void)hipSetDevice(s->staging_device);
            (void)hipFree(s->staging);
            (void)hipSetDevice(ctx->device);
        }
        s->staging = nullptr;
        s->staging_bytes = 0;
        if (hipMalloc((void**)&s->staging, total) != hipSuccess) {
            (void)hipGetLastError();
            return K3X_ERR_BACKEND_UNAVAILABLE;
        }
        s->staging_bytes = total;
        s->staging_device = ctx->device;
    }
    for (int i = 0; i < 6; ++i)
        if (!k3x_reader::read_at(s->dir.fd, off[i], len[i], s->pinned + at[i]))
            return K3X_ERR_TRUNCATED_FILE;
    if (hipMemcpyAsync(s->staging, s->pinned, total, hipMemcpyHostToDevice, ctx->stream) !=
        hipSuccess)
        return K3X_ERR_BACKEND_UNAVAILABLE;
    const uint8_t* ext[6];
    for (int i = 0; i < 6; ++i) ext[i] = s->staging + at[i];
    const uint64_t ids[3] = {rec[0]->id, rec[1]->id, rec[2]->id};
    const int st = k3x_hip_bank_upload_expert_device(bank, expert, ids, ext, crc);
    // A rejection may return before the copy above has been waited for:
    // drain it, so that no later call refills the pinned or staging buffer
    // while this copy still reads or writes it.
    if (st && hipStreamSynchronize(ctx->stream) != hipSuccess) return K3X_ERR_BACKEND_UNAVAILABLE;
    if (!st && bytes_read) *bytes_read = len[0] + len[1] + len[2] + len[3] + len[4] + len[5];
    if (!st && ordered_sha256) {
        // The digest load_storage_expert returns (storage_slice.cpp:80-90):
        // the six extents in order, from the bytes read into pinned memory.
        k3x_reader::Sha256 h;
        for (int i = 0; i < 6; ++i) h.update(s->pinned + at[i], len[i]);
        h.finish(ordered_sha256);
    }
    return st;
}

}  // extern "C"
