// k3x_select.hpp -- which kernels run a call's routed experts: a rule on
// sizes alone (host code, no HIP), so that it can be checked where the sizes
// themselves could not be allocated.
#pragma once

#include <cstdint>

namespace k3x_hip {

enum RoutedKind {
    kRoutedFew,     // few tokens: the decode path's gate/up and down
    kRoutedRows,    // few pairs: the same kernels, a slot's rows four at a time
    kRoutedStream,  // the streaming GEMM (stream_gemm.hip)
    kRoutedWide,    // many tokens: the wide GEMM (grouped_gemm.hip)
    kRoutedNarrow,  // operands past 32-bit offsets: expert_gemm
};

struct RoutedCall {
    uint32_t hidden, inter, experts, tokens, top_k;
    bool split_act, split_in;  // activation / input rows as [hi | lo] halves
    bool shared;               // a shared expert of the bank runs beside
    bool scaled;               // K3X_FLAG_SCALED_FP4 in effect
    bool few;                  // the decode path's kernels take these tokens
    bool rows;                 // ... and row chunks of this shape and so many tokens
    bool wide;                 // the wide GEMM's shape rules hold
};

// Tokens from which the wide GEMM can take routed experts at all.
constexpr uint32_t kWideMinTokens = 128;
// Whether the wide GEMM's class launches beat the streaming GEMM.  The wide
// GEMM takes 128 rows a pass at one workgroup a CU, so it needs enough of them
// to fill the device: the line is the pairs times the workgroups that a
// 128-row chunk has over both launches (inter / 128 + hidden / 256).  More
// experts at the same pairs are partial chunks, which it pads and the
// streaming GEMM does not, and weights, which the streaming GEMM reads faster;
// more so with a shared expert beside (its wide GEMMs want the same CUs).
// Where every token takes every expert the chunks are full and the line lies
// lower, except where their last part falls in the one class (65 to 96 rows)
// that runs behind the full chunks and not beside them.  From 448 tokens
// always.  Layer us over changing banks, streaming / wide, at (experts, top_k,
// tokens):
//   H=7168 I=2048  (16, 16, 128) 247 / 280, (16, 16, 192) 405 / 303, (16, 16,
//                  416) 823 / 598, (16, 8, 256) 341 / 392, (16, 8, 447) 565 /
//                  500, (64, 16, 192) 472 / 486, (64, 16, 300) 689 / 554, (128,
//                  16, 256) 717 / 747, (128, 16, 384) 909 / 813, (384, 16,
//                  331) 1120 / 1123, (8, 4, 447) 280 / 402, (8, 8, 300) 336 /
//                  296, (8, 8, 331) 409 / 435
//   + shared 2048  (128, 16, 256) 748 / 815, (128, 16, 384) 973 / 856, (64, 8,
//                  384) 542 / 581, (64, 8, 447) 606 / 578, (384, 16, 331)
//                  1161 / 1220
//   H=3584 I=3072  (16, 16, 192) 336 / 267, (64, 16, 192) 367 / 388, (64, 16,
//                  300) 556 / 458, split rows (8, 8, 300) 352 / 297, (16, 4,
//                  447) 337 / 456
//   H=4096 I=1536  (16, 16, 224) 239 / 305, (16, 16, 256) 256 / 229, (16, 8,
//                  447) 277 / 318, (64, 16, 384) 412 / 354
//   H=1024 I=512   (16, 16, 331) 111 / 178, (64, 16, 447) 124 / 185
// The scaled FP4 path is the wide GEMM's own and keeps its range.
constexpr uint32_t kStreamMaxTokens = 448;
constexpr bool wide_faster(uint32_t hidden, uint32_t inter, uint32_t experts, uint32_t tokens,
                           uint32_t top_k, bool shared) {
    const uint64_t groups = inter / 128 + hidden / 256, pairs = (uint64_t)tokens * top_k;
    const uint32_t last = tokens % 128;  // rows of each expert's last chunk, where all are used
    const uint64_t line = experts > top_k ? 101000 : last > 64 && last <= 96 ? 118000 : 89000;
    return tokens >= kStreamMaxTokens ||
           10 * pairs * groups >= 10 * line + (shared ? 16ull : 7ull) * experts * top_k * groups;
}

// Whether the decode kernels' row chunks beat the streaming GEMM: few pairs.
// There a slot's workgroups split K over their eight waves and walk its rows
// four at a time: the time grows with the pairs, and with one expert's rows
// where few experts share them.  The streaming GEMM walks all of K in one
// wave, a chain of tiles that a few experts' workgroups cannot hide: the
// longer the chain (H / 128 tiles), the further both lines.  Where every token
// takes every expert no slot has more rows than another and the line lies a
// little further still; with one or two such experts and a long chain, 33 rows
// make the streaming GEMM walk it twice, which the row chunks beat up to about
// 44 rows.  Layer us over changing banks, row chunks / streaming, at (experts,
// top_k, pairs):
//   H=7168 I=2048  (2, 1, 5) 45 / 68, (4, 2, 10) 52 / 70, (4, 2, 22) 66 / 73,
//                  (16, 4, 24) 88 / 93, (4, 4, 32) 69 / 72, (8, 2, 32) 80 / 74,
//                  (1, 1, 16) 64 / 73, (1, 1, 32) 93 / 81, (1, 1, 40) 107 / 113
//   H=3584 I=3072  (4, 2, 10) 49 / 59, (4, 2, 22) 61 / 60, (4, 2, 32) 67 / 61
//   H=1024 I=512   (16, 2, 16) 37 / 38, (16, 4, 24) 39 / 38, (4, 2, 44) 52 / 39
constexpr bool rows_faster(uint32_t hidden, uint32_t experts, uint32_t tokens, uint32_t top_k) {
    const uint32_t kt = hidden / 128;
    const bool all = experts <= top_k;
    const uint64_t pairs = (uint64_t)tokens * top_k;
    if (all && experts <= 2 && tokens > 32 && tokens <= kt * 4 / 5) return true;
    return pairs <= 20 + kt / 5 + (all ? kt / 16 : 0) && pairs <= experts * (4ull + kt / 4);
}

// The streaming GEMM addresses one expert's gate/up (or down) tiles, its
// scales and the activation rows by 32-bit byte offsets.
constexpr bool stream_addressable(const RoutedCall& c) {
    const uint64_t lim = 1ull << 32, K = c.top_k, T = c.tokens;
    return (uint64_t)c.inter * c.hidden < lim &&  // gate and up codes: half a byte each
           T * c.hidden * (c.split_in ? 4 : 2) < lim && T * K * c.inter * (c.split_act ? 4 : 2) < lim;
}

// The rows kernel of the dense projections addresses a chunk of 64 rows (stride
// in elements) and a 16-row block's tiles by 32-bit byte offsets.
constexpr bool dense_rows_addressable(uint64_t stride, uint64_t block_bytes) {
    return stride * 64 * 2 < (1ull << 32) && block_bytes < (1ull << 32);
}

constexpr RoutedKind select_routed(const RoutedCall& c) {
    if (!c.split_in && c.few) return kRoutedFew;
    if (!c.split_in && c.rows && rows_faster(c.hidden, c.experts, c.tokens, c.top_k))
        return kRoutedRows;
    if (!c.split_in && c.wide && c.tokens >= kWideMinTokens &&
        (c.scaled || wide_faster(c.hidden, c.inter, c.experts, c.tokens, c.top_k, c.shared)))
        return kRoutedWide;
    return stream_addressable(c) ? kRoutedStream : kRoutedNarrow;
}

}  // namespace k3x_hip
