// k3x_select.hpp -- which kernels run a call's routed experts: a rule on
// sizes alone (host code, no HIP), so that it can be checked where the sizes
// themselves could not be allocated.
#pragma once

#include <cstdint>

namespace k3x_hip {

enum RoutedKind {
    kRoutedFew,     // few tokens: the decode path's gate/up and down
    kRoutedStream,  // the streaming GEMM (stream_gemm.hip)
    kRoutedWide,    // many tokens: the wide GEMM (grouped_gemm.hip)
    kRoutedNarrow,  // operands past 32-bit offsets: expert_gemm
};

struct RoutedCall {
    uint32_t hidden, inter, tokens, top_k;
    bool split_act, split_in;  // activation / input rows as [hi | lo] halves
    bool scaled;               // K3X_FLAG_SCALED_FP4 in effect
    bool few;                  // the decode path's kernels take these tokens
    bool wide;                 // the wide GEMM's shape rules hold
};

// Tokens from which the wide GEMM can take routed experts at all.
constexpr uint32_t kWideMinTokens = 128;
// Tokens from which the wide GEMM's class launches beat the streaming GEMM
// (whole layer, H=7168, 384 experts of 2048, streaming / wide: T=160 872 /
// 1147 us, 331 1147 / 1281, 512 1484 / 1458, 768 1899 / 1773; the official
// layer's split rows, T=331 1598 / 1867, 512 2100 / 2036).  The scaled FP4
// path is the wide GEMM's own and keeps its range.
constexpr uint32_t kStreamMaxTokens = 448;

// The streaming GEMM addresses one expert's gate/up (or down) tiles, its
// scales and the activation rows by 32-bit byte offsets.
constexpr bool stream_addressable(const RoutedCall& c) {
    const uint64_t lim = 1ull << 32, K = c.top_k, T = c.tokens;
    return (uint64_t)c.inter * c.hidden < lim &&  // gate and up codes: half a byte each
           T * c.hidden * (c.split_in ? 4 : 2) < lim && T * K * c.inter * (c.split_act ? 4 : 2) < lim;
}

constexpr RoutedKind select_routed(const RoutedCall& c) {
    if (!c.split_in && c.few) return kRoutedFew;
    if (!c.split_in && c.wide && c.tokens >= (c.scaled ? kWideMinTokens : kStreamMaxTokens))
        return kRoutedWide;
    return stream_addressable(c) ? kRoutedStream : kRoutedNarrow;
}

}  // namespace k3x_hip
