// Loads from memory straight into LDS (buffer_load ... lds), for the K loops of the two quantised GEMMs.
#pragma once
#include "l2_internal.h"

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int kStepRow = 128; // bytes of a token in an activation tile of 64 k (16-bit values)

// Memory as a buffer of `bytes` from `base` (both the same in every lane).
__device__ __forceinline__ u4v buffer(const void *base, size_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    const uint32_t n = (uint32_t)(bytes < 0xFFFFFFFFull ? bytes : 0xFFFFFFFFull);
    return u4v{(uint32_t)__builtin_amdgcn_readfirstlane((int)p), (uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) & 0xFFFFu,
               (uint32_t)__builtin_amdgcn_readfirstlane((int)n), 0x00020000u};
}

__device__ __forceinline__ uint32_t lds_offset(void *p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)p; }

// From memory into LDS past the registers: lane l's piece (16 or 4 bytes) at `off` + `soff` bytes of the buffer goes to
// lds + `at` + size * l.  `at` (0..4095) shifts the source too, so callers have it taken off `off`; buffers therefore begin kBias
// bytes early and offsets are that much larger.  The destination goes through m0, set in the same statement: the compiler keeps
// what it holds there itself out of the way.  vmcnt counts these loads in order with all others, and since the compiler does
// not know of them, nothing else in a loop that waits for them by number may load from memory.
constexpr int kBias = 4096;
#define LDS_LOAD(n, lds, at, buf, off, soff) \
    asm volatile("s_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dword" n " %0, %1, %2 offen offset:%3 lds" \
                 ::"v"(off), "s"(buf), "s"(soff), "n"(at), "s"(lds) : "memory", "m0")

__device__ __forceinline__ u4v biased_buffer(const void *base, size_t bytes) { return buffer(reinterpret_cast<const char *>(base) - kBias, bytes + kBias); }

// By what the 16-byte pieces 0..7 of token t lie permuted (xor) in an activation tile of 128-byte rows.  A 16-byte LDS read takes
// the lanes 0-3, 12-15, 20-23 and 24-27 of each half of a wave together, then the others: with token r = l % 16 and piece
// 2 (l / 16 % 4) + s in the lanes, or piece l / 16 % 4 + 4 s, these sixteen then meet sixteen different places.
__device__ __forceinline__ int piece_xor(int t) {
    const int q = t >> 1;
    return (q & 1) | (q >> 1 & 2) | ((q << 1 ^ q) & 4);
}

// Blocks are dealt round-robin over the 8 XCDs, each with an L2 of its own: a contiguous range of the n items for each.
__device__ __forceinline__ int xcd_item(int b, int n) {
    const int per = n >> 3, over = n & 7, xcd = b & 7;
    return xcd * per + min(xcd, over) + (b >> 3);
}

} // namespace
