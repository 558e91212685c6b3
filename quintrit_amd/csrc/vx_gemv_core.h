// The velurex digit arithmetic shared by the GEMV kernels (the lone/batched GEMV of vx_gemv.hip and the decode-step
// GEMV of vx_decode.hip): the digit nibbles of a byte and the broadcast 4-bit dot products.
#pragma once

#include <type_traits>
#include <hip/hip_runtime.h>

#include <cstdint>

namespace vx {

// ---- digits of a velurex byte ---------------------------------------------------------------------------------------

// U = floor(B / 28) is the 2-trit group (d3, d4), L = B - 28 U the 3-trit group (d0, d1, d2); B is a velurex value iff
// B <= 250 and L <= 26 (docs/velurex-encoding.md sections 2-3).
__host__ __device__ constexpr bool byte_valid(uint32_t b) {
    const uint32_t u = b / 28u, l = b - 28u * u;
    return b <= 250u && l <= 26u;
}

__host__ __device__ constexpr uint32_t digit_nibbles(uint32_t b) {
    if (!byte_valid(b)) return 0x11111u;  // five zero trits
    const uint32_t u = b / 28u, l = b - 28u * u;
    return (l % 3u) | ((l / 3u % 3u) << 4) | ((l / 9u) << 8) | ((u % 3u) << 12) | ((u / 3u) << 16);
}

// digit_nibbles of every byte, built at compile time (a kernel copies it into its LDS table with loads instead of
// computing 256 entries in every thread).
struct DigitTable {
    uint32_t v[256];
};
constexpr DigitTable make_digit_table() {
    DigitTable t{};
    for (uint32_t b = 0; b < 256; ++b) t.v[b] = digit_nibbles(b);
    return t;
}

// t0..t3 of byte b as int8 in a dword (byte p = trit p); bytes that are not velurex values give zero trits.
__host__ __device__ constexpr uint32_t trits03_word(uint32_t b) {
    if (!byte_valid(b)) return 0u;
    const uint32_t e = digit_nibbles(b);
    uint32_t w = 0;
    for (uint32_t p = 0; p < 4; ++p) w |= ((((e >> (4 * p)) & 15u) - 1u) & 0xffu) << (8 * p);
    return w;
}
struct TritTable {
    uint32_t v[256];
};
constexpr TritTable make_trit_table() {
    TritTable t{};
    for (uint32_t b = 0; b < 256; ++b) t.v[b] = trits03_word(b);
    return t;
}

// t4 of each byte of w as int8: d4 = floor(B / 84) from B >= 84 and B >= 168, tested with 7-bit adds that cannot carry
// (the halved byte B >> 1 is below 128), then t4 = d4 - 1 per byte as (d4 + 0x7f) ^ 0x80, again without carries.
// Every byte must be a velurex value.
__host__ __device__ constexpr uint32_t t4_bytes(uint32_t w) {
    const uint32_t x = (w >> 1) & 0x7f7f7f7fu;
    const uint32_t d4 = (((x + 0x56565656u) >> 7) & 0x01010101u) + (((x + 0x2c2c2c2cu) >> 7) & 0x01010101u);
    return (d4 + 0x7f7f7f7fu) ^ 0x80808080u;
}

// One lane's 16 bytes of a B fragment of the batched GEMM (vx_gemm.hip): K block kb and half hs of K step ks of a token
// whose activations x[0..n) are in LDS, 4-byte aligned. In a whole 160-trit block K block kb < 4 takes, for byte-column
// 16 hs + 4 kb + d, its activations of planes 0..3 (dword d the bytes 160 ks + 32 e + 16 hs + 4 kb + d, e = 0..3), K
// block 4 plane 4 of the 16 byte-columns; in the packed tail byte-column c holds the activations from 160 ks + 5 c on.
// Zero past the row.
__device__ __forceinline__ uint4 gemm_fragment(const int8_t* x, uint32_t n, uint32_t ks, uint32_t kb, uint32_t hs) {
    if (ks < n / 160u) {
        const int8_t* b = x + ks * 160u + 16u * hs;
        if (kb == 4u) return *reinterpret_cast<const uint4*>(b + 128);
        const uint32_t a0 = *reinterpret_cast<const uint32_t*>(b + 4u * kb), a1 = *reinterpret_cast<const uint32_t*>(b + 4u * kb + 32u);
        const uint32_t a2 = *reinterpret_cast<const uint32_t*>(b + 4u * kb + 64u), a3 = *reinterpret_cast<const uint32_t*>(b + 4u * kb + 96u);
        const uint32_t lo01 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), hi01 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(a3, a2, 0x05010400u), hi23 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
        return make_uint4(__builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                          __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u));
    }
    uint32_t w[4];
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            const uint32_t i = ks * 160u + (kb < 4u ? 5u * (16u * hs + 4u * kb + d) + e : 5u * (16u * hs + 4u * d + e) + 4u);
            v |= (i < n ? static_cast<uint32_t>(static_cast<uint8_t>(x[i])) : 0u) << (8u * e);
        }
        w[d] = v;
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// f(std::integral_constant<uint32_t, k>) for k = 0 .. N - 1: a loop body with its index as a compile-time constant, so that
// arrays indexed by it stay in fixed registers (a counted loop may be kept rolled, with the registers rotated).
template <uint32_t N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<uint32_t, N - 1>{});
    }
}

__host__ __device__ inline int trit_of(uint32_t b, uint32_t p) {
    return static_cast<int>((digit_nibbles(b) >> (4 * p)) & 15u) - 1;
}

// Four bytes of a lane's weights against their activations: lo += dot8(L of byte K + j, t_j), hi += dot8(H, t_j) for
// j = 0..3, where t_j is the digit-nibble table entry of byte j and the activation dwords of the 16 byte-columns of a
// chunk sit in lanes 0..15 of every 16-lane row of L and H, broadcast by DPP row_newbcast. v_dot8c_i32_i4 multiplies
// signed nibbles: the digits (0..2), the high nibbles x >> 4 and the low nibbles (x & 15) - 8. L and H come from LDS
// loads; the s_nop keeps the two wait states a DPP read needs after any VALU write of its source.
template <int K>
__device__ __forceinline__ void dot4_bcast(int& lo, int& hi, uint32_t L, uint32_t H, uint32_t t0, uint32_t t1, uint32_t t2,
                                           uint32_t t3) {
    asm("s_nop 1\n\t"
        "v_dot8c_i32_i4_dpp %0, %2, %4 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %1, %3, %4 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %0, %2, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %1, %3, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %0, %2, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %1, %3, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %0, %2, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
        "v_dot8c_i32_i4_dpp %1, %3, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf"
        : "+v"(lo), "+v"(hi)
        : "v"(L), "v"(H), "v"(t0), "v"(t1), "v"(t2), "v"(t3), "n"(K), "n"(K + 1), "n"(K + 2), "n"(K + 3));
}

}  // namespace vx
