// int8 and int4 weight codes to f16 pairs, and bf16 scales: the conversions
// the weight-only kernels share.
#pragma once

#include "common.hpp"

namespace omni {

__device__ __forceinline__ u32 half2_bits(v2h h) {
    u32 u;
    __builtin_memcpy(&u, &h, 4);
    return u;
}
__device__ __forceinline__ v2h bits_half2(u32 u) {
    v2h h;
    __builtin_memcpy(&h, &u, 4);
    return h;
}

// Four int8 codes in `word` -> two f16 pairs (codes 0,1) and (codes 2,3), exact.
__device__ __forceinline__ void i8x4_to_f16x4(u32 word, v2h& lo, v2h& hi) {
    const u32 biased = word ^ 0x80808080u;  // w + 128 as unsigned bytes
    const u32 p0 = __builtin_amdgcn_perm(0x64646464u, biased, 0x04010400u);
    const u32 p1 = __builtin_amdgcn_perm(0x64646464u, biased, 0x04030402u);
    const v2h k1152 = {(_Float16)1152.0f, (_Float16)1152.0f};
    lo = bits_half2(p0) - k1152;
    hi = bits_half2(p1) - k1152;
}

// The same four codes as the f16 values 1152 + w (exact): three VALU per
// four codes. A dot product against them exceeds the true one by 1152 * (the
// sum of the activations), which the caller subtracts once per row.
__device__ __forceinline__ void i8x4_to_f16x4_biased(u32 word, v2h& lo, v2h& hi) {
    const u32 biased = word ^ 0x80808080u;
    lo = bits_half2(__builtin_amdgcn_perm(0x64646464u, biased, 0x04010400u));
    hi = bits_half2(__builtin_amdgcn_perm(0x64646464u, biased, 0x04030402u));
}

// Eight int4 codes of `word` (low nibble first, each stored plus 8, as
// crates/minicpm-v/src/quant.rs:22-29 unpacks them) -> four f16 pairs in k
// order (n0,n1) (n2,n3) (n4,n5) (n6,n7), exact: bytes [n, 0x64] are the f16
// 1024 + n, and one packed subtract of 1032 leaves n - 8.
// Byte t of word >> 4 holds code 2t + 1 in its low nibble: two v_perm_b32
// and two masks give the codes in k order one per byte, and one v_perm_b32
// per pair spreads two of them under 0x64 bytes (nine integer ops per word).
__device__ __forceinline__ void i4x8_to_f16x8(u32 word, v2h (&h)[4]) {
    const u32 sh = word >> 4;
    const u32 c0 = __builtin_amdgcn_perm(sh, word, 0x05010400u) & 0x0F0F0F0Fu;  // n0 n1 n2 n3
    const u32 c1 = __builtin_amdgcn_perm(sh, word, 0x07030602u) & 0x0F0F0F0Fu;  // n4 n5 n6 n7
    const u32 k64 = 0x64646464u;
    const v2h k1032 = {(_Float16)1032.0f, (_Float16)1032.0f};
    h[0] = bits_half2(__builtin_amdgcn_perm(k64, c0, 0x04010400u)) - k1032;
    h[1] = bits_half2(__builtin_amdgcn_perm(k64, c0, 0x04030402u)) - k1032;
    h[2] = bits_half2(__builtin_amdgcn_perm(k64, c1, 0x04010400u)) - k1032;
    h[3] = bits_half2(__builtin_amdgcn_perm(k64, c1, 0x04030402u)) - k1032;
}

// Eight int4 codes of `word` as the f16 values 1024 + nibble (exact), one
// v_perm_b32 per pair placing a nibble byte under the high byte 0x64 taken
// from k64 = 0x64646464, in the pairs (n0, n2), (n1, n3), (n4, n6), (n5, n7).
// The codes are nibble - 8, so a dot product against these values exceeds
// the true one by 1032 * (the sum of the activations), which the caller
// subtracts once per row of partial sums instead of once per pair.
__device__ __forceinline__ void i4x8_to_f16x8_biased(u32 word, u32 k64, v2h (&h)[4]) {
    const u32 lo = word & 0x0F0F0F0Fu;         // n0 n2 n4 n6
    const u32 hi = (word >> 4) & 0x0F0F0F0Fu;  // n1 n3 n5 n7
    h[0] = bits_half2(__builtin_amdgcn_perm(k64, lo, 0x04010400u));
    h[1] = bits_half2(__builtin_amdgcn_perm(k64, hi, 0x04010400u));
    h[2] = bits_half2(__builtin_amdgcn_perm(k64, lo, 0x04030402u));
    h[3] = bits_half2(__builtin_amdgcn_perm(k64, hi, 0x04030402u));
}

// A bf16 scale (quant.rs:74-81) as f32 (exact) and as f16 (exact for scales
// in f16's normal range, 2^-14 .. 65504).
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((u32)b << 16); }

// 16 int4 codes (two words) times one scale -> 16 halves in k order:
// f16(q * s), the dequantised value the reference's F16 route rounds to
// (quant.rs:186-200): q * s is exact in f32 and the packed f16 multiply
// rounds it once, like the f32 -> f16 cast.
__device__ __forceinline__ void i4x16_dequant(u32 w0, u32 w1, _Float16 s, v2h (&h)[8]) {
    v2h a[4], b[4];
    i4x8_to_f16x8(w0, a);
    i4x8_to_f16x8(w1, b);
    const v2h s2 = {s, s};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = a[i] * s2;
        h[4 + i] = b[i] * s2;
    }
}

}  // namespace omni
