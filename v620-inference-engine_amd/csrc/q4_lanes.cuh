// Register-level pieces of the kernels whose waves hold 64 weight rows: one
// row's scale and zero per lane, crossed to the lanes that need them, and the
// exact unpack of nibbles to q - z.
#pragma once

#include "q4_common.cuh"

namespace qwq4 {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// both halves' rows of a value each lane holds for its own row (rows 0-31 in
// lanes 0-31, 32-63 in lanes 32-63): a = row lane % 32, b = row 32 + lane % 32
__device__ __forceinline__ void split_halves(uint32_t v, uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = r[0];
    b = r[1];
}

// a value each lane holds for its own row (row = lane): v[j] = that of row
// 16 j + lane % 16
__device__ __forceinline__ void split_quarters(uint32_t x, uint32_t (&v)[4]) {
    uint32_t a, b;
    split_halves(x, a, b);
    const auto p = __builtin_amdgcn_permlane16_swap(a, a, false, false);
    const auto q = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    v[0] = p[0];
    v[1] = p[1];
    v[2] = q[0];
    v[3] = q[1];
}

// 8 packed nibbles -> 8 fp16 q - z, exact. zl: -(1024 + z), zh: -(64 + z).
// Byte pairs go under the high byte of 1024; the low nibbles then read
// 1024 + q, the high ones 1024 + 16 q.
__device__ __forceinline__ uint4 unpack8_exact(uint32_t w, h2 zl, h2 zh) {
    const uint32_t p01 = __builtin_amdgcn_perm(0u, w, 0x0c010c00u), p23 = __builtin_amdgcn_perm(0u, w, 0x0c030c02u);
    auto lo = [&](uint32_t p) { return __builtin_bit_cast(h2, (p & 0x000f000fu) | 0x64006400u) + zl; };
    auto hi = [&](uint32_t p) {
        return __builtin_elementwise_fma(__builtin_bit_cast(h2, (p & 0x00f000f0u) | 0x64006400u),
                                         h2{_Float16(0.0625f), _Float16(0.0625f)}, zh);
    };
    uint4 r;
    r.x = __builtin_bit_cast(uint32_t, lo(p01));
    r.y = __builtin_bit_cast(uint32_t, lo(p23));
    r.z = __builtin_bit_cast(uint32_t, hi(p01));
    r.w = __builtin_bit_cast(uint32_t, hi(p23));
    return r;
}

}  // namespace qwq4
