// Dense q4 GEMV for 9 to 32 rows, streamed: where the decode GEMV
// (q4_gemv_impl.cuh) stages every activation row of the whole K in LDS per 16
// weight rows, which outweighs the weights from about 8 rows on and no longer
// fits beyond 16 rows of 4096, a block here takes 64 WN weight rows and moves
// the rows' K in groups of 128 through a double buffer.
//
// The block's 8 waves are WN along the weight rows x WK = 8 / WN along K; a
// wave holds 64 weight rows (four 16-row subtiles) and the wk-th range of K
// groups, unpacks each weight once for all 16 MB rows (16x16x32 MFMA), and the
// parts' sums are added through LDS in part order. Each group goes out one
// group ahead: the part's A rows (direct global -> LDS loads, split over its WN
// waves) and the wave's weights, scale and zero (registers).
//
// Numerics as the decode GEMV's: exact products, fp32 sums, the group scale
// applied in fp32. fp16 rows take the exact q - z as operand, bf16 rows
// 128 + q with the zero point subtracted through the group's activation sum.
#pragma once

#include "q4_gemv_core.cuh"
#include "q4_lanes.cuh"

namespace qwq4 {

template <int MB, int WN>
struct Wide {
    static constexpr int WK = 8 / WN, ROWS = 64 * WN, BM = 16 * MB;
    static constexpr int NA = (BM / 4 + WN - 1) / WN;  // direct A loads per wave and group
    static constexpr int SLOT = 16 * 64 * 4;           // closing sums: 16 rows at a time per wave
    static constexpr int A = WK * BM * 256;            // bytes of a group's A
    static constexpr int SZ = WK > 1 && A < 4 * SLOT ? 4 * SLOT : A;
};

// 16-byte chunk c (0..15) of row r of a part's A tile [BM][128]
__device__ __forceinline__ int wide_swz(int r, int c) { return r * 256 + ((c ^ (r & 15)) << 4); }

template <typename XT, int MB, int WN, bool HAS_Z>
__device__ __forceinline__ void gemv_wide_block(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                const uint16_t *__restrict__ x, int xs, int M, int K, int N,
                                                void *__restrict__ y, int ys, int y_bf16, int accumulate, int n_lo) {
    using S = Wide<MB, WN>;
    constexpr int WK = S::WK, BM = S::BM, NA = S::NA;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    // Weights are read once: non-temporal loads are 1-5% faster (4096->12288 at 9
    // / 32 bf16 rows 10.7 / 13.3 -> 10.1 / 12.8 us; LM head at 32 fp16 rows 90.5 ->
    // 86.9), but not where they cost registers at the limit (LM head at 32 bf16
    // rows 88 -> 113).
    constexpr bool NT = !(MB == 2 && WN > 1 && __is_same(XT, BF16));
    __shared__ __align__(16) unsigned char a0[S::SZ], a1[S::SZ];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, n = lane % 16,
              q = lane / 16, wn = wave % WN, wk = wave / WN;
    const int nb = int(gridDim.x), xq = nb / 8, xr = nb % 8, xcd = int(blockIdx.x) % 8;
    const int item = xcd * xq + min(xcd, xr) + int(blockIdx.x) / 8;  // a contiguous range of row blocks per XCD
    const int n0 = item * S::ROWS + wn * 64, nsub = (N + 15) / 16;
    const int G = K / QGROUP, GC = (G + 3) / 4, per = G / WK, rem = G % WK;
    const int g0 = wk * per + min(wk, rem), ng = per + (wk < rem), ngmax = per + (rem > 0);

    // wave-uniform bases and 32-bit lane offsets (M xs fits: see the launch)
    const int sub0 = n0 / 16;
    const uint4 *w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = reinterpret_cast<const uint4 *>(Wt) + int64_t(min(sub0 + j, nsub - 1)) * G * 64;
    // this lane's own row's scale and zero words
    const int sb = min(sub0, nsub - 1), so = min(q, nsub - 1 - sb) * GC;
    const uint16_t *sp = St + int64_t(sb) * GC * 64, *zp = HAS_Z ? Zt + int64_t(sb) * GC * 16 : nullptr;
    const int s_off = so * 64 + n * 4, z_off = so * 16 + n;
    // A: instruction j of the wave moves rows 4 (j WN + wn) .. + 3 of its part
    int xo[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int r = (j * WN + wn) * 4 + q;
        xo[j] = min(r, M - 1) * xs + ((n ^ (r & 15)) * 8);
    }
    struct WR {
        uint4 w[4];
        uint16_t s, z;
    };
    auto group = [&](int i) { return min(g0 + min(i, max(ng, 1) - 1), G - 1); };  // past the end: a valid (unused) one
    auto issue = [&](int i, unsigned char *dst, WR &r) {
        const int g = group(i);
#pragma unroll
        for (int j = 0; j < NA; ++j)
            if ((j * WN + wn) * 4 < BM)  // (wave-uniform)
                __builtin_amdgcn_global_load_lds(x + g * QGROUP + xo[j], dst + wk * (BM * 256) + (j * WN + wn) * 1024, 16, 0,
                                                 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (NT) {
                const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w[j] + g * 64 + lane));
                r.w[j] = make_uint4(v[0], v[1], v[2], v[3]);
            } else {
                r.w[j] = w[j][g * 64 + lane];
            }
        }
        r.s = sp[(g >> 2) * 64 + (g & 3) + s_off];
        if constexpr (HAS_Z) r.z = zp[(g >> 2) * 16 + z_off];
    };
    f32x4 acc[4][MB];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const unsigned char *ab, const WR &r, int i) {
        const unsigned char *a = ab + wk * (BM * 256);
        uint32_t s = r.s, z = HAS_Z ? uint32_t(r.z) : 0u, sv[4], zv[4];
        asm volatile("" : "+v"(s), "+v"(z));  // taken here, not at their loads
        split_quarters(s, sv);
        if constexpr (HAS_Z) split_quarters((z >> (4 * (group(i) & 3))) & 0xfu, zv);
        else zv[0] = zv[1] = zv[2] = zv[3] = 8u;
        const uint4 one = make_uint4(XT::ONE, XT::ONE, XT::ONE, XT::ONE);
        f32x4 sum[MB];  // bf16: the group's activation sums
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) sum[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
        // two subtiles at a time, the fragments read again for the second two
        // (held across all four they would cost MB 2 its registers)
#pragma unroll
        for (int jp = 0; jp < 4; jp += 2) {
            asm volatile("" ::: "memory");
            h2 zl[2], zh[2];
            f32x4 p[2][MB];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                zl[j] = __builtin_bit_cast(h2, zv[jp + j] * 0x10001u | 0xe400e400u);         // -(1024 + z)
                zh[j] = __builtin_bit_cast(h2, (zv[jp + j] << 4) * 0x10001u + 0xd400d400u);  // -(64 + z)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) p[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                uint4 af[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    af[mb] = *reinterpret_cast<const uint4 *>(a + wide_swz(mb * 16 + n, q * 4 + t));
                    if constexpr (__is_same(XT, BF16))
                        if (jp == 0) sum[mb] = mfma16<XT>(af[mb], one, sum[mb]);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint4 &wj = r.w[jp + j];
                    const uint32_t word = t == 0 ? wj.x : t == 1 ? wj.y : t == 2 ? wj.z : wj.w;
                    uint4 f;
                    if constexpr (__is_same(XT, BF16)) f = unpack8_q<BF16>(word);
                    else f = unpack8_exact(word, zl[j], zh[j]);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) p[j][mb] = mfma16<XT>(af[mb], f, p[j][mb]);
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float sc = f16_bits_to_f32(uint16_t(sv[jp + j]));
                const float nz = -(BF16::BASE + float(zv[jp + j]));
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    if constexpr (__is_same(XT, BF16)) p[j][mb] += sum[mb] * nz;
                    acc[jp + j][mb] += sc * p[j][mb];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    WR w0, w1;
    issue(0, a0, w0);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](int i, const unsigned char *a, WR &cur, unsigned char *an, WR &next) {
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_below<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(i + 1, an, next);
        __builtin_amdgcn_sched_barrier(0);
        if (i < ng) compute(a, cur, i);
    };
    int i = 0;
    for (; i + 2 <= ngmax; i += 2) {
        step(i, a0, w0, a1, w1);
        step(i + 1, a1, w1, a0, w0);
    }
    if (i < ngmax) step(i, a0, w0, a1, w1);
    wait_vm_below<0>();

    if constexpr (WK == 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mb * 16 + 4 * q + r, row = n0 + 16 * j + n;
                    if (m < M && row < N && row >= n_lo)
                        store_y(y, int64_t(m) * ys + row, acc[j][mb][r], y_bf16, accumulate);
                }
    } else {
        // 16 rows at a time: the wave's sums to its slot ([row][64 weight
        // rows]), then each element's parts are added in part order
        auto slot = [&](int k) { return reinterpret_cast<float *>((k < 4 ? a0 : a1) + (k % 4) * S::SLOT); };
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            lds_barrier();
            float *mine = slot(wave);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[(4 * q + r) * 64 + 16 * j + n] = acc[j][mb][r];
            lds_barrier();
            for (int c = tid; c < 16 * S::ROWS; c += 512) {
                const int col = c % S::ROWS, tr = c / S::ROWS, m = mb * 16 + tr, row = item * S::ROWS + col;
                float v = 0.f;
#pragma unroll
                for (int k = 0; k < WK; ++k) v += slot(k * WN + col / 64)[tr * 64 + col % 64];
                if (m < M && row < N && row >= n_lo) store_y(y, int64_t(m) * ys + row, v, y_bf16, accumulate);
            }
        }
    }
}

// Two blocks per CU (128 VGPRs) where the buffers allow.
template <typename XT, int MB, int WN, bool HAS_Z>
__global__ __launch_bounds__(512, (2 * Wide<MB, WN>::SZ <= 80 * 1024 ? 4 : 2)) void q4_gemv_wide_kernel(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                              const uint16_t *x, int xs, int M, int K, int N,
                                                              void *__restrict__ y, int ys, int y_bf16, int accumulate,
                                                              int n_lo) {
    gemv_wide_block<XT, MB, WN, HAS_Z>(Wt, St, Zt, x, xs, M, K, N, y, ys, y_bf16, accumulate, n_lo);
}

}  // namespace qwq4
