// Dense GEMV on int8 weights with an fp32 scale per group of 16 or 32 along K.
//
// Reference role: gpu::gemv_rows_i8 (src/kernels/gemv.hip:75-136, declared
// src/kernels/gemv.hpp:15-23), the engine's int8 copy of its fp16 dense
// weights (QW_INT8_DENSE, src/engine/decode.hip:52-70,119-125), quantised by
// quantize_rows_i8 (src/engine/weight_convert.cpp:92-108):
//   y[m*ys + n] (+)= sum_g scale[n][g] * sum_{k in g} W8[n][k] * x[m*xs + off(n) + k]
// with off(n) = (n / rpg) * K when rows are grouped over activation slices.
//
// The weights are tiled once at load (qw_i8_tile, below; the role the q4
// path's qw_q4_tile plays for pack_int4_words) from the quantiser's row-major
// [N][K] int8 and [N][K/group] fp32 scales. Kernel shape as the 16-bit GEMV
// (w16_gemv.hip): a block holds one 16-row tile, its KS waves split K in
// 64-element steps, the activations (fp16) and the tile's scales are staged
// in LDS, the KS partial sums are added through LDS in k-part order. A wave
// instruction reads 1 KB of contiguous weights (row-major rows read 64 bytes
// per row per instruction measured 20% slower), 16 bytes per lane: lane
// (n, q) gets row n's weights arranged so that every MFMA operand covers
// exactly one scale group, and the MFMA's fp32 result is scaled once, as the
// reference scales each group's fp32 dot product (16x16x32 MFMAs for groups
// of 32, 16x16x16 for groups of 16).
// int8 -> fp16 is exact: the byte b ^ 0x80 = b + 128 becomes the low byte of
// fp16 1024 + (b + 128), minus 1152. Products with fp16 activations are exact
// in fp32, so a group's sum differs from the reference's only by summation
// order.
#include <algorithm>
#include <type_traits>

#include "q4_gemv_core.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

constexpr int I8_MAX_KS = 16;  // waves per block

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// four int8 weights (byte i = element i) -> four fp16 (two dwords), exactly
__device__ __forceinline__ uint2 i8x4_to_f16x4(uint32_t w) {
    const uint32_t u = w ^ 0x80808080u;
    const f16x2 off{(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);  // e0, e1
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);  // e2, e3
    return make_uint2(__builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, lo) - off),
                      __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, hi) - off));
}

__device__ __forceinline__ uint4 i8x8_to_f16x8(uint32_t a, uint32_t b) {
    const uint2 l = i8x4_to_f16x4(a), h = i8x4_to_f16x4(b);
    return make_uint4(l.x, l.y, h.x, h.y);
}

__device__ __forceinline__ f32x4 mfma16x16(const uint2 &a, const uint2 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0,
                                                 0);
}

// One 64-element step added to a sum: its groups' scaled products first
// (step_mul, then fused), so that the long sum has one term per step. No
// contraction but the fused ones written: both kernels below then give the same
// bits.
__device__ __forceinline__ float step_mul(float s, float r) {
#pragma clang fp contract(off)
    return s * r;
}
__device__ __forceinline__ float step_sum(float acc, float step) {
#pragma clang fp contract(off)
    return acc + step;
}
__device__ __forceinline__ float i8_add32(float acc, float s0, float r0, float s1, float r1) {
    return step_sum(acc, __builtin_fmaf(s0, r0, step_mul(s1, r1)));
}

// K split. Ungrouped rows of a K of whole 128-element groups: up to 8 parts of
// whole groups, the first ones a group longer where they do not divide, whatever
// the batch and the matrix's rows, in both kernels below: a token row's result
// does not depend on the batch it is in. Elsewhere (the staged kernel alone) KS
// parts of equally many 64-element steps.
__host__ __device__ inline bool i8_whole_groups(int K, int rpg) { return rpg == 0 && K % 128 == 0; }
struct I8Part {
    int s0, ns;  // 64-element steps s0 .. s0 + ns - 1
    __host__ __device__ I8Part(int K, int rpg, int KS, int kp) {
        if (i8_whole_groups(K, rpg)) {
            const int G = K / 128, per = G / KS, rem = G % KS;
            s0 = 2 * (kp * per + (kp < rem ? kp : rem));
            ns = 2 * (per + (kp < rem));
        } else {
            const int steps = K / 64, spw = (steps + KS - 1) / KS;
            s0 = kp * spw;
            ns = spw < steps - s0 ? spw : steps - s0;
        }
    }
};

// Direct global->LDS copy of `pieces` 16-byte pieces (whole waves of them are
// written: the LDS region is rounded up to 64 pieces).
__device__ __forceinline__ void stage_block_issue(const uint4 *src, int pieces, uint4 *dst) {
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, nw = blockDim.x / WAVE;
    for (int b = wave * WAVE; b < pieces; b += nw * WAVE)
        __builtin_amdgcn_global_load_lds(src + min(b + lane, pieces - 1), dst + b, 16, 0, 0);
}

// LDS pieces of a block's scales: 16 rows x K / GRP floats, whole waves
__host__ __device__ inline int i8_scale_pieces(int K, int group) { return (16 * (K / group) / 4 + WAVE - 1) / WAVE * WAVE; }

// GRP: scale group (16 or 32). MB row blocks of 16 tokens, MR rows of the
// last one formed. XPT: activation pieces per thread through registers (0:
// direct global->LDS). WS: 64-element steps a wave keeps in flight. NSL: row
// slices a 16-row tile can read (2 when rpg is not a multiple of 16).
template <int GRP, int MB, int MR, int XPT, int WS, int NSL>
__global__ __launch_bounds__(I8_MAX_KS *WAVE) void i8_gemv_kernel(const uint4 *Wt, const float *St, const uint16_t *x,
                                                                  int xs, int M, int K, int N, int rpg,
                                                                  void *__restrict__ y, int ys, int y_bf16,
                                                                  int accumulate) {
    static_assert(GRP == 16 || GRP == 32, "scale groups of 16 or 32");
    static_assert(NSL == 1 || XPT == 0, "two row slices are staged directly");
    extern __shared__ __align__(16) unsigned char smem[];
    const int KS = blockDim.x / WAVE;
    const int tid = threadIdx.x, kp = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, q = lane / 16,
              n = lane % 16;
    const I8Part part(K, rpg, KS, kp);
    const int steps = K / 64, s0 = part.s0, ns = part.ns;
    const int G = K / GRP, kc = x_row_stride(K);
    const int n0 = int(blockIdx.x) * 16;
    // activation slices of this tile: sl0 for its first row, sl1 for its last
    const int sl0 = rpg > 0 ? n0 / rpg : 0, sl1 = rpg > 0 ? min(n0 + 15, N - 1) / rpg : 0;
    uint4 *xl = reinterpret_cast<uint4 *>(smem);
    uint4 *sl = xl + x_pieces(NSL * M, K);
    float *red = reinterpret_cast<float *>(sl + i8_scale_pieces(K, GRP));
    const uint16_t *xb = x + int64_t(sl0) * K;
    XRegs xv;
    if constexpr (XPT > 0) stage_regs_issue<XPT>(xb, xs, M, K, xv);
    else if constexpr (NSL == 1) stage_x_issue(xb, xs, M, K, xl);
    else
        stage_rows_issue([&](int i) { return x + int64_t(i % M) * xs + int64_t(i < M ? sl0 : sl1) * K; }, NSL * M, K,
                         xl);
    // the tile's scales, [K / 64][16 rows][64 / GRP] floats, contiguous
    stage_block_issue(reinterpret_cast<const uint4 *>(St + int64_t(blockIdx.x) * 16 * G), 4 * G, sl);
    __builtin_amdgcn_sched_barrier(0);  // activations and scales go out before the weight loads
    // lane l of step s: 16 bytes of row n (see the tiled format above)
    const uint4 *wt = Wt + int64_t(blockIdx.x) * steps * WAVE + lane;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    uint4 w[WS];
    auto fetch = [&](int p) {  // steps p .. p + WS - 1 of the wave's range (clamped, no branches)
#pragma unroll
        for (int t = 0; t < WS; ++t) {
            const int s = min(s0 + min(p + t, max(ns - 1, 0)), steps - 1);
            const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wt + s * WAVE));
            w[t] = make_uint4(v[0], v[1], v[2], v[3]);
        }
    };
    f32x4 acc[NSL][MB];
#pragma unroll
    for (int j = 0; j < NSL; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (XPT > 0) stage_regs_commit<XPT>(xv, M, K, xl);
    wait_vm_below<WS>();  // this wave's activation and scale loads (its oldest)
    lds_barrier();
    // the second slice is computed only by tiles that straddle two
    const bool two = NSL == 2 && sl1 != sl0;
    const uint4 *xr[NSL][MB];
#pragma unroll
    for (int j = 0; j < NSL; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xr[j][mb] = xl + (j * M + min(mb * 16 + n, M - 1)) * kc;
    constexpr int SPS = 64 / GRP;  // scales per step
    typedef float sv_t __attribute__((ext_vector_type(SPS)));
    const sv_t *scl = reinterpret_cast<const sv_t *>(sl) + n;
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < ns; p += WS) {
        if (p > 0) fetch(p);
#pragma unroll
        for (int t = 0; t < WS; ++t)
            if (p + t < ns) {
                const int s = s0 + p + t;
                const sv_t sc = scl[s * 16];
                if constexpr (GRP == 32) {
                    // K of the lane's 8 weights: 8 q (first group), 32 + 8 q (second)
                    const uint4 wa = i8x8_to_f16x8(w[t].x, w[t].y), wb = i8x8_to_f16x8(w[t].z, w[t].w);
#pragma unroll
                    for (int j = 0; j < NSL; ++j)
                        if (j == 0 || two) {
#pragma unroll
                            for (int mb = 0; mb < MB; ++mb) {
                                const f32x4 ra = mfma16<F16>(xr[j][mb][s * 8 + q], wa, zero);
                                const f32x4 rb = mfma16<F16>(xr[j][mb][s * 8 + 4 + q], wb, zero);
                                const int rows = mb == MB - 1 ? MR : 4;
#pragma unroll
                                for (int r = 0; r < 4; ++r)
                                    if (r < rows) acc[j][mb][r] = i8_add32(acc[j][mb][r], sc[0], ra[r], sc[1], rb[r]);
                            }
                        }
                } else {
                    // dword g: K 16 g + 4 q .. + 3 of the step, group 4 s + g
                    const uint2 wg[4] = {i8x4_to_f16x4(w[t].x), i8x4_to_f16x4(w[t].y), i8x4_to_f16x4(w[t].z),
                                         i8x4_to_f16x4(w[t].w)};
#pragma unroll
                    for (int j = 0; j < NSL; ++j)
                        if (j == 0 || two) {
#pragma unroll
                            for (int mb = 0; mb < MB; ++mb) {
                                const uint2 *xh = reinterpret_cast<const uint2 *>(xr[j][mb]);
                                const int rows = mb == MB - 1 ? MR : 4;
                                f32x4 p;
#pragma unroll
                                for (int g = 0; g < 4; ++g) {
                                    const f32x4 rg = mfma16x16(xh[s * 16 + 4 * g + q], wg[g], zero);
#pragma unroll
                                    for (int r = 0; r < 4; ++r)
                                        if (r < rows) p[r] = g == 0 ? step_mul(sc[g], rg[r]) : __builtin_fmaf(sc[g], rg[r], p[r]);
                                }
#pragma unroll
                                for (int r = 0; r < 4; ++r)
                                    if (r < rows) acc[j][mb][r] = step_sum(acc[j][mb][r], p[r]);
                            }
                        }
                }
            }
    }
    // each lane keeps the slice of its own row
    if constexpr (NSL == 2) {
        if (min(n0 + n, N - 1) / rpg != sl0) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) acc[0][mb] = acc[1][mb];
        }
    }
    ksplit_sum<MB, MR>(acc[0], red, KS, kp, kp, lane);
    if (kp == 0) store_rows<MB, MR>(acc[0], y, ys, y_bf16, accumulate, M, N, blockIdx.x, lane);
}

// ------------------------------------------------------------ rows streamed
// The kernel above stages every activation row of the whole K per 16 weight
// rows: 8 KB a row of 4096 against 64 KB of weights, so the copy outweighs the
// weights from 8 rows on, nothing is requested while it is waited for, and past
// 16 rows of 4096 (9 of 6144) the batch no longer fits LDS and runs as several
// launches. Here a block takes 16 NS weight rows and moves the rows' K in
// groups of 128 through a double buffer: its 8 waves split K, each widens a
// weight once for 16 MB rows, and the next group's rows (direct global -> LDS
// loads), weights and scales (registers) are requested before a group is
// computed. The parts are added through LDS in part order. Products, the
// fp32 sum per scale group and its scaling are those above. K a multiple of
// 128, no row slices. Bound by the weight stream, which is read non-temporal
// and in block order (cached and in a range per XCD: 7% slower at 4096->12288).
// Before -> after on 1.2 GB of weights, groups of 32, us: 6144->4096 at 1 / 4 /
// 8 / 16 rows 8.8 / 9.7 / 10.2 / 19.7 -> 7.4 / 7.3 / 7.6 / 8.9, 4096->12288 12.2 /
// 13.2 / 15.1 / 21.9 -> 12.2 / 12.2 / 12.4 / 13.7 (4.6 TB/s at 4 rows).
template <int MB, int NS>
struct I8Wide {
    static constexpr int WK = 8, ROWS = 16 * NS, BM = 16 * MB;
    static constexpr int A = WK * BM * 256;      // bytes of a group's rows
    static constexpr int SLOT = 16 * ROWS * 4;   // closing sums: 16 rows at a time per wave
    static_assert(A >= 4 * SLOT, "four slots in each buffer");
};

// 8-byte half h (0..31) of row r of a part's tile [16 MB][128]
__device__ __forceinline__ int i8w_at(int r, int h) { return r * 256 + (((h >> 1) ^ (r & 15)) << 4) + (h & 1) * 8; }

template <int GRP, int MB, int NS>
__device__ __forceinline__ void i8_wide_block(const uint4 *Wt, const float *St, const uint16_t *__restrict__ x, int xs,
                                              int M, int K, int N, void *__restrict__ y, int ys, int y_bf16,
                                              int accumulate) {
    using S = I8Wide<MB, NS>;
    constexpr int WK = S::WK, SPS = 64 / GRP;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) unsigned char a0[S::A], a1[S::A];
    typedef float sv_t __attribute__((ext_vector_type(SPS)));
    const int tid = threadIdx.x, wk = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, n = lane % 16,
              q = lane / 16;
    const int item = int(blockIdx.x);
    const int nsub = (N + 15) / 16, steps = K / 64;
    const int G = K / 128, per = G / WK, rem = G % WK;  // (I8Part's split; parts past the last group are empty)
    const int g0 = wk * per + min(wk, rem), ng = per + (wk < rem), ngmax = per + (rem > 0);
    const uint4 *w[NS];
    const sv_t *sc[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int64_t sub = min(item * NS + j, nsub - 1);
        w[j] = Wt + sub * steps * WAVE;
        sc[j] = reinterpret_cast<const sv_t *>(St) + sub * steps * 16;
    }
    int xo[4 * MB];  // instruction j moves rows 4 j .. 4 j + 3 of the part
#pragma unroll
    for (int j = 0; j < 4 * MB; ++j) {
        const int r = j * 4 + q;
        xo[j] = min(r, M - 1) * xs + ((n ^ (r & 15)) * 8);
    }
    struct WR {
        uint4 w[NS][2];
        sv_t s[NS][2];
    };
    auto issue = [&](int i, unsigned char *dst, WR &r) {
        const int g = min(g0 + min(i, max(ng, 1) - 1), G - 1);  // past the end: a valid (unused) one
#pragma unroll
        for (int j = 0; j < 4 * MB; ++j)
            if (4 * j < M)  // (uniform)
                __builtin_amdgcn_global_load_lds(x + g * 128 + xo[j], dst + wk * (S::BM * 256) + j * 1024, 16, 0, 0);
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w[j] + (2 * g + t) * WAVE + lane));
                r.w[j][t] = make_uint4(v[0], v[1], v[2], v[3]);
                r.s[j][t] = sc[j][(2 * g + t) * 16 + n];
            }
    };
    int ar[MB];  // rows past M read the last one
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) ar[mb] = min(mb * 16 + n, M - 1);
    f32x4 acc[NS][MB];
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = zero;
    auto compute = [&](const unsigned char *ab, const WR &r) {
        const unsigned char *a = ab + wk * (S::BM * 256);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (GRP == 32) {
                uint4 fa[MB], fb[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    fa[mb] = *reinterpret_cast<const uint4 *>(a + i8w_at(ar[mb], 2 * (8 * t + q)));
                    fb[mb] = *reinterpret_cast<const uint4 *>(a + i8w_at(ar[mb], 2 * (8 * t + 4 + q)));
                }
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    const uint4 &v = r.w[j][t];
                    const uint4 wa = i8x8_to_f16x8(v.x, v.y), wb = i8x8_to_f16x8(v.z, v.w);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        const f32x4 ra = mfma16<F16>(fa[mb], wa, zero), rb = mfma16<F16>(fb[mb], wb, zero);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[j][mb][e] = i8_add32(acc[j][mb][e], r.s[j][t][0], ra[e], r.s[j][t][1], rb[e]);
                    }
                }
            } else {
                uint2 f[MB][4];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        f[mb][g] = *reinterpret_cast<const uint2 *>(a + i8w_at(ar[mb], 16 * t + 4 * g + q));
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    const uint32_t v[4] = {r.w[j][t].x, r.w[j][t].y, r.w[j][t].z, r.w[j][t].w};
                    const sv_t sj = r.s[j][t];
                    f32x4 p[MB];
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const uint2 wg = i8x4_to_f16x4(v[g]);
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) {
                            const f32x4 rg = mfma16x16(f[mb][g], wg, zero);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                p[mb][e] = g == 0 ? step_mul(sj[g], rg[e]) : __builtin_fmaf(sj[g], rg[e], p[mb][e]);
                        }
                    }
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[j][mb][e] = step_sum(acc[j][mb][e], p[mb][e]);
                }
            }
        }
    };
    WR w0, w1;
    issue(0, a0, w0);
    // a part's rows are written and read by one wave: the wait for its own loads
    // suffices for them, and the reads of the buffer being refilled are complete
    auto step = [&](int i, const unsigned char *a, WR &cur, unsigned char *an, WR &next) {
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_below<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(i + 1, an, next);
        __builtin_amdgcn_sched_barrier(0);
        if (i < ng) compute(a, cur);
    };
    int i = 0;
    for (; i + 2 <= ngmax; i += 2) {
        step(i, a0, w0, a1, w1);
        step(i + 1, a1, w1, a0, w0);
    }
    if (i < ngmax) step(i, a0, w0, a1, w1);
    wait_vm_below<0>();

    // 16 rows at a time: the wave's sums to its slot ([row][weight rows]), then
    // each element's parts are added in part order
    auto slot = [&](int k) { return reinterpret_cast<float *>((k < 4 ? a0 : a1) + (k % 4) * S::SLOT); };
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        lds_barrier();
        float *mine = slot(wk);
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) mine[(4 * q + r) * S::ROWS + 16 * j + n] = acc[j][mb][r];
        lds_barrier();
        for (int c = tid; c < 16 * S::ROWS; c += 512) {
            const int col = c % S::ROWS, tr = c / S::ROWS, m = mb * 16 + tr, row = item * S::ROWS + col;
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < WK; ++k) v += slot(k)[tr * S::ROWS + col];
            if (m < M && row < N) store_y(y, int64_t(m) * ys + row, v, y_bf16, accumulate);
        }
    }
}

template <int GRP, int MB, int NS>
__global__ __launch_bounds__(512, (MB == 1 && NS <= 2 ? 4 : 2)) void i8_wide_kernel(
    const uint4 *Wt, const float *St, const uint16_t *x, int xs, int M, int K, int N, void *__restrict__ y, int ys,
    int y_bf16, int accumulate) {
    i8_wide_block<GRP, MB, NS>(Wt, St, x, xs, M, K, N, y, ys, y_bf16, accumulate);
}

// ------------------------------------------------------------ tiled format
// Wt uint4 [ceil(N/16)][K/64][64]: entry (tile, s, lane l) holds 16 int8
// weights of row 16 tile + l % 16, q = l / 16, of the 64-element step s:
//   group 32: bytes 0-7 = K 64 s + 8 q .. + 7, bytes 8-15 = K 64 s + 32 + 8 q .. + 7
//   group 16: dword g = K 64 s + 16 g + 4 q .. + 3 (g = 0..3)
// so each 16x16x32 (16x16x16) MFMA operand covers one scale group. Rows past
// N are zero. St fp32 [ceil(N/16)][K/64][16][64/group]: the scales of the
// step's groups, per row.
__global__ void i8_tile_kernel(const int8_t *__restrict__ W8, const float *__restrict__ S, int N, int K, int group,
                               uint4 *__restrict__ Wt, float *__restrict__ St) {
    const int64_t steps = K / 64, total = int64_t((N + 15) / 16) * steps * WAVE;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
        const int l = int(i % WAVE), q = l / 16, nn = l % 16;
        const int64_t s = (i / WAVE) % steps, tile = i / (WAVE * steps), row = tile * 16 + nn;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (row < N) {
            const int8_t *r = W8 + row * K + s * 64;
            if (group == 32) {
                const uint2 a = *reinterpret_cast<const uint2 *>(r + 8 * q);
                const uint2 b = *reinterpret_cast<const uint2 *>(r + 32 + 8 * q);
                v = make_uint4(a.x, a.y, b.x, b.y);
            } else {
                const uint32_t *d = reinterpret_cast<const uint32_t *>(r + 4 * q);
                v = make_uint4(d[0], d[4], d[8], d[12]);
            }
        }
        Wt[i] = v;
        // scales: lane l < 16 writes row nn's scales of this step
        if (q == 0) {
            const int sps = 64 / group, G = K / group;
            for (int j = 0; j < sps; ++j)
                St[((tile * steps + s) * 16 + nn) * sps + j] = row < N ? S[row * G + s * sps + j] : 0.f;
        }
    }
}

void launch_i8_tile(const int8_t *W8, const float *S, int N, int K, int group, uint4 *Wt, float *St, hipStream_t s) {
    const int64_t total = int64_t((N + 15) / 16) * (K / 64) * WAVE;
    const unsigned blocks = unsigned(std::min<int64_t>((total + 255) / 256, 65536));
    i8_tile_kernel<<<blocks, 256, 0, s>>>(W8, S, N, K, group, Wt, St);
}

// Waves of the staged kernel: up to 8; 16 when the row tiles would not give
// every CU two blocks (fewer blocks leave the weight stream short of loads in
// flight). i8_ks_max: before the whole-group split (I8Part), which takes at most
// 8 parts; the LDS limit is sized by it.
static int i8_ks_max(int K, int N) {
    const int ks = (N + 15) / 16 < 512 ? 16 : 8;
    return K / 64 < ks ? K / 64 : ks;
}
static int i8_ks(int K, int N, int rpg) {
    if (i8_whole_groups(K, rpg)) return K / 128 < 8 ? K / 128 : 8;
    return i8_ks_max(K, N);
}

static int i8_nsl(int rpg) { return rpg > 0 && rpg % 16 != 0 ? 2 : 1; }

size_t i8_lds_bytes(int M, int K, int N, int group, int rpg) {
    const int KS = i8_ks_max(K, N), MB = M > 16 ? 2 : 1;
    return size_t(x_pieces(i8_nsl(rpg) * M, K) + i8_scale_pieces(K, group)) * 16 +
           size_t(red_slots(KS, KS)) * MB * WAVE * 16;  // one set of k-split slots (no persistent blocks)
}

template <int GRP, int MB, int MR, int NSL>
static void launch_i8_t(const I8Args &a, hipStream_t s) {
    const int KS = i8_ks(a.K, a.N, a.rpg), threads = KS * WAVE;
    const size_t lds = i8_lds_bytes(a.M, a.K, a.N, a.group, a.rpg);
    const int xpt = NSL == 1 ? (a.M * (a.K / 8) + threads - 1) / threads : 0;
    const unsigned blocks = unsigned((a.N + 15) / 16);
    auto go = [&](auto kern) {
        if (lds > 64 * 1024) (void)persistent_shape(reinterpret_cast<const void *>(kern), threads, lds);
        kern<<<blocks, threads, lds, s>>>(a.W, a.S, a.x, a.xs, a.M, a.K, a.N, a.rpg, a.y, a.ys, a.y_bf16,
                                          a.accumulate);
    };
    const int spw = I8Part(a.K, a.rpg, KS, 0).ns;  // (the first part is the longest)
    auto pick = [&](auto ws) {
        constexpr int W = decltype(ws)::value;
        if constexpr (NSL == 2) go(i8_gemv_kernel<GRP, MB, MR, 0, W, 2>);
        else {
            if (xpt <= 1) go(i8_gemv_kernel<GRP, MB, MR, 1, W, 1>);
            else if (xpt <= 2) go(i8_gemv_kernel<GRP, MB, MR, 2, W, 1>);
            else if (xpt <= 4) go(i8_gemv_kernel<GRP, MB, MR, 4, W, 1>);
            else go(i8_gemv_kernel<GRP, MB, MR, 0, W, 1>);
        }
    };
    if (spw <= 4) pick(std::integral_constant<int, 4>());
    else pick(std::integral_constant<int, 8>());
}

template <int GRP, int NSL>
static void launch_i8_m(const I8Args &a, hipStream_t s) {
    if (a.M > 16) launch_i8_t<GRP, 2, 4, NSL>(a, s);
    else if (a.M == 1) launch_i8_t<GRP, 1, 1, NSL>(a, s);
    else if (a.M == 2) launch_i8_t<GRP, 1, 2, NSL>(a, s);
    else launch_i8_t<GRP, 1, 4, NSL>(a, s);
}

static void launch_i8_fit(const I8Args &a, hipStream_t s) {
    const bool two = i8_nsl(a.rpg) == 2;
    if (a.group == 32) two ? launch_i8_m<32, 2>(a, s) : launch_i8_m<32, 1>(a, s);
    else two ? launch_i8_m<16, 2>(a, s) : launch_i8_m<16, 1>(a, s);
}

bool i8_fits(int M, int K, int N, int group, int rpg) { return i8_lds_bytes(M, K, N, group, rpg) <= 160 * 1024; }

template <int GRP, int MB, int NS>
static void launch_i8_wide_t(const I8Args &a, hipStream_t s) {
    constexpr int R = I8Wide<MB, NS>::ROWS;
    i8_wide_kernel<GRP, MB, NS><<<unsigned((a.N + R - 1) / R), 512, 0, s>>>(a.W, a.S, a.x, a.xs, a.M, a.K, a.N, a.y,
                                                                            a.ys, a.y_bf16, a.accumulate);
}

// Row tiles per block: the fewest that make one round of a block per CU
// (4096->12288, 768 tiles, at 16 rows 16.1 / 15.3 / 13.0 / 14.3 us with 1 / 2 / 3
// / 4; 3072->6144, 384 tiles, 7.6 / 6.6 / 8.0 / 9.1; 6144->4096, 256 tiles, 8.0 /
// 9.6 / 12.1 / 14.4). Beyond three rounds of single tiles 2 up to 16 rows, where
// two blocks share a CU, and 4 above (2048->32000 18.6 against 18.7-23.5, and
// 24.1 against 28.5-40.7).
template <int GRP>
static void launch_i8_wide(const I8Args &a, hipStream_t s) {
    const int ns = ((a.N + 15) / 16 + 255) / 256;
    if (a.M <= 16) {
        if (ns == 1) launch_i8_wide_t<GRP, 1, 1>(a, s);
        else if (ns == 3) launch_i8_wide_t<GRP, 1, 3>(a, s);
        else launch_i8_wide_t<GRP, 1, 2>(a, s);
    } else {
        if (ns == 1) launch_i8_wide_t<GRP, 2, 1>(a, s);
        else if (ns == 2) launch_i8_wide_t<GRP, 2, 2>(a, s);
        else if (ns == 3) launch_i8_wide_t<GRP, 2, 3>(a, s);
        else launch_i8_wide_t<GRP, 2, 4>(a, s);
    }
}

// The streamed kernel takes every batch where its blocks are one round of the
// CUs, and batches above 8 beyond. Up to 8 rows of more than 768 tiles the
// staged kernel's small blocks keep more of the weight stream in flight
// (2048->32000 at 1 / 8 / 16 rows 14.0 / 16.9 / 22.9 us against 15.8 / 16.8 /
// 18.6), as with groups of 16 (a quarter more bytes and twice the MFMAs) for one
// row of more than 640 tiles (4096->12288 at 1 / 2 / 4 rows 13.1 / 13.6 / 15.2
// against 14.0 / 13.5 / 13.7; 2560->10000, 625 tiles, 9.1 / 9.2 / 10.1 against
// 8.1 / 8.1 / 8.3).
// xs: 32-bit row offsets.
static bool i8_wide(const I8Args &a) {
    const int nt = (a.N + 15) / 16;
    if (a.rpg != 0 || a.K % 128 != 0 || a.xs > 1 << 25) return false;
    if (a.M > 8) return true;
    return nt <= 768 && !(a.group == 16 && a.M == 1 && nt > 640);
}

// Batches whose activations exceed LDS run as several launches of fewer rows
// (the caller has checked that one row fits).
void launch_i8_gemv(const I8Args &a, hipStream_t s) {
    if (i8_wide(a)) {
        a.group == 32 ? launch_i8_wide<32>(a, s) : launch_i8_wide<16>(a, s);
        return;
    }
    if (i8_fits(a.M, a.K, a.N, a.group, a.rpg)) {
        launch_i8_fit(a, s);
        return;
    }
    int mc = 16;
    while (mc > 1 && !i8_fits(mc, a.K, a.N, a.group, a.rpg)) --mc;
    const size_t ysz = a.y_bf16 ? 2 : 4;
    for (int m0 = 0; m0 < a.M; m0 += mc) {
        I8Args b = a;
        b.M = a.M - m0 < mc ? a.M - m0 : mc;
        b.x = a.x + int64_t(m0) * a.xs;
        b.y = static_cast<char *>(a.y) + int64_t(m0) * a.ys * ysz;
        launch_i8_fit(b, s);
    }
}

}  // namespace qwq4
