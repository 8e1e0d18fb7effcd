// q4-dequant GEMM tiles for chunks whose 128- to 256-token tiles are too few to
// fill the chip (short prompts, the rest of a prompt, narrow projections). Every
// tile runs over the whole K with gemm_tile's operands, MFMA and K order, so a
// token row's result is the same bits in a chunk of any length. (K split over the
// waves of a block and added at the end, which these replace, gave other bits for
// a few microseconds: 6144->4096 at 80 / 601 tokens 16 / 42 us against 22 / 51,
// 4096->12288 25 / 61 against 24 / 74; the 128 x 256 tiles 86 / 89 and 61 / 75.)
//
// Roles form (up to a few hundred tokens): NP waves move A (direct global -> LDS
// loads) and dequantise the block's weight rows into LDS, a group (128 K) ahead;
// the others hold 32 NI x 32 NJ results each and only read fragments and run
// MFMAs. Bound by the latency of a group's turn (8 MFMAs in a chain, fragment
// reads, barrier): about 650 cycles for 32 x 32 (6144->4096 at 16 tokens 16 us),
// which neither twice the loading waves nor two fragment sets shorten. With loads,
// dequantisation and MFMAs in the same waves it was the sum of them (22 us).
//
// Register form (beyond that): a wave holds 32 weight rows and every token row of
// the tile and dequantises its weights in registers (each lane one tiled q4 entry
// per 64-K stage); only A goes through LDS, shared by the 4 waves. Bound by LDS
// reads (a fragment serves one MFMA) and the matrix core.
//
// Loads are requested 3 stages or P groups ahead, A and weights together: vector
// loads complete in order, so a shallower A would also cut the weights' time in
// flight.
#pragma once

#include "q4_gemm_core.cuh"

namespace qwq4 {

// Register form: BM tokens x 128 weight rows in 4 waves of 32 rows.
template <int BM>
struct RegTile {
    static_assert(BM % 32 == 0 && BM <= 128, "");
    static constexpr int WN = 4, THREADS = WN * WAVE, BN = 32 * WN, NI = BM / 32, NST = 4;  // NST: K stages in LDS and registers
    static constexpr int NA = BM / 8 / WN;  // direct A loads per wave and stage
    static constexpr int SZ = BM * 128;     // bytes of one stage's A
    static constexpr int SLOTS = SZ / 4096; // epilogue slots (32 x 32 fp32) per stage buffer
};

// one output element as stored (yt: 0 fp32, 1 bf16, 2 fp16 saturated)
__device__ __forceinline__ uint32_t cvt_y16(float v, int yt) {
    return yt == 1 ? f32_to_bf16_rne(v) : __builtin_bit_cast(uint16_t, f32_to_f16_satfinite(v));
}

// Weight-row-major tile order, a contiguous range of tiles per XCD: the token
// tiles over the same weights run together and share an L2.
__device__ __forceinline__ int small_item() {
    const int nb = int(gridDim.x), xq = nb / 8, xr = nb % 8, xcd = int(blockIdx.x) % 8;
    return xcd * xq + min(xcd, xr) + int(blockIdx.x) / 8;
}

// A wave's results, 32 x 32 at a time through its 4 KB slot: 8 weight rows per lane and store.
template <int NI, int NJ>
__device__ __forceinline__ void store_slots(const f32x16 (&acc)[NI][NJ], unsigned char *slot, int lane, int t0, int n0,
                                            int T, int N, void *Y, int ldy, int yt) {
    const int l32 = lane % 32, lh = lane / 32;
    const int ye = yt == 0 ? 4 : 2;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int r = 0; r < 16; ++r)
                *reinterpret_cast<float *>(slot + ((r / 4) * 8 + lh * 4 + r % 4) * 128 + l32 * 4) = acc[i][j][r];
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int tr = h * 16 + lane / 4, col = lane % 4 * 8;
                const unsigned char *q = slot + tr * 128 + col * 4;
                const f32x4 v0 = *reinterpret_cast<const f32x4 *>(q), v1 = *reinterpret_cast<const f32x4 *>(q + 16);
                const int t = t0 + i * 32 + tr, n = n0 + j * 32 + col;
                if (t < T && n < N) {
                    unsigned char *o = static_cast<unsigned char *>(Y) + (int64_t(t) * ldy + n) * ye;
                    if (yt == 0) {
                        *reinterpret_cast<f32x4 *>(o) = v0;
                        *reinterpret_cast<f32x4 *>(o + 16) = v1;
                    } else {
                        uint32_t d[4];
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            d[e] = cvt_y16(v0[2 * e], yt) | (cvt_y16(v0[2 * e + 1], yt) << 16);
                            d[2 + e] = cvt_y16(v1[2 * e], yt) | (cvt_y16(v1[2 * e + 1], yt) << 16);
                        }
                        *reinterpret_cast<uint4 *>(o) = make_uint4(d[0], d[1], d[2], d[3]);
                    }
                }
            }
        }
}

template <int BM, bool HAS_Z>
__device__ __forceinline__ void gemm_reg_block(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                               const uint16_t *__restrict__ Xh, int lda, int T, void *__restrict__ Y,
                                               int ldy, int yt, int N, int K, int nby) {
    using S = RegTile<BM>;
    constexpr int NI = S::NI, NA = S::NA, SZ = S::SZ, WN = S::WN, NST = S::NST;
    // (distinct objects: see lds_a0)
    __shared__ __align__(16) unsigned char b0[SZ], b1[SZ], b2[SZ], b3[SZ];
    auto buf = [&](int i) -> unsigned char * { return i == 0 ? b0 : i == 1 ? b1 : i == 2 ? b2 : b3; };
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / WAVE), lane = int(threadIdx.x) % WAVE;
    const int l32 = lane % 32, lh = lane / 32, nk = K / GB_K, G = K / QGROUP;
    const int item = small_item(), n0 = item / nby * S::BN + wave * 32, t0 = item % nby * BM;

    const uint16_t *xb = Xh + int64_t(t0) * lda;
    int aoff[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int r = (j * WN + wave) * 8 + lane / 8;
        aoff[j] = min(r, T - 1 - t0) * lda + ((lane % 8) ^ swz_x(r)) * 8;
    }
    const BRow b(Wt, St, Zt, min(n0 + l32, N - 1), G);
    struct SZr {  // a group's scale and zero word, as loaded
        uint16_t s;
        uint32_t z;
    };
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    u32x4 wr[NST];
    SZr sz[NST / 2];
    constexpr int NLD = NA + 1, NSZ = 1 + HAS_Z;  // vector loads per stage, and per group beside them
    auto issue = [&](int s, int u, unsigned char *dst) {
        const int g = min(s / 2, G - 1), h = u & 1;  // past the end: a valid (unused) one
        const uint16_t *xs = xb + g * QGROUP + h * GB_K;
#pragma unroll
        for (int j = 0; j < NA; ++j)
            __builtin_amdgcn_global_load_lds(xs + aoff[j], dst + (j * WN + wave) * 1024, 16, 0, 0);
        wr[u] = *reinterpret_cast<const u32x4 *>(b.w + g * 64 + (h * 2 + lh) * 16);
        if (h == 0) {
            sz[u / 2].s = b.s[(g >> 2) * 64 + (g & 3)];
            if constexpr (HAS_Z) sz[u / 2].z = b.z[(g >> 2) * 8];
        }
    };
    f32x16 acc[NI][1];
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[i][0] = f32x16{};
    // the row's packed fp16 scale and zero point of the group at hand
    uint32_t sv = 0, zv = 0;
    auto open_group = [&](const SZr &q, int g) {
        zv = HAS_Z ? ((q.z >> (b.zs + 4 * (g & 3))) & 0xfu) * 0x10001u : 0x80008u;
        sv = uint32_t(q.s) * 0x10001u;
    };
    auto compute = [&](const unsigned char *a, const u32x4 &r) {
        // step kk takes the stage's chunks 2 kk (lanes 0-31) and 2 kk + 1, as
        // gemm_tile; a lane holds chunks 4 lh .. 4 lh + 3
        const auto p = __builtin_amdgcn_permlane32_swap(r[0], r[1], false, false);
        const auto q = __builtin_amdgcn_permlane32_swap(r[2], r[3], false, false);
        const uint32_t w[4] = {p[0], q[0], p[1], q[1]};
        const h2 zl = __builtin_bit_cast(h2, zv | 0xe400e400u);         // -(1024 + z)
        const h2 zh = __builtin_bit_cast(h2, (zv << 4) + 0xd400d400u);  // -(64 + z)
        const h2 s2 = __builtin_bit_cast(h2, sv);
        uint4 af[2][NI], f[2];
        auto rd = [&](int kk, uint4 (&d)[NI]) {
#pragma unroll
            for (int i = 0; i < NI; ++i) d[i] = *reinterpret_cast<const uint4 *>(a + swz(i * 32 + l32, 2 * kk + lh));
        };
        rd(0, af[0]);
        f[0] = dequant8_light(w[0], zl, zh, s2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < GB_K / 16; ++kk) {
            const int c = kk & 1;
            const bool more = kk + 1 < GB_K / 16;
            if (more) {
                rd(kk + 1, af[c ^ 1]);
                f[c ^ 1] = dequant8_light(w[kk + 1], zl, zh, s2);
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) acc[i][0] = mfma32<F16>(af[c][i], f[c], acc[i][0]);
            // the next step's fragment reads, then its dequant spread over
            // this step's MFMAs: in order of issue a wave would wait for the
            // matrix core with its VALU work still to come
            if (more) {
                __builtin_amdgcn_sched_group_barrier(0x100, NI, 0);
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (14 + NI - 1) / NI, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

#pragma unroll
    for (int s = 0; s < NST - 1; ++s) {
        issue(s, s, buf(s));
        __builtin_amdgcn_sched_barrier(0);
    }
    auto stage = [&](int s, int u) {  // u = s % NST, a constant
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_below<(NST - 2) * NLD + (NST / 2 - 1) * NSZ>();  // stage s arrived (this wave's part of it)
        // ... every wave's, and stage s - 1 is consumed (its fragment reads
        // were waited for by its MFMAs). A fence here would drain the direct
        // loads in flight, so only the compiler is held back.
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(s + NST - 1, (u + NST - 1) % NST, buf((u + NST - 1) % NST));
        __builtin_amdgcn_sched_barrier(0);
        // taken here, not at its load, and as one: single words are copied right
        // after the load, which drains every load in flight
        asm volatile("" : "+v"(wr[u]));
        if (u % 2 == 0) {
            asm volatile("" : "+v"(sz[u / 2].s));
            if constexpr (HAS_Z) asm volatile("" : "+v"(sz[u / 2].z));
            open_group(sz[u / 2], s / 2);
        }
        compute(buf(u), wr[u]);
    };
    // Whole rounds of the stage buffers, then the rest: with an exit inside
    // the round the compiler sees paths on which a stage does not follow its
    // predecessor's requests, and drains every load in flight before it
    // reuses a stage's registers.
    int s = 0;
    for (; s + NST <= nk; s += NST) {
#pragma unroll
        for (int u = 0; u < NST; ++u) stage(s + u, u);
    }
#pragma unroll
    for (int u = 0; u < NST - 1; ++u)
        if (s + u < nk) stage(s + u, u);
    wait_vm_below<0>();
    lds_barrier();  // every wave is done with the buffers, and its loads into them have landed
    store_slots<NI, 1>(acc, buf(wave / S::SLOTS) + wave % S::SLOTS * 4096, lane, t0, n0, T, N, Y, ldy, yt);
}

// (waves per SIMD that the accumulators leave registers for)
template <int BM, bool HAS_Z>
__global__ __launch_bounds__(RegTile<BM>::THREADS, (BM <= 64 ? 4 : BM <= 96 ? 3 : 2)) void q4_gemm_reg_kernel(
    const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt, const uint16_t *__restrict__ Xh, int lda, int T,
    void *__restrict__ Y, int ldy, int yt, int N, int K, int nby) {
    gemm_reg_block<BM, HAS_Z>(Wt, St, Zt, Xh, lda, T, Y, ldy, yt, N, K, nby);
}

// Roles form: NP waves load and dequantise, WM x WN waves hold the results. P:
// groups that the loads are ahead.
template <int BM, int BN, int NI, int NJ, int NP, int P>
struct RoleTile {
    static constexpr int U = P + 1;  // A buffers and register sets
    static constexpr int WM = BM / (32 * NI), WN = BN / (32 * NJ), NC = WM * WN, THREADS = (NC + NP) * WAVE;
    static constexpr int NA = BM / 4 / NP;   // direct A loads per producer wave and group
    static constexpr int WPT = BN / 4 / NP;  // weight words per producer thread and group
    static constexpr int SA = BM * 256, SB = BN * 256, SLOTS = SA / 4096;
    static_assert(BM % (32 * NI) == 0 && BN % (32 * NJ) == 0 && BM / 4 % NP == 0 && BN <= NP * WAVE, "");
    static_assert((WPT == 1 || WPT == 2 || WPT == 4 || WPT == 8) && P >= 1 && P <= 3 && SLOTS * U >= NC, "");
    static_assert(U * SA + 2 * SB <= 160 * 1024, "");
};

template <int BM, int BN, int NI, int NJ, int NP, int P, bool HAS_Z>
__device__ __forceinline__ void gemm_roles_block(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                 const uint16_t *__restrict__ Xh, int lda, int T,
                                                 void *__restrict__ Y, int ldy, int yt, int N, int K, int nby) {
    using S = RoleTile<BM, BN, NI, NJ, NP, P>;
    constexpr int U = S::U, NA = S::NA, WPT = S::WPT, SA = S::SA, SB = S::SB;
    __shared__ __align__(16) unsigned char a0[SA], a1[SA], a2[U > 2 ? SA : 16], a3[U > 3 ? SA : 16], w0[SB], w1[SB];
    auto abuf = [&](int i) -> unsigned char * { return i == 0 ? a0 : i == 1 ? a1 : i == 2 ? a2 : a3; };
    auto bbuf = [&](int i) -> unsigned char * { return i == 0 ? w0 : w1; };
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / WAVE), lane = int(threadIdx.x) % WAVE;
    const int l32 = lane % 32, lh = lane / 32, G = K / QGROUP;
    const int item = small_item(), n0 = item / nby * BN, t0 = item % nby * BM;
    constexpr int RND = U % 2 ? 2 * U : U;  // periods after which the buffers repeat

    if (wave >= S::NC) {
        const int pw = wave - S::NC, tid = pw * WAVE + lane;
        // instruction j of the wave moves 8 rows x 64 K: piece i = j NP + pw: rows
        // 8 (i % (BM / 8)), half i / (BM / 8) of the group
        const uint16_t *xb = Xh + int64_t(t0) * lda;
        int aoff[NA];
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            const int i = j * NP + pw, r = i % (BM / 8) * 8 + lane / 8;
            aoff[j] = min(r, T - 1 - t0) * lda + i / (BM / 8) * 64 + ((lane % 8) ^ swz_x(r)) * 8;
        }
        // the thread's weights: words WPT part .. of the group of row tid % BN
        const int brow = tid % BN, part = tid / BN;
        const BRow b(Wt, St, Zt, min(n0 + brow, N - 1), G);
        const uint32_t *bw = reinterpret_cast<const uint32_t *>(b.w) + part * WPT / 4 * 64 + part * WPT % 4;
        struct WR {
            uint32_t w[WPT];
            uint16_t s;
            uint32_t z;
        };
        WR wr[U];
        constexpr int NLD = NA + (WPT + 3) / 4 + 1 + HAS_Z;
        auto issue_w = [&](int g, WR &r) {
            g = min(g, G - 1);  // past the end: a valid (unused) one
            const uint32_t *q = bw + g * 256;
            if constexpr (WPT >= 4) {
#pragma unroll
                for (int i = 0; i < WPT / 4; ++i) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(q + i * 64);
                    r.w[4 * i] = v.x, r.w[4 * i + 1] = v.y, r.w[4 * i + 2] = v.z, r.w[4 * i + 3] = v.w;
                }
            } else if constexpr (WPT == 2) {
                const uint2 v = *reinterpret_cast<const uint2 *>(q);
                r.w[0] = v.x, r.w[1] = v.y;
            } else {
                r.w[0] = *q;
            }
            r.s = b.s[(g >> 2) * 64 + (g & 3)];
            if constexpr (HAS_Z) r.z = b.z[(g >> 2) * 8];
        };
        auto issue_a = [&](int g, unsigned char *dst) {
            const uint16_t *xs = xb + min(g, G - 1) * QGROUP;
#pragma unroll
            for (int j = 0; j < NA; ++j)
                __builtin_amdgcn_global_load_lds(xs + aoff[j], dst + (j * NP + pw) * 1024, 16, 0, 0);
        };
        auto commit = [&](const WR &r, int g, unsigned char *dst) {
            uint32_t s = r.s, z = HAS_Z ? r.z : 0u;
            asm volatile("" : "+v"(s), "+v"(z));  // taken here, not at their loads
            const uint32_t zv = HAS_Z ? ((z >> (b.zs + 4 * (g & 3))) & 0xfu) * 0x10001u : 0x80008u;
            const h2 zl = __builtin_bit_cast(h2, zv | 0xe400e400u), zh = __builtin_bit_cast(h2, (zv << 4) + 0xd400d400u);
            const h2 s2 = __builtin_bit_cast(h2, s * 0x10001u);
#pragma unroll
            for (int i = 0; i < WPT; ++i) {
                const int c = part * WPT + i;
                *reinterpret_cast<uint4 *>(dst + c / 8 * (BN * 128) + swz(brow, c % 8)) = dequant8_light(r.w[i], zl, zh, s2);
            }
        };
        // every load but the last V of this wave landed, its weights written
        auto meet = [&](auto left) {
            constexpr int V = decltype(left)::value;
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt((V & 15) | ((V >> 4) << 14) | (7 << 4));  // vmcnt V, lgkmcnt 0
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        issue_w(0, wr[0]);
#pragma unroll
        for (int g = 0; g < P; ++g) {
            issue_a(g, abuf(g));
            issue_w(g + 1, wr[(g + 1) % U]);
            __builtin_amdgcn_sched_barrier(0);
        }
        commit(wr[0], 0, bbuf(0));
        meet(std::integral_constant<int, (P - 1) * NLD>());
        auto period = [&](int g, int u) {  // u = g % RND, a constant
            issue_a(g + P, abuf((u + P) % U));
            issue_w(g + P + 1, wr[u % U]);
            __builtin_amdgcn_sched_barrier(0);
            commit(wr[(u + 1) % U], g + 1, bbuf((u + 1) % 2));
            meet(std::integral_constant<int, (P - 1) * NLD>());
        };
        int g = 0;
        for (; g + RND <= G; g += RND) {
#pragma unroll
            for (int u = 0; u < RND; ++u) period(g + u, u);
        }
#pragma unroll
        for (int u = 0; u < RND - 1; ++u)
            if (g + u < G) period(g + u, u);
        meet(std::integral_constant<int, 0>());  // the loads into LDS past the last group
        return;
    }

    const int wm = wave / S::WN, wn = wave % S::WN;
    f32x16 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x16{};
    // A group's fragments, each read again for the next group once its MFMAs are
    // out. (Two sets, read ahead of the MFMAs: 6144->4096 at 16 tokens 18.6 us
    // against 16.1.)
    uint4 af[8][NI], bf[8][NJ];
    auto read = [&](int kk, const unsigned char *a, const unsigned char *w) {
        const int c = 2 * kk % 8 + lh, h = kk / 4;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            af[kk][i] = *reinterpret_cast<const uint4 *>(a + h * (BM * 128) + swz((wm * NI + i) * 32 + l32, c));
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            bf[kk][j] = *reinterpret_cast<const uint4 *>(w + h * (BN * 128) + swz((wn * NJ + j) * 32 + l32, c));
    };
    auto mul = [&](int kk) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = mfma32<F16>(af[kk][i], bf[kk][j], acc[i][j]);
    };
    auto meet = [&] {  // this wave's reads are done
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt 0
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    meet();
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) read(kk, abuf(0), bbuf(0));
    meet();
    auto period = [&](int u) {  // u = g % RND: the MFMAs of group g - 1, the reads of g
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            mul(kk);
            __builtin_amdgcn_sched_barrier(0);
            read(kk, abuf(u % U), bbuf(u % 2));
            __builtin_amdgcn_sched_barrier(0);
        }
        meet();
    };
    int g = 1;
    for (; g + RND <= G; g += RND) {
#pragma unroll
        for (int u = 0; u < RND; ++u) period((u + 1) % RND);
    }
#pragma unroll
    for (int u = 0; u < RND - 1; ++u)
        if (g + u < G) period((u + 1) % RND);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) mul(kk);
    meet();
    store_slots<NI, NJ>(acc, abuf(wave / S::SLOTS) + wave % S::SLOTS * 4096, lane, t0 + wm * NI * 32, n0 + wn * NJ * 32, T,
                        N, Y, ldy, yt);
}

template <int BM, int BN, int NI, int NJ, int NP, int P, bool HAS_Z>
__global__ __launch_bounds__((RoleTile<BM, BN, NI, NJ, NP, P>::THREADS)) void q4_gemm_roles_kernel(
    const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt, const uint16_t *__restrict__ Xh, int lda, int T,
    void *__restrict__ Y, int ldy, int yt, int N, int K, int nby) {
    gemm_roles_block<BM, BN, NI, NJ, NP, P, HAS_Z>(Wt, St, Zt, Xh, lda, T, Y, ldy, yt, N, K, nby);
}

}  // namespace qwq4
