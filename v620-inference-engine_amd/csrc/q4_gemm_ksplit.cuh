// q4-dequant GEMM tiles with K split over the waves of a block, for chunks
// whose 128- to 256-token tiles are too few to fill the chip (short prompts,
// the rest of a prompt, narrow projections).
//
// A block computes BM tokens x 32 NG WN weight rows. Its 8 waves are WN along
// the weight rows x WK = 8 / WN along K: wave (wn, wk) holds 32 NG weight rows
// and the wk-th range of whole 128-wide K groups, dequantises its weights in
// registers (each lane one tiled q4 entry per 32 rows and 64-K stage) and
// computes every token row of the tile against them. The parts' sums are
// added through LDS in part order at the end (deterministic), so no workspace
// and no second pass over memory.
//
// Pipeline. K runs in stages of 64 per part. The stage's A rows (direct
// global -> LDS loads, split over the part's WN waves) and the wave's raw
// weights, scales and zeros (registers) are requested together, NST - 1
// stages ahead: vector loads complete in order, so a shallower A would also
// cut the weights' time in flight. One barrier per stage.
#pragma once

#include "q4_gemm_core.cuh"

namespace qwq4 {

template <int BM, int NG, int WN, int NST>
struct KSplit {
    static_assert(BM % 32 == 0 && BM <= 128 && 8 % WN == 0 && (NG == 1 || NG == 2), "");
    static constexpr int WK = 8 / WN, ROWS = 32 * NG * WN, NI = BM / 32;
    static constexpr int NA = BM / 8 / WN;      // direct A loads per wave and stage
    static constexpr int SZ = WK * BM * 128;    // bytes of one stage's A
    static_assert(NA >= 1 && NST % 2 == 0 && NST * SZ <= 160 * 1024, "");
    // the closing sum runs over PT tokens at a time: one slot of PT x 32 NG
    // floats per wave, whole slots per stage buffer
    static constexpr int PT = BM % 64 == 0 && 64 * 32 * NG * 4 * 8 <= SZ / (64 * 32 * NG * 4) * (64 * 32 * NG * 4) * NST ? 64 : 32;
    static constexpr int SLOT = PT * 32 * NG * 4, PER = SZ / SLOT;
    static_assert(PER >= 1 && PER * NST >= 8, "the partial sums fit the stage buffers");
};

// one output element as stored (yt: 0 fp32, 1 bf16, 2 fp16 saturated)
__device__ __forceinline__ uint32_t cvt_y16(float v, int yt) {
    return yt == 1 ? f32_to_bf16_rne(v) : __builtin_bit_cast(uint16_t, f32_to_f16_satfinite(v));
}

template <int BM, int NG, int WN, int NST, bool HAS_Z>
__device__ __forceinline__ void gemm_ksplit_block(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                  const uint16_t *__restrict__ Xh, int lda, int T,
                                                  void *__restrict__ Y, int ldy, int yt, int N, int K, int nby) {
    using S = KSplit<BM, NG, WN, NST>;
    constexpr int NI = S::NI, NA = S::NA, SZ = S::SZ;
    __shared__ __align__(16) unsigned char b0[SZ], b1[SZ], b2[NST > 2 ? SZ : 16], b3[NST > 3 ? SZ : 16];
    auto buf = [&](int i) -> unsigned char * { return i == 0 ? b0 : i == 1 ? b1 : i == 2 ? b2 : b3; };
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int l32 = lane % 32, lh = lane / 32, wn = wave % WN, wk = wave / WN;

    // weight-row-major tile order, a contiguous range of tiles per XCD: the
    // token tiles over the same weights run together and share an L2
    const int nb = int(gridDim.x), xq = nb / 8, xr = nb % 8, xcd = int(blockIdx.x) % 8;
    const int item = xcd * xq + min(xcd, xr) + int(blockIdx.x) / 8;
    const int n0 = item / nby * S::ROWS, t0 = item % nby * BM;

    // this wave's K range: groups g0 .. g0 + ng - 1 of G (ng may be 0)
    const int G = K / QGROUP, per = G / S::WK, rem = G % S::WK;
    const int g0 = wk * per + min(wk, rem), ns = 2 * (per + (wk < rem)), nsmax = 2 * (per + (rem > 0));

    const uint16_t *xb = Xh + int64_t(t0) * lda;
    int aoff[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int r = (j * WN + wn) * 8 + lane / 8;
        aoff[j] = min(r, T - 1 - t0) * lda + ((lane % 8) ^ swz_x(r)) * 8;
    }
    const int64_t row0 = n0 + wn * 32 * NG;
    const BRow bs(Wt, St, Zt, min(row0 + (NG == 2 ? lane : l32), int64_t(N - 1)), G);
    const uint4 *bw[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) bw[j] = BRow(Wt, St, Zt, min(row0 + j * 32 + l32, int64_t(N - 1)), G).w;

    struct WR {
        uint4 w[NG];
    };
    struct SZr {  // a group's scale and zero word, as loaded
        uint16_t s;
        uint32_t z;
    };
    WR wr[NST];
    SZr sz[NST / 2];
    constexpr int NLD = NA + NG, NSZ = 1 + HAS_Z;  // vector loads per stage, and per group beside them
    auto group = [&](int s) { return min(g0 + min(s, max(ns, 1) - 1) / 2, G - 1); };  // past the end: a valid (unused) one
    auto issue = [&](int s, int u, unsigned char *dst) {
        const int g = group(s), h = u & 1;
        const uint16_t *xs = xb + g * QGROUP + h * GB_K;
#pragma unroll
        for (int j = 0; j < NA; ++j)
            __builtin_amdgcn_global_load_lds(xs + aoff[j], dst + wk * (BM * 128) + (j * WN + wn) * 1024, 16, 0, 0);
#pragma unroll
        for (int j = 0; j < NG; ++j) wr[u].w[j] = bw[j][g * 64 + (h * 2 + lh) * 16];
        if (h == 0) {
            sz[u / 2].s = bs.s[(g >> 2) * 64 + (g & 3)];
            if constexpr (HAS_Z) sz[u / 2].z = bs.z[(g >> 2) * 8];
        }
    };
    f32x16 acc[NI][NG];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j) acc[i][j] = f32x16{};
    // the rows' packed fp16 scales and 1024 + z of the group at hand
    uint32_t sv[2] = {}, zv[2] = {};
    auto open_group = [&](const SZr &q, int s) {
        const uint32_t z = HAS_Z ? (q.z >> (bs.zs + 4 * (group(s) & 3))) & 0xfu : 8u;
        if constexpr (NG == 2) {  // each lane's own row's, then both halves' rows
            split_halves(uint32_t(q.s) * 0x10001u, sv[0], sv[1]);
            if constexpr (HAS_Z) split_halves(z * 0x10001u | 0x64006400u, zv[0], zv[1]);
            else zv[0] = zv[1] = 0x64086408u;
        } else {
            sv[0] = uint32_t(q.s) * 0x10001u;
            zv[0] = z * 0x10001u | 0x64006400u;
        }
    };
    auto compute = [&](const unsigned char *ab, const WR &r) {
        const unsigned char *a = ab + wk * (BM * 128);
        uint4 af[2][NI], f[2][NG];
        auto rd = [&](int kk, uint4 (&d)[NI]) {
#pragma unroll
            for (int i = 0; i < NI; ++i) d[i] = *reinterpret_cast<const uint4 *>(a + swz(i * 32 + l32, kk + 4 * lh));
        };
        auto dq = [&](int kk, uint4 (&d)[NG]) {
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                const uint32_t w = kk == 0 ? r.w[j].x : kk == 1 ? r.w[j].y : kk == 2 ? r.w[j].z : r.w[j].w;
                d[j] = dequant8(w, __builtin_bit_cast(h2, zv[j]), __builtin_bit_cast(h2, sv[j]));
            }
        };
        rd(0, af[0]);
        dq(0, f[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < GB_K / 16; ++kk) {
            const int c = kk & 1;
            const bool more = kk + 1 < GB_K / 16;
            if (more) {
                rd(kk + 1, af[c ^ 1]);
                dq(kk + 1, f[c ^ 1]);
            }
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < NG; ++j) acc[i][j] = mfma32<F16>(af[c][i], f[c][j], acc[i][j]);
            // the next step's fragment reads, then its dequant spread over
            // this step's MFMAs: in order of issue a wave would wait for the
            // matrix core with its VALU work still to come, and so would the
            // other wave of its SIMD, which the stage barrier keeps in step
            if (more) {
                __builtin_amdgcn_sched_group_barrier(0x100, NI, 0);
#pragma unroll
                for (int q = 0; q < NI * NG; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (15 * NG + NI * NG - 1) / (NI * NG), 0);
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
        // the stage's registers count as arrived also where its compute is
        // skipped (a part with fewer groups than the longest)
        asm volatile("" : "+v"(wr[u].w[0].x), "+v"(wr[u].w[NG - 1].x));
        if (u % 2 == 0) {
            asm volatile("" : "+v"(sz[u / 2].s));
            if constexpr (HAS_Z) asm volatile("" : "+v"(sz[u / 2].z));
            open_group(sz[u / 2], s);
        }
        if (s < ns) compute(buf(u), wr[u]);
    };
    // Whole rounds of the stage buffers, then the rest: with an exit inside
    // the round the compiler sees paths on which a stage does not follow its
    // predecessor's requests, and drains every load in flight before it
    // reuses a stage's registers.
    int s = 0;
    for (; s + NST <= nsmax; s += NST) {
#pragma unroll
        for (int u = 0; u < NST; ++u) stage(s + u, u);
    }
#pragma unroll
    for (int u = 0; u < NST - 1; ++u)
        if (s + u < nsmax) stage(s + u, u);
    wait_vm_below<0>();

    // closing sum: PT tokens at a time, the wave's sums to its slot, then
    // every wave adds the WK parts of its share in part order and stores it
    constexpr int PT = S::PT, SLOT = S::SLOT, PER = S::PER, RB = 32 * NG * 4;  // RB: bytes of a slot row
    auto slot = [&](int w) { return buf(w / PER) + (w % PER) * SLOT; };
    const int ye = yt == 0 ? 4 : 2;
#pragma unroll
    for (int p = 0; p < BM / PT; ++p) {
        lds_barrier();
        unsigned char *mine = slot(wave);
#pragma unroll
        for (int i = 0; i < PT / 32; ++i)
#pragma unroll
            for (int j = 0; j < NG; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int tr = i * 32 + (r / 4) * 8 + lh * 4 + (r % 4);
                    *reinterpret_cast<float *>(mine + tr * RB + (j * 32 + l32) * 4) = acc[p * (PT / 32) + i][j][r];
                }
        lds_barrier();
        // pieces of 8 weight rows: PT x 4 NG per weight-row slice
        constexpr int PCS = PT * 4 * NG * WN;
        for (int c = tid; c < PCS; c += G_THREADS) {
            const int pc = c % (4 * NG * WN), tr = c / (4 * NG * WN), sl = pc / (4 * NG), col = pc % (4 * NG) * 8;
            f32x4 v0{}, v1{};
#pragma unroll
            for (int k = 0; k < S::WK; ++k) {
                const unsigned char *q = slot(k * WN + sl) + tr * RB + col * 4;
                v0 += *reinterpret_cast<const f32x4 *>(q);
                v1 += *reinterpret_cast<const f32x4 *>(q + 16);
            }
            const int t = t0 + p * PT + tr, n = n0 + sl * 32 * NG + col;
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

template <int BM, int NG, int WN, int NST, bool HAS_Z>
__global__ __launch_bounds__(G_THREADS) void q4_gemm_ksplit_kernel(const uint32_t *Wt, const uint16_t *St,
                                                                   const uint16_t *Zt,
                                                                   const uint16_t *__restrict__ Xh, int lda, int T,
                                                                   void *__restrict__ Y, int ldy, int yt, int N, int K,
                                                                   int nby) {
    gemm_ksplit_block<BM, NG, WN, NST, HAS_Z>(Wt, St, Zt, Xh, lda, T, Y, ldy, yt, N, K, nby);
}

}  // namespace qwq4
