// Dense q4 GEMV for 9 to 32 rows, streamed: where the decode GEMV
// (q4_gemv_impl.cuh) stages every activation row of the whole K in LDS per 16
// weight rows, which outweighs the weights from about 8 rows on and no longer
// fits beyond 16 rows of 4096, a wave here holds 64 weight rows (four 16-row
// subtiles), unpacks each weight once for all 16 MB rows (16x16x32 MFMA) and
// moves the rows' K in groups of 128 through a double buffer. Each group goes
// out one group ahead: the A rows (direct global -> LDS loads) and the wave's
// weights, scale and zero (registers).
//
// Sums are the decode GEMV's, bit for bit: the K parts of dense_gpk groups, each
// group's product started at -(BASE + UNIT z) times its activation sum, the
// parts added in part order. So a row does not depend on its batch. Two forms:
//   split: a block holds 64 weight rows, its waves the K parts, added through LDS.
//     Each wave moves and reads its own A rows, so nothing is waited for between
//     the waves until the end.
//   chain: a block holds 256 weight rows, four waves on the even parts and four on
//     the odd ones, the running sum handed from one to the other through LDS
//     after each part; the A rows of a part are shared by its four waves.
#pragma once

#include "q4_gemv_core.cuh"
#include "q4_lanes.cuh"

namespace qwq4 {


// 16-byte chunk c (0..15) of row r of an A tile [16 MB][128]
__device__ __forceinline__ int wide_swz(int r, int c) { return r * 256 + ((c ^ (r & 15)) << 4); }

// A wave's 64 weight rows from row n0: wave-uniform bases and 32-bit lane offsets.
template <typename XT, int MB, bool HAS_Z, bool HOLD>
struct WideRows {
    const uint4 *w[4];
    const uint16_t *sp, *zp;  // the lane's own row's scales and zero words, at s_off / z_off
    int s_off, z_off;
    struct Group {  // a group as loaded
        uint4 w[4];
        uint16_t s, z;
    };
    __device__ __forceinline__ WideRows(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt, int n0, int nsub, int G,
                                        int lane) {
        const int sub0 = n0 / 16, GC = (G + 3) / 4, n = lane % 16, q = lane / 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = reinterpret_cast<const uint4 *>(Wt) + int64_t(min(sub0 + j, nsub - 1)) * G * 64;
        const int sb = min(sub0, nsub - 1), so = min(q, nsub - 1 - sb) * GC;
        sp = St + int64_t(sb) * GC * 64;
        zp = HAS_Z ? Zt + int64_t(sb) * GC * 16 : nullptr;
        s_off = so * 64 + n * 4;
        z_off = so * 16 + n;
    }
    __device__ __forceinline__ void issue(int g, int lane, Group &r) const {
        typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w[j] + g * 64 + lane));
            r.w[j] = make_uint4(v[0], v[1], v[2], v[3]);
        }
        r.s = sp[(g >> 2) * 64 + (g & 3) + s_off];
        if constexpr (HAS_Z) r.z = zp[(g >> 2) * 16 + z_off];
    }
    // acc[j] += subtile j's rows over group g (A rows at a), as compute_zq
    __device__ __forceinline__ static void compute(const unsigned char *a, const Group &r, int g, int lane,
                                                   f32x4 (&acc)[4][MB]) {
        const int n = lane % 16, q = lane / 16;
        uint32_t s = r.s, z = HAS_Z ? uint32_t(r.z) : 0u, sv[4], zv[4];
        asm volatile("" : "+v"(s), "+v"(z));  // taken here, not at their loads
        split_quarters(s, sv);
        if constexpr (HAS_Z) split_quarters((z >> (4 * (g & 3))) & 0xfu, zv);
        else zv[0] = zv[1] = zv[2] = zv[3] = 8u;
        const uint4 one = make_uint4(XT::ONE, XT::ONE, XT::ONE, XT::ONE);
        auto frag = [&](int t, int mb) { return *reinterpret_cast<const uint4 *>(a + wide_swz(mb * 16 + n, q * 4 + t)); };
        // HOLD: the fragments stay in registers, else they are read again for
        // each pair of subtiles (held they cost the two blocks per CU)
        uint4 held[HOLD ? 4 : 1][MB];
        f32x4 sum[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) sum[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const uint4 f = frag(t, mb);
                if constexpr (HOLD) held[t][mb] = f;
                sum[mb] = mfma16<XT>(f, one, sum[mb]);
            }
#pragma unroll
        for (int jp = 0; jp < 4; jp += 2) {
            if constexpr (!HOLD) asm volatile("" ::: "memory");
            f32x4 p[2][MB];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float nz = -(XT::BASE + XT::UNIT * float(zv[jp + j]));
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) p[j][mb] = sum[mb] * nz;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                uint4 af[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    if constexpr (HOLD) af[mb] = held[t][mb];
                    else af[mb] = frag(t, mb);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint4 &wj = r.w[jp + j];
                    const uint4 f = unpack8_q<XT>(t == 0 ? wj.x : t == 1 ? wj.y : t == 2 ? wj.z : wj.w);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) p[j][mb] = mfma16<XT>(af[mb], f, p[j][mb]);
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float sc = f16_bits_to_f32(uint16_t(sv[jp + j])) * (1.f / XT::UNIT);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[jp + j][mb][e] = __builtin_fmaf(sc, p[j][mb][e], acc[jp + j][mb][e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

template <int MB>
__device__ __forceinline__ void wide_clear(f32x4 (&acc)[4][MB]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// A contiguous range of the row blocks per XCD.
__device__ __forceinline__ int wide_item() {
    const int nb = int(gridDim.x), xq = nb / 8, xr = nb % 8, xcd = int(blockIdx.x) % 8;
    return xcd * xq + min(xcd, xr) + int(blockIdx.x) / 8;
}

// Group i of a double-buffered run: its data arrived (wait), group i + 1 requested,
// then its products.
template <class Group, class IssueFn, class WaitFn, class ComputeFn>
__device__ __forceinline__ void wide_step(int i, const unsigned char *a, const Group &cur, unsigned char *an, Group &next,
                                          IssueFn issue, WaitFn wait, ComputeFn compute) {
    __builtin_amdgcn_sched_barrier(0);
    wait();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue(i + 1, an, next);
    __builtin_amdgcn_sched_barrier(0);
    compute(i, a, cur);
}

// NW waves, a part each (waves past the last part none). TWO: up to 2 NW parts,
// wave w takes parts w and w + NW.
// Grid (64-row blocks, blocks of 16 MB rows).
template <typename XT, int MB, bool HAS_Z, int NW, bool TWO>
__device__ __forceinline__ void gemv_wide_split(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                const uint16_t *__restrict__ x, int xs, int M, int K, int N,
                                                void *__restrict__ y, int ys, int y_bf16, int accumulate, int n_lo) {
    constexpr int BM = 16 * MB, SLOT = 16 * 64 * 4;  // SLOT: a part's sums of 16 rows
    __shared__ __align__(16) unsigned char a0[NW * BM * 256], a1[NW * BM * 256];
    static_assert(sizeof a0 >= (TWO ? 2 : 1) * NW * SLOT, "a slot per part");
    using R = WideRows<XT, MB, HAS_Z, MB == 2>;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, n = lane % 16,
              q = lane / 16;
    const int n0 = wide_item() * 64, G = K / QGROUP, gpk = dense_gpk(G), KS = (G + gpk - 1) / gpk;
    const int m0 = int(blockIdx.y) * BM;
    x += int64_t(m0) * xs;
    M = min(M - m0, BM);
    const R rows(Wt, St, Zt, n0, (N + 15) / 16, G, lane);
    int xo[BM / 4];  // instruction j moves rows 4 j .. 4 j + 3
#pragma unroll
    for (int j = 0; j < BM / 4; ++j) {
        const int r = j * 4 + q;
        xo[j] = min(r, M - 1) * xs + ((n ^ (r & 15)) * 8);
    }
    // the wave's groups: n1 of its first part, then n2 of its second
    const int g0 = wave * gpk, n1 = min(gpk, G - g0), n2 = TWO && wave + NW < KS ? min(gpk, G - g0 - NW * gpk) : 0;
    auto group = [&](int i) { return g0 + i + (TWO && i >= gpk ? (NW - 1) * gpk : 0); };
    unsigned char *const t0 = a0 + wave * (BM * 256), *const t1 = a1 + wave * (BM * 256);
    f32x4 acc[4][MB], first[4][MB];  // first: a first part's sums beside a second part's
    wide_clear(acc);
    if constexpr (TWO) wide_clear(first);
    if (wave < KS) {
        auto issue = [&](int i, unsigned char *dst, typename R::Group &r) {
            const int g = min(group(i), G - 1);  // past the end: a valid (unused) one
#pragma unroll
            for (int j = 0; j < BM / 4; ++j)
                __builtin_amdgcn_global_load_lds(x + g * QGROUP + xo[j], dst + j * 1024, 16, 0, 0);
            rows.issue(g, lane, r);
        };
        // the wave reads what it moved itself: its own loads are waited for, and
        // the reads of the buffer being refilled are complete
        auto wait = [] { wait_vm_below<0>(); };
        auto compute = [&](int i, const unsigned char *a, const typename R::Group &r) {
            R::compute(a, r, group(i), lane, acc);
        };
        typename R::Group w0, w1;
        issue(0, t0, w0);
        int i = 0;
        auto run = [&](int end) {
            for (; i + 2 <= end; i += 2) {
                wide_step(i, t0, w0, t1, w1, issue, wait, compute);
                wide_step(i + 1, t1, w1, t0, w0, issue, wait, compute);
            }
            if (i < end) wide_step(i, t0, w0, t1, w1, issue, wait, compute);  // (the last part's only)
        };
        run(n1);
        if (TWO && n2 > 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) first[j][mb] = acc[j][mb];
            wide_clear(acc);
            run(n1 + n2);
        }
        wait_vm_below<0>();
    }
    // 16 rows at a time: the parts' sums to their slots ([row][64 weight rows]),
    // then each element's parts are added in part order
    const int lo = opaque_lane();
    auto slot = [&](int k) { return reinterpret_cast<float *>(a0 + k * SLOT); };
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        lds_barrier();
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = (4 * (lo / 16) + r) * 64 + 16 * j + lo % 16;
                if (TWO && n2 > 0) {
                    slot(wave)[o] = first[j][mb][r];
                    slot(wave + NW)[o] = acc[j][mb][r];
                } else {
                    slot(wave)[o] = acc[j][mb][r];
                }
            }
        lds_barrier();
        for (int c = wave * WAVE + lo; c < 16 * 64; c += NW * WAVE) {
            const int m = mb * 16 + c / 64, row = n0 + c % 64;
            float v = slot(0)[c];
#pragma unroll
            for (int k = 1; k < (TWO ? 2 : 1) * NW; ++k)
                if (k < KS) v += slot(k)[c];
            if (m < M && row < N && row >= n_lo) store_y(y, int64_t(m0 + m) * ys + row, v, y_bf16, accumulate);
        }
    }
}

template <typename XT, int MB, bool HAS_Z>
__device__ __forceinline__ void gemv_wide_chain(const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt,
                                                const uint16_t *__restrict__ x, int xs, int M, int K, int N,
                                                void *__restrict__ y, int ys, int y_bf16, int accumulate, int n_lo) {
    constexpr int BM = 16 * MB, NA = BM / 16;  // NA: direct A loads per wave and group
    __shared__ __align__(16) unsigned char a0[2 * BM * 256], a1[2 * BM * 256];
    __shared__ f32x4 tot[4][4 * MB][WAVE];  // the running sums, per row group and lane
    using R = WideRows<XT, MB, HAS_Z, MB == 2>;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, n = lane % 16,
              q = lane / 16, wn = wave % 4, wk = wave / 4;
    const int n0 = (wide_item() * 4 + wn) * 64, G = K / QGROUP, gpk = dense_gpk(G), KS = (G + gpk - 1) / gpk;
    const R rows(Wt, St, Zt, n0, (N + 15) / 16, G, lane);
    int xo[NA];  // instruction j moves rows 4 (4 j + wn) .. + 3 of the part's
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int r = (j * 4 + wn) * 4 + q;
        xo[j] = min(r, M - 1) * xs + ((n ^ (r & 15)) * 8);
    }
    f32x4 acc[4][MB];
    wide_clear(acc);
    int g0 = wk * gpk;  // the wave's part of the pair at hand
    auto issue = [&](int i, unsigned char *dst, typename R::Group &r) {
        const int g = min(g0 + i + (i >= gpk ? gpk : 0), G - 1);  // i = gpk: the next pair's; past the end: a valid (unused) one
#pragma unroll
        for (int j = 0; j < NA; ++j)
            __builtin_amdgcn_global_load_lds(x + g * QGROUP + xo[j], dst + wk * (BM * 256) + (j * 4 + wn) * 1024, 16, 0, 0);
        rows.issue(g, lane, r);
    };
    auto wait = [] {
        wait_vm_below<0>();
        __builtin_amdgcn_s_barrier();  // every wave's rows have landed, and the other buffer is read
    };
    auto compute = [&](int i, const unsigned char *a, const typename R::Group &r) {
        if (g0 + i < G) R::compute(a + wk * (BM * 256), r, g0 + i, lane, acc);
    };
    typename R::Group w0, w1;
    issue(0, a0, w0);
    for (int p = 0; p < KS; p += 2) {  // parts p and p + 1: gpk groups each, the last part of all shorter
        const int steps = min(gpk, G - p * gpk);
        int i = 0;
        for (; i + 2 <= steps; i += 2) {
            wide_step(i, a0, w0, a1, w1, issue, wait, compute);
            wide_step(i + 1, a1, w1, a0, w0, issue, wait, compute);
        }
        if (i < steps) wide_step(i, a0, w0, a1, w1, issue, wait, compute);
        // the running sum: through part p, then through part p + 1
        auto add = [&](bool take) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    if (take) acc[j][mb] = tot[wn][j * MB + mb][lane] + acc[j][mb];
                    tot[wn][j * MB + mb][lane] = acc[j][mb];
                }
        };
        if (wk == 0) add(p > 0);
        lds_barrier();
        if (wk == 1 && p + 1 < KS) add(true);
        lds_barrier();
        if (p + 2 < KS) wide_clear(acc);
        g0 += 2 * gpk;
    }
    wait_vm_below<0>();
    if (wk != (KS - 1) % 2) return;
    const int lo = opaque_lane();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = mb * 16 + 4 * (lo / 16) + r, row = n0 + 16 * j + lo % 16;
                if (m < M && row < N && row >= n_lo) store_y(y, int64_t(m) * ys + row, acc[j][mb][r], y_bf16, accumulate);
            }
}

template <typename XT, int MB, bool HAS_Z, int NW, bool TWO>
__global__ __launch_bounds__(NW *WAVE, (MB == 1 && NW != 12 ? 4 : MB == 1 ? 3 : 2)) void q4_gemv_wide_split_kernel(
    const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt, const uint16_t *__restrict__ x, int xs, int M, int K, int N,
    void *__restrict__ y, int ys, int y_bf16, int accumulate, int n_lo) {
    gemv_wide_split<XT, MB, HAS_Z, NW, TWO>(Wt, St, Zt, x, xs, M, K, N, y, ys, y_bf16, accumulate, n_lo);
}

template <typename XT, int MB, bool HAS_Z>
__global__ __launch_bounds__(8 * WAVE, (MB == 1 ? 4 : 2)) void q4_gemv_wide_chain_kernel(
    const uint32_t *Wt, const uint16_t *St, const uint16_t *Zt, const uint16_t *__restrict__ x, int xs, int M, int K, int N,
    void *__restrict__ y, int ys, int y_bf16, int accumulate, int n_lo) {
    gemv_wide_chain<XT, MB, HAS_Z>(Wt, St, Zt, x, xs, M, K, N, y, ys, y_bf16, accumulate, n_lo);
}

}  // namespace qwq4
