// Launch of the small prefill tiles (q4_gemm_small.cuh) and the choice among
// them.
#include "q4_gemm_small.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

namespace {

// A tile of bm tokens x bn weight rows and its launch time in us over nb blocks
// and G groups of 128 K: base + G (per_k + per_round R + per_load nb / CUs) + round R,
// with R rounds of one block per CU. Fitted to 138 launches of seeded random shapes
// (N 512-14336, K 1024-8192, 1-3900 tokens): the tile predicted fastest is within
// 0.3% of the one measured fastest on average, at worst 13% (4672 rows of K = 7040,
// 435 tokens). The last is the 128 x 256 whole-chip tile (q4_gemm.hip).
struct Shape {
    int bm, bn;
    float base, per_k, per_round, per_load, round;
};
constexpr Shape SHAPES[] = {
    {32, 32, 2.231f, 0.104f, 0.148f, 0.033f, 1.011f}, {32, 64, 1.818f, 0.046f, 0.310f, 0.064f, 1.708f},
    {64, 64, 1.436f, 0.f, 0.411f, 0.102f, 2.454f},    {96, 64, 0.084f, 0.f, 0.529f, 0.099f, 4.245f},
    {128, 64, 0.f, 0.f, 0.595f, 0.167f, 4.296f},      {64, 128, 3.076f, 0.370f, 0.334f, 0.217f, 0.943f},
    {96, 128, 3.084f, 0.302f, 0.543f, 0.218f, 1.156f}, {128, 128, 5.737f, 0.123f, 0.806f, 0.260f, 0.207f},
    {128, 256, 0.f, 0.f, 1.642f, 0.589f, 5.009f},
};

template <class Kern>
void launch_tile(Kern kern, int bm, int bn, int threads, const GemmArgs &a, const uint16_t *Xh, int lda, hipStream_t s) {
    const int nbx = (a.N + bn - 1) / bn, nby = (a.T + bm - 1) / bm;
    kern<<<unsigned(nbx * nby), threads, 0, s>>>(a.W, a.S, a.Z, Xh, lda, a.T, a.Y, a.ldy, a.y_type, a.N, a.K, nby);
}

template <int BM>
void launch_reg(const GemmArgs &a, const uint16_t *Xh, int lda, hipStream_t s) {
    using S = RegTile<BM>;
    launch_tile(a.Z ? q4_gemm_reg_kernel<BM, true> : q4_gemm_reg_kernel<BM, false>, BM, S::BN, S::THREADS, a, Xh, lda, s);
}

template <int BM, int BN, int NI, int NJ, int NP, int P>
void launch_roles(const GemmArgs &a, const uint16_t *Xh, int lda, hipStream_t s) {
    using S = RoleTile<BM, BN, NI, NJ, NP, P>;
    launch_tile(a.Z ? q4_gemm_roles_kernel<BM, BN, NI, NJ, NP, P, true> : q4_gemm_roles_kernel<BM, BN, NI, NJ, NP, P, false>,
                BM, BN, S::THREADS, a, Xh, lda, s);
}

}  // namespace

bool launch_gemm_small(const GemmArgs &a, const uint16_t *Xh, int lda, int cus, hipStream_t s) {
    if (lda > (1 << 23)) return false;  // (token rows within a tile are addressed by 32-bit offsets)
    int best = 0;
    float t = 0.f;
    const float G = float(a.K / QGROUP);
    for (int i = 0; i < int(sizeof SHAPES / sizeof SHAPES[0]); ++i) {
        const Shape &p = SHAPES[i];
        const int64_t nb = (int64_t(a.N) + p.bn - 1) / p.bn * ((int64_t(a.T) + p.bm - 1) / p.bm);
        const float R = float((nb + cus - 1) / cus);
        const float ti = p.base + G * (p.per_k + p.per_round * R + p.per_load * (float(nb) / float(cus))) + p.round * R;
        if (i == 0 || ti < t) {
            best = i;
            t = ti;
        }
    }
    switch (best) {
        case 0: launch_roles<32, 32, 1, 1, 4, 3>(a, Xh, lda, s); break;
        case 1: launch_roles<32, 64, 1, 1, 4, 3>(a, Xh, lda, s); break;
        case 2: launch_roles<64, 64, 1, 1, 4, 3>(a, Xh, lda, s); break;
        case 3: launch_roles<96, 64, 1, 2, 4, 3>(a, Xh, lda, s); break;
        case 4: launch_roles<128, 64, 2, 1, 4, 2>(a, Xh, lda, s); break;
        case 5: launch_reg<64>(a, Xh, lda, s); break;
        case 6: launch_reg<96>(a, Xh, lda, s); break;
        case 7: launch_reg<128>(a, Xh, lda, s); break;
        default: return false;
    }
    return true;
}

}  // namespace qwq4
