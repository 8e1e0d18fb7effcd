// Launch of the small prefill tiles (q4_gemm_small.cuh) and the choice among
// them.
#include "q4_gemm_small.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

namespace {

struct Shape {  // a tile of bm tokens x bn weight rows
    int bm, bn;
    TileTime t;
};
constexpr Shape SHAPES[] = {
    {32, 32, {1.244f, 0.110f, 0.139f, 0.038f, 1.931f}},  {32, 64, {1.185f, 0.044f, 0.311f, 0.066f, 2.353f}},
    {64, 64, {0.823f, 0.029f, 0.383f, 0.103f, 3.072f}},  {96, 64, {0.480f, 0.f, 0.555f, 0.064f, 3.823f}},
    {128, 64, {0.202f, 0.f, 0.620f, 0.136f, 3.879f}},    {64, 128, {3.008f, 0.307f, 0.330f, 0.274f, 1.020f}},
    {96, 128, {2.171f, 0.265f, 0.498f, 0.320f, 1.453f}}, {128, 128, {2.871f, 0.144f, 0.750f, 0.325f, 1.985f}},
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

bool launch_gemm_small(const GemmArgs &a, const uint16_t *Xh, int lda, int cus, float large_us, hipStream_t s) {
    if (lda > (1 << 23)) return false;  // (token rows within a tile are addressed by 32-bit offsets)
    int best = -1;
    for (int i = 0; i < int(sizeof SHAPES / sizeof SHAPES[0]); ++i) {
        const Shape &p = SHAPES[i];
        const int64_t nb = (int64_t(a.N) + p.bn - 1) / p.bn * ((int64_t(a.T) + p.bm - 1) / p.bm);
        const float t = p.t.us(a.K / QGROUP, float(nb) / float(cus), float((nb + cus - 1) / cus));
        if (t < large_us) {
            best = i;
            large_us = t;
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
