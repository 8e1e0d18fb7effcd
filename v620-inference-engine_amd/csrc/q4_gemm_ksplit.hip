// Launch of the K-split prefill tiles (q4_gemm_ksplit.cuh) and the choice
// among them.
#include "q4_gemm_ksplit.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

namespace {

// A tile shape (KSplit) and its launch time in us over nb blocks of st 64-K
// stages per part: base + st (per_round R + per_load nb / 256) + round R, with
// R rounds of one block per CU (256 CUs). Fitted to 110 launches of seeded
// random shapes (N 1024-12288, K 1024-8192, 1-2427 tokens): every prediction
// within 0.77-1.15 of its measurement, and the shape predicted fastest within
// 1.7% of the one measured fastest (0.02% on average).
struct Shape {
    int bm, ng, wn;
    float base, per_round, per_load, round;
};
constexpr Shape SHAPES[] = {
    {32, 1, 1, 1.95f, 0.512f, 0.207f, 2.38f},  {32, 2, 1, 2.05f, 0.804f, 0.220f, 2.65f},
    {64, 1, 2, 1.59f, 0.602f, 0.149f, 2.85f},  {64, 2, 2, 0.56f, 0.923f, 0.231f, 4.51f},
    {64, 2, 4, 0.07f, 0.845f, 0.199f, 5.57f},  {96, 2, 2, 0.88f, 1.112f, 0.399f, 4.52f},
    {96, 2, 4, 0.00f, 0.999f, 0.329f, 6.73f},  {128, 2, 2, 0.43f, 1.363f, 0.571f, 5.94f},
    {128, 2, 4, 0.00f, 1.209f, 0.498f, 7.61f},
};

template <int BM, int NG, int WN, int NST>
void launch_shape(const GemmArgs &a, const uint16_t *Xh, int lda, hipStream_t s) {
    using S = KSplit<BM, NG, WN, NST>;
    const int nbx = (a.N + S::ROWS - 1) / S::ROWS, nby = (a.T + BM - 1) / BM;
    auto kern = a.Z ? q4_gemm_ksplit_kernel<BM, NG, WN, NST, true> : q4_gemm_ksplit_kernel<BM, NG, WN, NST, false>;
    kern<<<unsigned(nbx * nby), G_THREADS, 0, s>>>(a.W, a.S, a.Z, Xh, lda, a.T, a.Y, a.ldy, a.y_type, a.N, a.K, nby);
}

}  // namespace

bool launch_gemm_ksplit(const GemmArgs &a, const uint16_t *Xh, int lda, int cus, hipStream_t s) {
    // below two rounds of 128 x 256 tiles: measured faster than the whole-K
    // tiles at every one of those 110 shapes (N = 4096, K = 6144, fp16 rows:
    // 80 tokens 16 against 87 us, 601 tokens 42 against 88, 1500 tokens 82
    // against 99; N = 12288, K = 4096: 23 against 60, 67 against 76, 168
    // against 171). Token rows within a tile are addressed by 32-bit offsets.
    const int64_t nb128 = (int64_t(a.N) + 255) / 256 * ((int64_t(a.T) + 127) / 128);
    if (nb128 >= 2 * int64_t(cus) || lda > (1 << 23)) return false;
    // exactly one round of 256 x 128 tiles keeps every CU at its largest tile
    // (2048 rows of K = 3712, 4050 tokens: 3% faster than the K-split tiles)
    if ((int64_t(a.N) + 127) / 128 * ((int64_t(a.T) + 255) / 256) == cus) return false;
    int best = 0;
    float t = 0.f;
    for (int i = 0; i < int(sizeof SHAPES / sizeof SHAPES[0]); ++i) {
        const Shape &p = SHAPES[i];
        const int rows = 32 * p.ng * p.wn, wk = G_WAVES / p.wn, G = a.K / QGROUP;
        const int64_t nb = (int64_t(a.N) + rows - 1) / rows * ((int64_t(a.T) + p.bm - 1) / p.bm);
        const float st = float(2 * ((G + wk - 1) / wk)), R = float((nb + cus - 1) / cus);
        const float ti = p.base + st * (p.per_round * R + p.per_load * (float(nb) / float(cus))) + p.round * R;
        if (i == 0 || ti < t) {
            best = i;
            t = ti;
        }
    }
    switch (best) {
        case 0: launch_shape<32, 1, 1, 4>(a, Xh, lda, s); break;
        case 1: launch_shape<32, 2, 1, 4>(a, Xh, lda, s); break;
        case 2: launch_shape<64, 1, 2, 4>(a, Xh, lda, s); break;
        case 3: launch_shape<64, 2, 2, 4>(a, Xh, lda, s); break;
        case 4: launch_shape<64, 2, 4, 4>(a, Xh, lda, s); break;
        case 5: launch_shape<96, 2, 2, 2>(a, Xh, lda, s); break;
        case 6: launch_shape<96, 2, 4, 4>(a, Xh, lda, s); break;
        case 7: launch_shape<128, 2, 2, 2>(a, Xh, lda, s); break;
        default: launch_shape<128, 2, 4, 4>(a, Xh, lda, s); break;
    }
    return true;
}

}  // namespace qwq4
