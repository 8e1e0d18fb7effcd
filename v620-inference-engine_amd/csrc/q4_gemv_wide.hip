// Launch of the streamed GEMV (q4_gemv_wide.cuh).
#include "q4_gemv_wide.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

namespace {

// The form and its blocks (every one gives the same bits), us at fp32 results:
//   up to 16 rows: split, a wave per part (two blocks of 8 waves per CU, one of 12
//     or 16), up to three rounds of a block per CU, chain beyond (65536 rows of
//     K = 6144 at 16 rows 43.4 against 56.3; 35920 of 2560 20.4 against 17.7).
//   17 to 32 rows: split with the 16-row blocks on CUs of their own where both
//     fill one round of them (8192 rows of K = 4096 at 32 9.8 against 13.2 with both
//     in a block, 4096 of 6144 12.3 against 17.5), else both in a block up to two
//     rounds (12288 of 4096 14.2 against 16.3; beyond 8 parts some waves take two),
//     chain beyond (35920 of 2560 23.6 against 28.9, 151936 of 4096 90 against 120;
//     20480 of 4096 29.8 against 24.7).
template <typename XT, bool HAS_Z>
void launch_wide(const GemvArgs &a, hipStream_t s) {
    const int nb = (a.N + 63) / 64, G = a.K / QGROUP, gpk = dense_gpk(G), KS = (G + gpk - 1) / gpk;
    auto go = [&](auto kern, dim3 grid, int waves) {
        kern<<<grid, waves * WAVE, 0, s>>>(a.W, a.S, a.Z, a.x, a.xs, a.M, a.K, a.N, a.y, a.ys, a.y_bf16, a.accumulate,
                                           a.n_lo);
    };
    const bool two = a.M > 16, apart = !two || nb <= 128;
    if (nb > (two ? 512 : 768)) {
        const dim3 grid((nb + 3) / 4);
        if (two) go(q4_gemv_wide_chain_kernel<XT, 2, HAS_Z>, grid, 8);
        else go(q4_gemv_wide_chain_kernel<XT, 1, HAS_Z>, grid, 8);
    } else if (apart) {
        const dim3 grid(nb, two ? 2 : 1);
        if (KS <= 8) go(q4_gemv_wide_split_kernel<XT, 1, HAS_Z, 8, false>, grid, 8);
        else if (KS <= 12) go(q4_gemv_wide_split_kernel<XT, 1, HAS_Z, 12, false>, grid, 12);
        else go(q4_gemv_wide_split_kernel<XT, 1, HAS_Z, 16, false>, grid, 16);
    } else {
        if (KS <= 8) go(q4_gemv_wide_split_kernel<XT, 2, HAS_Z, 8, false>, dim3(nb), 8);
        else go(q4_gemv_wide_split_kernel<XT, 2, HAS_Z, 8, true>, dim3(nb), 8);
    }
}

}  // namespace

void launch_gemv_wide(const GemvArgs &a, hipStream_t s) {
    if (a.x_f16) a.Z ? launch_wide<F16, true>(a, s) : launch_wide<F16, false>(a, s);
    else a.Z ? launch_wide<BF16, true>(a, s) : launch_wide<BF16, false>(a, s);
}

}  // namespace qwq4
