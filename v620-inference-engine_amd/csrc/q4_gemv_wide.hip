// Launch of the streamed GEMV (q4_gemv_wide.cuh).
#include "q4_gemv_wide.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

namespace {

template <typename XT, int MB, int WN>
void launch_wide(const GemvArgs &a, hipStream_t s) {
    auto kern = a.Z ? q4_gemv_wide_kernel<XT, MB, WN, true> : q4_gemv_wide_kernel<XT, MB, WN, false>;
    kern<<<unsigned((a.N + Wide<MB, WN>::ROWS - 1) / Wide<MB, WN>::ROWS), 512, 0, s>>>(
        a.W, a.S, a.Z, a.x, a.xs, a.M, a.K, a.N, a.y, a.ys, a.y_bf16, a.accumulate, a.n_lo);
}

// Row blocks of 64 (K split 8 ways) up to two rounds of the chip's resident
// blocks (one per CU above 16 rows, two up to 16), wider ones beyond, which
// move the rows' K fewer times: 32 rows of 4096->151936 88 us with 256 weight
// rows against 114 with 64, 2560->35920 22 against 27; 4096->12288 12.4 with 64
// against 29 with 256. n_all: the matrix's rows, so that the row slices of one
// product take the same K split as the whole.
template <typename XT>
void launch_wide_t(const GemvArgs &a, int n_all, hipStream_t s) {
    const int nb = (n_all + 63) / 64;
    if (a.M <= 16) {
        if (nb <= 1024) launch_wide<XT, 1, 1>(a, s);
        else launch_wide<XT, 1, 2>(a, s);
    } else {
        if (nb <= 512) launch_wide<XT, 2, 1>(a, s);
        else launch_wide<XT, 2, 4>(a, s);
    }
}

}  // namespace

void launch_gemv_wide(const GemvArgs &a, int n_all, hipStream_t s) {
    if (a.x_f16) launch_wide_t<F16>(a, n_all, s);
    else launch_wide_t<BF16>(a, n_all, s);
}

}  // namespace qwq4
