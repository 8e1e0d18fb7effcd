// Grouped q4 expert GEMMs for prefill chunks (reference role:
// gpu::moe_experts_T, src/kernels/moe_experts.hip:17-171, which dequantises
// the expert's q4 weights into an fp16 LDS tile and multiplies gathered
// token rows).
//
// Work is the (expert, tile) list written by the routing kernel
// (qw_moe_route with tile_m = GROUPED_TILE_M = -32: mixed tiles of 32 to 160
// slots); slots of one expert are contiguous (offsets[e] ..), slot p
// carries token pair_tok[p]. A tile's height follows from its start and the
// expert's slot count (tile_rows). Each block runs the register-dequant MFMA
// core (gemm_tile_rd2, q4_gemm_core.cuh) at that height on one list entry
// and 512 weight rows:
//   gate/up  A = the tile's gathered token rows of x (fp16 copy in the
//            workspace); wave w holds the gate and the up rows of the same 32
//            columns j0 + 32 w .., so h = silu(g) * u (fp16, saturated, the
//            reference's fp16 intermediate) is formed in the wave.
//   down     A = the tile's h rows (contiguous slots), 512 down rows; yp fp32
//            or fp16.
// Chunks with few tokens per expert take kernels of 32 slots per block instead
// (gemm_tile_light below) on the same list.
// Blocks past the list's length (n_tiles, known only on the device) exit at
// once; the grid is sized for the largest possible list (they are dispatched
// after every real tile).
#include "q4_gemm_core.cuh"
#include "q4_kernels.hpp"

namespace qwq4 {

// 32 to 160 slots. Before the 96- and 160-slot tiles (128, 64 or 32 slots):
// same box, config 5, 1.82-1.86 ms per chunk against
// 1.96 with tiles of 256 (role-split core), 128 and 64 (one 32-row weight
// group per wave); the finer remainders cut the padded rows from 1.25 to 1.12
// of the real ones, and each A fragment feeds two MFMAs.
constexpr int GROUPED_TILE_M = -32;

int moe_grouped_tile_m() { return GROUPED_TILE_M; }

size_t moe_grouped_workspace_bytes(int T, int, int, int H, int) { return gemm_workspace_bytes(T, H); }

static __device__ __forceinline__ uint16_t f32_to_f16_sat(float v) {
    return __builtin_bit_cast(uint16_t, f32_to_f16_satfinite(v));
}

static __device__ __forceinline__ float silu_mul(float g, float u) { return silu_ref(g) * u; }

struct GateUpTile {
    const uint32_t *gw, *uw;
    const uint16_t *gs, *gz, *us, *uz;
    const int32_t *pair_tok;
    const uint16_t *xh;
    int H, F;
    uint16_t *h;
};

// ---- a tile of 32 to 160 slots by 512 weight rows (gemm_tile_rd2)
// gate/up: wave w holds gate and up rows of the same 32 columns j0 + 32 w ..
// (group 0 gate, group 1 up), so h = silu(g) * u is formed in the wave.
template <int BM, bool HAS_Z>
__device__ __forceinline__ void gate_up_tile(const GateUpTile &a, int e, int base, int M, int j0) {
    constexpr int NI = BM / 32, NA = (BM + 63) / 64;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
    const int64_t wrow = int64_t(e) * a.F + min(j0 + wave * 32 + lane % 32, a.F - 1);
    const int G = a.H / QGROUP;
    const BRow bg(a.gw, a.gs, a.gz, wrow, G), bu(a.uw, a.us, a.uz, wrow, G);
    // the lane's own row: gate in lanes 0-31, up in 32-63
    const bool up = lane >= 32;
    const BRow bs(a.gw, up ? a.us : a.gs, up ? a.uz : a.gz, wrow, G);
    const uint16_t *arow[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) arow[j] = a.xh + int64_t(a.pair_tok[base + min(64 * j + wave * 8 + lane / 8, M - 1)]) * a.H;
    f32x16 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[i][0] = acc[i][1] = f32x16{};
    gemm_tile_rd2<BM, HAS_Z, 0>(arow, bg, bu, bs, a.H, acc);
    auto cvt = [](float v, int, int) { return f32_to_f16_sat(v); };
#pragma unroll
    for (int hh = 0; hh < (NI + 1) / 2; ++hh) {
        f32x16 hv[2][1];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q)
                hv[i][0][q] = 2 * hh + i < NI ? silu_mul(acc[min(2 * hh + i, NI - 1)][0][q], acc[min(2 * hh + i, NI - 1)][1][q]) : 0.f;
        emit_tile<1, 2>(epi_slot(wave), hv, cvt, [&](int tr, int c, uint4 v) {
            const int m = hh * 64 + tr, j = j0 + wave * 32 + c;
            if (m < M && j < a.F) *reinterpret_cast<uint4 *>(a.h + int64_t(base + m) * a.F + j) = v;
        });
    }
}

template <int BM, bool HAS_Z, bool YP16>
__device__ __forceinline__ void down_tile(const uint32_t *dw, const uint16_t *ds, const uint16_t *dz, int e, int base,
                                           int M, const uint16_t *h, int H, int F, void *yp) {
    constexpr int NI = BM / 32, NA = (BM + 63) / 64, YB = YP16 ? 2 : 4;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
    const int n0 = blockIdx.x * 512 + wave * 64;
    const int G = F / QGROUP;
    const BRow b0(dw, ds, dz, int64_t(e) * H + min(n0 + lane % 32, H - 1), G),
        b1(dw, ds, dz, int64_t(e) * H + min(n0 + 32 + lane % 32, H - 1), G),
        bs(dw, ds, dz, int64_t(e) * H + min(n0 + lane, H - 1), G);
    const uint16_t *arow[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) arow[j] = h + int64_t(base + min(64 * j + wave * 8 + lane / 8, M - 1)) * F;
    f32x16 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[i][0] = acc[i][1] = f32x16{};
    gemm_tile_rd2<BM, HAS_Z, 1 + YP16>(arow, b0, b1, bs, F, acc);
#pragma unroll
    for (int hh = 0; hh < (NI + 1) / 2; ++hh) {
        f32x16 o[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) o[i][j] = 2 * hh + i < NI ? acc[min(2 * hh + i, NI - 1)][j] : f32x16{};
        emit_tile<2, YB>(
            epi_slot(wave), o, [](float v, int, int) { return f32_to_f16_sat(v); },
            [&](int tr, int c, uint4 v) {
                const int m = hh * 64 + tr, n = n0 + c;
                if (m < M && n < H)
                    *reinterpret_cast<uint4 *>(static_cast<unsigned char *>(yp) + (int64_t(base + m) * H + n) * YB) = v;
            });
    }
}

template <bool HAS_Z>
__global__ __launch_bounds__(G_THREADS) void moe_gate_up_gemm_kernel(GateUpTile a, const int32_t *__restrict__ offsets,
                                                                      const int32_t *__restrict__ tile_e,
                                                                      const int32_t *__restrict__ tile_m0,
                                                                      const int32_t *__restrict__ n_tiles) {
    const int tile = blockIdx.y;
    if (tile >= *n_tiles) return;
    const int e = tile_e[tile], m0 = tile_m0[tile], rem = offsets[e + 1] - offsets[e] - m0;
    const int base = offsets[e] + m0, rows = tile_rows(rem, GROUPED_TILE_M), M = min(rows, rem);
    const int j0 = blockIdx.x * 256;
    if (rows == 160) gate_up_tile<160, HAS_Z>(a, e, base, M, j0);
    else if (rows == 128) gate_up_tile<128, HAS_Z>(a, e, base, M, j0);
    else if (rows == 96) gate_up_tile<96, HAS_Z>(a, e, base, M, j0);
    else if (rows == 64) gate_up_tile<64, HAS_Z>(a, e, base, M, j0);
    else gate_up_tile<32, HAS_Z>(a, e, base, M, j0);
}

template <bool HAS_Z, bool YP16>
__global__ __launch_bounds__(G_THREADS) void moe_down_gemm_kernel(
    const uint32_t *__restrict__ dw, const uint16_t *__restrict__ ds, const uint16_t *__restrict__ dz,
    const int32_t *__restrict__ offsets, const int32_t *__restrict__ tile_e, const int32_t *__restrict__ tile_m0,
    const int32_t *__restrict__ n_tiles, const uint16_t *__restrict__ h, int H, int F, void *__restrict__ yp) {
    const int tile = blockIdx.y;
    if (tile >= *n_tiles) return;
    const int e = tile_e[tile], m0 = tile_m0[tile], rem = offsets[e + 1] - offsets[e] - m0;
    const int base = offsets[e] + m0, rows = tile_rows(rem, GROUPED_TILE_M), M = min(rows, rem);
    if (rows == 160) down_tile<160, HAS_Z, YP16>(dw, ds, dz, e, base, M, h, H, F, yp);
    else if (rows == 128) down_tile<128, HAS_Z, YP16>(dw, ds, dz, e, base, M, h, H, F, yp);
    else if (rows == 96) down_tile<96, HAS_Z, YP16>(dw, ds, dz, e, base, M, h, H, F, yp);
    else if (rows == 64) down_tile<64, HAS_Z, YP16>(dw, ds, dz, e, base, M, h, H, F, yp);
    else down_tile<32, HAS_Z, YP16>(dw, ds, dz, e, base, M, h, H, F, yp);
}

// ---- chunks with few tokens per expert: 32 slots by 512 weight rows, bound
// by the weight stream
// A wave holds 64 weight rows (two 32-row groups, as gemm_tile_rd2) and every
// slot of the block, so each weight is read and dequantised once per 32 slots.
// What the stream needs is requests in flight: with 32 accumulator registers a
// wave fits 128 VGPRs, so a CU holds two blocks (of the taller tiles one), each
// wave a whole group (128 K) ahead; a group's A rows are 8 KB, one direct load
// per wave. Operands, MFMA and K order are gemm_tile_rd2's, so a slot's sums
// are the same bits in a chunk of any length.
constexpr int LIGHT_A = 32 * 256;  // bytes of a group's A: [32][128] fp16

// 16-byte chunk c (0..15) of row r of the A tile: a fragment read takes 32
// rows at one chunk of each 128-byte half
__device__ __forceinline__ int light_swz(int r, int c) { return r * 256 + ((c ^ (r & 15)) << 4); }

// acc[j] += the tile's 32 slots (A rows arow, this lane's of the loads) times
// row group j's rows (b0, b1: row lane % 32) over all G groups; bs: the lane's
// own row (its scales and zeros).
template <bool HAS_Z, int USE>
__device__ __forceinline__ void gemm_tile_light(const uint16_t *arow, const BRow &b0, const BRow &b1, const BRow &bs,
                                                int G, int lane, f32x16 (&acc)[2]) {
    __shared__ __align__(16) unsigned char a0[LIGHT_A], a1[LIGHT_A];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), l32 = lane % 32, lh = lane / 32;
    struct WR {
        uint4 w0[2], w1[2];  // 64-K halves of the group
        uint16_t s;
        uint32_t z;
    };
    // wave w moves rows 4 w .. 4 w + 3 (lane: row 4 w + lane / 16, slot lane % 16)
    const int ac = ((lane % 16) ^ ((wave * 4 + lane / 16) & 15)) * 8;
    auto issue = [&](int g, unsigned char *dst, WR &r) {
        g = min(g, G - 1);  // past the end: a valid (unused) one
        __builtin_amdgcn_global_load_lds(arow + g * QGROUP + ac, dst + wave * 1024, 16, 0, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            r.w0[h] = b0.w[g * 64 + (h * 2 + lh) * 16];
            r.w1[h] = b1.w[g * 64 + (h * 2 + lh) * 16];
        }
        r.s = bs.s[(g >> 2) * 64 + (g & 3)];
        if constexpr (HAS_Z) r.z = bs.z[(g >> 2) * 8];
    };
    auto compute = [&](const unsigned char *a, const WR &r, int g) {
        uint32_t s = r.s, z = HAS_Z ? r.z : 0u, sv[2], zv[2] = {8u, 8u};
        asm volatile("" : "+v"(s), "+v"(z));  // taken here, not at their loads
        split_halves(s * 0x10001u, sv[0], sv[1]);
        if constexpr (HAS_Z) split_halves(((z >> (bs.zs + 4 * (g & 3))) & 0xfu) * 0x10001u, zv[0], zv[1]);
        else zv[0] = zv[1] = 0x80008u;
        h2 zl[2], zh[2], s2[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            zl[j] = __builtin_bit_cast(h2, zv[j] | 0xe400e400u);         // -(1024 + z)
            zh[j] = __builtin_bit_cast(h2, (zv[j] << 4) + 0xd400d400u);  // -(64 + z)
            s2[j] = __builtin_bit_cast(h2, sv[j]);
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {  // 16-K steps: 64-K half t / 4, word t % 4
            const uint4 af = *reinterpret_cast<const uint4 *>(a + light_swz(l32, (t / 4) * 8 + t % 4 + 4 * lh));
            const uint4 &w0 = r.w0[t / 4], &w1 = r.w1[t / 4];
            auto word = [&](const uint4 &w) { return t % 4 == 0 ? w.x : t % 4 == 1 ? w.y : t % 4 == 2 ? w.z : w.w; };
            acc[0] = mfma32<F16>(af, dequant8_light(word(w0), zl[0], zh[0], s2[0]), acc[0]);
            acc[1] = mfma32<F16>(af, dequant8_light(word(w1), zl[1], zh[1], s2[1]), acc[1]);
        }
    };
    WR w0, w1;
    issue(0, a0, w0);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](int g, const unsigned char *a, const WR &cur, unsigned char *an, WR &next) {
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_below<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(g + 1, an, next);
        __builtin_amdgcn_sched_barrier(0);
        compute(a, cur, g);
    };
    int g = 0;
    for (; g + 2 <= G; g += 2) {
        step(g, a0, w0, a1, w1);
        step(g + 1, a1, w1, a0, w0);
    }
    if (g < G) step(g, a0, w0, a1, w1);
    wait_vm_below<0>();
    __builtin_amdgcn_s_barrier();  // every wave is done with the buffers, and its loads into them have landed
}

// The lane index as a value the compiler cannot see through: the epilogue's
// per-lane addresses are then formed after the loop, not held across it.
__device__ __forceinline__ int light_lane() {
    int l = int(threadIdx.x) % WAVE;
    asm volatile("" : "+v"(l));
    return l;
}

// Grid (column blocks, list entries, 5): the z-th block of an entry of up to
// 160 slots takes its z-th 32 slots. Entries above 32 are experts far above the
// average; blocks past an entry's slots exit, after every first block.
// gate/up: wave w holds the gate and the up rows of columns j0 + 32 w .. + 31
// (groups 0 and 1), so h = silu(g) * u is formed in the wave.
template <bool HAS_Z>
__device__ __forceinline__ void gate_up_light(const GateUpTile &a, int e, int base, int mc) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = light_lane(), G = a.H / QGROUP;
    const int ar = min(wave * 4 + lane / 16, mc - 1), col0 = int(blockIdx.x) * 256 + wave * 32;
    const int64_t wrow = int64_t(e) * a.F + min(col0 + lane % 32, a.F - 1);
    const BRow bg(a.gw, a.gs, a.gz, wrow, G), bu(a.uw, a.us, a.uz, wrow, G);
    const bool up = lane >= 32;
    const BRow bs(a.gw, up ? a.us : a.gs, up ? a.uz : a.gz, wrow, G);
    f32x16 acc[2] = {};
    gemm_tile_light<HAS_Z, 0>(a.xh + int64_t(a.pair_tok[base + ar]) * a.H, bg, bu, bs, G, lane, acc);
    const int lo = light_lane(), c = col0 + lo % 32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = (r / 4) * 8 + lo / 32 * 4 + r % 4;
        if (m < mc && c < a.F) a.h[int64_t(base + m) * a.F + c] = f32_to_f16_sat(silu_mul(acc[0][r], acc[1][r]));
    }
}

template <bool HAS_Z, bool YP16>
__device__ __forceinline__ void down_light(const uint32_t *dw, const uint16_t *ds, const uint16_t *dz, int e, int base,
                                           int mc, const uint16_t *h, int H, int F, void *yp) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = light_lane(), G = F / QGROUP;
    const int ar = min(wave * 4 + lane / 16, mc - 1), n0 = int(blockIdx.x) * 512 + wave * 64;
    const int64_t row0 = int64_t(e) * H;
    const BRow b0(dw, ds, dz, row0 + min(n0 + lane % 32, H - 1), G),
        b1(dw, ds, dz, row0 + min(n0 + 32 + lane % 32, H - 1), G), bs(dw, ds, dz, row0 + min(n0 + lane, H - 1), G);
    f32x16 acc[2] = {};
    gemm_tile_light<HAS_Z, 1 + YP16>(h + int64_t(base + ar) * F, b0, b1, bs, G, lane, acc);
    const int lo = light_lane(), n = n0 + lo % 32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = (r / 4) * 8 + lo / 32 * 4 + r % 4;
        const int64_t o = int64_t(base + m) * H + n;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (m < mc && n + 32 * j < H) {
                if constexpr (YP16) static_cast<uint16_t *>(yp)[o + 32 * j] = f32_to_f16_sat(acc[j][r]);
                else static_cast<float *>(yp)[o + 32 * j] = acc[j][r];
            }
    }
}

template <bool HAS_Z>
__global__ __launch_bounds__(G_THREADS, 4) void moe_gate_up_light_kernel(GateUpTile a,
                                                                          const int32_t *__restrict__ offsets,
                                                                          const int32_t *__restrict__ tile_e,
                                                                          const int32_t *__restrict__ tile_m0,
                                                                          const int32_t *__restrict__ n_tiles) {
    const int tile = blockIdx.y;
    if (tile >= *n_tiles) return;
    const int e = tile_e[tile], m0 = tile_m0[tile], rem = offsets[e + 1] - offsets[e] - m0;
    const int base = offsets[e] + m0, M = min(tile_rows(rem, GROUPED_TILE_M), rem);
    const int c0 = int(blockIdx.z) * 32;
    if (c0 >= M) return;
    gate_up_light<HAS_Z>(a, e, base + c0, min(32, M - c0));
}

template <bool HAS_Z, bool YP16>
__global__ __launch_bounds__(G_THREADS, 4) void moe_down_light_kernel(
    const uint32_t *__restrict__ dw, const uint16_t *__restrict__ ds, const uint16_t *__restrict__ dz,
    const int32_t *__restrict__ offsets, const int32_t *__restrict__ tile_e, const int32_t *__restrict__ tile_m0,
    const int32_t *__restrict__ n_tiles, const uint16_t *__restrict__ h, int H, int F, void *__restrict__ yp) {
    const int tile = blockIdx.y;
    if (tile >= *n_tiles) return;
    const int e = tile_e[tile], m0 = tile_m0[tile], rem = offsets[e + 1] - offsets[e] - m0;
    const int base = offsets[e] + m0, M = min(tile_rows(rem, GROUPED_TILE_M), rem);
    const int c0 = int(blockIdx.z) * 32;
    if (c0 >= M) return;
    down_light<HAS_Z, YP16>(dw, ds, dz, e, base + c0, min(32, M - c0), h, H, F, yp);
}

// Up to 7 tokens per expert on average: the light kernels, where their gate/up
// blocks give most CUs two (elsewhere a block waits for its groups one by one;
// the longer K, the more). Same box, both expert GEMMs, tiles of up to 160
// slots against these: 256 experts of 4096 / 1536, top 8, uneven loads, 2
// tokens per expert 408 -> 371 us, 5 468 -> 445; 256 of 2048 / 1152, 6.5 per
// expert 223 -> 207; 128 of 4096 / 1024 with zeros, 5 per expert 190 -> 174; at 8
// per expert gains and losses balance (256 of 3072 / 896 267 -> 275), at 19 they
// lose 11%; 64 of 4096 / 768, 5 per expert 89 -> 93.
static bool light_load(int T, int topk, int E, int H, int F) {
    const int64_t fill = int64_t((F + 255) / 256) * E * 4096 / H;  // gate/up blocks, at 4096 K
    return int64_t(T) * topk <= int64_t(7) * E && fill >= 320;
}

void launch_moe_grouped(const MoeGroupedArgs &a, hipStream_t s) {
    // bf16 rows through the fp16 pre-pass into the workspace; fp16 rows as they are
    const uint16_t *xh = a.x;
    if (!a.x_f16) {
        uint16_t *w = static_cast<uint16_t *>(a.ws);
        launch_x_to_f16(a.x, a.H, a.T, a.H, w, s);
        xh = w;
    }
    const int max_tiles = a.T * a.topk / -GROUPED_TILE_M + a.E;
    const dim3 g1(unsigned((a.F + 255) / 256), unsigned(max_tiles)), g2(unsigned((a.H + 511) / 512), unsigned(max_tiles));
    const GateUpTile gu{a.gw, a.uw, a.gs, a.gz, a.us, a.uz, a.pair_tok, xh, a.H, a.F, a.h};
    if (light_load(a.T, a.topk, a.E, a.H, a.F)) {
        // (an entry has at most T slots)
        const unsigned nz = unsigned(a.T < 160 ? (a.T + 31) / 32 : 5);
        const dim3 l1(g1.x, g1.y, nz), l2(g2.x, g2.y, nz);
        auto gate_up = a.gz ? moe_gate_up_light_kernel<true> : moe_gate_up_light_kernel<false>;
        gate_up<<<l1, G_THREADS, 0, s>>>(gu, a.offsets, a.tile_e, a.tile_m0, a.n_tiles);
        auto down = a.dz ? (a.yp_f16 ? moe_down_light_kernel<true, true> : moe_down_light_kernel<true, false>)
                         : (a.yp_f16 ? moe_down_light_kernel<false, true> : moe_down_light_kernel<false, false>);
        down<<<l2, G_THREADS, 0, s>>>(a.dw, a.ds, a.dz, a.offsets, a.tile_e, a.tile_m0, a.n_tiles, a.h, a.H, a.F, a.yp);
        return;
    }
    if (a.gz) moe_gate_up_gemm_kernel<true><<<g1, G_THREADS, 0, s>>>(gu, a.offsets, a.tile_e, a.tile_m0, a.n_tiles);
    else moe_gate_up_gemm_kernel<false><<<g1, G_THREADS, 0, s>>>(gu, a.offsets, a.tile_e, a.tile_m0, a.n_tiles);
    auto down = [&](auto kern) {
        kern<<<g2, G_THREADS, 0, s>>>(a.dw, a.ds, a.dz, a.offsets, a.tile_e, a.tile_m0, a.n_tiles, a.h, a.H, a.F, a.yp);
    };
    if (a.dz) {
        if (a.yp_f16) down(moe_down_gemm_kernel<true, true>);
        else down(moe_down_gemm_kernel<true, false>);
    } else {
        if (a.yp_f16) down(moe_down_gemm_kernel<false, true>);
        else down(moe_down_gemm_kernel<false, false>);
    }
}

}  // namespace qwq4
