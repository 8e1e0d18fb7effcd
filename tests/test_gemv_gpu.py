"""q4 GEMV (qw_q4_gemv) against the CPU oracle (decode projections, LM head)."""
import numpy as np
import pytest

import qwq4
from qwq4 import synth
from _gpu_util import TOL, bf16_err_ok, host, rel_err, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(256, 512), (384, 128), (4096, 4096), (12288, 4096), (4096, 6144), (1536, 4096), (4096, 1536)]


def _setup(dev, N, K, M, zeros=True, seed=11):
    W, S, Z = synth.q4_weights(seed, f"w{N}x{K}", N, K, zeros)
    xb, xf = synth.acts(seed, f"x{M}x{K}", M, K)
    dW, dS, dZ = qwq4.tile(to_dev(W, dev), to_dev(S, dev), to_dev(Z, dev), N, K)
    return (W, S, Z, xb, xf), (dW, dS, dZ, to_dev(xb, dev))


@pytest.mark.parametrize("N,K", SHAPES)
@pytest.mark.parametrize("M", [1, 2, 4, 6, 8])
def test_gemv_fp32(gpu, oracle, N, K, M):
    print(f"gemv N={N} K={K} M={M}", flush=True)
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M)
    y = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M))
    r = oracle.q4_linear(W, S, Z, N, K, xf)
    assert rel_err(y, r) <= TOL


@pytest.mark.parametrize("N,K", [(12288, 4096), (4096, 6144)])
@pytest.mark.parametrize("M", [3, 5, 7])
def test_gemv_odd_batches(gpu, oracle, N, K, M):
    """Batches between the benchmarked ones (packed corrections with clamped
    rows, register or direct activation staging)."""
    print(f"gemv odd N={N} K={K} M={M}", flush=True)
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M, seed=13)
    y = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M))
    r = oracle.q4_linear(W, S, Z, N, K, xf)
    assert rel_err(y, r) <= TOL


@pytest.mark.parametrize("M,K", [(1, 2048), (8, 2048), (16, 2048), (17, 2048), (32, 2048), (32, 6144), (13, 640)])
def test_gemv_symmetric_and_wide(gpu, oracle, M, K):
    N = 1024
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M, zeros=False)
    y = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M))
    r = oracle.q4_linear(W, S, None, N, K, xf)
    assert rel_err(y, r) <= TOL


def test_gemv_bf16_out_is_rne_of_fp32(gpu, oracle):
    N, K, M = 4096, 4096, 4
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M)
    y32 = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M))
    y16 = qwq4.gemv(dW, dS, dZ, dx, N, K, M, y_bf16=True)
    bits = host(y16).view(np.uint32) >> 16
    assert np.array_equal(bits.astype(np.uint16), synth.bf16_bits(y32))
    assert bf16_err_ok(host(y16), oracle.q4_linear(W, S, Z, N, K, xf))


@pytest.mark.parametrize("M", [1, 2, 4, 6, 8])
def test_gemv_lm_head(gpu, oracle, M):
    """The LM head at every benchmarked batch: batches 4-8 run the persistent
    prefetching kernel (blocks take items grid-stride), 1-2 one item per
    block over many rounds."""
    N, K = 151936, 4096
    print(f"gemv lm head M={M}", flush=True)
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M)
    y = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M, y_bf16=True))
    r = oracle.q4_linear(W, S, Z, N, K, xf)
    assert bf16_err_ok(y, r)


@pytest.mark.parametrize("N,K,rpg,M", [(1296, 1024, 324, 1), (1296, 1024, 324, 8), (12288, 4096, 3076, 1),
                                        (12288, 4096, 3076, 8), (4096, 6144, 2048, 4), (2000, 512, 130, 3),
                                        (4096, 4096, 64, 32)])
def test_gemv_row_slices(gpu, oracle, N, K, rpg, M):
    """gemv_rows' row grouping (rpg: row n reads activation slice n // rpg,
    src/kernels/gemv.hip:16-17) on q4 weights: the engine's hyper-connection
    shape (4 slices of 324 rows: tiles straddle two slices), config 2's
    4096->12288 in 4 slices of 3076 rows (not a multiple of 16) at batches 1
    and 8, slices of whole tiles, and 64 slices at batch 32 (two launches
    per slice). Rows strided over every slice, accumulated into y; against
    the oracle; rows past N untouched; each row equal, bit for bit, to the
    ungrouped GEMV of its own slice."""
    import torch
    print(f"gemv rpg N={N} K={K} rpg={rpg} M={M}", flush=True)
    ns = (N + rpg - 1) // rpg
    W, S, Z = synth.q4_weights(15, f"r{N}x{K}", N, K)
    xs = ns * K + 8
    xb, xf = synth.acts(15, f"rx{M}x{xs}", M, xs)
    dW, dS, dZ = qwq4.tile(to_dev(W, gpu), to_dev(S, gpu), to_dev(Z, gpu), N, K)
    dx = to_dev(xb, gpu)
    y = torch.full((M, N + 16), 0.5, dtype=torch.float32, device=gpu)
    qwq4.gemv(dW, dS, dZ, dx, N, K, M, y=y, accumulate=True, xs=xs, ys=N + 16, rpg=rpg)
    yh = host(y)
    assert np.all(yh[:, N:] == 0.5)
    ref = oracle.q4_linear(W, S, Z, N, K, xf[:, :ns * K], rpg=rpg) + 0.5
    assert rel_err(yh[:, :N], ref) <= TOL
    # each slice's rows equal the plain GEMV of that slice (same arithmetic)
    for sl in sorted({0, ns - 1, ns // 2}):
        y1 = host(qwq4.gemv(dW, dS, dZ, dx[:, sl * K:].contiguous(), N, K, M))
        r0, r1 = sl * rpg, min(N, (sl + 1) * rpg)
        assert np.array_equal((y1[:, r0:r1] + np.float32(0.5)).view(np.uint32), yh[:, r0:r1].view(np.uint32))


def test_gemv_rows_independent_bit_exact(gpu):
    N, K, M = 2048, 4096, 8
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M)
    y8 = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M))
    for m in (0, 5, 7):
        y1 = host(qwq4.gemv(dW, dS, dZ, dx[m:m + 1].contiguous(), N, K, 1))
        assert np.array_equal(y1[0].view(np.uint32), y8[m].view(np.uint32))


def test_gemv_strides_accumulate_and_guard(gpu, oracle):
    import torch
    N, K, M = 1008, 1024, 3   # N not a multiple of 128
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M)
    xs = K + 64
    xpad = torch.zeros((M, xs), dtype=torch.int16, device=gpu)
    xpad[:, :K] = dx
    ys = N + 24
    y = torch.full((M, ys), 12345.0, device=gpu)
    y[:, :N] = 1.5
    qwq4.gemv(dW, dS, dZ, xpad, N, K, M, y=y, accumulate=True, xs=xs, ys=ys)
    yh = host(y)
    assert np.all(yh[:, N:] == 12345.0)  # no stray writes past N
    r = oracle.q4_linear(W, S, Z, N, K, xf) + 1.5
    assert rel_err(yh[:, :N], r) <= TOL


def test_gemv_special_inputs(gpu, oracle):
    import torch
    N, K = 512, 1024
    W, S, Z = synth.q4_weights(12, "sp", N, K)
    dW, dS, dZ = qwq4.tile(to_dev(W, gpu), to_dev(S, gpu), to_dev(Z, gpu), N, K)
    x = np.zeros((2, K), np.float32)
    x[1, 777] = 1.0
    y = host(qwq4.gemv(dW, dS, dZ, to_dev(synth.bf16_bits(x), gpu), N, K, 2))
    assert np.all(y[0] == 0)
    deq = oracle.q4_dequant(W, S, Z, N, K)
    assert np.array_equal(y[1], deq[:, 777])  # one-hot: a column, exactly


def _random_shapes(n, seed=2024):
    r = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        out.append((16 * int(r.integers(1, 641)), 128 * int(r.integers(1, 65)), int(r.integers(1, 33)),
                    bool(r.integers(0, 2)), bool(r.integers(0, 2))))
    return out


@pytest.mark.parametrize("N,K,M,zeros,y_bf16", _random_shapes(16))
def test_gemv_random_shapes(gpu, oracle, N, K, M, zeros, y_bf16):
    """Seeded random shapes (N a multiple of 16 up to 10240, K a multiple of
    128 up to 8192, batch 1-32, with and without zeros, fp32 or bf16 out):
    exercises the launch-shape choices (K split, block width, register or
    direct staging, one round or persistent, row-split launches) against
    the oracle."""
    print(f"gemv random N={N} K={K} M={M} zeros={zeros} bf16={y_bf16}", flush=True)
    (W, S, Z, xb, xf), (dW, dS, dZ, dx) = _setup(gpu, N, K, M, zeros=zeros, seed=N + K + M)
    y = host(qwq4.gemv(dW, dS, dZ, dx, N, K, M, y_bf16=y_bf16))
    r = oracle.q4_linear(W, S, Z if zeros else None, N, K, xf)
    if y_bf16:
        assert bf16_err_ok(y, r)
    else:
        assert rel_err(y, r) <= TOL


@pytest.mark.gpu
def test_read_probe_runs():
    """The measurement aid the bench times beside the GEMV: launches and
    rejects sizes that are not whole 32 KB blocks."""
    import torch
    t = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    qwq4.read_probe(t)
    qwq4.read_probe()
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        qwq4.read_probe(t[:1000])


# K whose group count leaves the last wave a part of its chunk (5, 13, 29, 43
# groups), more than 16 chunks (86 groups: two passes per wave), staged rows
# that end inside a wave instruction (K / 8 not a multiple of 64) and rows
# shorter than one (K = 384); N giving one and several subtiles per block.
@pytest.mark.parametrize("K", [384, 640, 1664, 3712, 5504, 11008])
@pytest.mark.parametrize("N,M,f16", [(16, 1, False), (1040, 5, True), (4112, 3, False), (528, 17, False), (4128, 16, True)])
def test_gemv_ragged_k(gpu, oracle, N, K, M, f16):
    import torch
    print(f"gemv ragged N={N} K={K} M={M} f16={f16}", flush=True)
    W, S, Z = synth.q4_weights(K + N, f"rk{N}x{K}", N, K)
    _, xf = synth.acts(K + M, f"rkx{M}x{K}", M, K)
    dW, dS, dZ = qwq4.tile(to_dev(W, gpu), to_dev(S, gpu), to_dev(Z, gpu), N, K)
    x = torch.from_numpy(xf).to(gpu).to(torch.float16 if f16 else torch.bfloat16)
    xf = host(x.float())
    y = torch.full((M, N), 7.0, dtype=torch.float32, device=gpu)
    qwq4.gemv(dW, dS, dZ, x, N, K, M, y=y)
    assert rel_err(host(y), oracle.q4_linear(W, S, Z, N, K, xf)) <= 1e-5  # fp32 sums of exact products


def _staged_fits(M, K):
    """Whether a batch's rows fit the staging LDS (gemv_fits, q4_gemv.hip): else 9 to 32 rows are streamed."""
    G = K // 128
    gpk = 4 * -(-G // 64)
    ks = -(-G // gpk)
    nw = next((w for w in (8, 12, 16) if w % ks == 0), 12 if 8 < ks <= 12 else 16)
    waves = nw // ks * ks
    stride = K // 8 | 1 if K // 8 >= 64 else K // 8
    return -(-M * stride // 64) * 1024 + 2 * (waves - waves // ks) * (1 if M <= 16 else 2) * 1024 <= 160 * 1024


# Rows streamed in K groups (batches of 9 to 32 whose rows do not fit LDS). Up to
# 16 rows: 12 and 16 parts, parts longer than a chunk, a last part of 3 groups, and
# chained blocks (N above 48 Ki) with an even and an odd number of parts. Above: the
# 16-row blocks apart (N up to 8 Ki), together with one and with two parts per wave,
# chained (N above 32 Ki). Weight rows off every block size.
@pytest.mark.parametrize("N,K,M", [(1040, 6144, 12), (16, 11008, 16), (2064, 7040, 16), (65584, 6144, 13), (49232, 5504, 15),
                                   (4112, 5504, 17), (528, 4096, 32), (3076 // 16 * 16, 3712, 25),
                                   (8208, 3712, 32), (12304, 4096, 21), (8208, 6144, 32), (8224, 7040, 19),
                                   (32848, 4096, 21), (32864, 2560, 32), (32784, 8320, 17)])
@pytest.mark.parametrize("f16,zeros", [(False, True), (True, True), (False, False), (True, False)])
def test_gemv_wide(gpu, oracle, N, K, M, f16, zeros):
    import torch
    print(f"gemv wide N={N} K={K} M={M} f16={f16} zeros={zeros}", flush=True)
    assert M > 8 and not _staged_fits(M, K)
    g = torch.Generator(device=gpu)
    g.manual_seed(N + K)
    W = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device=gpu, dtype=torch.int32)
    S = (torch.randn((N, K // 128), generator=g, device=gpu) * 0.02).abs().to(torch.float16)
    Z = torch.randint(-2**31, 2**31, (N, (K // 128 + 7) // 8), generator=g, device=gpu, dtype=torch.int32) if zeros else None
    d = qwq4.tile(W, S, Z, N, K)
    x = torch.full((M, K + 64), float("nan"), device=gpu).to(torch.float16 if f16 else torch.bfloat16)
    x[:, :K] = torch.randn((M, K), generator=g, device=gpu).to(x.dtype)
    y = torch.full((M, N + 3), 7.0, dtype=torch.float32, device=gpu)
    qwq4.gemv(*d, x, N, K, M, y=y)
    assert bool((y[:, N:] == 7.0).all())
    rows = np.unique(np.r_[0, N - 1, np.random.default_rng(N).choice(N, min(N, 512), replace=False)])
    np_ = lambda t, v: None if t is None else host(t[torch.from_numpy(rows).to(gpu)]).view(v)
    ref = oracle.q4_linear_f64(np_(W, np.uint32), np_(S, np.uint16), np_(Z, np.uint32), len(rows), K, host(x[:, :K].float().contiguous()))
    assert rel_err(host(y)[:, rows], ref) <= 1e-5  # fp32 sums of exact products
    acc = y.clone()
    qwq4.gemv(*d, x, N, K, M, y=acc, accumulate=True)
    assert torch.equal(acc[:, :N], 2 * y[:, :N])
    yb = torch.zeros((M, N), dtype=torch.bfloat16, device=gpu)
    qwq4.gemv(*d, x, N, K, M, y=yb, y_bf16=True)
    assert torch.equal(yb, y[:, :N].to(torch.bfloat16))


def test_gemv_wide_row_slices(gpu):
    """Rows grouped over activation slices: each equals the ungrouped product
    with its slice, bit for bit, whichever block sizes its slice alone would get."""
    import torch
    N, K, M, rpg = 36864, 4096, 20, 3076
    print("gemv wide row slices", flush=True)
    W, S, Z = synth.q4_weights(93, "wrs", N, K)
    d = qwq4.tile(to_dev(W, gpu), to_dev(S, gpu), to_dev(Z, gpu), N, K)
    ns = -(-N // rpg)
    x = torch.randn((M, ns * K), device=gpu).to(torch.bfloat16)
    y = qwq4.gemv(*d, x, N, K, M, rpg=rpg)
    for sl in (0, 5, ns - 1):
        whole = qwq4.gemv(*d, x[:, sl * K:(sl + 1) * K], N, K, M)
        assert torch.equal(y[:, sl * rpg:(sl + 1) * rpg], whole[:, sl * rpg:(sl + 1) * rpg])


# Batches on both sides of every change of kernel (staged, streamed split and
# chained): parts that cover K exactly and not, one and two parts per wave.
@pytest.mark.parametrize("N,K,f16,zeros", [(1040, 4096, False, True), (4112, 6144, True, True), (4112, 6144, False, False),
                                           (12304, 4096, True, False), (8208, 5504, False, True), (32848, 4096, False, True),
                                           (32864, 2560, True, True), (49232, 7040, False, True), (1040, 8320, True, True)])
def test_gemv_rows_independent_of_batch(gpu, N, K, f16, zeros):
    """A token row's result is the same bits in every batch of 1 to 32 rows, infinities and NaN in
    other rows and in its own included."""
    import torch
    print(f"gemv rows independent N={N} K={K} f16={f16} zeros={zeros}", flush=True)
    assert not _staged_fits(32, K)
    g = torch.Generator(device=gpu)
    g.manual_seed(N + K)
    W = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device=gpu, dtype=torch.int32)
    S = (torch.randn((N, K // 128), generator=g, device=gpu) * 0.02).abs().to(torch.float16)
    Z = torch.randint(-2**31, 2**31, (N, (K // 128 + 7) // 8), generator=g, device=gpu, dtype=torch.int32) if zeros else None
    d = qwq4.tile(W, S, Z, N, K)
    x = torch.randn((32, K), generator=g, device=gpu).to(torch.float16 if f16 else torch.bfloat16)
    x[2, 130], x[20, K - 1], x[30, 0] = float("inf"), float("-inf"), float("nan")
    y32 = qwq4.gemv(*d, x, N, K, 32)
    ok = torch.ones(32, dtype=torch.bool, device=gpu)
    ok[[2, 20, 30]] = False
    assert bool(torch.isfinite(y32[ok]).all()) and not bool(torch.isfinite(y32[~ok]).any())
    for M in (1, 2, 4, 8, 9, 11, 12, 16, 17, 20):
        for m0 in {0, 32 - M}:
            y, r = qwq4.gemv(*d, x[m0:m0 + M], N, K, M), y32[m0:m0 + M]
            assert torch.equal(torch.isnan(y), torch.isnan(r)), (M, m0)
            assert torch.equal(y.nan_to_num(nan=0.0).view(torch.int32), r.nan_to_num(nan=0.0).view(torch.int32)), (M, m0)


@pytest.mark.parametrize("G", [512, 530, 631])
def test_gemv_longest_rows(gpu, oracle, G):
    """K of 64 Ki, where a single row fits the staging LDS, and above, where none does beside the K parts'
    sums: one row against the oracle, batches the same bits."""
    import torch
    N, K = 48, 128 * G
    print(f"gemv longest rows K={K}", flush=True)
    W, S, Z = synth.q4_weights(G, "long", N, K)
    _, xf = synth.acts(G, "longx", 10, K)
    d = qwq4.tile(to_dev(W, gpu), to_dev(S, gpu), to_dev(Z, gpu), N, K)
    x = torch.from_numpy(xf).to(gpu).to(torch.bfloat16)
    y = qwq4.gemv(*d, x[:1], N, K, 1)
    assert rel_err(host(y), oracle.q4_linear_f64(W, S, Z, N, K, host(x[:1].float()))) <= 1e-5  # fp32 sums of exact products
    for M in (2, 10):
        assert torch.equal(qwq4.gemv(*d, x[:M], N, K, M)[:1], y)
