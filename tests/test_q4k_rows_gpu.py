"""The Q4_K products for several rows at the sizes where their tiles end.

Values: within the f32 bound 1e-5 * sum_k (|w_k| + 2|dmin*min_k|) |x_k| of the
f64 product (the bound of test_q4k_gpu.py), and, over a whole result, no
further from it (2-norm) than 3e-7: f32 sums of a few thousand products in any
order stay below that (2^-24 times a small factor), operands rounded to 16
bits do not (4e-3) and two-part ones hardly (4e-6).
Infinities, NaN and sums that overflow on the way come out as the product of
the dequantised weights has them.
"""
import numpy as np
import pytest
import torch

import oracle
import sts_attn
from test_depformer_gpu import q4k_bound

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda")


def host(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def quantised(seed, N, K):
    return oracle.q4k_quantize(oracle.normal(seed, (N, K)) / np.float32(np.sqrt(K)))


def check(got, blocks, x, N, res=None):
    ref = oracle.q4k_matvec_f64(blocks, x, N)
    tol = 1e-5 * q4k_bound(blocks, x, N)
    if res is not None:
        ref = ref + res.astype(np.float64)
        tol = tol + 1e-6 * np.abs(res)
    d = got.astype(np.float64) - ref
    assert (np.abs(d) <= tol).all(), np.abs(d).max()
    assert np.linalg.norm(d) <= 3e-7 * np.linalg.norm(ref)


# Rows about the 16-row tile; weight rows about the 16-row tile and the groups
# of 2, 3, 4 and 6 tiles; K below, at and above one half super-block a wave.
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (2, 15, 256), (15, 17, 512), (16, 16, 1024),
                                   (17, 33, 768), (31, 5000, 256), (33, 4097, 512),
                                   (48, 3000, 1280), (65, 4111, 256), (5, 47, 16384),
                                   (129, 1001, 2816)])
def test_rows_edges(gpu, M, N, K):
    print(f"q4k rows M={M} N={N} K={K}", flush=True)
    blocks = quantised(M + N + K, N, K)
    x = oracle.normal(N + 3 * M, (M, K))
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    check(host(sts_attn.q4k_gemm(dev(x), w)), blocks, x, N)


# One or two rows: a weight row per 16, 32 or 64 lanes (K up to 1024, 2048,
# 4096), one or four of them a wave; with and without RMSNorm, SwiGLU, residual.
@pytest.mark.parametrize("M,N,K,norm,swiglu,res", [
    (1, 1, 256, False, False, False), (2, 30, 768, True, True, False),
    (1, 3073, 1024, True, False, True), (2, 9001, 1024, False, False, True),
    (1, 20002, 512, True, True, False), (1, 66, 1280, False, True, False),
    (2, 6003, 2048, True, False, False), (1, 1024, 2816, False, False, True),
    (2, 5001, 3072, True, False, True), (1, 2817, 4096, True, False, False),
    (2, 1500, 3328, False, True, False), (1, 515, 4352, False, False, True),
    (2, 4096, 2304, True, False, False), (2, 4097, 2304, True, False, False)])
def test_single_rows(gpu, M, N, K, norm, swiglu, res):
    print(f"q4k M={M} N={N} K={K} norm={norm} swiglu={swiglu} res={res}", flush=True)
    blocks = oracle._random_q4k_scaled(M + N + K, N, K)
    x = oracle.normal(N + M, (M, K)) * np.float32(2.0)
    alpha = (1 + 0.1 * oracle.normal(K, (K,))).astype(np.float32)
    r = oracle.normal(N + 3, (M, N)) if res else None
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    got = host(sts_attn.q4k_gemm(dev(x), w, residual=dev(r) if res else None, swiglu=swiglu,
                                 norm_alpha=dev(alpha) if norm else None, norm_eps=1e-8))
    xn = oracle.rmsnorm_wgsl(x, alpha, 1e-8) if norm else x
    y = oracle.q4k_matvec_f64(blocks, xn, N)
    b = 1e-5 * q4k_bound(blocks, xn, N)
    if swiglu:
        F = N // 2
        g, v = y[:, :F], y[:, F:]
        sig = 1 / (1 + np.exp(-g))
        want = g * sig * v
        tol = (np.abs(sig * (1 + g * (1 - sig))) * np.abs(v) * b[:, :F]
               + np.abs(g * sig) * b[:, F:] + 1e-6 * np.abs(want) + 1e-30)
    else:
        want, tol = y, b
    if res:
        want, tol = want + r, tol + 1e-6 * np.abs(r)
    d = got.astype(np.float64) - want
    assert (np.abs(d) <= tol).all(), (np.abs(d) / tol).max()
    if not norm and not swiglu:
        assert np.linalg.norm(d) <= 3e-7 * np.linalg.norm(want)


def test_single_rows_not_finite(gpu):
    N, K = 300, 1024
    blocks = oracle._random_q4k_scaled(8, N, K)
    wt = oracle.q4k_dequant(blocks, N, K).astype(np.float64)
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    x = oracle.normal(9, (2, K))
    x[0, 37] = np.inf
    x[1] = 0
    x[1, 5], x[1, K - 2] = np.float32(3e38), np.float32(-1e38)
    got = host(sts_attn.q4k_gemm(dev(x), w))
    with np.errstate(invalid="ignore"):
        want = np.where(wt[:, 37] == 0, np.nan, np.inf * np.sign(wt[:, 37]))
    np.testing.assert_array_equal(got[0], want.astype(np.float32))
    big = x[1].astype(np.float64) @ wt.T
    np.testing.assert_allclose(got[1], big, rtol=1e-5, atol=1e-5 * np.abs(big).max())


# The tiles of many rows: 64 x 128 outputs, up to 1024 rows at a time, one or
# several ranges of K.
@pytest.mark.parametrize("M,N,K,res", [(33, 1921, 16384, True), (65, 4601, 4096, False),
                                       (64, 11265, 2304, True), (130, 41001, 256, False),
                                       (1025, 1501, 1024, True), (1088, 127, 11264, False)])
def test_tiles_edges(gpu, M, N, K, res):
    print(f"q4k tiles M={M} N={N} K={K} res={res}", flush=True)
    blocks = oracle._random_q4k_scaled(M + N + K, N, K)
    x = oracle.normal(N + 3 * M, (M, K))
    x[M // 2, :K // 2] *= np.float32(1000.0)  # rows and super-blocks of other sizes
    x[M - 1] *= np.float32(1e-12)
    r = oracle.normal(N + 7, (M, N)) if res else None
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    got = host(sts_attn.q4k_gemm(dev(x), w, residual=dev(r) if res else None))
    wt = torch.from_numpy(oracle.q4k_dequant(blocks, N, K)).cuda().double()
    xd = dev(x).double()
    ref = (xd @ wt.T.contiguous()).cpu().numpy() + (r.astype(np.float64) if res else 0.0)
    tol = 1e-5 * q4k_bound(blocks, x, N) + (1e-6 * np.abs(r) if res else 0.0)
    assert (np.abs(got - ref) <= tol).all(), (np.abs(got - ref) / tol).max()
    # Row by row, the residual's own rounding aside.
    d, own = got - ref, ref - (r.astype(np.float64) if res else 0.0)
    off, norm = np.linalg.norm(d, axis=1), np.linalg.norm(own, axis=1)
    print(f"  worst row {(off / norm).max():.2e}", flush=True)
    assert (off <= 3e-7 * norm + (2.0 ** -24 * np.linalg.norm(got, axis=1) if res else 0.0)).all()
    again = host(sts_attn.q4k_gemm(dev(x), w, residual=dev(r) if res else None))
    np.testing.assert_array_equal(again, got)


def test_tiles_captured_without_workspace(gpu):
    """A stream whose workspace does not hold the tiles' operands yet: captured,
    the product runs without them; every replay gives the same values."""
    M, N, K = 128, 4096, 4096
    blocks = oracle._random_q4k_scaled(5, N, K)
    x = oracle.normal(6, (M, K))
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    xd, out = dev(x), torch.empty((M, N), device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        sts_attn.q4k_gemm(xd, w, out=out, stream=s)
    ref = oracle.q4k_matvec_f64(blocks, x, N)
    tol = 1e-5 * q4k_bound(blocks, x, N)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert (np.abs(host(out) - ref) <= tol).all()
        eager = host(sts_attn.q4k_gemm(xd, w))
        assert (np.abs(eager - ref) <= tol).all()
        for y in (host(out), eager):
            assert (np.linalg.norm(y - ref, axis=1) <= 3e-7 * np.linalg.norm(ref, axis=1)).all()


@pytest.mark.parametrize("N,K,B,res", [(4096, 1024, 3, True), (4096, 1024, 4, True),
                                       (300, 11264, 7, False), (300, 11264, 8, True),
                                       (2048, 512, 70, False)])
def test_matvec_batches(gpu, N, K, B, res):
    """Rows of a batch on either side of the batch size from which they share
    the weights: each within the bound of the f64 product."""
    blocks = quantised(N + K, N, K)
    x = oracle.normal(N + B, (B, K))
    r = oracle.normal(N + 9, (B, N)) if res else None
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    got = host(sts_attn.q4k_matmul(dev(x[:, None]), w,
                                   residual=dev(r[:, None]) if res else None))[:, 0]
    check(got, blocks, x, N, r)


# (40, 2400, 16384): the tiles of many rows, their K in several ranges;
# (40, 41001, 1024): in one.
@pytest.mark.parametrize("M,N,K", [(3, 40, 512), (20, 700, 1024), (40, 2400, 16384),
                                   (40, 41001, 1024)])
def test_rows_not_finite(gpu, M, N, K):
    """Row 0 holds an infinity, row 1 a NaN, row 2 values whose 15-fold
    overflows though the products do not; the others are ordinary."""
    blocks = (quantised if N * K < 1 << 20 else oracle._random_q4k_scaled)(M * N + K, N, K)
    wt = oracle.q4k_dequant(blocks, N, K).astype(np.float64)
    x = oracle.normal(N + M, (M, K))
    x[0, 37] = -np.inf
    x[1, K - 1] = np.nan
    x[2] = 0
    x[2, 5] = np.float32(3e38)
    x[2, K - 2] = np.float32(-1e38)
    w = sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))
    got = host(sts_attn.q4k_gemm(dev(x), w))
    want = np.where(wt[:, 37] == 0, np.nan, -np.inf * np.sign(wt[:, 37]))
    np.testing.assert_array_equal(got[0], want.astype(np.float32))
    assert np.isnan(got[1]).all()
    big = x[2].astype(np.float64) @ wt.T
    np.testing.assert_allclose(got[2], big, rtol=1e-5, atol=1e-5 * np.abs(big).max())
    if M > 3:
        d = got[3:] - x[3:].astype(np.float64) @ wt.T
        assert (np.abs(d) <= 1e-5 * q4k_bound(blocks, x[3:], N)).all()


def test_threads_on_one_stream(gpu):
    """Two host threads with products of many rows and one with prefills whose
    key ranges are split, all on the one stream that torch gives every thread:
    each result is that of the call alone, bit for bit."""
    import threading

    M, N, K, H, D, cached, S = 128, 4096, 4096, 8, 128, 1500, 24
    g = torch.Generator(device="cuda").manual_seed(3)
    w = sts_attn.Q4KTensor.from_q4k_bytes(oracle._random_q4k_scaled(11, N, K), (N, K))
    xs = [torch.randn((M, K), generator=g, device="cuda") for _ in range(2)]
    q = torch.randn((S, H, D), generator=g, device="cuda")
    kc, vc = (torch.randn((H, cached + S, D), generator=g, device="cuda") for _ in range(2))
    calls = [lambda: sts_attn.q4k_gemm(xs[0], w), lambda: sts_attn.q4k_gemm(xs[1], w),
             lambda: sts_attn.prefill_attention(q, kc, vc, 0, cached + S, 0.09,
                                                sts_attn.PREC_BF16_MFMA)]
    alone = [c() for c in calls]
    torch.cuda.synchronize()
    start, got, errors = threading.Barrier(3), [[] for _ in calls], []

    def work(i):
        try:
            start.wait()
            for _ in range(40):
                got[i].append(calls[i]())
        except Exception as e:  # reported below, in the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(3):
        assert all(torch.equal(y, alone[i]) for y in got[i]), i


def near_zero_blocks(seed, N, K, cols):
    """Random Q4_K matrix whose even rows have dmin = 8 d and every min equal to
    its scale, and whose weights in the given columns (one or more of each
    super-block) are the ones nearest to zero: exactly zero in the even rows, less
    than half a quant step in the others (where the min is within the quants'
    range)."""
    blk = oracle._random_q4k_scaled(seed, N, K).reshape(N, K // 256, 144).copy()
    s = blk[..., 4:16]
    even = slice(0, None, 2)
    dm = np.float16(8 * float(blk[0, 0, :2].view(np.float16)[0]))
    blk[even, :, 2:4] = np.array([dm]).view(np.uint8)
    s[even, :, 4:8] = s[even, :, 0:4]
    s[even, :, 8:12] = (s[even, :, 8:12] & 15) * 17
    d = blk[..., 0:2].copy().view(np.float16)[..., 0].astype(np.float64)
    dmin = blk[..., 2:4].copy().view(np.float16)[..., 0].astype(np.float64)
    for c in cols:
        b, j, i = c // 256, c // 32 % 8, c % 32
        if j < 4:
            sc, mn = s[:, b, j] & 63, s[:, b, 4 + j] & 63
        else:
            sc = (s[:, b, 4 + j] & 15) | (s[:, b, j - 4] >> 6 << 4)
            mn = (s[:, b, 4 + j] >> 4) | (s[:, b, j] >> 6 << 4)
        with np.errstate(divide="ignore", invalid="ignore"):
            q = np.nan_to_num(np.rint(dmin[:, b] * mn / (d[:, b] * sc)), posinf=15)
        q = q.clip(0, 15).astype(np.uint8)
        byte = 16 + 32 * (j // 2) + i
        old = blk[:, b, byte]
        blk[:, b, byte] = (old & 0xF0) | q if j % 2 == 0 else (old & 0x0F) | (q << 4)
    return blk.reshape(-1)


# One and two rows; a few rows; the tiles of many rows (the last two).
@pytest.mark.parametrize("M,N,K", [(1, 515, 1024), (2, 301, 2304), (1, 130, 4096), (5, 200, 512),
                                   (13, 700, 2816), (40, 130, 5120), (64, 11265, 2304),
                                   (130, 41001, 512)])
def test_small_weights_under_large_x(gpu, M, N, K):
    """Channels of x up to 1e12 times the others at weights that are zero or
    nearly: each output is within 2e-6 of sum |w x|, 33 roundings of f32 at that
    size (a sum of thousands of terms of random sign stays below), with no
    allowance for the mins.  Sums over quants and mins apart, or x held to fewer
    bits of the largest value of its block, are off by far more."""
    print(f"q4k large channels M={M} N={N} K={K}", flush=True)
    cols = [256 * b + (37 * b + 11) % 256 for b in range(K // 256)]
    blocks = near_zero_blocks(M + N + K, N, K, cols)
    x = oracle.normal(N + 3 * M, (M, K))
    for m in range(M):
        x[m, cols] *= np.float32(10.0 ** (12 - m % 13))
    wt = torch.from_numpy(oracle.q4k_dequant(blocks, N, K)).cuda().double()
    assert (wt[::2, cols] == 0).all()
    got = host(sts_attn.q4k_gemm(dev(x), sts_attn.Q4KTensor.from_q4k_bytes(blocks, (N, K))))
    xd = dev(x).double()
    ref = (xd @ wt.T.contiguous()).cpu().numpy()
    size = (xd.abs() @ wt.abs().T.contiguous()).cpu().numpy()
    worst = (np.abs(got - ref) / size).max()
    print(f"  worst error over sum |w x|: {worst:.2e}", flush=True)
    assert worst <= 2e-6


@pytest.mark.parametrize("M,N,K", [(1, 601, 1024), (2, 601, 2304), (7, 601, 1280),
                                   (65, 11265, 2304)])
def test_unusual_headers(gpu, M, N, K):
    """Scales that no quantiser writes: d and dmin zero, of either sign, subnormal,
    the largest half, an infinity or NaN; sub-block scales and mins of 0, 1 and 63.
    Finite outputs within 2e-6 of sum |w x| (33 roundings of f32), the others as
    the dequantised weights have them."""
    print(f"q4k headers M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N)
    blk = oracle._random_q4k_scaled(M + N + K, N, K).reshape(N, K // 256, 144).copy()
    vals = np.array([0x0000, 0x8000, 0x0001, 0x83FF, 0x0400, 0x2C00, 0xAC00, 0x3C00, 0x7BFF, 0xFBFF],
                    np.uint16)
    for off in (0, 2):
        blk[..., off:off + 2] = rng.choice(vals, blk.shape[:2])[..., None].view(np.uint8)
    blk[7, 0, 0:2] = np.array([0x7C00], np.uint16).view(np.uint8)   # d = inf
    blk[9, -1, 2:4] = np.array([0x7E00], np.uint16).view(np.uint8)  # dmin = NaN
    blk[1::5, :, 4:16] = 0          # every scale and min 0
    blk[2::5, :, 4:12], blk[2::5, :, 12:16] = 1, 0x11  # 1
    blk[3::5, :, 4:16] = 0xFF       # 63
    blk[4::5, :, 4:8] = 0           # low scales 0, mins as they are
    x = oracle.normal(N + M, (M, K))
    wt = torch.from_numpy(oracle.q4k_dequant(blk.reshape(-1), N, K)).cuda().double()
    got = host(sts_attn.q4k_gemm(dev(x), sts_attn.Q4KTensor.from_q4k_bytes(blk.reshape(-1), (N, K))))
    xd = dev(x).double()
    ref = (xd @ wt.T.contiguous()).cpu().numpy()
    size = (xd.abs() @ wt.abs().T.contiguous()).cpu().numpy()
    finite = np.isfinite(ref)
    assert not finite[:, 9].any() and not finite[:, 7].any()
    assert finite[:, np.delete(np.arange(N), [7, 9])].all()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    assert (got[~finite & ~np.isnan(ref)] == ref[~finite & ~np.isnan(ref)]).all()
    off = np.abs(got[finite] - ref[finite])
    print(f"  worst error over sum |w x|: {(off / (size[finite] + 1e-300)).max():.2e}", flush=True)
    assert (off <= 2e-6 * size[finite]).all()
