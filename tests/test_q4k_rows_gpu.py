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


@pytest.mark.parametrize("M,N,K", [(3, 40, 512), (20, 700, 1024)])
def test_rows_not_finite(gpu, M, N, K):
    """Row 0 holds an infinity, row 1 a NaN, row 2 values whose 15-fold
    overflows though the products do not; the others are ordinary."""
    blocks = quantised(M * N + K, N, K)
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
        check(got[3:], blocks, x[3:], N)
