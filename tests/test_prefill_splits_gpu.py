"""Short chunks after long windows: the launches whose key ranges are split over
several workgroups, at the window lengths and chunk sizes where the number of
splits changes, wrapped windows and grouped heads among them.  f32 and
split-bf16 within 1e-4 of the f64 oracle, bf16 within 2e-2 (the bounds of
test_prefill_gpu.py; the fold adds one f32 rounding per split)."""
import numpy as np
import pytest
import torch

import oracle
import sts_attn
from cases import prefill_inputs, scale_for
from test_prefill_gpu import TOL_F32, dev, host, run, tol
from test_workspace_gpu import _stream_pool, fresh_stream  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu

F32, BF16, SPLIT = (sts_attn.PREC_F32, sts_attn.PREC_BF16_MFMA, sts_attn.PREC_F32_SPLIT_BF16)


# H, D, M, cached rows, chunk rows, first slot.  One block more or less than the
# six that a split has to save; a last block of one key; tiles of one query;
# more splits than sixteen would give; windows that wrap inside a split.
CASES = [(4, 128, 1200, 1100, 1, 700), (4, 128, 1200, 1000, 33, 900), (8, 64, 900, 800, 65, 850),
         (32, 128, 520, 488, 24, 100), (32, 128, 600, 488, 25, 590), (32, 128, 513, 512, 1, 0),
         (2, 128, 3000, 2930, 64, 2999), (1, 64, 2200, 2100, 100, 3), (16, 128, 1600, 1400, 130, 1599),
         (3, 128, 400, 381, 3, 0)]


@pytest.mark.parametrize("prec", [F32, BF16, SPLIT])
@pytest.mark.parametrize("H,D,M,cached,S,start", CASES)
def test_split_windows(gpu, H, D, M, cached, S, start, prec):
    print(f"prefill H={H} D={D} cached={cached} S={S} start={start} prec={prec}", flush=True)
    q, kc, vc = prefill_inputs(H + cached + S, H, D, M, cached, S, start)
    L, scale = cached + S, scale_for(D)
    got = run(q, kc, vc, start, L, scale, prec)
    ref = oracle.prefill_f64(q, kc, vc, start, L, scale)
    assert np.abs(got - ref).max() < tol(prec)
    np.testing.assert_array_equal(run(q, kc, vc, start, L, scale, prec), got)
    if prec == BF16:
        k16, v16 = dev(kc).bfloat16(), dev(vc).bfloat16()
        mir = sts_attn.prefill_attention_bf16kv(dev(q), k16, v16, start, L, scale)
        np.testing.assert_array_equal(host(mir), got)


@pytest.mark.parametrize("prec", [F32, BF16])
def test_captured_with_a_smaller_workspace(gpu, prec):
    """A chunk captured on a stream that ran only a short window before (or, the
    bf16 kernel, nothing at all): the launch makes do with the splits it has
    room for, and every replay gives the eager call's result within rounding."""
    H, D, M, cached, S, start = 8, 128, 2600, 2500, 24, 77
    q, kc, vc = prefill_inputs(5, H, D, M, cached, S, start)
    scale = scale_for(D)
    ref = oracle.prefill_f64(q, kc, vc, start, cached + S, scale)
    qd, kd, vd, out = dev(q), dev(kc), dev(vc), torch.empty((S, H, D), device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    if prec == F32:
        sts_attn.prefill_attention(qd, kd, vd, start, S + 3, scale, prec, out=out, stream=s)
        s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        sts_attn.prefill_attention(qd, kd, vd, start, cached + S, scale, prec, out=out, stream=s)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        assert np.abs(host(out) - ref).max() < tol(prec)
        eager = sts_attn.prefill_attention(qd, kd, vd, start, cached + S, scale, prec)
        assert np.abs(host(eager) - ref).max() < tol(prec)


def test_grouped_heads_split(gpu):
    """Grouped-query prefill of a short chunk equals the same call on the
    expanded heads bit for bit (each query head has its own tiles)."""
    Hk, G, D, M, cached, S = 2, 4, 128, 1500, 1300, 20
    q, kc, vc = prefill_inputs(9, Hk * G, D, M, cached, S, 0)
    kc, vc = kc[:Hk], vc[:Hk]
    rows = lambda c: dev(np.ascontiguousarray(c[:, :cached].transpose(1, 0, 2))[None])
    new = lambda c: dev(np.ascontiguousarray(c[:, cached:cached + S].transpose(1, 0, 2)))
    outs = []
    for heads, rep in ((Hk, 1), (Hk * G, G)):
        k, v = np.repeat(kc, rep, 0), np.repeat(vc, rep, 0)
        c = sts_attn.KVCache(M, heads, D, n_heads=Hk * G)
        c.update(rows(k), rows(v))
        outs.append(host(c.prefill(dev(q), new(k), new(v), scale_for(D), F32)))
    np.testing.assert_array_equal(outs[0], outs[1])


# H, D, M, cached rows, chunk rows, first slot: short chunks whose last block
# leaves a key slice empty, wrapped windows, and long chunks of few heads, where
# a split's only block lies past the window of some of its tile's queries.
@pytest.mark.parametrize("prec", [BF16, SPLIT])
@pytest.mark.parametrize("H,D,M,cached,S,start", [
    (32, 128, 3000, 2500, 24, 100), (4, 128, 1200, 1100, 1, 700), (8, 64, 900, 800, 65, 850),
    (2, 128, 3000, 2930, 64, 2999), (1, 64, 800, 0, 800, 3), (2, 128, 1000, 30, 900, 970)])
def test_splits_round_as_one(gpu, fresh_stream, H, D, M, cached, S, start, prec):
    """The splits' weights are rounded relative to the base that one workgroup
    walking the whole tile has, so a launch with splits differs from one without
    (a captured one on a stream that has no workspace) by its f32 sums alone:
    about 2^-22 of the result, and a weight next to a rounding boundary now and
    then, where bases of each split's own are 2e-3 apart (bf16)."""
    print(f"prefill H={H} D={D} cached={cached} S={S} start={start} prec={prec}", flush=True)
    q, kc, vc = prefill_inputs(H + cached + S, H, D, M, cached, S, start)
    scale = scale_for(D)
    qd, kd, vd, out = dev(q), dev(kc), dev(vc), torch.empty((S, H, D), device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=fresh_stream):
        sts_attn.prefill_attention(qd, kd, vd, start, cached + S, scale, prec, out=out,
                                   stream=fresh_stream)
    ref = oracle.prefill_f64(q, kc, vc, start, cached + S, scale)
    split = host(sts_attn.prefill_attention(qd, kd, vd, start, cached + S, scale, prec))
    assert np.abs(split - ref).max() < tol(prec)
    for _ in range(2):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        one = host(out)
        d = np.linalg.norm(split.astype(np.float64) - one) / np.linalg.norm(one)
        print(f"  splits against one: {d:.2e}", flush=True)
        assert d <= 5e-5
