"""What the prefill attention with shared tiles keeps of its softmax weights, against 64 bits."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu

# (KV heads, heads per KV head, rows, pos): 64 query rows a workgroup on tiles of 128 keys, 128 on tiles of 64
SHAPES = [(8, 3, 512, 256), (8, 4, 1100, 1)]


def inputs(kv, hpk, M, pos, std):
    stride = (kv * hpk + 2 * kv) * 128
    qkv = synth.normal_f32(71, 1, M * stride, std=std).reshape(M, stride)
    K = synth.normal_f32(71, 2, (pos + M) * kv * 128).astype(np.float16)
    V = synth.normal_f32(71, 3, (pos + M) * kv * 128).astype(np.float16)
    return qkv, K, V


def attend(ctx, qkv, K, V, kv, hpk, pos, step):
    """`step` rows a call; 64 and fewer take the per-head form."""
    M, stride = qkv.shape
    row = kv * hpk * 512
    q, kc, vc, out = ctx.to_device(qkv), ctx.to_device(K), ctx.to_device(V), ctx.alloc(M * row)
    for m in range(0, M, step):
        n = min(step, M - m)
        qv, ov = ctx.view(q, m * stride * 4, n * stride * 4), ctx.view(out, m * row, n * row)
        ctx.attention_prefill(qv, n, kc, vc, ov, pos + m, kv, hpk, 128)
        qv.free(), ov.free()
    y = ctx.download(out).reshape(M, kv * hpk, 128).astype(np.float64)
    for b in (q, kc, vc, out):
        b.free()
    return y


@pytest.mark.parametrize("kv,hpk,M,pos", SHAPES)
def test_weights_lose_nothing_on_average(ctx, kv, hpk, M, pos):
    """V = 1: every output is the sum of the halves of P over the sum of P.  Halves rounded to nearest err to both
    sides, so the mean over half a million outputs is 1 to a few 1e-9; a half cut off instead is short by 2^-22 of
    a weight on average where its last bit counts (measured: 7e-8 in all)."""
    qkv, K, V = inputs(kv, hpk, M, pos, 1.5)
    V[:] = 1.0
    assert abs(attend(ctx, qkv, K, V, kv, hpk, pos, M).mean() - 1.0) < 2.0 ** -25


@pytest.mark.parametrize("kv,hpk,M,pos", SHAPES)
def test_no_further_off_than_the_per_head_form(ctx, kv, hpk, M, pos):
    """Small scores: weights near 1, whose exponents have an argument near 0.  The forms differ in the order of
    their sums only: to 64 bits both are about 1.3e-7 off.  The longer sums of the shared tiles (twice the keys a
    wave) may cost a factor of up to sqrt(2) where the sums are all of the error; with 2^12 in the exponent's
    argument the factor was 2."""
    qkv, K, V = inputs(kv, hpk, M, pos, 0.3)
    tiles, heads = attend(ctx, qkv, K, V, kv, hpk, pos, M), attend(ctx, qkv, K, V, kv, hpk, pos, 64)
    n = pos + M
    q, k, v = (a.astype(np.float64) for a in (qkv[:, :kv * hpk * 128].reshape(M, kv * hpk, 128),
                                              K.reshape(n, kv, 128), V.reshape(n, kv, 128)))
    seen = np.arange(n)[None] <= pos + np.arange(M)[:, None]
    err = {"tiles": 0.0, "heads": 0.0}
    for h in range(0, kv * hpk, 5):
        p = np.where(seen, np.exp(q[:, h] @ k[:, h // hpk].T / np.sqrt(128.0)), 0.0)
        ref = (p / p.sum(1, keepdims=True)) @ v[:, h // hpk]
        err["tiles"] += ((tiles[:, h] - ref) ** 2).sum()
        err["heads"] += ((heads[:, h] - ref) ** 2).sum()
    assert err["tiles"] <= 2.0 * err["heads"], err
