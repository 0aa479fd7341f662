"""Causal prefill attention with cache rows that are not finite: token t sees keys 0 .. pos0 + t and nothing else, so
a V or K row of inf or NaN (an f16 overflow of the KV store) leaves every earlier token as it is, bit for bit, and of
the later ones only the dims it touches.  All forms: the per-head form, the tiles shared by two and by four waves a
row group, and the per-token form of large groups."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv,hpk,M,pos", [
    (8, 3, 75, 0), (2, 1, 60, 30),          # per head, 16 tokens a workgroup
    (8, 3, 300, 0), (8, 1, 700, 45), (3, 4, 400, 100),      # 64 query rows a workgroup, tiles of 128 keys
    (32, 1, 1040, 0), (8, 4, 1100, 17),     # 128 query rows, tiles of 64 keys
    (2, 6, 60, 3)])                         # one token a workgroup
def test_later_rows_stay_out(ctx, kv, hpk, M, pos):
    H, n = kv * hpk, pos + M
    qkv = synth.normal_f32(61, 1, M * (H + 2 * kv) * 128, std=1.5)
    K = synth.normal_f32(61, 2, n * kv * 128).astype(np.float16).reshape(n, kv, 128)
    V = synth.normal_f32(61, 3, n * kv * 128).astype(np.float16).reshape(n, kv, 128)
    q, kc, vc, out = ctx.to_device(qkv), ctx.to_device(K), ctx.to_device(V), ctx.alloc(M * H * 512)

    def run(k, v):
        ctx.upload(kc, k)
        ctx.upload(vc, v)
        ctx.fill_u32(out, 0x7F7F7F7F)
        ctx.attention_prefill(q, M, kc, vc, out, pos, kv, hpk, 128)
        return ctx.download(out, np.uint32).reshape(M, kv, hpk, 128)

    want = run(K, V)
    for tok in sorted({1, 15, M // 2, M // 2 + 21, M - 1}):
        t = pos + tok
        v = V.copy()
        v[t, 0, 5] = np.inf
        v[t, 0, 70] = -np.inf
        v[t, kv - 1, 96:] = np.nan
        got = run(K, v)
        hit = np.zeros((kv, 128), bool)
        hit[0, [5, 70]] = True
        hit[kv - 1, 96:] = True
        assert np.array_equal(got[:tok], want[:tok]), tok
        later = np.moveaxis(got[tok:], 2, 1).reshape(-1, kv, 128), np.moveaxis(want[tok:], 2, 1).reshape(-1, kv, 128)
        assert np.array_equal(later[0][:, ~hit], later[1][:, ~hit]), tok
        assert not np.isfinite(later[0][:, hit].view(np.float32)).any(), tok
        k = K.copy()
        k[t, kv - 1] = np.inf
        k[t, 0, 3] = np.nan
        got = run(k, V)
        assert np.array_equal(got[:tok], want[:tok]), tok
        assert not np.isfinite(got[tok:, [0, kv - 1]].view(np.float32)).any(), tok
    for b in (q, kc, vc, out):
        b.free()
