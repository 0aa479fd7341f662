"""Causal prefill attention where a workgroup's waves share each K/V tile (csrc/attn_flash.hip), at its edges: every
group size it takes, query rows that end inside a 32-row wave, keys that end inside a tile of 64 or 128, a cached
prefix, and the last cache row.

Tolerance: K and V are exact in f16, the query and the softmax weights are carried in two f16 halves (22 bits), the
sums are f32 over at most 2,048 keys: a few 1e-6 of the row's largest output; 1e-5 leaves a factor of about five.
A score is off by about 2^-22 of the row's largest score (its query's 22 bits, f32 accumulation), and a weight by the
same as a relative error, which counts where scores are large: four times that is added per row.  The f16 output is the f32 one rounded to nearest."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


def reference(q, k, v, pos):
    M, H, hd = q.shape
    seen = np.arange(k.shape[0])[None] <= pos + np.arange(M)[:, None]
    out, top = np.empty((M, H, hd)), np.empty((M, H))
    for h in range(H):
        s = q[:, h] @ k[:, h // (H // k.shape[1])].T / np.sqrt(hd)
        top[:, h] = np.abs(np.where(seen, s, 0.0)).max(1)
        s = np.where(seen, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ v[:, h // (H // k.shape[1])]
    return out, top


@pytest.mark.parametrize("kv,hpk,M,pos", [
    (8, 3, 171, 0),        # just past the per-head form; 513 query rows a KV head
    (8, 1, 513, 0), (8, 2, 257, 127), (8, 4, 130, 62), (3, 2, 777, 5), (1, 4, 1025, 300),
    (8, 3, 700, 1348),     # up to the last cache row
    (8, 4, 1100, 1),       # 128 query rows a workgroup
    (16, 3, 690, 63)])
def test_attention_rows_sharing_tiles(kv, hpk, M, pos):
    H, stride = kv * hpk, (kv * hpk + 2 * kv) * 128
    qkv = synth.normal_f32(41, 1, M * stride, std=1.5).reshape(M, stride)
    qkv[::7] *= np.float32(1e-3)
    qkv[3::11] *= np.float32(30.0)      # near one-hot rows
    K = synth.normal_f32(41, 2, 2048 * kv * 128).astype(np.float16)
    V = synth.normal_f32(41, 3, 2048 * kv * 128).astype(np.float16)
    with rrr.Context(0) as ctx:
        q, kc, vc = ctx.to_device(qkv), ctx.to_device(K), ctx.to_device(V)
        o32, o16 = ctx.alloc((M + 1) * H * 512), ctx.alloc((M + 1) * H * 256)
        ctx.fill_u32(o32, 0x7F7F7F7F)
        ctx.fill_u32(o16, 0x7B7B7B7B)
        ctx.attention_prefill(q, M, kc, vc, o32, pos, kv, hpk, 128)
        ctx.attention_prefill(q, M, kc, vc, o16, pos, kv, hpk, 128, out_type=rrr.F16)
        got = ctx.download(o32).reshape(M + 1, H, 128)
        half = ctx.download(o16, np.float16).reshape(M + 1, H, 128)
    assert np.all(got[M].view(np.uint32) == 0x7F7F7F7F) and np.all(half[M].view(np.uint16) == 0x7B7B)
    assert np.array_equal(half[:M].view(np.uint16), got[:M].astype(np.float16).view(np.uint16))
    n = pos + M
    ref, top = reference(qkv[:, :H * 128].reshape(M, H, 128).astype(np.float64), K.reshape(2048, kv, 128)[:n].astype(np.float64),
                         V.reshape(2048, kv, 128)[:n].astype(np.float64), pos)
    assert np.all(np.abs(got[:M] - ref).max(2) <= (1e-5 + 4 * 2.0 ** -22 * top) * np.abs(ref).max(2))
