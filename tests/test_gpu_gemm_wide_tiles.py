"""The GEMM on expanded weights (csrc/gemm_wide.hip), every tile width: its outputs are those of the GEMM that
dequantizes as it goes, without split K, bit for bit, so the fused calls, which take either, keep the bits of their
parts.  The routes are asked for, so a change of the estimates cannot empty a case."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def plain():
    """A context that never expands weights."""
    with rrr.Context(0) as c:
        c.probe_drop_optional()
        yield c


# (tile, K, N, M): tiles that divide N and not, rows that end inside a 256-row tile and not; where K = 256 the ring's
# depth covers every step
CASES = [(64, 1536, 1088, 2048), (64, 256, 8192, 1408),
         (96, 1024, 2112, 2048), (96, 256, 16448, 896), (96, 3072, 3072, 1920),
         (128, 512, 4160, 1536), (128, 512, 5696, 1152), (128, 3072, 5120, 1152),
         (160, 256, 5184, 1664), (160, 3072, 5120, 1920),
         (192, 256, 5184, 2048), (192, 256, 5696, 1920), (192, 3072, 16384, 1152),
         (256, 256, 9024, 1408), (256, 256, 16448, 768), (256, 3072, 8192, 1536),
         (96, 10240, 8192, 1152)]     # 160 MiB of f16 weights: two column parts


@pytest.mark.parametrize("tile,K,N,M", CASES)
@pytest.mark.parametrize("qtype", [12, 13, 14])
def test_tiles_keep_the_bits(ctx, plain, qtype, tile, K, N, M):
    assert ctx.probe_gemm_route(K, N, M) == (tile, 1) and plain.probe_gemm_route(K, N, M) == (0, 1)
    raw = synth.weight(34, qtype, qtype, K, N)
    X = synth.normal_f32(34, 1, M * K).astype(np.float16)
    sc = (2.0 ** np.arange(-4, 4)).astype(np.float32)[np.arange(M) % 8]
    Y0 = synth.normal_f32(34, 2, M * N)
    out = []
    for c in (ctx, plain):
        W, Xb, Sb, Y = c.weight_upload(qtype, K, N, raw), c.to_device(X), c.to_device(sc), c.to_device(Y0)
        c.gemm_f16(Xb, W, qtype, Y, K, N, M)
        a = c.download(Y, np.uint32)
        c.upload(Y, Y0)
        c.gemm_f16(Xb, W, qtype, Y, K, N, M, accumulate=True, row_scale=Sb)
        out.append((a, c.download(Y, np.uint32)))
        for b in (W, Xb, Sb, Y):
            b.free()
    for with_it, without in zip(*out):
        assert np.array_equal(with_it, without)


@pytest.mark.parametrize("qtype,K,N,M,acc,scaled", [(14, 3072, 3072, 1920, True, True), (12, 2048, 4096, 1024, False, False)])
def test_rmsnorm_after_it_is_the_two_calls(ctx, qtype, K, N, M, acc, scaled):
    assert ctx.probe_gemm_route(K, N, M)[0]
    raw = synth.weight(35, qtype, qtype, K, N)
    X = synth.normal_f32(35, 1, M * K).astype(np.float16)
    sc = (2.0 ** np.arange(-4, 4)).astype(np.float32)[np.arange(M) % 8]
    Y0, g = synth.normal_f32(35, 2, M * N), synth.normal_f32(35, 3, N, 1.0, 0.1)
    W, Xb, Sb, Gb = ctx.weight_upload(qtype, K, N, raw), ctx.to_device(X), ctx.to_device(sc), ctx.to_device(g)
    Ya, Yb, Na, Nb = ctx.to_device(Y0), ctx.to_device(Y0), ctx.alloc(M * N * 2), ctx.alloc(M * N * 2)
    rs = Sb if scaled else None
    ctx.gemm_f16(Xb, W, qtype, Ya, K, N, M, accumulate=acc, row_scale=rs)
    ctx.rmsnorm_f16(Ya, Gb, Na, M, N, 1e-5)
    ctx.gemm_f16_rmsnorm(Xb, W, qtype, Yb, K, N, M, Gb, Nb, 1e-5, accumulate=acc, row_scale=rs)
    assert np.array_equal(ctx.download(Ya, np.uint32), ctx.download(Yb, np.uint32))
    assert np.array_equal(ctx.download(Na, np.uint16), ctx.download(Nb, np.uint16))
    for b in (W, Xb, Sb, Gb, Ya, Yb, Na, Nb):
        b.free()


def test_rope_kv_after_it_is_the_two_calls(ctx):
    K, nh, nkv, hd, rd, M, rows, pos0 = 3072, 24, 8, 128, 96, 1152, 1111, 9
    q_dim, kv = nh * hd, nkv * hd
    N = q_dim + 2 * kv
    assert ctx.probe_gemm_route(K, N, M)[0]
    raw = synth.weight(36, 13, rrr.Q5_K, K, N)
    X = synth.normal_f32(36, 1, M * K).astype(np.float16)
    fac = (1.0 + np.abs(synth.normal_f32(36, 2, rd // 2))).astype(np.float32)
    W, Xb, Fb = ctx.weight_upload(rrr.Q5_K, K, N, raw), ctx.to_device(X), ctx.to_device(fac)
    c0 = synth.normal_f32(36, 3, (pos0 + rows) * kv).astype(np.float16)
    qa, qb = ctx.alloc(M * N * 4), ctx.alloc(M * N * 4)
    ka, va, kb, vb = (ctx.to_device(c0) for _ in range(4))
    ctx.gemm_f16(Xb, W, rrr.Q5_K, qa, K, N, M)
    ctx.rope_kv_store_rows(qa, rows, Fb, rd // 2, ka, va, pos0, nh, nkv, hd, rd, q_dim, kv)
    ctx.gemm_f16_rope_kv_rows(Xb, W, rrr.Q5_K, qb, K, M, rows, Fb, rd // 2, kb, vb, pos0, nh, nkv, hd, rd, q_dim, kv)
    for a, b, t in ((qa, qb, np.uint32), (ka, kb, np.uint16), (va, vb, np.uint16)):
        assert np.array_equal(ctx.download(a, t), ctx.download(b, t))
    for b in (W, Xb, Fb, qa, qb, ka, va, kb, vb):
        b.free()


@pytest.mark.parametrize("qtype,K,F,M", [(12, 512, 2752, 1536), (13, 3072, 1664, 1280), (14, 3072, 2048, 1024)])
def test_silu_gate_is_the_two_calls(ctx, qtype, K, F, M):
    """The fused call dequantizes as it goes; the plain GEMM of the two calls takes the wide form."""
    assert ctx.probe_gemm_route(K, 2 * F, M)[0]
    raw = synth.weight(37, qtype, qtype, K, 2 * F)
    W, Xb = ctx.weight_upload(qtype, K, 2 * F, raw), ctx.to_device(synth.normal_f32(37, 1, M * K).astype(np.float16))
    gu, ma, mb = ctx.alloc(M * 2 * F * 4), ctx.alloc(M * F * 2), ctx.alloc(M * F * 2)
    sa, sb = ctx.alloc(M * 4), ctx.alloc(M * 4)
    ctx.gemm_f16(Xb, W, qtype, gu, K, 2 * F, M)
    ctx.silu_gate_f16(gu, ma, sa, M, F)
    ctx.gemm_f16_silu_gate_f16(Xb, W, qtype, mb, sb, K, F, M)
    assert np.array_equal(ctx.download(ma, np.uint16), ctx.download(mb, np.uint16))
    assert np.array_equal(ctx.download(sa, np.uint32), ctx.download(sb, np.uint32))
    for b in (W, Xb, gu, ma, mb, sa, sb):
        b.free()
