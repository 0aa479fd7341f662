"""Long-prompt GEMMs, whose weights are expanded to f16 first (csrc/gemm_wide.hip): tile widths that do and do not
divide N, row counts that end inside a 256-row tile, accumulate, row scales and caller rows short of the padding,
and weights taken in several column parts.

The expanded weights are the f16 values the in-kernel dequant makes and every output adds the same products over K,
so the rows agree with calls of 128 rows (which never expand, and may split K) to the order of f32 sums over K
terms.  Each of the K / 16 accumulations rounds by at most 2^-24 of a partial sum (about the row's largest output),
so two orders differ by at most 2 (K / 16) 2^-24 of it, and, the roundings being independent, by a few sqrt(K / 16)
2^-24: four of them are allowed.  Against the oracle the matrix-core bar, 2e-3."""
import numpy as np
import pytest

import oracle.oracle as orc
import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu

MFMA_TOL = 2e-3


@pytest.fixture(scope="module")
def ctx():
    with rrr.Context(0) as c:
        yield c


def close(a, b, tol):
    big = np.max(np.abs(b), axis=1)
    assert np.all(np.max(np.abs(a - b), axis=1) <= tol * np.where(big > 0, big, 1.0))


@pytest.mark.parametrize("qtype,K,N,M,acc,scaled", [
    (12, 3072, 5696, 896, False, False),     # N not a multiple of any wider tile
    (13, 1024, 5184, 1792, True, True),
    (14, 2816, 1088, 2048, True, False),
    (12, 3072, 3072, 2048, False, True),
    (14, 11264, 4096, 640, False, False),    # 92 MB of expanded weights
    (12, 10240, 8192, 1152, True, False)])   # 168 MB: two column parts
def test_long_rows_match_short_calls(ctx, qtype, K, N, M, acc, scaled):
    raw = synth.weight(31, qtype, qtype, K, N)
    X = synth.normal_f32(31, 7, M * K).astype(np.float16).reshape(M, K)
    Y0 = synth.normal_f32(31, 8, M * N).reshape(M, N)
    sc = (2.0 ** np.arange(-4, 4)).astype(np.float32)[np.arange(M) % 8]
    W, Xb, Sb = ctx.weight_upload(qtype, K, N, raw), ctx.to_device(X), ctx.to_device(sc)
    Y, P = ctx.to_device(Y0), ctx.to_device(Y0)
    ctx.gemm_f16(Xb, W, qtype, Y, K, N, M, accumulate=acc, row_scale=Sb if scaled else None)
    for m in range(0, M, 128):
        views = [ctx.view(Xb, m * K * 2, 128 * K * 2), ctx.view(P, m * N * 4, 128 * N * 4), ctx.view(Sb, m * 4, 512)]
        ctx.gemm_f16(views[0], W, qtype, views[1], K, N, 128, accumulate=acc, row_scale=views[2] if scaled else None)
        for v in views:
            v.free()
    got, want = ctx.download(Y).reshape(M, N), ctx.download(P).reshape(M, N)
    for b in (W, Xb, Sb, Y, P):
        b.free()
    base = Y0 if acc else 0.0
    sums = 4 * (K / 16) ** 0.5 * 2.0 ** -24
    if acc:   # the add of Y0 and its removal here round once more each
        sums += 2.0 ** -22
    close(got - base, want - base, sums)
    rows = [0, 127, 255, 256, M - 129, M - 1]
    ref = orc.gemv(qtype, raw, X[rows].astype(np.float32).reshape(-1), K, N, len(rows), 16, f64=True)
    if scaled:
        ref = ref * sc[rows][:, None]
    close((got - base)[rows], ref, MFMA_TOL)


@pytest.mark.parametrize("qtype,K,N,M", [(14, 8192, 3072, 1111), (13, 1536, 2688, 641)])
def test_ragged_bf16_rows(ctx, qtype, K, N, M):
    raw = synth.weight(32, qtype, qtype, K, N)
    xb = synth.normal_bf16(32, 9, M * K)
    X = (xb.astype(np.uint32) << 16).view(np.float32).reshape(M, K)
    W, Xb, Y = ctx.weight_upload(qtype, K, N, raw), ctx.to_device(xb), ctx.alloc((M + 1) * N * 4)
    ctx.fill_u32(Y, 0x7F7F7F7F)
    ctx.gemm_bf16(Xb, W, qtype, Y, K, N, M)
    got = ctx.download(Y).reshape(M + 1, N)
    for b in (W, Xb, Y):
        b.free()
    assert np.all(got[M].view(np.uint32) == 0x7F7F7F7F)     # nothing past the caller's rows
    rows = [0, 255, 256, M // 2, M - 2, M - 1]
    ref = orc.gemv(qtype, raw, np.ascontiguousarray(X[rows]).reshape(-1), K, N, len(rows), 16, f64=True)
    close(got[rows], ref, MFMA_TOL)
