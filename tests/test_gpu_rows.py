"""A few token rows on the skinny kernel (csrc/skinny.hip) at its edges: one and several super-block columns a
wave, one to more than four tiles a workgroup, a ragged last tile, blocks at odd offsets (Q6_K), the row counts
where its A tiles fill up, and the row runs above 16 that keep f32 accuracy.

Tolerance: hi/lo activations hold 22 bits of a slice's maximum and the sums are f32 over at most K terms, so an
output is off by a few 1e-7 of the row's largest; 2e-6 leaves a factor of about five.  Rows taken as f16 keep
the matrix-core bar, 2e-3."""
import numpy as np
import pytest

import oracle.oracle as orc
import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu

F32_TOL, F16_TOL = 2e-6, 2e-3


@pytest.fixture(scope="module")
def ctx():
    with rrr.Context(0) as c:
        yield c


def rows(ctx, qtype, K, N, X):
    M = X.shape[0]
    raw = synth.weight(23, qtype, qtype, K, N)
    W, Xb, Yb = ctx.weight_upload(qtype, K, N, raw), ctx.to_device(X), ctx.alloc(M * N * 4)
    ctx.fill_u32(Yb, 0x7FC00000)
    ctx.gemv(Xb, W, qtype, Yb, K, N, M)
    Y = ctx.download(Yb).reshape(M, N)
    for b in (W, Xb, Yb):
        b.free()
    return raw, Y


@pytest.mark.parametrize("qtype,K,N", [
    (14, 256, 16), (14, 3072, 4111),        # one column; a ragged tile
    (14, 3328, 8200),                       # 13 columns on 7 waves, odd blocks, three tiles a workgroup
    (12, 3584, 12300), (13, 3840, 16900),   # four tiles a workgroup; more than four
    (12, 8192, 96), (14, 11008, 100)])      # three and four columns a wave
@pytest.mark.parametrize("M", [5, 8, 9, 16, 17, 33])
def test_rows_at_the_edges(ctx, qtype, K, N, M):
    X = synth.normal_f32(24, M, M * K).reshape(M, K)
    raw, Y = rows(ctx, qtype, K, N, X)
    ref = orc.gemv(qtype, raw, X.reshape(-1), K, N, M, 16, f64=True)
    f16 = M > 16 and (N % 64 == 0 or (M <= 32 and qtype != 14 and K <= 3072))
    for m in range(M):
        assert orc.normwise_err(Y[m], ref[m]) < (F16_TOL if f16 else F32_TOL), m


@pytest.mark.parametrize("qtype,K,N", [(14, 8192, 48), (12, 4096, 64)])
def test_rows_of_any_size(ctx, qtype, K, N):
    """Rows at both ends of the exponent range, a zero row, and rows with inf and NaN, which keep to themselves."""
    X = synth.normal_f32(25, 1, 9 * K).reshape(9, K)
    X[0] *= np.float32(1e30)
    X[1] *= np.float32(1e-36)
    X[2] = 0.0
    X[3, 5] = np.inf
    X[4, K - 1] = np.nan
    raw, Y = rows(ctx, qtype, K, N, X)
    assert not np.any(np.isfinite(Y[3])) and not np.any(np.isfinite(Y[4]))
    assert np.all(Y[2] == 0.0)
    fin = [0, 1, 5, 6, 7, 8]
    ref = orc.gemv(qtype, raw, np.ascontiguousarray(X[fin]).reshape(-1), K, N, len(fin), 16, f64=True)
    for i, m in enumerate(fin):
        assert orc.normwise_err(Y[m], ref[i]) < F32_TOL, m


@pytest.mark.parametrize("qtype,K,N", [(12, 4096, 4111), (13, 3328, 96), (14, 4096, 12300), (12, 4096, 16900)])
@pytest.mark.parametrize("M", [3, 8])
def test_rows_one_column_a_wave(ctx, qtype, K, N, M):
    """13 to 16 columns with one A tile: one a wave, one to more than four tiles a workgroup."""
    X = synth.normal_f32(26, M, M * K).reshape(M, K)
    raw, Y = rows(ctx, qtype, K, N, X)
    ref = orc.gemv(qtype, raw, X.reshape(-1), K, N, M, 16, f64=True)
    for m in range(M):
        assert orc.normwise_err(Y[m], ref[m]) < F32_TOL, m


@pytest.mark.parametrize("qtype,K,N", [(14, 256, 16), (12, 256, 8200), (13, 1024, 4111), (14, 1280, 12300),
                                       (12, 2048, 20000), (13, 2048, 100)])
def test_operands_built_in_the_wave(ctx, qtype, K, N):
    """To 8 columns and 8 rows a wave builds its operands itself: bit for bit those of the encoding pass, which calls
    of more rows take (two A tiles; the same products and sums for each row)."""
    X = synth.normal_f32(30, 1, 12 * K).reshape(12, K)
    X[1] *= np.float32(1e30)
    X[2] *= np.float32(1e-36)
    X[3] = 0.0
    X[4, ::7] *= np.float32(100.0)
    Y12 = rows(ctx, qtype, K, N, X)[1]
    for M in (5, 7, 8):
        raw, Y = rows(ctx, qtype, K, N, X[:M].copy())
        assert np.array_equal(Y.view(np.uint32), Y12[:M].view(np.uint32)), M
    ref = orc.gemv(qtype, raw, X[:8].reshape(-1), K, N, 8, 16, f64=True)
    for m in (0, 1, 4, 5, 6, 7):
        assert orc.normwise_err(Y[m], ref[m]) < F32_TOL, m
    assert np.all(Y[3] == 0.0)


@pytest.mark.parametrize("qtype,K,N,M", [
    (14, 4096, 1024, 3), (12, 6144, 1000, 3), (13, 8192, 2048, 2), (14, 16384, 16, 2),      # VALU kernel
    (12, 4096, 512, 16), (13, 5120, 680, 12), (12, 3328, 500, 9),
    (14, 4096, 1032, 3), (12, 16640, 64, 3), (12, 12544, 64, 2), (14, 4096, 512, 16), (12, 5376, 512, 16)])   # past it
def test_long_rows_of_few_weights(ctx, qtype, K, N, M):
    """Both sides of the rule that leaves few weights and long rows to the VALU kernel."""
    X = synth.normal_f32(32, M, M * K).reshape(M, K)
    raw, Y = rows(ctx, qtype, K, N, X)
    ref = orc.gemv(qtype, raw, X.reshape(-1), K, N, M, 16, f64=True)
    for m in range(M):
        assert orc.normwise_err(Y[m], ref[m]) < F32_TOL, m
