"""Batched rows up to 16 against 64 bits: no further off than f32 activations and f32 sums are.  The bounds are the
errors of the VALU kernel (f32 throughout) measured on these very inputs, over rows of one magnitude, of uneven
magnitude, and with a mean; weights of mean zero as trained matrices have (each sub-block's min code its scale code,
min step the middle of the quants times the scale step), where a mean of x makes d sc q and dmin mn nearly cancel."""
import numpy as np
import pytest

import oracle.oracle as orc
import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu

K, N = 8192, 384
VALU = {  # (type, rows): relative 2-norm error over the outputs of 5 and of 16 rows
    (12, "even"): (2.023e-07, 1.891e-07), (12, "uneven"): (2.077e-07, 1.860e-07), (12, "mean"): (4.289e-07, 4.177e-07),
    (13, "even"): (2.122e-07, 1.932e-07), (13, "uneven"): (2.281e-07, 1.844e-07), (13, "mean"): (4.110e-07, 4.184e-07),
    (14, "even"): (2.014e-07, 2.030e-07), (14, "uneven"): (2.204e-07, 1.956e-07), (14, "mean"): (4.068e-07, 4.089e-07),
}


def mean_zero(qtype, seed):
    raw = np.array(synth.weight(seed, qtype, qtype, K, N), np.uint8).reshape(N * K // 256, -1).copy()
    if qtype != rrr.Q6_K:
        raw[:, 8:12] = raw[:, 4:8]
        low = raw[:, 12:16] & 15
        raw[:, 12:16] = low | (low << 4)
        d = raw[:, 0:2].copy().view(np.float16).astype(np.float32)
        raw[:, 2:4] = (d * (7.5 if qtype == rrr.Q4_K else 15.5)).astype(np.float16).view(np.uint8)
    return raw


def rows(kind, M):
    X = synth.normal_f32(28, M, M * K).reshape(M, K)
    if kind == "mean":
        return np.abs(X)
    if kind == "uneven":
        return (X * np.exp(2 * synth.normal_f32(29, M, M * K).reshape(M, K))).astype(np.float32)
    return X


@pytest.mark.parametrize("kind", ["even", "uneven", "mean"])
@pytest.mark.parametrize("qtype", [12, 13, 14])
def test_rows_as_exact_as_f32(ctx, qtype, kind):
    raw = mean_zero(qtype, 27)
    W, Y = ctx.weight_upload(qtype, K, N, raw), ctx.alloc(16 * N * 4)
    for M, bound in zip((5, 16), VALU[qtype, kind]):
        X = rows(kind, M)
        Xb = ctx.to_device(X)
        ctx.gemv(Xb, W, qtype, Y, K, N, M)
        y = ctx.download(Y, np.float32, M * N).reshape(M, N)
        Xb.free()
        ref = orc.gemv(qtype, raw.reshape(-1), X.reshape(-1), K, N, M, 16, f64=True)
        err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        assert err <= bound, (M, err)
    W.free(), Y.free()
