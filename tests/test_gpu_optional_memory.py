"""A context without the memory that only makes calls faster (no room at rrr_init): the long-prompt GEMMs dequantize
inside the GEMM, rrr_matmul_kquant copies through pageable memory; results as before."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


def test_calls_without_optional_memory():
    K, N, M = 3072, 5120, 1152
    raw = synth.weight(33, 12, rrr.Q4_K, K, N)
    X = synth.normal_f32(33, 1, M * K).astype(np.float16)
    x = synth.normal_f32(33, 2, K)
    out = []
    for drop in (False, True):
        with rrr.Context(0) as ctx:
            W, Xb, Y = ctx.weight_upload(rrr.Q4_K, K, N, raw), ctx.to_device(X), ctx.alloc(M * N * 4)
            if drop:
                ctx.probe_drop_optional()
                ctx.probe_drop_optional()       # nothing left to give back
            ctx.gemm_f16(Xb, W, rrr.Q4_K, Y, K, N, M)
            y = ctx.download(Y, np.uint32)
            a, c = ctx.alloc(K * 4), ctx.alloc(N * 4)
            out.append((y, ctx.matmul_kquant(a, W, c, rrr.Q4_K, x, K, N).view(np.uint32)))
    for with_it, without in zip(*out):
        assert np.array_equal(with_it, without)
