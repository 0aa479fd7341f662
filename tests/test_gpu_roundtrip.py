"""rrr_matmul_kquant: vectors through the pinned staging (to 32,768 floats, N not a multiple of 4 too) and past it,
called in turn with other vectors: the same bits as upload, GEMV and download, in either wait mode."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("async_", [False, True])
@pytest.mark.parametrize("qtype,K,N", [(12, 256, 1), (13, 512, 37), (14, 2048, 1030), (12, 256, 32768), (12, 256, 32769),
                                       (0, 33024, 5)])
def test_roundtrip_is_upload_gemv_download(qtype, K, N, async_):
    raw = (synth.normal_f32(51, 1, K * N) if qtype == 0 else synth.weight(51, qtype, qtype, K, N))
    with rrr.Context(0) as ctx:
        ctx.set_async(async_)
        W, a, c = ctx.weight_upload(qtype, K, N, raw), ctx.alloc(K * 4), ctx.alloc((N + 4) * 4)
        a2, c2 = ctx.alloc(K * 4), ctx.alloc(N * 4)
        ctx.fill_u32(c, 0x7F7F7F7F)
        for i in range(3):
            x = synth.normal_f32(52, i, K)
            y = ctx.matmul_kquant(a, W, c, qtype, x, K, N)
            ctx.upload(a2, x)
            ctx.gemv(a2, W, qtype, c2, K, N)
            assert np.array_equal(y, ctx.download(c2))
            assert np.array_equal(ctx.download(a), x)
            left = ctx.download(c, np.uint32)
            assert np.array_equal(left[:N], y.view(np.uint32)) and np.all(left[N:] == 0x7F7F7F7F)
