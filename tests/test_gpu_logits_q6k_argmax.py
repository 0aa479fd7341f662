"""rrr_logits_rmsnorm_argmax on Q6_K rows: the logits of rrr_logits_rmsnorm bit for bit and the first index of their
maximum, from one row to several tiles a workgroup, either side of a wave's one and two super-blocks and past the widest
K of the epilogue; with ties across workgroups, without a live candidate, eager and in a replayed graph.  And the GEMV
below it where two workgroups share a CU."""
import numpy as np
import pytest

import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu
EPS = 1e-5


@pytest.mark.parametrize("K,V", [(256, 1), (256, 17), (512, 4097), (1024, 32064), (3072, 1000), (3072, 32064), (4096, 4099),
                                 (4352, 5000), (8192, 2561), (8192, 70000), (8448, 300)])
@pytest.mark.parametrize("same", [False, True])
def test_token_is_first_max_of_the_same_logits(K, V, same):
    raw = np.frombuffer(synth.weight(61, 1, rrr.Q6_K, K, V), np.uint8)
    if same:   # rows repeat every 7: the maximum is in many workgroups
        rows = raw.reshape(V, -1)
        raw = np.ascontiguousarray(rows[np.arange(V) % 7]).reshape(-1)
    with rrr.Context(0) as ctx:
        E, g = ctx.weight_upload(rrr.Q6_K, K, V, raw), ctx.alloc(K * 4)
        x, y, y2 = ctx.alloc(K * 4), ctx.alloc((V + 4) * 4), ctx.alloc(V * 4)
        token = ctx.alloc(4)
        ctx.upload(g, 1.0 + 0.1 * synth.normal_f32(62, 1, K))
        issue = lambda t=token: ctx.logits_rmsnorm_argmax(x, g, EPS, E, y, K, V, t, rrr.LOGITS_Q6K, 0)
        ctx.upload(x, synth.normal_f32(62, 2, K))
        ctx.graph_begin()
        issue()
        graph = ctx.graph_end()
        for i, run in enumerate([issue, graph.launch, issue, graph.launch, graph.launch]):
            ctx.upload(x, synth.normal_f32(63, i, K))
            ctx.fill_u32(y, 0x7F7F7F7F)
            ctx.fill_u32(token, 0xFFFFFFFF)
            run()
            got = ctx.download(y, np.uint32)
            ctx.logits_rmsnorm(x, g, EPS, E, y2, K, V, rrr.LOGITS_Q6K, 0)
            ref = ctx.download(y2)
            assert np.array_equal(got[:V], ref.view(np.uint32)) and np.all(got[V:] == 0x7F7F7F7F)
            assert ctx.download(token, np.uint32)[0] == np.argmax(ref)
        graph.destroy()
        for bad in (0.0, np.nan):   # all logits zero: index 0; all NaN: no candidate, index 0
            v = synth.normal_f32(63, 9, K) * (0.0 if bad == 0.0 else 1.0)
            v[K // 2] = bad
            ctx.upload(x, v.astype(np.float32))
            ctx.fill_u32(token, 0xFFFFFFFF)
            issue()
            assert ctx.download(token, np.uint32)[0] == 0
        # a token stored over one of the logits: the token is what stays
        ctx.upload(x, synth.normal_f32(63, 10, K))
        issue()
        want = ctx.download(token, np.uint32)[0]
        issue(ctx.view(y, (V // 2) * 4, 4))
        assert ctx.download(y, np.uint32)[V // 2] == want


@pytest.mark.parametrize("qtype,K,N", [(12, 1024, 4097), (13, 256, 8193), (14, 1024, 16397), (14, 768, 20480)])
def test_two_workgroups_a_cu_give_the_bits_of_one(qtype, K, N):
    rows = np.frombuffer(synth.weight(64, 1, qtype, K, N), np.uint8).reshape(N, -1)
    with rrr.Context(0) as ctx:
        x, y, g = ctx.alloc(K * 4), ctx.alloc((N + 4) * 4), ctx.alloc(K * 4)
        ctx.upload(x, synth.normal_f32(65, 1, K))
        ctx.upload(g, 1.0 + 0.1 * synth.normal_f32(65, 2, K))
        W = ctx.weight_upload(qtype, K, N, rows.reshape(-1))
        part = ctx.alloc(4096 * 4)
        ctx.fill_u32(y, 0x7F7F7F7F)
        ctx.gemv_rmsnorm(x, g, EPS, W, qtype, y, K, N)
        got = ctx.download(y, np.uint32)
        assert np.all(got[N:] == 0x7F7F7F7F)
        for r in range(0, N, 4096):   # 16 rows a CU: one workgroup each
            n = min(4096, N - r)
            Wr = ctx.weight_upload(qtype, K, n, np.ascontiguousarray(rows[r:r + n]).reshape(-1))
            ctx.gemv_rmsnorm(x, g, EPS, Wr, qtype, part, K, n)
            assert np.array_equal(got[r:r + n], ctx.download(part, np.uint32)[:n])
