"""Dequant of block counts around a workgroup's 16 blocks and a wave's 4, from a buffer and from views that start
at any block (Q6_K blocks at odd 2-byte offsets): bit-exact with the oracle, and nothing written past the end."""
import numpy as np
import pytest

import oracle.oracle as orc
import rrr_hip as rrr
from rrr_hip import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [0, 12, 13, 14])
@pytest.mark.parametrize("blocks,first", [(1, 0), (3, 0), (4, 2), (5, 0), (15, 4), (16, 0), (17, 6), (63, 0)])
def test_dequant_block_counts(qtype, blocks, first):
    n, size = blocks * 256, rrr.BLOCK_BYTES[qtype]
    raw = (synth.normal_f32(26, 1, (blocks + first) * 256).view(np.uint8) if qtype == 0
           else synth.kquant(26, qtype, qtype, blocks + first))
    with rrr.Context(0) as ctx:
        whole = ctx.to_device(raw)
        W = ctx.view(whole, first * size, blocks * size)
        out = ctx.alloc((n + 64) * 4)
        ctx.fill_u32(out, 0xABCDEF01)
        ctx.dequant(qtype, W, out, n)
        got = ctx.download(out, np.uint32)
    part = np.ascontiguousarray(raw[first * size:])
    want = part.view(np.float32) if qtype == 0 else orc.dequant(qtype, part, n)
    assert np.array_equal(got[:n], want.view(np.uint32))
    assert np.all(got[n:] == 0xABCDEF01)
