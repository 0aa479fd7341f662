"""The prefill GEMM's choice of form, asked for without a device, and its probes' argument checks."""
import ctypes

import pytest

import rrr_hip as rrr
from rrr_hip import _lib


@pytest.fixture(scope="module")
def vctx():
    with rrr.Context(-1) as c:
        yield c


def test_route(vctx):
    """Few rows dequantize inside the GEMM, long prompts expand the weights first, in tiles that fit the CUs; a matrix
    past the workspace goes in column parts, each with tiles of its own."""
    for K, N in ((3072, 5120), (3072, 16384), (8192, 3072)):
        assert vctx.probe_gemm_route(K, N, 128)[0] == 0
        tile, splits = vctx.probe_gemm_route(K, N, 2048)
        assert tile in (64, 96, 128, 160, 192, 256) and splits == 1
    assert vctx.probe_gemm_route(3072, 3072, 512)[1] > 1        # K split over idle CUs
    assert vctx.probe_gemm_route(10240, 8192, 1152)[0] > 0      # 160 MiB of f16 weights


def test_route_arguments(vctx):
    for K, N, M in ((3072, 5120, 100), (3072, 5121, 128), (3072, 5120, 0), (100, 64, 128), (0, 64, 128)):
        with pytest.raises(rrr.RrrError):
            vctx.probe_gemm_route(K, N, M)
    lib, n = _lib.hip(), ctypes.c_uint32()
    assert lib.rrr_probe_gemm_route(vctx._h, 256, 64, 128, None, ctypes.byref(n)) != 0
    assert lib.rrr_probe_gemm_route(vctx._h, 256, 64, 128, ctypes.byref(n), None) != 0
    with pytest.raises(rrr.RrrError):
        vctx.probe_drop_optional()      # no device
