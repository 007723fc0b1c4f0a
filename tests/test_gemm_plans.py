"""Which GEMM kernels the shapes of the GPU parity tests reach: the tiles are
picked by cost models, so a change of their constants could leave a kernel
without a test (no device is needed: the choice is made for 256 compute units).
"""
import ctypes

import pytest

from gollek_amd import _native
from gollek_amd import synthetic as syn
from tests.test_gpu_gemm import K_QUANT_TILES, RAGGED_K, SPLIT_REPEATS
from tests.test_zz_no_alloc import SPLIT


def plan(type_id, rows, cols, m):
    p = (ctypes.c_int32 * 4)()
    assert _native.load().gollek_hip_testing_gemm_plan(type_id, m, rows, cols, p) == _native.OK
    return tuple(p)


@pytest.mark.parametrize("tid", [syn.Q4_K, syn.Q5_K, syn.Q6_K])
def test_k_quant_tile_shapes_reach_every_plan(tid):
    plans = {plan(tid, *shape) for shape in K_QUANT_TILES}
    assert {p[:3] for p in plans} == {(1, 1, 4), (1, 1, 8), (1, 2, 4), (2, 2, 2), (2, 2, 4), (2, 4, 2), (4, 4, 2),
                                      (4, 8, 1), (6, 8, 1), (8, 8, 1)}
    # split over K: one row tile, and six (three quads of X rows per wave)
    assert {(1, 1, 4), (6, 8, 1)} <= {p[:3] for p in plans if p[3] > 1}


@pytest.mark.parametrize("tid", [syn.Q8_0, syn.Q4_0])
def test_ragged_k_shapes_reach_every_tile_height(tid):
    assert {plan(tid, *s)[0] for s in RAGGED_K if s[1] // 32 % 2 == 1} == {1, 2, 4, 8}


def test_split_shapes_split():
    for tid, rows, m in SPLIT_REPEATS:
        assert plan(tid, rows, 4096, m)[3] > 1, (tid, rows, m)
    for tid, rows, cols, ms in SPLIT:
        for m in ms:  # (up to 32 rows of Q8_0 never do)
            assert plan(tid, rows, cols, m)[3] > 1, (tid, rows, cols, m)


def test_plan_checks_arguments():
    lib, p = _native.load(), (ctypes.c_int32 * 4)()
    assert lib.gollek_hip_testing_gemm_plan(syn.Q4_K, 16, 64, 256, None) == _native.ERR_ARG
    assert lib.gollek_hip_testing_gemm_plan(syn.Q4_K, 0, 64, 256, p) == _native.ERR_ARG
    assert lib.gollek_hip_testing_gemm_plan(0, 16, 64, 256, p) == _native.ERR_UNSUPPORTED
