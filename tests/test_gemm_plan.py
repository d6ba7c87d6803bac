"""The plain GEMM's launch plan (host code only, no GPU)."""
import ctypes as C

import pytest

from mnemocuda_amd import lib as mlib
from tests.test_gpu_gemm import RAGGED

BLOCK = {12: 144, 14: 210}


def plan(type_id, M, K, N, cus=256):
    """(shape, rows and tokens of its tile, slices of K, rows and tokens of one launch)"""
    out = (C.c_int * 5)()
    shape = mlib.load_library().mnemo_internal_gemm_plan(type_id, M, K, N, cus, out)
    return (shape, *out)


@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("M", [1, 3, 33, 300, 8192, 1 << 20])
@pytest.mark.parametrize("K", [256, 16384, 1 << 24, 5 << 22, 1 << 27, 5 << 25, (1 << 31) - 256])
@pytest.mark.parametrize("N", [1, 17, 2000, 1 << 21])
def test_a_tile_spans_less_than_4_gib(type_id, M, K, N):
    # offsets within a workgroup's rows are 32 bits
    _, rows, toks, _, launch_rows, launch_toks = plan(type_id, M, K, N)
    assert 1 <= launch_rows <= M and 1 <= launch_toks <= N
    assert min(rows, launch_rows) * (K // 256) * BLOCK[type_id] < 1 << 32
    assert min(toks, launch_toks) * (K // 128) * 144 < 1 << 32
    if launch_rows < M:  # the next launch's output stays 16-byte aligned where the stores are 16 bytes
        assert launch_rows % 4 == 0 or launch_rows < 4
    if K <= 1 << 24:
        assert (launch_rows, launch_toks) == (M, N)


@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("shape", range(12))
def test_gpu_sizes_reach_every_shape(type_id, shape):
    """Each shape and type runs with ragged rows and tokens, once with slices of at most one super-block
    (two pairs are never taken for those) and once with unequal slices of more than a window (four)."""
    short = long = False
    for M, K, N in RAGGED:
        got, rows, toks, slices, *_ = plan(type_id, M, K, N)
        if got == shape and M % rows and M % 4 and N % toks:
            nsb = K // 256
            short |= nsb <= slices
            long |= nsb > 4 * slices and (slices == 1 or nsb % slices != 0)
    assert short or (type_id, shape) in ((12, 1), (14, 2))
    assert long
