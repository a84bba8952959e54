"""CPU: which kernel a shape takes (the rules are host code: hk_*_route asks them without a context)."""
import pytest

from rust_ascend_hip import _lib
from rust_ascend_hip._lib import BF16, F32

CUS = 256
T256, T256x192, T256x128, T128, T128_PAIR, T64x128, T128x64, T64, T32x64 = range(9)


def gemm(m, n, k, ta=0, dtype=BF16, batch=1, scratch=1 << 62):
    r = _lib.load().hk_gemm_route(batch, m, n, k, ta, dtype, scratch, CUS)
    return r if r < 0 else (r % 256, r // 256)


# few rows against a weight past the caches whose column tiles fill 3/4 of the CUs: one unsplit row tile
@pytest.mark.parametrize("m,n,k,ta,want", [(64, 14336, 4096, 0, T64), (48, 14192, 4288, 0, T64), (32, 12320, 11488, 0, T32x64),
                                           (16, 16384, 4096, 0, T32x64), (16, 12288, 4096, 1, T64)])
def test_streamed_weight_is_not_split(m, n, k, ta, want):
    assert gemm(m, n, k, ta) == gemm(m, n, k, ta, scratch=0) == (want, 1)


def test_streamed_weight_of_few_columns_is_split():
    assert gemm(16, 4096, 14336) == (T32x64, 4)
    assert gemm(16, 4096, 14336, scratch=0)[1] == 1
