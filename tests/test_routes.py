"""CPU: which kernel a shape takes (the rules are host code: hk_*_route asks them without a context)."""
import pytest

import tile_cases as cases
from rust_ascend_hip import _lib
from rust_ascend_hip._lib import BF16, F32
from tile_cases import CUS, T32x64, T64


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


# ------------------------------------------------------------------ the shapes of tests/tile_cases.py

def epilogue(m, n, k, qkv):
    return _lib.load().hk_epilogue_route(m, n, k, qkv, CUS)


def matmul(a, b, which, scratch=1 << 62):
    t = [_lib.tensor_desc(1 << 20, F32, s) for s in (a, b)]
    r = _lib.load().hk_tensor_matmul_route(t[0], t[1], which, scratch, CUS)
    return r if r < 0 else (r % 1024, r // 1024)


def test_every_tile_has_a_case():
    mid = set(range(cases.T256x128, cases.T32x64 + 1))
    assert set(cases.PLAIN) == mid and set(cases.SPLIT) == mid - {cases.T128_PAIR}  # its pairs are never the cheapest split
    assert set(cases.TWO_OUTPUTS) == mid - {cases.T32x64} | {cases.T256}  # A MN-major: tiles of 64 rows or more
    assert set(cases.PAIR) == mid - {cases.T32x64}
    assert set(cases.EPILOGUE) == {cases.T256x128, cases.T128_PAIR, cases.T64x128, cases.T64}
    assert set(cases.QKV) == {cases.T128_PAIR, cases.T64x128}
    assert mid - {cases.T64, cases.T32x64} <= {t for ts in cases.CROPPED.values() for t in ts}  # those two: small shapes
    assert {r for rs in cases.F32.values() for r in rs} >= {(64, 1), (64, 16), (128, 1), (128, 4)}


def test_gemm_tile_cases():
    for tile, dims in cases.PLAIN.items():
        for dtype in (BF16, F32):
            assert gemm(*dims, 0, dtype) == (tile, 1), dims
        assert gemm(*dims, 1, F32) == (cases.T64 if tile == cases.T32x64 else tile, 1), dims
    for tile, (m, n, k, splits) in cases.SPLIT.items():
        assert gemm(m, n, k, 0, F32) == gemm(m, n, k, 0, BF16) == (tile, splits)
        assert gemm(m, n, k, 0, F32, scratch=0)[1] == 1
    for tile, (m, k, h) in cases.TWO_OUTPUTS.items():
        assert gemm(2 * h, k, m, 1, F32, scratch=0) == (tile, 1)
    for tile, (heads, rows, keys, d) in cases.PAIR.items():
        assert gemm(keys, d, rows, 1, F32, batch=2 * heads, scratch=0) == (tile, 1)


def test_epilogue_tile_cases():
    for tile, dims in cases.EPILOGUE.items():
        assert epilogue(*dims, 0) == tile
    for tile, (tokens, hq, hkv, hidden) in cases.QKV.items():
        assert epilogue(tokens, (hq + 2 * hkv) * 128, hidden, 1) == tile


def test_cropped_tile_cases():
    up = lambda x: (x + 15) // 16 * 16  # noqa: E731
    for (m, k, n), tiles in cases.CROPPED.items():
        m, k, n = up(m), up(k), up(n)
        for tile, route in zip(tiles, (gemm(m, n, k, 0, F32), gemm(m, k, n, 0, F32), gemm(n, k, m, 1, F32))):
            assert tile is None or route == (tile, 1)


def test_f32_matmul_tile_cases():
    for (a, b), routes in cases.F32.items():
        assert tuple(matmul(a, b, which) for which in range(3)) == routes, (a, b)
