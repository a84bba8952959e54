"""GPU parity of the F32 generic matmul read in place (any extents, batch strides and alignment, K split over
workgroups, batches folded into M or the contraction) and its gradients, against float64.

A sum of K products rounded to F32 at each step has a relative 2-norm error of about sqrt(K) 2^-24; four
times that is allowed."""
import os

import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime

pytestmark = pytest.mark.gpu


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def randn(shape, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV)


def unbroadcast(t, shape):
    while t.dim() > len(shape):
        t = t.sum(0)
    for d, n in enumerate(shape):
        if n == 1 and t.shape[d] != 1:
            t = t.sum(d, keepdim=True)
    return t


def check(a, b):
    y = HipRuntime.tensor_matmul(a, b)
    dy = randn(y.shape, 3)
    da, db = HipRuntime.tensor_matmul_backward(a, b, dy)
    k, n, rows = a.shape[-1], b.shape[-1], y.numel() // b.shape[-1]
    want = torch.matmul(a.double(), b.double())
    wa = unbroadcast(torch.matmul(dy.double(), b.double().transpose(-1, -2).contiguous()), a.shape)
    wb = unbroadcast(torch.matmul(a.double().transpose(-1, -2).contiguous(), dy.double()), b.shape)
    for got, ref, terms in ((y, want, k), (da, wa, n * max(1, y[..., 0, 0].numel())), (db, wb, rows)):
        assert rel(got, ref) <= 4 * terms ** 0.5 * 2 ** -24


# edges of tiles and of a 16-step, one element, odd strides, split K (all of these on 64x64 tiles; the 128x128
# ones are in test_gpu_gemm_tiles.py)
@pytest.mark.parametrize("a,b", [((1, 1), (1, 1)), ((3, 5), (5, 7)), ((64, 16), (16, 64)), ((65, 17), (17, 129)), ((130, 1001), (1001, 67)), ((130, 1001), (1001, 68)), ((130, 1004), (1004, 67)),
                                 ((31, 4097), (4097, 33)), ((2050, 70), (70, 1999)), ((1100, 64), (64, 4099)),
                                 ((4, 77, 130), (130, 95)), ((3, 2, 40, 33), (33, 20)), ((6, 50, 64), (6, 64, 70)),
                                 ((1, 30, 20), (5, 20, 40)), ((2, 1, 17, 9), (3, 9, 11)), ((4, 1, 16, 8), (1, 5, 8, 16)),
                                 ((2, 300, 257), (2, 257, 301))])
def test_f32_matmul_and_gradients(a, b):
    print(f"f32 matmul {a} @ {b}", flush=True)
    check(randn(a, 1), randn(b, 2))


def test_f32_matmul_off_16_byte_alignment():
    buf = randn((1 + 70 * 45,), 5)
    a, b = buf[1:].view(70, 45), randn((45, 80), 6)
    assert rel(HipRuntime.tensor_matmul(a, b), a.double() @ b.double()) <= 4 * 45 ** 0.5 * 2 ** -24


def test_f32_matmul_non_finite_values_stay_in_their_rows():
    a, b = randn((100, 70), 7), randn((70, 90), 8)
    a[3, 10], a[70, 69], b[5, 44] = float("inf"), float("nan"), float("-inf")
    y, want = HipRuntime.tensor_matmul(a, b), a.double() @ b.double()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want))


def test_f32_matmul_split_within_a_workspace_limit():
    a, b = randn((31, 4097), 9), randn((4097, 33), 10)
    HipRuntime.trim_workspace()
    os.environ["HK_WORKSPACE_LIMIT"] = "16"
    try:
        y = HipRuntime.tensor_matmul(a, b)
        assert HipRuntime.workspace_size() == 0
    finally:
        del os.environ["HK_WORKSPACE_LIMIT"]
    assert rel(y, a.double() @ b.double()) <= 4 * 4097 ** 0.5 * 2 ** -24
