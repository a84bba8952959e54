"""GPU parity of the GEMMs that 256x256 tiles cannot fill: every tile shape from 256x128 to 32x64, K
split over workgroups or not, every transpose read in place, at edges of tiles and of K stages.

Against float64 products of the same BF16 values. F32 outputs: a sum of K products rounded to F32 at
each of K steps in the worst order has a relative 2-norm error of at most about sqrt(K) 2^-24 against
the rounding's random walk; four times that is allowed. BF16 outputs add one rounding, 2^-9 of each
value."""
import os

import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime

pytestmark = pytest.mark.gpu

# batch, M, N, K: one row tile and skinny weights (32x64 tiles, split K), tails of every tile shape,
# a K tail (K % 64 != 0), K of one stage, many small batches, grids around one tile per CU
SHAPES = [(1, 16, 64, 16), (1, 16, 4096, 2048), (1, 48, 1056, 7312), (1, 144, 272, 336), (1, 272, 400, 1040),
          (1, 512, 2048, 704), (1, 784, 2288, 592), (1, 848, 1264, 3952), (1, 1120, 5360, 1152), (1, 2000, 2048, 80),
          (1, 2064, 2032, 1840), (4, 176, 816, 128), (16, 240, 64, 176), (32, 144, 352, 64)]


def operands(g, m, n, k, ta, tb, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)

    def randn(r, c):
        return torch.randn((r, c) if g == 1 else (g, r, c), generator=gen, device=DEV).to(torch.bfloat16)
    a, b = randn(*((k, m) if ta else (m, k))), randn(*((n, k) if tb else (k, n)))
    op = lambda t, tr: (t.transpose(-1, -2) if tr else t).double().contiguous()  # noqa: E731
    return a, b, torch.matmul(op(a, ta), op(b, tb))


def err(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def bound(k, dtype):
    return 4 * k ** 0.5 * 2 ** -24 + (2 ** -9 if dtype == torch.bfloat16 else 0.0)


@pytest.mark.parametrize("g,m,n,k", SHAPES)
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_small_grid_gemm(g, m, n, k, ta, tb):
    a, b, want = operands(g, m, n, k, ta, tb, m + n + k)
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full(want.shape, float("nan"), device=DEV, dtype=dtype)
        print(f"gemm {g}x{m}x{n}x{k} ta{ta} tb{tb} {dtype}", flush=True)
        HipRuntime.gemm_into(a, b, ta, tb, out)
        assert err(out, want) <= bound(k, dtype)


def test_split_k_falls_back_within_a_workspace_limit():
    """A product that would split K runs unsplit when its partial planes may not be allocated."""
    m, n, k = 16, 1200, 6096
    a, b, want = operands(1, m, n, k, 0, 1, 5)
    HipRuntime.trim_workspace()
    os.environ["HK_WORKSPACE_LIMIT"] = "1024"
    try:
        out = HipRuntime.gemm(a, b, 0, 1, torch.float32)
        assert HipRuntime.workspace_size() == 0
    finally:
        del os.environ["HK_WORKSPACE_LIMIT"]
    assert err(out, want) <= bound(k, torch.float32)
    again = HipRuntime.gemm(a, b, 0, 1, torch.float32)
    assert HipRuntime.workspace_size() > 0 and err(again, want) <= bound(k, torch.float32)


def test_split_k_under_graph_capture_allocates_nothing():
    m, n, k = 16, 1200, 6096
    a, b, want = operands(1, m, n, k, 0, 1, 6)
    out = torch.zeros((m, n), device=DEV, dtype=torch.float32)
    HipRuntime.trim_workspace()
    HipRuntime.set_async(True)
    try:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            HipRuntime.gemm_into(a, b, 0, 1, out)
        assert HipRuntime.workspace_size() == 0
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert err(out, want) <= bound(k, torch.float32)
    finally:
        HipRuntime.set_async(False)


@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0)])
def test_unaligned_operands(ta, tb):
    """Operands off 16-byte alignment take the kernel with per-lane loads."""
    m, n, k = 80, 96, 208
    a, b, want = operands(1, m, n, k, ta, tb, 7)
    buf = torch.empty(a.numel() + 1, device=DEV, dtype=torch.bfloat16)
    buf[1:] = a.reshape(-1)
    shifted = buf[1:].view(a.shape)
    out = HipRuntime.gemm(shifted, b, ta, tb, torch.float32)
    assert err(out, want) <= bound(k, torch.float32)


def test_grouped_small_grid():
    ends = [256, 256, 768]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(9)
    a = torch.randn((768, 320), generator=gen, device=DEV).to(torch.bfloat16)
    w = torch.randn((3, 208, 320), generator=gen, device=DEV).to(torch.bfloat16)
    groups = HipRuntime.upload_group_ends(ends)
    out = HipRuntime.grouped_nt(a, w, groups, torch.float32)
    want = torch.cat([a[:256].double() @ w[0].double().t().contiguous(), a[256:].double() @ w[2].double().t().contiguous()])
    assert err(out, want) <= bound(320, torch.float32)
    groups.close()
