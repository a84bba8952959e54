"""GPU parity of the GEMMs that 256x256 tiles cannot fill, over small and ragged shapes: K split over
workgroups or not, every transpose read in place, at edges of tiles and of K stages (each tile shape in each
of its forms: test_gpu_gemm_tiles.py).

Against float64 products of the same BF16 values. F32 outputs: a sum of K products rounded to F32 at
each of K steps in the worst order has a relative 2-norm error of at most about sqrt(K) 2^-24 against
the rounding's random walk; four times that is allowed. BF16 outputs add one rounding, 2^-9 of each
value."""
import os

import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime, runtime

pytestmark = pytest.mark.gpu

# batch, M, N, K: one row tile and skinny weights (32x64 tiles, split K), tails of several tile shapes,
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


# ------------------------------------------------------------------ fused epilogues below a full grid

def bf(shape, seed, scale=1.0):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return (torch.randn(shape, generator=gen, device=DEV) * scale).to(torch.bfloat16)


def call(name, *args):
    runtime._call(name, *(runtime.desc(t) if isinstance(t, torch.Tensor) else t for t in args))


def rounded(t):
    return t.to(torch.bfloat16).double()


# a product that lands within its sum's error of a BF16 tie rounds the other way in float64: one BF16
# step (2^-8) of few values, so the rounded results are compared to 2^-8 of the norm
@pytest.mark.parametrize("t,h,f", [(130, 264, 96), (512, 2048, 1408), (1000, 1024, 2944), (1, 128, 16)])
def test_small_fused_ffn(t, h, f):
    x, wg, wu, wd, res = bf((t, h), 1), bf((f, h), 2, h ** -0.5), bf((f, h), 3, h ** -0.5), bf((h, f), 4, 0.1), bf((t, h), 5)
    w_gu = torch.stack([wg.view(f // 16, 16, h), wu.view(f // 16, 16, h)], 1).reshape(2 * f, h).contiguous()
    gate, up, act = (torch.empty((t, f), device=DEV, dtype=torch.bfloat16) for _ in range(3))
    print(f"fused ffn {t}x{h}x{f}", flush=True)
    call("hk_swiglu_projection", x, w_gu, gate, up, act)
    g = rounded(x.double() @ wg.double().t().contiguous())
    u = rounded(x.double() @ wu.double().t().contiguous())
    assert err(gate, g) <= 2 ** -8 and err(up, u) <= 2 ** -8
    assert torch.equal(act, HipRuntime.silu_mul(gate, up))
    if h % 16 == 0:
        y = torch.empty((t, h), device=DEV, dtype=torch.bfloat16)
        call("hk_linear_residual", act, wd, res, y)
        assert err(y, rounded(act.double() @ wd.double().t().contiguous()) + res.double()) <= 2 ** -8
    dy, dgu = bf((t, h), 6), torch.empty((t, 2 * f), device=DEV, dtype=torch.bfloat16)
    call("hk_swiglu_projection_backward", dy, wd, gate, up, dgu)
    dm = dy.double() @ wd.double()
    sg = torch.sigmoid(gate.double())
    d = dgu.view(t, f // 16, 2, 16)
    assert err(d[:, :, 0].reshape(t, f), dm * up.double() * sg * (1 + gate.double() * (1 - sg))) <= 2 ** -7
    assert err(d[:, :, 1].reshape(t, f), dm * gate.double() * sg) <= 2 ** -7


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("b,s,h,hq,hkv", [(1, 512, 2048, 16, 4), (2, 72, 264, 2, 1), (1, 1, 128, 1, 1), (3, 100, 1024, 8, 8)])
def test_small_fused_qkv_rope(b, s, h, hq, hkv, layout):
    """The rotated head planes of the fused projection against the BF16 product split and rotated."""
    x, w = bf((b * s, h), 1), bf(((hq + 2 * hkv) * 128, h), 2, h ** -0.5)
    ang = torch.arange(s, device=DEV)[:, None] * 5e5 ** (-torch.arange(0, 128, 2, device=DEV) / 128)
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    print(f"fused qkv {b}x{s}x{h} {hq}/{hkv} layout {layout}", flush=True)
    q, k, v = HipRuntime.qkv_projection_rope(x, w, cos, sin, b, hq, hkv, layout)
    rows = (x.double() @ w.double().t().contiguous()).to(torch.bfloat16).view(b, s, -1)
    for got, want in zip((q, k, v), HipRuntime.qkv_rope_split(rows, cos, sin, hq, hkv, layout)):
        assert err(got, want.double()) <= 2 ** -8
