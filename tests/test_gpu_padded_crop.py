"""GPU parity: padded linear products whose GEMM stores only the logical rows and columns, at every
remainder of the columns modulo 4, on 32x64 and 64x64 tiles, split, and on the 256x256 tiles (the tiles
between: test_gpu_gemm_tiles.py), with K off its stages; and row padding of odd lengths. Against float64 on the BF16-rounded operands: F32 accumulation
over K terms, so 1e-5 of the norm; nothing outside the logical output is written."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import Transpose, nn, runtime

pytestmark = pytest.mark.gpu

SHAPES = [(1, 515, 1), (17, 33, 70), (100, 700, 301), (300, 600, 1030), (33, 4000, 95), (777, 1001, 515), (4083, 70, 4091)]


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_padded_linear_at_remainders(m, k, n):
    g = torch.Generator(device=DEV)
    g.manual_seed(m + k + n)
    x, w, dy = (torch.randn(s, generator=g, device=DEV) for s in ((m, k), (n, k), (m, n)))
    xr, wr, dr = (t.to(torch.bfloat16).double() for t in (x, w, dy))
    x.requires_grad_(), w.requires_grad_()
    print(f"padded {m} {k} {n}", flush=True)
    y = nn.linear_padded_bf16_fp32(x, w)
    y.backward(dy)
    for name, a, b in (("y", y, xr @ wr.t()), ("dx", x.grad, dr @ wr), ("dw", w.grad, dr.t() @ xr)):
        assert rel(a.detach(), b) <= 1e-5, name


@pytest.mark.parametrize("ta", [Transpose.No, Transpose.Yes])
@pytest.mark.parametrize("tb", [Transpose.No, Transpose.Yes])
def test_batched_transposes(ta, tb):
    b, m, k, n = 3, 130, 77, 201
    g = torch.Generator(device=DEV)
    g.manual_seed(5)
    x = torch.randn((b, k, m) if ta else (b, m, k), generator=g, device=DEV)
    w = torch.randn((b, n, k) if tb else (b, k, n), generator=g, device=DEV)
    xr, wr = x.to(torch.bfloat16).double(), w.to(torch.bfloat16).double()
    want = torch.matmul(xr.transpose(1, 2).contiguous() if ta else xr, wr.transpose(1, 2).contiguous() if tb else wr)
    assert rel(nn.matmul_padded_bf16_fp32(x, w, ta, tb), want) <= 1e-5


def test_unaligned_output_and_neighbours():
    m, k, n = 50, 48, 37
    g = torch.Generator(device=DEV)
    g.manual_seed(9)
    x, w = torch.randn((m, k), generator=g, device=DEV), torch.randn((n, k), generator=g, device=DEV)
    buf = torch.full((m * n + 9,), 7.0, device=DEV)
    xp = torch.empty((64, 48), device=DEV, dtype=torch.bfloat16)
    wp = torch.empty((48, 48), device=DEV, dtype=torch.bfloat16)
    out = buf[5:5 + m * n].view(m, n)
    runtime._call("hk_gemm_padded_bf16_fp32", runtime.desc(x), runtime.desc(w), 0, 1, runtime.desc(out), runtime.desc(xp),
                  runtime.desc(wp))
    assert rel(out, x.to(torch.bfloat16).double() @ w.to(torch.bfloat16).double().t()) <= 1e-5
    assert bool((buf[:5] == 7).all()) and bool((buf[5 + m * n:] == 7).all())
