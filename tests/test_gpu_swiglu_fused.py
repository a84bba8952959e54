"""GPU parity of the FP32 SwiGLU block as one node with its composition of linears and silu_mul.

The products are the same; where one splits its contraction or adds the two halves of dX in another order,
a last-bit difference can move a BF16 rounding of the next operand (2^-9 of that value). Few values move, so
results agree to 2^-12 of their norm."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime, HkError, nn

pytestmark = pytest.mark.gpu


def rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def inputs(m, k, h, n, seed=8):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    r = lambda *s, std=1.0: (torch.randn(s, generator=g, device=DEV) * std)  # noqa: E731
    return r(m, k), r(h, k, std=k ** -0.5), r(h, k, std=k ** -0.5), r(n, h, std=h ** -0.5), r(m, n)


def composed(x, gate, up, down):
    return nn.linear_bf16_fp32(nn.silu_mul(nn.linear_bf16_fp32(x, gate), nn.linear_bf16_fp32(x, up)), down)


# one tile and less, K tails, split K, the gate/up boundary inside a tile (H % 256, H % 64), full grids
@pytest.mark.parametrize("m,k,h,n", [(16, 16, 16, 16), (48, 80, 112, 144), (16, 1024, 2816, 1024), (272, 400, 1040, 208),
                                     (512, 1024, 2832, 1024), (2000, 2048, 5632, 2048)])
def test_fused_swiglu_matches_composition(m, k, h, n):
    *ins, dy = inputs(m, k, h, n)
    a = [t.clone().requires_grad_(True) for t in ins]
    b = [t.clone().requires_grad_(True) for t in ins]
    print(f"swiglu {m}x{k}x{h}x{n}", flush=True)
    y, want = nn.swiglu_bf16_fp32(*a), composed(*b)
    assert rel(y, want) <= 2 ** -12
    for name, got, ref in zip(("dx", "dgate", "dup", "ddown"), torch.autograd.grad(y, a, dy), torch.autograd.grad(want, b, dy)):
        assert got.is_contiguous() and rel(got, ref) <= 2 ** -12, name


def test_fused_swiglu_inputs():
    x, gate, up, down, dy = inputs(32, 64, 48, 80)
    want = composed(x, gate, up, down)
    buf = torch.empty(x.numel() + 1, device=DEV)
    shifted = buf[1:].view(x.shape).copy_(x)  # off 16-byte alignment: the composition
    assert torch.equal(nn.swiglu_bf16_fp32(shifted, gate, up, down), want)
    w = gate.clone().requires_grad_(True)  # one weight for gate and up: both gradients reach it
    y = nn.swiglu_bf16_fp32(x, w, w, down)
    dbuf = torch.empty(dy.numel() + 1, device=DEV)
    (g1,) = torch.autograd.grad(y, [w], dbuf[1:].view(dy.shape).copy_(dy))
    w2 = gate.clone().requires_grad_(True)
    (g2,) = torch.autograd.grad(composed(x, w2, w2, down), [w2], dy)
    assert rel(g1, g2) <= 2 ** -12
    with pytest.raises(ValueError):
        nn.swiglu_bf16_fp32(x, gate, up[:, :48], down)
    with pytest.raises(HkError):
        HipRuntime.swiglu_bf16_fp32(x.to(torch.bfloat16), gate, up, down)
