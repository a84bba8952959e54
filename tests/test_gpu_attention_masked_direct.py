"""GPU parity: the materialized attention with its scores in registers, at the edges of its split of the
keys (fewer blocks than waves, four and eight waves, the last key count it takes and the next), of its
widths (a half column step, more than one chunk of output columns, an odd tile, the last width sum and
the next), with BF16 operands and results, and off 16-byte alignment, against float64.

P, dS and the operands are BF16 in the products: relative 2-norm errors below 2^-7, as for the row passes;
a BF16 result adds its own rounding of 2^-9, inside the same bound. dMask is F32 throughout: 1e-5, as there."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime
from test_gpu_attention_masked_rows import case, reference, rel

pytestmark = pytest.mark.gpu

NAMES = ("o", "dq", "dk", "dv", "dmask")


@pytest.mark.parametrize("n,d,dv", [(32, 16, 16), (96, 80, 144), (1152, 48, 96), (1184, 96, 80), (2304, 144, 16), (2336, 32, 32),
                                    (64, 512, 256), (64, 512, 272)])
@pytest.mark.parametrize("mask_grad", [True, False])
def test_edges(n, d, dv, mask_grad):
    q, k, v, dy, mask = case(2, 4, 2, 80, n, d, dv, seed=n + d)
    print(f"masked direct n {n} d {d} dv {dv} grad {mask_grad}", flush=True)
    o = HipRuntime.attention_masked_forward(q, k, v, d ** -0.5, mask)
    got = (o,) + tuple(HipRuntime.attention_masked_backward(q, k, v, mask, dy, d ** -0.5, mask_grad=mask_grad))
    for name, a, b in zip(NAMES, got, reference(q, k, v, dy, mask, d ** -0.5)):
        if a is not None:
            assert rel(a, b) <= (1e-5 if name == "dmask" else 2 ** -7), name


@pytest.mark.parametrize("shift", [0, 1])
def test_bf16_operands_and_results(shift):
    """Operands one element off their alignment take the GEMMs and give the same to rounding."""
    args = [t.to(torch.bfloat16) for t in case(1, 4, 2, 48, 160, 48, 64)[:4]]
    mask = case(1, 4, 2, 48, 160, 48, 64)[4]
    want = reference(*[t.float() for t in args], mask, 0.2)
    moved = []
    for t in args:
        buf = torch.empty(t.numel() + 8, device=DEV, dtype=t.dtype)
        moved.append(buf[shift:shift + t.numel()].view(t.shape).copy_(t))
    q, k, v, dy = moved
    o = HipRuntime.attention_masked_forward(q, k, v, 0.2, mask, out_dtype=torch.bfloat16)
    got = (o,) + tuple(HipRuntime.attention_masked_backward(q, k, v, mask, dy, 0.2, grad_dtype=torch.bfloat16))
    for name, a, b in zip(NAMES, got, want):
        if a is not None:
            assert rel(a, b) <= 2 ** -7, name


def test_extreme_values():
    """Infinities of the mask and rows without a key keep to their rows; the mask's lowest value is finite."""
    q, k, v, dy, mask = case(1, 2, 1, 32, 96, 32, 32)
    mask[0, 0, 1] = float("-inf")                            # no key: NaN
    mask[0, 0, 2] = torch.finfo(torch.float32).min           # every key at the lowest value: equal weights
    mask[0, 1, 3, 5] = float("inf")                          # NaN
    want = reference(q, k, v, dy, mask, 0.2)[0]
    o = HipRuntime.attention_masked_forward(q, k, v, 0.2, mask)
    nan_rows = torch.isnan(o).all(-1)
    assert torch.equal(nan_rows, torch.isnan(want).all(-1)) and int(nan_rows.sum()) == 2
    assert int(torch.isnan(o).sum()) == 2 * o.shape[-1]
    ok = ~nan_rows
    assert rel(o[ok], want[ok]) <= 2 ** -7
    dq, dk, dv, dmask = HipRuntime.attention_masked_backward(q, k, v, mask, dy, 0.2, mask_grad=True)
    assert torch.equal(torch.isnan(dq).any(-1), nan_rows) and torch.equal(torch.isnan(dmask).any(-1), nan_rows)


def test_small_probabilities_keep_f32_accuracy():
    """dMask of keys far below the row's maximum, element by element. The scores are 0 and the maximum is 0, so the
    exponents are the mask's values, exactly; dP is small whole numbers, exact too. What is left is the
    exponential (1.5 ulp), the row's sum and reciprocal, dP - rowsum(P dP) (at least 1 here, values up to 8) and
    two products: 8 roundings of 2^-24, 5e-7 of each element. An exponent rounded once more, at 2^-24 of up
    to 115, would be off by 2e-6."""
    m, n, d = 32, 96, 16
    q = torch.zeros((1, 2, m, d), device=DEV)
    k, v = (torch.zeros((1, 1, n, d), device=DEV) for _ in range(2))
    dy = torch.zeros((1, 2, m, d), device=DEV)
    g = torch.Generator(device=DEV)
    g.manual_seed(2)
    dy[..., 0] = 1.0
    v[..., 0] = torch.randint(2, 7, (n,), generator=g, device=DEV).float()
    v[0, 0, 0, 0] = 0.0  # the one heavy key: rowsum(P dP) stays near 0
    mask = -80 + 60 * torch.rand((1, 2, m, n), generator=g, device=DEV)
    mask[..., 0] = 0.0
    got = HipRuntime.attention_masked_backward(q, k, v, mask, dy, 1.0, mask_grad=True)[3].double()
    want = reference(q, k, v, dy, mask, 1.0)[4]
    far = ((got - want).abs() / want.abs())[..., 1:]
    assert far.max().item() <= 5e-7
