"""GPU parity of the materialized attention's row passes (scale, mask, softmax, its gradient and the BF16
rounding in one kernel each up to 4096 keys, one kernel per step above) against float64.

P, dS and the operands are BF16 in the GEMMs: relative 2-norm errors below 2^-7 (two or three roundings of
2^-9 each). dMask is dS in F32 and both sides round its operands alike: what is left is F32 arithmetic, of
which an exponent of up to 16 matters most (its 2^-24 a dozen times over, in the scores' sum, the scale and
mask, the maximum and the exponential): 1e-5."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime

pytestmark = pytest.mark.gpu


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def case(b, hq, hkv, m, n, d, dv, seed=11):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    q, k, v, dy = (torch.randn(s, generator=g, device=DEV) for s in ((b, hq, m, d), (b, hkv, n, d), (b, hkv, n, dv), (b, hq, m, dv)))
    mask = torch.randn((b, hq, m, n), generator=g, device=DEV)
    mask[:, :, :, n - n // 4:] = float("-inf")
    mask[0, 0, 0, 1:] = torch.finfo(torch.float32).min  # one key left, the others at the type's lowest value
    return q, k, v, dy, mask


def reference(q, k, v, dy, mask, scale):
    r = q.shape[1] // k.shape[1]
    bf = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    qq, kk, vv, dd = bf(q), bf(k).repeat_interleave(r, 1), bf(v).repeat_interleave(r, 1), bf(dy)
    s = torch.matmul(qq, kk.transpose(-1, -2).contiguous()) * scale
    p = torch.softmax(s if mask is None else s + mask.double(), -1)
    dp = torch.matmul(dd, vv.transpose(-1, -2).contiguous())
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    fold = lambda t: t.view(k.shape[0], k.shape[1], r, *t.shape[2:]).sum(2)  # noqa: E731
    dst, pt = ds.transpose(-1, -2).contiguous(), p.transpose(-1, -2).contiguous()
    return (torch.matmul(p, vv), torch.matmul(ds, kk) * scale, fold(torch.matmul(dst, qq)) * scale, fold(torch.matmul(pt, dd)), ds)


# one chunk per lane, partial chunks, every register count, the last fused width and the first unfused
@pytest.mark.parametrize("n", [32, 288, 1056, 1504, 2080, 4096, 4128])
@pytest.mark.parametrize("with_mask,mask_grad", [(True, True), (True, False), (False, False)])
def test_masked_rows(n, with_mask, mask_grad):
    q, k, v, dy, mask = case(1, 4, 2, 48, n, 32, 48)
    mask = mask if with_mask else None
    print(f"masked rows n {n} mask {with_mask} grad {mask_grad}", flush=True)
    o = HipRuntime.attention_masked_forward(q, k, v, 0.2, mask)
    got = (o,) + tuple(HipRuntime.attention_masked_backward(q, k, v, mask, dy, 0.2, mask_grad=mask_grad))
    for name, a, b in zip(("o", "dq", "dk", "dv", "dmask"), got, reference(q, k, v, dy, mask, 0.2)):
        if a is not None:
            assert rel(a, b) <= (1e-5 if name == "dmask" else 2 ** -7), name


@pytest.mark.parametrize("n", [64, 4128])
def test_fully_masked_rows_are_nan(n):
    q, k, v, dy, mask = case(1, 2, 2, 16, n, 16, 16)
    mask[0, 1, 3] = float("-inf")
    o = HipRuntime.attention_masked_forward(q, k, v, 0.25, mask)
    bad = torch.isnan(o).all(-1)
    assert bool(bad[0, 1, 3]) and int(bad.sum()) == 1 and int(torch.isnan(o).sum()) == o.shape[-1]


def test_unaligned_mask():
    """A mask off 16-byte alignment takes the step-by-step kernels."""
    q, k, v, dy, mask = case(1, 2, 2, 16, 64, 16, 16)
    buf = torch.empty(mask.numel() + 1, device=DEV)
    buf[1:] = mask.reshape(-1)
    shifted = buf[1:].view(mask.shape)
    assert rel(HipRuntime.attention_masked_forward(q, k, v, 0.25, shifted), reference(q, k, v, dy, mask, 0.25)[0]) <= 2 ** -7
