"""GPU parity of the fused cross entropy (log-softmax with the NLL row term in one pass, the logits'
gradient in one pass) with its composition, nll_loss(log_softmax(logits)), and with float64.

Log-probabilities and gradients differ from the composition by the order of the row's sum of
exponentials alone: F32 values within 2^-20 of the largest log-probability."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime, HkError, LossReduction, nn

pytestmark = pytest.mark.gpu


def inputs(rows, classes, dtype=torch.int64, seed=4):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    x = torch.randn((rows, classes), generator=g, device=DEV) * 3
    t = torch.randint(0, classes, (rows,), generator=g, device=DEV).to(dtype)
    w = torch.rand((classes,), generator=g, device=DEV) + 0.5
    return x, t, w


def composed(x, t, w, reduction, ignore):
    y = nn.log_softmax(x)
    return nn.nll_loss(y, t, torch.ones_like(x[0]) if w is None else w, reduction, ignore)


# widths: one chunk or less, every row alignment, edges of each register count and of the widest, past it
@pytest.mark.parametrize("classes", [1, 2, 3, 5, 7, 64, 1001, 1024, 1027, 4096, 4098, 8193, 16384, 16387, 32000, 32771, 65536, 65539])
@pytest.mark.parametrize("reduction", [LossReduction.None_, LossReduction.Mean, LossReduction.Sum])
@pytest.mark.parametrize("weighted", [False, True])
def test_fused_matches_composed(classes, reduction, weighted):
    rows = 9
    x, t, w = inputs(rows, classes, torch.int32 if weighted else torch.int64)
    t[3] = 0
    w, ignore = (w if weighted else None), (0 if classes > 1 else None)
    x[1, classes // 2] = 40.0
    if classes > 2:
        x[5, 1:] = float("-inf")
        x[2, 0] = torch.finfo(torch.float32).min
    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    fused = nn._cross_entropy(a, t, w, reduction, ignore)
    want = composed(b, t, w, reduction, ignore)
    g = torch.linspace(0.5, 1.5, fused.numel(), device=DEV)
    (da,), (db,) = torch.autograd.grad(fused, [a], g), torch.autograd.grad(want, [b], g)
    for got, ref in ((fused.detach(), want.detach()), (da, db)):
        finite = torch.isfinite(ref)
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        assert torch.equal(got[~finite & ~torch.isnan(ref)], ref[~finite & ~torch.isnan(ref)])
        scale = ref[finite].abs().max().clamp_min(1.0) if bool(finite.any()) else 1.0
        assert bool(((got - ref).abs()[finite] <= 2 ** -20 * scale).all())


def test_logits_may_change_after_the_forward():
    """The backward reads the saved log-probabilities, never the logits."""
    x, t, _ = inputs(5, 300)
    leaf = x.clone().requires_grad_(True)
    logits = leaf * 1.0
    loss = nn.cross_entropy(logits, t)
    with torch.no_grad():
        logits.zero_()
    (got,) = torch.autograd.grad(loss, [leaf])
    want = (torch.softmax(x.double(), -1) - torch.nn.functional.one_hot(t, 300)) / 5
    assert ((got.double() - want).norm() / want.norm()).item() <= 1e-6


def test_unaligned_logits_and_bad_labels():
    x, t, w = inputs(6, 130)
    buf = torch.empty(x.numel() + 1, device=DEV)
    buf[1:] = x.reshape(-1)
    shifted = buf[1:].view(x.shape)
    loss, y, total = HipRuntime.cross_entropy(shifted, t, w)
    want = torch.nn.functional.cross_entropy(x.double(), t, weight=w.double())
    assert abs(loss.item() - want.item()) <= 1e-6 * abs(want.item())
    dy = torch.empty(x.numel() + 1, device=DEV)
    ys = dy[1:].view(x.shape).copy_(y)
    g = torch.ones(1, device=DEV)
    assert torch.equal(HipRuntime.cross_entropy_backward(g, ys, t, w, total), HipRuntime.cross_entropy_backward(g, y, t, w, total))
    t[2] = 130
    with pytest.raises(HkError):
        nn.cross_entropy(x, t)
    with pytest.raises(HkError):
        nn.cross_entropy(x[0:1], t)


# the last widths of the two passes and the first of the one, on either row alignment
@pytest.mark.parametrize("classes,two_passes", [(3, True), (100, True), (255, True), (256, True), (257, False), (300, True),
                                                (768, True), (769, False), (772, False)])
def test_narrow_rows_take_the_faster_passes(classes, two_passes):
    """Rows too narrow for the one-pass kernel run the log-softmax and the NLL one after the other: the bits of
    that composition (the widths past the line agree with it as above)."""
    x, t, w = inputs(67, classes)
    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    fused, want = nn.weighted_cross_entropy(a, t, w), composed(b, t, w, LossReduction.Mean, None)
    _, y, _ = HipRuntime.cross_entropy(x, t, w)
    logp = nn.log_softmax(x)
    if two_passes:
        assert torch.equal(y, logp) and torch.equal(fused, want)
    assert bool(((y - logp).abs() <= 2 ** -20 * logp.abs().max()).all())
    assert abs((fused - want).item()) <= 2 ** -20 * abs(want.item())
    (da,), (db,) = torch.autograd.grad(fused, [a]), torch.autograd.grad(want, [b])
    assert ((da - db).norm() / db.norm()).item() <= 2 ** -20
    x64 = torch.log_softmax(x.double(), -1)
    assert ((logp.double() - x64).norm() / x64.norm()).item() <= 1e-6
