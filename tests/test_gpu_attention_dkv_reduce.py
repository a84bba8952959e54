"""GPU parity: the sum of the dK/dV splits' F32 partials, which rounds, rotates and stores what the
unsplit kernel does. Shapes: grids small enough for 8 splits by themselves, ragged key counts, every
head width; the rows output must equal the planes followed by qkv_rope_merge bit for bit, and the
F32 planes the unsplit result up to the order of the additions (at most 8 terms more a sum: 1e-5 of
a row's norm, as for 2 and 4 splits)."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, dev_f32
import oracle
from rust_ascend_hip import HipRuntime, RotaryLayout

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 2, 512, 128), (1, 2, 1, 577, 64), (2, 2, 2, 520, 32), (1, 4, 1, 700, 16)]  # b, hq, hkv, s, d


def inputs(b, hq, hkv, s, d):
    g = torch.Generator(device=DEV)
    g.manual_seed(s + d)
    q, k, v, do = (torch.randn(shape, generator=g, device=DEV).to(torch.bfloat16)
                   for shape in ((b, hq, s, d), (b, hkv, s, d), (b, hkv, s, d), (b, hq, s, d)))
    o, lse = HipRuntime.attention_forward(q, k, v, d ** -0.5, True)
    return q, k, v, o, lse, do


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_small_grid_splits_match_unsplit(shape, monkeypatch):
    d = shape[-1]
    args = inputs(*shape)
    monkeypatch.delenv("HK_ATTN_DKV_SPLITS", raising=False)
    got = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.float32)
    got16 = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.bfloat16)
    monkeypatch.setenv("HK_ATTN_DKV_SPLITS", "1")
    want = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.float32)
    for name, a, b, c in zip(("dq", "dk", "dv"), got, want, got16):
        err = (a - b).reshape(-1, d).norm(dim=1) / b.reshape(-1, d).norm(dim=1).clamp_min(1e-30)
        assert float(err.max()) <= 1e-5, (name, float(err.max()))
        assert torch.equal(a.to(torch.bfloat16), c), name


@pytest.mark.parametrize("shape", SHAPES[:2], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("splits", ["2", None])
def test_rows_output_bit_exact_with_merge(shape, layout, splits, monkeypatch):
    d = shape[-1]
    args = inputs(*shape)
    if splits is None:
        monkeypatch.delenv("HK_ATTN_DKV_SPLITS", raising=False)
    else:
        monkeypatch.setenv("HK_ATTN_DKV_SPLITS", splits)
    cos, sin = (dev_f32(t) for t in oracle.rope_tables(np.arange(shape[3]), d, 5e5))
    rows = HipRuntime.attention_backward_qkv_rows(*args, cos, sin, d ** -0.5, True, layout=RotaryLayout(layout))
    dq, dk, dv = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.bfloat16)
    assert torch.equal(rows, HipRuntime.qkv_rope_merge(dq, dk, dv, cos, sin, RotaryLayout(layout)))


def test_eight_splits_past_the_workspace_limit_become_four(monkeypatch):
    """A limit that holds the partial sums of four splits but not of eight: four, with the stored dS, not the
    unsplit recompute form."""
    shape = SHAPES[0]
    d = shape[-1]
    args = inputs(*shape)

    def run(splits=None, limit=None):
        for name, value in (("HK_ATTN_DKV_SPLITS", splits), ("HK_WORKSPACE_LIMIT", limit)):
            monkeypatch.delenv(name, raising=False) if value is None else monkeypatch.setenv(name, str(value))
        HipRuntime.trim_workspace()
        return HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.float32), HipRuntime.workspace_size()
    _, eight = run()
    four, limit = run(splits=4)
    assert limit < eight
    got, held = run(limit=limit)
    assert held == limit
    for a, b in zip(got, four):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", SHAPES + [(2, 4, 4, 300, 64)], ids=lambda s: "x".join(map(str, s)))
def test_eight_splits_forced(shape, monkeypatch):
    """HK_ATTN_DKV_SPLITS=8: the choice of the small grids, and five query steps over eight splits (empty shares)."""
    d = shape[-1]
    args = inputs(*shape)
    monkeypatch.delenv("HK_ATTN_DKV_SPLITS", raising=False)
    own = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.float32)
    held = {}
    for splits in ("4", "8"):
        monkeypatch.setenv("HK_ATTN_DKV_SPLITS", splits)
        HipRuntime.trim_workspace()
        got = HipRuntime.attention_backward(*args, d ** -0.5, True, grad_dtype=torch.float32)
        held[splits] = HipRuntime.workspace_size()
    assert held["8"] > held["4"]
    for a, b in zip(got, own):
        err = (a - b).reshape(-1, d).norm(dim=1) / b.reshape(-1, d).norm(dim=1).clamp_min(1e-30)
        assert float(err.max()) <= 1e-5
        assert shape not in SHAPES or torch.equal(a, b)
