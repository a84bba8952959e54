"""GPU: a captured call holds no optional scratch, however much the context's workspace holds already.

The split forms of these calls keep F32 partial sums in the workspace, which a later call may grow or trim
(free). Captured after a warm-up, each must record the unsplit form: bit for bit what a run without scratch
gives, and not what the eager split gives. Only once that is shown is the workspace grown and trimmed and
the graph replayed again."""
import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime, runtime

pytestmark = pytest.mark.gpu


def randn(shape, seed, dtype):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV).to(dtype)


def gemm():
    a, b = randn((16, 6096), 1, torch.bfloat16), randn((1200, 6096), 2, torch.bfloat16)
    out = torch.zeros((16, 1200), device=DEV)
    return out, lambda: HipRuntime.gemm_into(a, b, 0, 1, out)


def linear_backward():
    x, w, dy = (randn(s, i, torch.bfloat16) for i, s in enumerate(((8192, 64), (48, 64), (8192, 48))))
    dx, dw = torch.zeros((8192, 64), device=DEV, dtype=torch.bfloat16), torch.zeros((48, 64), device=DEV)
    return dw, lambda: runtime._call("hk_linear_nt_backward", *(runtime.desc(t) for t in (x, w, dy, dx, dw)))


def matmul():
    a, b = randn((31, 4097), 1, torch.float32), randn((4097, 33), 2, torch.float32)
    out = torch.zeros((31, 33), device=DEV)
    return out, lambda: runtime._call("hk_tensor_matmul", *(runtime.desc(t) for t in (a, b, out)))


def decode():
    q, k, v = (randn(s, i, torch.bfloat16) for i, s in enumerate(((1, 8, 1, 128), (1, 2, 4096, 128), (1, 2, 4096, 128))))
    out = torch.zeros_like(q)
    held = {}

    def run():
        held["o"], held["lse"] = HipRuntime.attention_forward(q, k, v, 128 ** -0.5, True, 4095, 0)
        out.copy_(held["o"])
    return out, run


@pytest.mark.parametrize("make", [gemm, linear_backward, matmul, decode], ids=lambda f: f.__name__)
def test_warm_capture_takes_the_unsplit_form(make, monkeypatch):
    out, run = make()

    def result():
        out.zero_()
        run()
        torch.cuda.synchronize()
        return out.clone()
    HipRuntime.trim_workspace()
    monkeypatch.setenv("HK_WORKSPACE_LIMIT", "16")
    unsplit = result()
    assert HipRuntime.workspace_size() == 0
    monkeypatch.delenv("HK_WORKSPACE_LIMIT")
    split = result()
    warm = HipRuntime.workspace_size()
    assert warm > 0 and not torch.equal(split, unsplit)  # the two forms are told apart by their bits
    HipRuntime.set_async(True)
    try:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            run()
        assert HipRuntime.workspace_size() == warm
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, unsplit)  # no partial sums in the workspace, which is still the warm one
        assert torch.equal(result(), split)
        HipRuntime.trim_workspace()
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, unsplit)
            assert torch.equal(result(), split)
    finally:
        HipRuntime.set_async(False)


def test_scratch_does_not_depend_on_earlier_calls(monkeypatch):
    """A limit between two splits' needs: unsplit, whether or not the workspace already holds something."""
    out, run = gemm()
    full = 4 * 16 * 1200  # one F32 plane
    monkeypatch.setenv("HK_WORKSPACE_LIMIT", str(full * 2 + 4096))
    results = []
    for warm in (0, full, full * 2):
        HipRuntime.trim_workspace()
        if warm:
            # an F32 product off 16-byte alignment needs its transposed operand as scratch
            buf = randn((warm // 2 + 1,), 5, torch.bfloat16)
            a = buf[1:1 + warm // 2].view(16, warm // 32)
            HipRuntime.gemm(randn((16, 16), 6, torch.bfloat16), a, 0, 0, torch.float32)
            assert warm <= HipRuntime.workspace_size()
        run()
        torch.cuda.synchronize()
        results.append(out.clone())
    assert all(torch.equal(results[0], r) for r in results[1:])
