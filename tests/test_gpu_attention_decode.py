"""GPU parity of the attention forward for a few queries per head (the generation step), whose keys are
split over workgroups: against float64 attention on the same BF16 values.

O: P and O are each rounded to BF16 (2^-9 of a value), so its relative 2-norm error stays below 2^-8.
lse: F32 scores of a D-long BF16 dot product and an F32 sum of exponentials: absolute 1e-5 x the largest
score magnitude."""
import os

import pytest
import torch

from gpu_util import DEV
from rust_ascend_hip import HipRuntime

pytestmark = pytest.mark.gpu


def reference(q, k, v, scale, causal, qs, ks):
    hq, m, hkv, n = q.shape[1], q.shape[2], k.shape[1], k.shape[2]
    kk, vv = (t.double().repeat_interleave(hq // hkv, 1) for t in (k, v))
    s = torch.matmul(q.double(), kk.transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(ks + torch.arange(n, device=DEV)[None, :] > qs + torch.arange(m, device=DEV)[:, None], float("-inf"))
    lse = torch.logsumexp(s, -1)
    return torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), vv), lse


def inputs(b, hq, hkv, m, n, d, seed=3):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return [torch.randn(s, generator=g, device=DEV).to(torch.bfloat16) for s in ((b, hq, m, d), (b, hkv, n, d), (b, hkv, n, d))]


def check(o, lse, q, k, v, scale, causal, qs, ks):
    want, want_lse = reference(q, k, v, scale, causal, qs, ks)
    assert ((o.double() - want).norm() / want.norm().clamp_min(1e-30)).item() <= 2 ** -8
    seen = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse), seen) and bool((lse[~seen] == float("-inf")).all())
    if bool(seen.any()):
        assert (lse.double() - want_lse)[seen].abs().max().item() <= 1e-5 * max(1.0, want_lse[seen].abs().max().item() * 4)
    assert bool((o[~seen] == 0).all())


# query rows per KV head 1, 16, 17, 32, 33 and 64; keys below, at and past a 32-key tile and a split
@pytest.mark.parametrize("b,hq,hkv,m,n", [(1, 1, 1, 1, 1), (1, 4, 4, 1, 31), (2, 8, 2, 1, 33), (1, 16, 1, 1, 200), (3, 17, 1, 1, 4097),
                                          (1, 8, 2, 4, 640), (1, 32, 8, 8, 1000), (2, 33, 1, 1, 129), (1, 16, 2, 8, 5000),
                                          (40, 8, 8, 2, 257)])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_attention(b, hq, hkv, m, n, d):
    q, k, v = inputs(b, hq, hkv, m, n, d)
    for causal, qs, ks in ((True, max(n - m, 0), 0), (False, 0, 0), (True, n // 2, 0), (True, 0, min(n, 2))):
        print(f"decode {b}x{hq}/{hkv} m{m} n{n} d{d} causal {causal} {qs} {ks}", flush=True)
        o, lse = HipRuntime.attention_forward(q, k, v, d ** -0.5, causal, qs, ks)
        check(o, lse, q, k, v, d ** -0.5, causal, qs, ks)


# 33 to 64 query rows on either side of the line between the two kernels, told apart by the workspace: the
# split decode keeps its partials there, the ping-pong kernel takes none
@pytest.mark.parametrize("hq,hkv,m,n,d,decodes", [(4, 4, 64, 512, 128, False), (4, 4, 64, 520, 128, True), (4, 4, 33, 192, 64, False),
                                                  (4, 4, 33, 200, 64, None), (8, 4, 24, 384, 128, False), (4, 4, 32, 512, 128, True),
                                                  (4, 4, 64, 2048, 64, True), (8, 4, 32, 2000, 128, True)])
def test_rows_where_the_query_kernel_is_faster(hq, hkv, m, n, d, decodes):
    q, k, v = inputs(2, hq, hkv, m, n, d)
    HipRuntime.trim_workspace()
    print(f"rows {hq}/{hkv} m{m} n{n} d{d}", flush=True)
    o, lse = HipRuntime.attention_forward(q, k, v, d ** -0.5, True, n - m, 0)
    if decodes is not None:
        assert (HipRuntime.workspace_size() > 0) == decodes
    check(o, lse, q, k, v, d ** -0.5, True, n - m, 0)


def test_decode_attention_f32_surface_and_negative_scale():
    q, k, v = (t.float() for t in inputs(2, 8, 2, 1, 700, 128))
    o, lse = HipRuntime.attention_forward(q, k, v, -0.1, True, 699, 0, out_dtype=torch.float32)
    check(o, lse, q, k, v, -0.1, True, 699, 0)


def test_decode_attention_without_scratch_and_under_capture():
    """Where its partials may not be allocated (a limit, a capturing stream) the keys are not split."""
    q, k, v = inputs(1, 8, 2, 1, 4096, 128)
    scale = 128 ** -0.5
    HipRuntime.trim_workspace()
    os.environ["HK_WORKSPACE_LIMIT"] = "64"
    try:
        o, lse = HipRuntime.attention_forward(q, k, v, scale, True, 4095, 0)
        assert HipRuntime.workspace_size() == 0
    finally:
        del os.environ["HK_WORKSPACE_LIMIT"]
    check(o, lse, q, k, v, scale, True, 4095, 0)
    HipRuntime.set_async(True)
    try:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            o, lse = HipRuntime.attention_forward(q, k, v, scale, True, 4095, 0)
        assert HipRuntime.workspace_size() == 0
        for _ in range(3):
            o.zero_()
            graph.replay()
            torch.cuda.synchronize()
            check(o, lse, q, k, v, scale, True, 4095, 0)
    finally:
        HipRuntime.set_async(False)
