"""GPU parity of every output tile that the GEMM's rules can take below the 256x256 grids, in each form that it
has: plain in every transpose, K split, cropped, two outputs, a pair, each fused epilogue; and the F32
matmul's 64x64 and 128x128 tiles with 16- and 4-byte loads of either operand, split and unsplit. The rules
are asked first, so a shape that no longer reaches its tile fails here. Bounds as in the tests of the
small shapes, whose helpers these are."""
import pytest
import torch

import tile_cases as cases
from gpu_util import DEV
from rust_ascend_hip import HipRuntime, _lib, nn, runtime
from test_gpu_attention_masked_rows import case as masked_case, reference as masked_reference
from test_gpu_gemm_mid import bf, bound, call, err, operands, rounded
from test_gpu_matmul_f32 import check as check_f32, randn
from test_gpu_swiglu_fused import composed, inputs as swiglu_inputs, rel

pytestmark = pytest.mark.gpu

INF = 1 << 62


def cus():
    return torch.cuda.get_device_properties(DEV).multi_processor_count


def gemm_route(m, n, k, ta, dtype, batch=1, scratch=INF):
    r = _lib.load().hk_gemm_route(batch, m, n, k, ta, _lib.BF16 if dtype == torch.bfloat16 else _lib.F32, scratch, cus())
    return r % 256, r // 256


@pytest.mark.parametrize("tile", sorted(cases.PLAIN))
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_plain(tile, ta, tb):
    m, n, k = cases.PLAIN[tile]
    a, b, want = operands(1, m, n, k, ta, tb, tile)
    for dtype in (torch.float32, torch.bfloat16):
        assert gemm_route(m, n, k, ta, dtype) == (cases.T64 if ta and tile == cases.T32x64 else tile, 1)
        out = torch.full((m, n), float("nan"), device=DEV, dtype=dtype)
        HipRuntime.gemm_into(a, b, ta, tb, out)
        assert err(out, want) <= bound(k, dtype)


@pytest.mark.parametrize("tile", sorted(cases.SPLIT))
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split(tile, ta, tb):
    m, n, k, splits = cases.SPLIT[tile]
    a, b, want = operands(1, m, n, k, ta, tb, tile)
    for dtype in (torch.float32, torch.bfloat16):
        route = gemm_route(m, n, k, ta, dtype)
        assert route[1] > 1 and (ta or route == (tile, splits))
        out = torch.full((m, n), float("nan"), device=DEV, dtype=dtype)
        HipRuntime.gemm_into(a, b, ta, tb, out)
        assert err(out, want) <= bound(k, dtype)


@pytest.mark.parametrize("dims", cases.CROPPED, ids=lambda d: "x".join(map(str, d)))
def test_cropped(dims):
    m, k, n = dims
    up = lambda x: (x + 15) // 16 * 16  # noqa: E731
    x, w, dy = (torch.randn(s, generator=torch.Generator(DEV).manual_seed(i), device=DEV) for i, s in enumerate(((m, k), (n, k), (m, n))))
    routes = [gemm_route(up(m), up(n), up(k), 0, torch.float32), gemm_route(up(m), up(k), up(n), 0, torch.float32),
              gemm_route(up(n), up(k), up(m), 1, torch.float32)]
    for tile, route in zip(cases.CROPPED[dims], routes):
        assert tile is None or route == (tile, 1)
    x.requires_grad_(), w.requires_grad_()
    print(f"cropped {dims} {routes}", flush=True)
    y = nn.linear_padded_bf16_fp32(x, w)
    dx, dw = torch.autograd.grad(y, [x, w], dy)
    xr, wr, dr = (t.detach().to(torch.bfloat16).double() for t in (x, w, dy))
    for got, want, terms in ((y.detach(), xr @ wr.t(), k), (dx, dr @ wr, n), (dw, dr.t() @ xr, m)):
        assert err(got, want) <= bound(terms, torch.float32)


@pytest.mark.parametrize("tile", sorted(cases.TWO_OUTPUTS))
def test_two_outputs(tile):
    m, k, h = cases.TWO_OUTPUTS[tile]
    assert gemm_route(2 * h, k, m, 1, torch.float32, scratch=0) == (tile, 1)
    *ins, dy = swiglu_inputs(m, k, h, 48)
    a, b = ([t.clone().requires_grad_(True) for t in ins] for _ in range(2))
    print(f"two outputs {m} {k} {h}", flush=True)
    got = torch.autograd.grad(nn.swiglu_bf16_fp32(*a), a, dy)
    for name, g, ref in zip(("dx", "dgate", "dup", "ddown"), got, torch.autograd.grad(composed(*b), b, dy)):
        assert rel(g, ref) <= 2 ** -12, name


@pytest.mark.parametrize("tile", sorted(cases.PAIR))
def test_pair(tile):
    heads, rows, keys, d = cases.PAIR[tile]
    assert gemm_route(keys, d, rows, 1, torch.float32, batch=2 * heads, scratch=0) == (tile, 1)
    q, k, v, dy, mask = masked_case(1, heads, heads, rows, keys, d, d)
    print(f"pair {heads} {rows} {keys} {d}", flush=True)
    got = HipRuntime.attention_masked_backward(q, k, v, mask, dy, d ** -0.5)
    for g, want in zip(got[:3], masked_reference(q, k, v, dy, mask, d ** -0.5)[1:4]):
        assert err(g, want) <= 2 ** -7


@pytest.mark.parametrize("tile", sorted(cases.EPILOGUE))
def test_epilogues(tile):
    m, n, k = cases.EPILOGUE[tile]
    assert _lib.load().hk_epilogue_route(m, n, k, 0, cus()) == tile
    print(f"epilogues {m} {n} {k}", flush=True)
    x, w, res = bf((m, k), 1), bf((n, k), 2, k ** -0.5), bf((m, n), 3)
    y = torch.empty_like(res)
    call("hk_linear_residual", x, w, res, y)
    product = x.double() @ w.double().t().contiguous()
    assert err(y, rounded(product) + res.double()) <= 2 ** -8
    f = n // 2
    gate, up, act = (torch.empty((m, f), device=DEV, dtype=torch.bfloat16) for _ in range(3))
    call("hk_swiglu_projection", x, w, gate, up, act)  # w's rows: 16 of gate, 16 of up, in turn
    both = rounded(product).view(m, f // 16, 2, 16)
    assert err(gate, both[:, :, 0].reshape(m, f)) <= 2 ** -8 and err(up, both[:, :, 1].reshape(m, f)) <= 2 ** -8
    assert torch.equal(act, HipRuntime.silu_mul(gate, up))
    gate, up, wd = bf((m, n), 4), bf((m, n), 5), bf((k, n), 6, k ** -0.5)
    dgu = torch.empty((m, 2 * n), device=DEV, dtype=torch.bfloat16)
    call("hk_swiglu_projection_backward", x, wd, gate, up, dgu)
    dm, sg = x.double() @ wd.double(), torch.sigmoid(gate.double())
    got = dgu.view(m, n // 16, 2, 16)
    assert err(got[:, :, 0].reshape(m, n), dm * up.double() * sg * (1 + gate.double() * (1 - sg))) <= 2 ** -7
    assert err(got[:, :, 1].reshape(m, n), dm * gate.double() * sg) <= 2 ** -7


@pytest.mark.parametrize("tile", sorted(cases.QKV))
@pytest.mark.parametrize("layout", [0, 1])
def test_qkv_rope(tile, layout):
    s, hq, hkv, h = cases.QKV[tile]
    assert _lib.load().hk_epilogue_route(s, (hq + 2 * hkv) * 128, h, 1, cus()) == tile
    x, w = bf((s, h), 1), bf(((hq + 2 * hkv) * 128, h), 2, h ** -0.5)
    ang = torch.arange(s, device=DEV)[:, None] * 5e5 ** (-torch.arange(0, 128, 2, device=DEV) / 128)
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    print(f"qkv {s} {hq}/{hkv} {h} layout {layout}", flush=True)
    got = HipRuntime.qkv_projection_rope(x, w, cos, sin, 1, hq, hkv, layout)
    rows = (x.double() @ w.double().t().contiguous()).to(torch.bfloat16).view(1, s, -1)
    for g, want in zip(got, HipRuntime.qkv_rope_split(rows, cos, sin, hq, hkv, layout)):
        assert err(g, want.double()) <= 2 ** -8


@pytest.mark.parametrize("a,b", cases.F32, ids=str)
def test_f32_matmul(a, b):
    x, y = randn(a, 1), randn(b, 2)
    r = [_lib.load().hk_tensor_matmul_route(runtime.desc(x), runtime.desc(y), which, INF, cus()) for which in range(3)]
    assert tuple((v % 1024, v // 1024) for v in r) == cases.F32[(a, b)]
    print(f"f32 {a} @ {b}", flush=True)
    check_f32(x, y)
