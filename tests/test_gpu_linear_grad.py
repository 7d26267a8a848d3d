"""Gradient kernels of the straight-through linear (linear_grad_x / linear_grad_w) against float64 products of the
same codes and scales: edges of the 64 / 128 / 256-row tiles, rows that are not 16-byte aligned, every gradient type,
sums short enough for one stage and long enough to be split.

Bound: every product is exact in fp32 and the sums are fp32, so the normwise error is that of an fp32 sum of C terms,
at most about sqrt(3 C / 16) roundings of 2^-24 (three planes, 16 terms per matrix instruction) plus the rounding of
g * a_scale and the result's own: below 1e-6 for C <= 2048 (measured 0.3-4e-7); 16-bit outputs are the fp32 result
rounded once, bit for bit."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 8, 128), (5, 257, 129), (63, 65, 512), (129, 1000, 640), (300, 96, 2057),
                                   (2048, 136, 257), (70, 2040, 384)])
def test_linear_grads_match_float64(pkg, dev, m, n, k, dtype):
    ops = pkg.ops
    g = torch.Generator(device=dev).manual_seed(m * n + k)
    rand = lambda *s: torch.randn(s, generator=g, device=dev)  # noqa: E731
    k_pad = (k + 127) // 128 * 128
    qw, scale = ops.pack_ternary_i2s((rand(n, k) * 0.02), k_pad=k_pad)
    codes, a_scale = ops.quantize_activations_i8_per_token(rand(m, k) * (1 + rand(m, 1).abs()), k_pad=k_pad)
    gy = rand(m, n).to(dtype)
    t = ops.unpack_i2s(qw)[:, :k].double()
    gx = ops.linear_grad_x(qw, scale, gy, k, torch.float32)
    gw = ops.linear_grad_w(codes, a_scale, gy, k, torch.float32)
    assert _rel(gx, (gy.double() @ t) * scale.double()) <= 1e-6
    assert _rel(gw, (gy.double() * a_scale.double()[:, None]).t().contiguous() @ codes[:, :k].double()) <= 1e-6
    for out in (torch.bfloat16, torch.float16):
        assert torch.equal(ops.linear_grad_x(qw, scale, gy, k, out), gx.to(out))
        assert torch.equal(ops.linear_grad_w(codes, a_scale, gy, k, out), gw.to(out))


# One case for every form that the plan picks: each tile size, its tiles summed whole, all of them in parts, or only
# those past the last full round of workgroups; every edge ragged.
_FORMS = [
    ("x", torch.bfloat16, (70, 84, 69), (64, 128, "whole")), ("x", torch.bfloat16, (77, 787, 78), (64, 128, "parts")),
    ("x", torch.bfloat16, (7254, 74, 799), (128, 128, "whole")),
    ("x", torch.bfloat16, (962, 1697, 1163), (128, 128, "parts")),
    ("x", torch.bfloat16, (3867, 1265, 2116), (128, 128, "rest")),
    ("x", torch.bfloat16, (5831, 68, 2087), (256, 256, "whole")),
    ("x", torch.bfloat16, (1421, 5384, 1960), (256, 256, "parts")),
    ("x", torch.bfloat16, (3545, 1512, 4821), (256, 256, "rest")),
    ("x", torch.float32, (70, 84, 69), (64, 128, "whole")), ("x", torch.float32, (72, 211, 72), (64, 128, "parts")),
    ("x", torch.float32, (1691, 493, 4781), (64, 128, "rest")),
    ("x", torch.float32, (2382, 78, 3339), (128, 256, "whole")),
    ("x", torch.float32, (1374, 1547, 1960), (128, 256, "parts")),
    ("x", torch.float32, (3122, 325, 5264), (128, 256, "rest")),
    ("w", torch.bfloat16, (70, 84, 69), (64, 128, "whole")), ("w", torch.bfloat16, (226, 72, 71), (64, 128, "parts")),
    ("w", torch.bfloat16, (479, 3118, 2617), (64, 128, "rest")),
    ("w", torch.bfloat16, (75, 4729, 1722), (128, 256, "whole")),
    ("w", torch.bfloat16, (1541, 1266, 2224), (128, 256, "parts")),
    ("w", torch.bfloat16, (344, 6602, 2551), (128, 256, "rest")),
]


@pytest.mark.parametrize("which,dtype,size,form", _FORMS)
def test_every_tile_form_matches_float64(pkg, dev, which, dtype, size, form):
    ops, (m, n, k) = pkg.ops, size
    plan = (ctypes.c_int64 * 5)()
    ptr = ctypes.addressof(plan)
    pkg._lib.call("wfb_linear_grad_plan", m, n, k, 0 if dtype == torch.float32 else 1, ptr if which == "x" else None,
                  ptr if which == "w" else None)
    bi, bj, tiles, full, parts = plan
    how = "whole" if full == tiles else "rest" if full else "parts"
    assert (bi, bj, how) == form and (parts > 1) == (how != "whole")
    g = torch.Generator(device=dev).manual_seed(m)
    rand = lambda *s: torch.randn(s, generator=g, device=dev)  # noqa: E731
    k_pad = (k + 127) // 128 * 128
    gy = rand(m, n).to(dtype)
    # sums of C terms, P planes of 16 terms per matrix instruction: that many roundings of 2^-24, and two more
    planes, terms = (1 if dtype == torch.bfloat16 else 3, n) if which == "x" else (3, m)
    tol = 2.0 ** -24 * ((planes * terms / 16) ** 0.5 + 2)
    if which == "x":
        qw, scale = ops.pack_ternary_i2s(rand(n, k) * 0.02, k_pad=k_pad)
        got = ops.linear_grad_x(qw, scale, gy, k, torch.float32)
        want = (gy.double() @ ops.unpack_i2s(qw)[:, :k].double()) * scale.double()
    else:
        codes, a_scale = ops.quantize_activations_i8_per_token(rand(m, k) * (1 + rand(m, 1).abs()), k_pad=k_pad)
        got = ops.linear_grad_w(codes, a_scale, gy, k, torch.float32)
        want = (gy.double() * a_scale.double()[:, None]).t().contiguous() @ codes[:, :k].double()
    assert _rel(got, want) <= tol


@pytest.mark.parametrize("m,k", [(1, 20), (6, 20), (70, 131), (65, 127)])
def test_grad_w_codes_may_end_with_their_last_row(pkg, dev, m, k):
    """Rows 16-byte aligned whose storage ends with the last row's codes (no padding behind them)."""
    ops, n, ld = pkg.ops, 40, (k + 15) // 16 * 16
    g = torch.Generator(device=dev).manual_seed(k)
    flat = torch.randint(-127, 128, ((m - 1) * ld + k,), generator=g, device=dev, dtype=torch.int8)
    codes = flat.as_strided((m, k), (ld, 1))
    a_scale = torch.rand(m, generator=g, device=dev) + 0.1
    gy = torch.randn((m, n), generator=g, device=dev)
    want = (gy.double() * a_scale.double()[:, None]).t().contiguous() @ codes.double()
    assert _rel(ops.linear_grad_w(codes, a_scale, gy, k, torch.float32), want) <= 1e-6


@pytest.mark.parametrize("m", [520, 1030])
def test_grad_w_splits_only_the_last_tiles(pkg, dev, m):
    """605 tiles: 512 summed by one workgroup each and the last 93 in 2 or 5 parts, at ragged edges of both."""
    ops, n, k = pkg.ops, 6950, 2570
    g = torch.Generator(device=dev).manual_seed(m)
    codes, a_scale = ops.quantize_activations_i8_per_token(torch.randn((m, k), generator=g, device=dev), k_pad=2688)
    gy = torch.randn((m, n), generator=g, device=dev).to(torch.bfloat16)
    gw, gb = ops.linear_grad_w(codes, a_scale, gy, k, torch.float32, torch.float32)
    want = (gy.double() * a_scale.double()[:, None]).t().contiguous() @ codes[:, :k].double()
    assert float((gw - want).abs().max()) <= 1e-5 * float(want.abs().max()) and _rel(gw, want) <= 1e-6
    assert _rel(gb, gy.double().sum(0)) <= 1e-6


def test_non_finite_gradients_reach_the_products(pkg, dev):
    """An infinite or NaN gradient gives what an fp32 product gives: inf * code, NaN where a code is 0."""
    ops = pkg.ops
    m, n, k = 6, 40, 256
    g = torch.Generator(device=dev).manual_seed(3)
    qw, scale = ops.pack_ternary_i2s(torch.randn((n, k), generator=g, device=dev))
    codes, a_scale = ops.quantize_activations_i8_per_token(torch.randn((m, k), generator=g, device=dev))
    gy = torch.randn((m, n), generator=g, device=dev)
    gy[1, 3], gy[4, 7] = float("inf"), float("nan")
    gx = ops.linear_grad_x(qw, scale, gy, k, torch.float32)
    gw = ops.linear_grad_w(codes, a_scale, gy, k, torch.float32)
    ex = (gy.double() @ ops.unpack_i2s(qw).double()) * scale.double()
    ew = (gy.double() * a_scale.double()[:, None]).t().contiguous() @ codes.double()
    for got, want in ((gx, ex), (gw, ew)):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        fine = want.isfinite()
        assert torch.allclose(got[fine].double(), want[fine], rtol=0, atol=1e-5 * float(want[fine].abs().max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [0.02, 2.0 ** -20, -0.3, 1.5, 3e-40, 0.0])
@pytest.mark.parametrize("n", [72, 4040])
def test_grad_x_is_bounded_by_its_result_not_by_the_unscaled_sum(pkg, dev, dtype, scale, n):
    """Gradients whose sum against the ternary weight (standard deviation sd) leaves fp32's range before the weight
    scale brings it back, and scales that are negative, above 1, subnormal or zero, summed whole and in parts."""
    ops, m, k = pkg.ops, 40, 264
    g = torch.Generator(device=dev).manual_seed(n)
    qw, _ = ops.pack_ternary_i2s(torch.randn((n, k), generator=g, device=dev), k_pad=384)
    t = ops.unpack_i2s(qw)[:, :k].double()
    sd = 1.2e38 if abs(scale) < 1 else 3e37
    gy = (torch.randn((m, n), generator=g, device=dev) * (sd / float(t.pow(2).sum(0).mean().sqrt()))).to(dtype)
    s = torch.full((1,), scale, device=dev)
    sums = gy.double() @ t
    assert abs(scale) > 1 or float(sums.abs().max()) > torch.finfo(torch.float32).max
    got, want = ops.linear_grad_x(qw, s, gy, k, torch.float32), sums * s.double()
    # (a subnormal result is rounded to 2^-149)
    assert torch.isfinite(got).all()
    assert float((got.double() - want).norm()) <= 1e-6 * float(want.norm()) + 2.0 ** -149 * (m * k) ** 0.5


def test_gradients_of_gradients_and_batched_gradients_keep_working(pkg, dev):
    """create_graph and is_grads_batched go through the torch products that autograd and vmap see through."""
    torch.manual_seed(5)
    mod = pkg.BitLinear(256, 96, device=dev)
    x = torch.randn(7, 256, device=dev, requires_grad=True)
    gy = torch.randn(7, 96, device=dev, requires_grad=True)
    plain = torch.autograd.grad(mod(x), [x, mod.weight], gy.detach())
    (gx,) = torch.autograd.grad(mod(x), x, gy, create_graph=True)
    (ggy,) = torch.autograd.grad(gx.square().sum(), gy)
    w = pkg.unpack_i2s(mod.qweight)[:, :256].float() * mod.weight_scale
    assert _rel(gx.detach(), plain[0].double()) <= 1e-6
    assert _rel(ggy, 2 * (gx.detach() @ w.t()).double()) <= 1e-5
    both = torch.stack([gy.detach(), 2 * gy.detach()])
    bx, bw = torch.autograd.grad(mod(x), [x, mod.weight], both, is_grads_batched=True)
    assert _rel(bx[0], plain[0].double()) <= 1e-6 and _rel(bw[1], 2 * plain[1].double()) <= 1e-6


def _module(pkg, dev, subln):
    """(module with a bias, input, the tensors to differentiate) of a small layer."""
    torch.manual_seed(11)
    mod = (pkg.SubLNBitLinear if subln else pkg.BitLinear)(256, 96, bias=True, device=dev)
    lin = mod.linear if subln else mod
    x = torch.randn(7, 256, device=dev, requires_grad=True)
    return mod, x, [x, lin.weight, lin.bias] + ([mod.norm_weight] if subln else [])


@pytest.mark.parametrize("subln", [False, True])
def test_forward_mode_tangents_pass_through_the_backward(pkg, dev, subln):
    """Every gradient is linear in the output's: its tangent is the gradient at the tangent (the two routes' fp32
    sums differ by 1e-6 at most)."""
    from torch.autograd import forward_ad as fw

    mod, x, wrt = _module(pkg, dev, subln)
    gy, t = torch.randn(7, 96, device=dev), torch.randn(7, 96, device=dev)
    with fw.dual_level():
        grads = torch.autograd.grad(mod(x), wrt, fw.make_dual(gy, t))
        tangents = [fw.unpack_dual(g).tangent for g in grads]
    for got, want in zip(tangents, torch.autograd.grad(mod(x), wrt, t)):
        assert got is not None and _rel(got, want.double()) <= 1e-6


@pytest.mark.parametrize("subln", [False, True])
def test_traced_backward_computes_the_weight_gradients(pkg, dev, subln):
    """A traced backward holds the products of its inputs: on another output gradient it gives that one's weight and
    bias gradients (fp32 sums in another order: 1e-6)."""
    from torch.fx.experimental.proxy_tensor import make_fx

    mod, x, wrt = _module(pkg, dev, subln)
    y = mod(x)
    gy, other = torch.randn(7, 96, device=dev), torch.randn(7, 96, device=dev)
    traced = make_fx(lambda g: torch.autograd.grad(y, wrt[1:3], g, retain_graph=True))(gy)
    for got, want in zip(traced(other), torch.autograd.grad(y, wrt[1:3], other)):
        assert _rel(got, want.double()) <= 1e-6


class _Wrapped(torch.Tensor):
    """A tensor subclass without memory of its own: every operation runs on the tensor inside."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype, device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        from torch.utils._pytree import tree_map

        def unwrap(v):
            return v.inner if isinstance(v, cls) else v

        out = func(*tree_map(unwrap, args), **tree_map(unwrap, kwargs or {}))
        return tree_map(lambda v: cls(v) if isinstance(v, torch.Tensor) else v, out)


@pytest.mark.parametrize("subln", [False, True])
def test_subclass_gradients_take_the_torch_products(pkg, dev, subln):
    mod, x, wrt = _module(pkg, dev, subln)
    gy = torch.randn(7, 96, device=dev)
    grads = torch.autograd.grad(mod(x), wrt, _Wrapped(gy))
    for got, want in zip(grads, torch.autograd.grad(mod(x), wrt, gy)):
        assert _rel(got.inner, want.double()) <= 1e-6


def _negated_view(t):
    """t's values as a lazily negated, strided view (what .imag of a conjugate is)."""
    return torch.complex(torch.zeros_like(t), -t).conj().imag


@pytest.mark.parametrize("subln", [False, True])
@pytest.mark.parametrize("form", ["negated", "columns"])
def test_saved_tensor_hooks_may_change_the_form(pkg, dev, subln, form):
    """Hooks that give the float tensors back as negated views (the one-element weight scale among them), or the
    activations and their codes column by column: the same values, the same gradients."""
    def unpack(t):
        if form == "negated":
            return _negated_view(t) if t.dtype == torch.float32 else t
        return t.t().contiguous().t() if t.dim() == 2 and t.dtype != torch.uint8 else t

    mod, x, wrt = _module(pkg, dev, subln)
    gy = torch.randn(7, 96, device=dev)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = mod(x)
    for got, want in zip(torch.autograd.grad(y, wrt, gy), torch.autograd.grad(mod(x), wrt, gy)):
        assert _rel(got, want.double()) <= 1e-6


@pytest.mark.parametrize("subln", [False, True])
def test_negated_gradients_keep_their_sign(pkg, dev, subln):
    """A lazily negated gradient, as strides let it through to the kernels: one element, whose view counts as
    contiguous."""
    mod = (pkg.SubLNBitLinear if subln else pkg.BitLinear)(256, 1, device=dev)
    x = torch.randn(1, 256, device=dev, requires_grad=True)
    wrt = [x, (mod.linear if subln else mod).weight]
    gy = torch.randn(1, 1, device=dev)
    view = _negated_view(gy)
    assert view.is_neg() and view.is_contiguous() and torch.equal(view, gy)
    for got, want in zip(torch.autograd.grad(mod(x), wrt, view), torch.autograd.grad(mod(x), wrt, gy)):
        assert _rel(got, want.double()) <= 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,h", [(1, 8), (3, 2048), (7, 2056), (513, 576), (1100, 4104), (20, 8200), (5, 16384)])
def test_rmsnorm_grad_matches_float64(pkg, dev, m, h, dtype):
    """Vector remainders of the 256-thread rows, more rows than workgroups, every row-length form.  fp32 sums of H
    and of M terms: normwise error below 1e-6; 16-bit results are rounded once (2^-9 at most)."""
    g = torch.Generator(device=dev).manual_seed(m + h)
    x = torch.randn((m, h), generator=g, device=dev).to(dtype)
    w = (1 + 0.1 * torch.randn(h, generator=g, device=dev)).to(dtype)
    gy = torch.randn((m, h), generator=g, device=dev)
    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y = x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-6) * w64
    want = torch.autograd.grad(y, [x64, w64], gy.double())
    got = pkg.ops.rmsnorm_grad(x, w, gy, 1e-6)
    tol = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for a, b in zip(got, want):
        assert a.dtype == dtype and _rel(a, b) <= tol
    only = pkg.ops.rmsnorm_grad(x, w, gy, 1e-6, need_x=False)
    assert only[0] is None and torch.equal(only[1], got[1])


def test_gradient_ops_refuse_what_they_cannot_read(pkg, dev):
    ops = pkg.ops
    qw, scale = torch.zeros((8, 64), dtype=torch.uint8, device=dev), torch.ones(1, device=dev)
    gy, codes = torch.zeros((4, 8), device=dev), torch.zeros((4, 256), dtype=torch.int8, device=dev)
    a_scale, f32 = torch.ones(4, device=dev), torch.float32
    for bad in ((qw.int(), scale, gy, 256, f32), (qw, scale.double(), gy, 256, f32), (qw, scale, gy[:, :7], 256, f32),
                (qw, scale, gy, 257, f32), (qw, scale, gy, 0, f32), (qw, scale, gy.double(), 256, f32),
                (qw, scale, gy, 256, torch.float64), (qw.cpu(), scale, gy, 256, f32)):
        with pytest.raises(RuntimeError):
            ops.linear_grad_x(*bad)
    for bad in ((codes.short(), a_scale, gy, 256, f32), (codes.t().contiguous().t(), a_scale, gy, 256, f32),
                (codes[:3], a_scale, gy, 256, f32), (codes, a_scale[:3], gy, 256, f32), (codes, a_scale, gy, 257, f32),
                (codes, a_scale, gy, 256, f32, torch.int32), (codes.cpu(), a_scale, gy, 256, f32)):
        with pytest.raises(RuntimeError):
            ops.linear_grad_w(*bad)
    x, w = torch.zeros((4, 256), device=dev), torch.ones(256, device=dev)
    for bad in ((x, w, x.bfloat16()), (x, w[:128], x), (x, w, x[:3]), (x.double(), w, x), (x[:, :252].contiguous(), w[:252], x[:, :252].contiguous())):
        with pytest.raises(RuntimeError):
            ops.rmsnorm_grad(*bad, 1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h", [8, 1000, 16384])
def test_rmsnorm_grad_of_no_rows_is_zero(pkg, dev, dtype, h):
    gw = torch.full((h,), 7.0, dtype=dtype, device=dev)
    code = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    pkg._lib.call("wfb_rmsnorm_grad", None, code, None, code, None, 1e-6, 0, h, None, gw.data_ptr(), code, None,
                  torch.cuda.current_stream().cuda_stream)
    assert torch.equal(gw, torch.zeros_like(gw))
    x, w = torch.empty((0, h), dtype=dtype, device=dev), torch.ones(h, dtype=dtype, device=dev)
    gx, gw = pkg.ops.rmsnorm_grad(x, w, torch.empty((0, h), device=dev), 1e-6)
    assert gx.shape == (0, h) and torch.equal(gw, torch.zeros_like(w))
