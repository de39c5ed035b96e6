"""The native call path of the shims against their Python path: the same bits, the same shapes, the same errors."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


def _on(native, f):
    """f() on the native call path, or on the Python path."""
    from triton_funcs import _lib as L
    assert L.call_path(), "the native call path did not load"
    host = L._host
    L._host = host if native else False
    try:
        return f()
    finally:
        L._host = host


def _both(f):
    """f() on the native call path and on the Python path, as tuples of tensors."""
    outs = [_on(native, f) for native in (True, False)]
    return [o if isinstance(o, tuple) else (o,) for o in outs]


def _same(f):
    a, b = _both(f)
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


def _ops(dtype):
    from triton_funcs import blast_kernels as B, blast_sym_quant_kernels as Q, dense_kernels as D, low_rank_kernels as R, monarch_kernels as M
    g = torch.Generator("cuda").manual_seed(0)
    t = lambda *s: (torch.randn(*s, device="cuda", generator=g) / 8).to(dtype)
    b, p, q, r = 4, 32, 48, 64
    full, bmm = (t(b, r, q), t(b, p, r), t(b, b, r)), (t(b, q, r), t(b, p, r), t(r, b, b))
    w1, w2 = t(b, p, r), t(b, r, q)
    a, bb, w = t(b * p, r), t(r, b * q), t(b * p, b * q)
    if dtype == torch.float32:
        return [(B.triton_blast_full_fp32, full), (B.triton_blast_bmm_fp32, bmm), (M.triton_monarch_right_left_fp32, (w1, w2)),
                (R.triton_low_rank_fp32, (a, bb)), (D.triton_dense_fp32, (w,))]
    uq, vq = Q.quantize_blast_factors(bmm[0].float(), bmm[1].float(), 8)
    return [(B.triton_blast_full_fp16, full), (B.triton_blast_bmm_fp16, bmm), (M.triton_monarch_right_left_fp16, (w1, w2)),
            (M.triton_monarch_right_fp16, (w1, t(b, q, r))), (R.triton_low_rank_fp16, (a, bb)), (D.triton_dense_fp16, (w,)),
            (Q.triton_blast_bmm_int8_fp16, (uq, vq, bmm[2]))]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lead", [(1, 1), (1, 5), (3, 7), (33,), (130,)])
def test_same_results(lead, dtype):
    for f, w in _ops(dtype):
        say(f"[case] call path {f.__name__} {dtype} {lead}")
        x = torch.randn(*lead, 128, device="cuda").to(dtype)
        _same(lambda: f(x, *w))
        wide = torch.randn(*lead, 256, device="cuda").to(dtype)
        _same(lambda: f(wide[..., :128], *w))                      # rows of a wider matrix
        if len(lead) == 1:
            _same(lambda: f(x.t().contiguous().t(), *w))           # columns apart: takes a copy


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 6, 40, 200])
def test_same_output_stage(rows, dtype):
    from triton_funcs import _lib as L
    for f, w in _ops(dtype):
        if not hasattr(f, "with_epilogue") or "int8" in f.__name__:
            continue
        images = 3
        x = torch.randn(images, rows, 128, device="cuda").to(dtype)
        bias = torch.randn(192, device="cuda").to(dtype)
        mod = torch.randn(images, 5 * 192, device="cuda").to(dtype)
        resid = torch.randn(images * rows, 2 * 192, device="cuda").to(dtype)[:, 192:]
        for act in (None, "gelu_tanh", "silu_mul"):
            say(f"[case] output stage {f.__name__} {dtype} rows={rows} {act}")
            _same(lambda: f.with_epilogue(x, *w, (bias, L.ACTS[act], None, 0, None)))
        gate = mod[:, 192:384]                                     # a row for each image, both operands rows of a wider matrix
        assert not gate.is_contiguous() and not resid.is_contiguous()
        want = f.with_epilogue(x, *w, (bias, 0, gate.contiguous(), rows, resid.contiguous()))
        rest = f(x, *w).reshape(-1, 192).double() + bias.double()
        ref = resid.double() + gate.double().repeat_interleave(rows, 0) * rest
        # (op + bias and the result are each rounded; the factor 8 leaves room for the operator's own rounding points)
        unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
        assert (want.reshape(-1, 192).double() - ref).abs().max() <= 8 * unit * (ref.abs().max() + gate.abs().max().double() * rest.abs().max())
        for g, r in ((gate, resid), (gate, resid.contiguous()), (gate.contiguous(), resid)):
            for got in _both(lambda: f.with_epilogue(x, *w, (bias, 0, g, rows, r))):
                assert torch.equal(got[0], want)
        _same(lambda: f.with_epilogue(x, *w, (None, 0, gate, rows, resid)))


@pytest.mark.parametrize("rows", [1, 6, 40, 200])
def test_expanded_gate_and_residual(rows):
    """One row of modulation, or of the residual, for everything: a view without a stride between its rows."""
    from triton_funcs import _lib as L
    images = 3
    for f, w in _ops(torch.float16):
        if not hasattr(f, "with_epilogue") or "int8" in f.__name__:
            continue
        say(f"[case] expanded gate {f.__name__} {images} x {rows}")
        x = torch.randn(images, rows, 128, device="cuda").half()
        gate, resid = torch.randn(192, device="cuda").half(), torch.randn(192, device="cuda").half()
        full = resid.expand(images * rows, 192)
        want = f.with_epilogue(x, *w, (None, 0, gate.repeat(images, 1), rows, full.contiguous()))
        for g, r in ((gate.expand(images, 192), full.contiguous()), (gate.expand(images, 192), full), (gate.repeat(images, 1), full)):
            for got in _both(lambda: f.with_epilogue(x, *w, (None, 0, g, rows, r))):
                assert torch.equal(got[0], want)
            with L.fused_epilogue(None, None, g, rows, r):
                assert torch.equal(f(x, *w).reshape(want.shape), want)
        # a single row, whose stride torch is free to choose
        one = torch.as_strided(gate, (1, 192), (0, 1))
        x1 = x[:1].contiguous()
        want = f.with_epilogue(x1, *w, (None, 0, gate.reshape(1, 192), rows, None))
        for got in _both(lambda: f.with_epilogue(x1, *w, (None, 0, one, rows, None))):
            assert torch.equal(got[0], want)


def test_quantized_module_bias_and_activation():
    """QuantBlastLinear's bias and activation in the kernel's output stage: as the separate passes leave them."""
    from models.wrappers import QuantBlastLinear
    torch.manual_seed(0)
    for act in (None, "gelu_tanh", "silu", "silu_mul"):
        for rows in (1, 9, 70, 150):
            m = QuantBlastLinear(128, 192, b=4, rank=64, func_path="triton_funcs.blast_sym_quant_kernels.triton_blast_bmm_int8_fp16", device="cuda", dtype=torch.float16)
            m.fused_act = act
            x = torch.randn(1, rows, 128, device="cuda").half()
            with torch.no_grad():
                a, b = _both(lambda: m(x))
                m.fused_act = None
                v = m(x).float()                                   # what the activation is applied to, rounded
                m.fused_act = act
            # The separate passes round op + bias before the activation, the output stage does not: half a unit of v, times the
            # activation's slope (at most 1.13) and, gated, the other factor; then one rounding of each side (gated: of silu too).
            half = 2.0 ** -11
            slope = 0.0 if act is None else 1.13 * half * v.abs()
            if act == "silu_mul":
                slope = slope[..., :96] * v[..., 96:].abs()
            err = (a[0].float() - b[0].float()).abs()
            assert (err <= slope + 4 * half * b[0].float().abs() + 1e-6).all(), (act, rows, float(err.max()))


def test_quantized_module_bias_gradient():
    """A bias that wants a gradient, or carries a tangent, is added by torch: the kernel's output stage has neither."""
    from models.wrappers import QuantBlastLinear
    torch.manual_seed(0)
    m = QuantBlastLinear(128, 192, b=4, rank=64, func_path="triton_funcs.blast_sym_quant_kernels.triton_blast_bmm_int8_fp16", device="cuda", dtype=torch.float16)
    for rows in (1, 9, 150):
        x = torch.randn(1, rows, 128, device="cuda").half()
        m.bias.grad = None
        m(x).float().sum().backward()
        assert torch.equal(m.bias.grad, torch.full_like(m.bias, rows))
    m.fused_act, m.bias.grad = "silu", None
    m(x).float().sum().backward()
    assert m.bias.grad is not None and bool((m.bias.grad != 0).any())
    m.fused_act = None
    bias = m.bias.detach()
    del m.bias
    with torch.autograd.forward_ad.dual_level():
        m.bias = torch.autograd.forward_ad.make_dual(bias, torch.ones_like(bias))
        assert torch.autograd.forward_ad.unpack_dual(m(x)).tangent is not None


def test_irregular_calls_raise_as_before():
    from triton_funcs import _lib as L, blast_kernels as B, dense_kernels as D
    (f, (U, V, S)), = _ops(torch.float16)[:1]
    x = torch.randn(1, 4, 128, device="cuda").half()
    for bad in (lambda: f(x[..., :96].contiguous(), U, V, S), lambda: f(x, U, V, S[:, :2].contiguous()), lambda: f(x.float(), U, V, S),
                lambda: f(x, U.transpose(1, 2), V, S), lambda: D.triton_dense_fp16(x.float(), torch.randn(128, 64, device="cuda")),
                lambda: B.triton_blast_full_fp32(x, U, V, S)):
        with pytest.raises(AssertionError):
            bad()
    with pytest.raises(L.BlrError):
        f(x.cpu(), U, V, S)
    f(x, U, V, S)
    cfg = B.get_triton_blast_full_fp16_config()
    assert cfg["M"] == 4 and cfg["in_f"] == 128 and cfg["out_f"] == 192 and cfg["rank"] == 64 and cfg["dtype"] == "torch.float16"
    f(x[:, :3], U, V, S)
    assert B.get_triton_blast_full_fp16_config()["M"] == 3


def test_gates_and_residuals_that_are_too_short_are_refused():
    from triton_funcs import _lib as L
    for f, w in _ops(torch.float16):
        if not hasattr(f, "with_epilogue") or "int8" in f.__name__:
            continue
        for rows in (7, 100):
            x = torch.randn(rows, 128, device="cuda").half()
            t = lambda n: torch.randn(n, 192, device="cuda").half()
            for gate, every, resid in ((t(2), 3, None), (t(1), rows - 1, None), (t(1), 0, None), (None, 0, t(rows - 1)), (t(1), rows, t(1))):
                say(f"[case] too short {f.__name__} {rows} rows, one gate row for {every}")
                for host in (True, False):
                    with pytest.raises(L.BlrError):
                        _on(host, lambda: f.with_epilogue(x, *w, (None, 0, gate, every, resid)))
            f.with_epilogue(x, *w, (None, 0, t(2), -(-rows // 2), t(rows)))


def test_transformed_tensors_raise():
    """Tensors of vmap, grad and jvp have no memory: an error, as on the Python path, and the next call is as good as the one before."""
    for f, w in _ops(torch.float16):
        say(f"[case] transforms of {f.__name__}")
        x = torch.randn(2, 5, 128, device="cuda").half()
        want = f(x[0], *w)
        for call in (lambda: torch.func.vmap(lambda t: f(t, *w))(x),
                     lambda: torch.func.grad(lambda t: f(t, *w).float().sum())(x[0]),
                     lambda: torch.func.jvp(lambda t: f(t, *w), (x[0],), (x[1],))):
            for native in (True, False):
                with pytest.raises(RuntimeError):
                    _on(native, call)
        assert torch.equal(f(x[0], *w), want)
