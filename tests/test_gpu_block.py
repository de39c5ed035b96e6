"""The kernels between the linears of a DiT block against torch in 64 bits, and which calls are left to torch."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from gpu_util import say

pytestmark = pytest.mark.gpu

HALF = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}       # one rounding of a result, relatively


def _host():
    from triton_funcs import _lib as L
    host = L.call_path()
    assert host, "the native call path did not load"
    return host


# columns: one piece of a lane, the edges of its pieces per lane, the most; rows that do not fill a workgroup
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("images,tokens,cols", [(1, 1, 8), (3, 5, 504), (2, 64, 512), (1, 7, 520), (16, 256, 1152), (5, 3, 1544), (1, 2, 2048)])
def test_ln_modulate(images, tokens, cols, dtype):
    say(f"[case] ln_modulate {images} x {tokens} x {cols} {dtype}")
    x = (torch.randn(images, tokens, cols, device="cuda") * 2 + 1).to(dtype)
    mod = torch.randn(images, 3 * cols, device="cuda").to(dtype)
    shift, scale, _ = mod.chunk(3, dim=1)
    got = _host().ln_modulate(x, shift, scale, 1e-6)
    ref = F.layer_norm(x.double(), (cols,), eps=1e-6) * (1 + scale.double().unsqueeze(1)) + shift.double().unsqueeze(1)
    # fp32 inside: a few 2^-24 of the terms before the sum with the shift may cancel them, then one rounding
    slack = 2.0 ** -20 * (ref.abs() + shift.double().abs().unsqueeze(1) + 1)
    assert ((got.double() - ref).abs() <= HALF[dtype] * ref.abs() + slack).all()


def test_ln_modulate_is_left_to_torch():
    """fp32, odd columns, gradients, autocast, transforms, a norm with hooks: as before."""
    from models import dit_xl as D
    h = _host()
    x, s = torch.randn(2, 4, 64, device="cuda").half(), torch.randn(2, 64, device="cuda").half()
    assert h.ln_modulate(x, s, s, 1e-6) is not None
    assert h.ln_modulate(x.float(), s.float(), s.float(), 1e-6) is None
    assert h.ln_modulate(x[..., :60], s[:, :60], s[:, :60], 1e-6) is None
    assert h.ln_modulate(x.transpose(0, 1), s[:, :], s, 1e-6) is None
    assert h.ln_modulate(x.clone().requires_grad_(), s, s, 1e-6) is None
    with torch.no_grad():
        assert h.ln_modulate(x.clone().requires_grad_(), s, s, 1e-6) is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert h.ln_modulate(x, s, s, 1e-6) is None
    norm = nn.LayerNorm(64, elementwise_affine=False, eps=1e-6)
    want = D.modulate(norm(x), s, s)
    got = torch.func.vmap(lambda xx, ss: D._norm_modulate(norm, xx[None], ss[None], ss[None])[0])(x, s)
    assert torch.allclose(got.float(), want.float(), atol=2e-2)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x.float().half(), torch.ones_like(x))
        assert h.ln_modulate(dual, s, s, 1e-6) is None
    seen = []
    norm.register_forward_hook(lambda *a: seen.append(1))
    D._norm_modulate(norm, x, s, s)
    assert seen


def _attention64(qkv, heads):
    B, N, C3 = qkv.shape
    q, k, v = qkv.double().cpu().reshape(B, N, 3, heads, C3 // 3 // heads).permute(2, 0, 3, 1, 4)
    p = torch.softmax(q @ k.transpose(-1, -2) * q.shape[-1] ** -0.5, dim=-1)
    return (p @ v).transpose(1, 2).reshape(B, N, C3 // 3), (p @ v.abs()).transpose(1, 2).reshape(B, N, C3 // 3)


def _close(got, ref, mag, half, slack):
    """The result's rounding (half a place; at least half of fp16's smallest value, 2^-25), and the probabilities': each is off by at
    most half a place, their errors add up to at most that of p |v|; slack * p |v| for the exponentials' arguments in fp32."""
    err, bound = (got - ref).abs(), half * (ref.abs() + 1.01 * mag) + slack * mag + 2.0 ** -25
    at = (err - bound).argmax()
    assert (err <= bound).all(), (got.flatten()[at], ref.flatten()[at], mag.flatten()[at], err.flatten()[at], bound.flatten()[at])


# tokens: one, the edges of a wave's queries, of a step of keys and of a workgroup's queries, several steps
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [64, 72])
@pytest.mark.parametrize("images,heads,tokens", [(1, 1, 1), (2, 3, 31), (1, 2, 33), (3, 16, 64), (1, 5, 65), (2, 2, 127), (1, 1, 129), (2, 16, 256), (1, 3, 700)])
def test_attention(images, heads, tokens, dim, dtype):
    say(f"[case] attention {images} x {heads} x {tokens} x {dim} {dtype}")
    qkv = (torch.randn(images, tokens, 3 * heads * dim, device="cuda") * 1.5).to(dtype)
    got = _host().attention(qkv, heads).double().cpu()
    ref, mag = _attention64(qkv, heads)
    _close(got, ref, mag, HALF[dtype], 2.0 ** -16)


def test_attention_large_scores_and_infinities():
    """Scores far apart (the running maximum moves, exponentials underflow), and a key of minus infinity takes no part."""
    heads, dim, n = 2, 72, 200
    qkv = torch.randn(1, n, 3 * heads * dim, device="cuda").half()
    qkv[:, :, : heads * dim] *= 12
    qkv[:, :, heads * dim: 2 * heads * dim] *= torch.linspace(0.1, 4, n, device="cuda")[None, :, None].half()
    ref, mag = _attention64(qkv, heads)
    got = _host().attention(qkv, heads).double().cpu()
    _close(got, ref, mag, 2.0 ** -11, 2.0 ** -14)
    # the first value of every query is positive and of one key minus infinity
    qkv[:, :, 0] = qkv[:, :, dim] = 1.0
    for key in (0, 63, 64, 199):
        one = qkv.clone()
        one[0, key, heads * dim] = one[0, key, heads * dim + dim] = -float("inf")
        ref, mag = _attention64(one, heads)
        got = _host().attention(one, heads).double().cpu()
        assert torch.isfinite(got).all()
        _close(got, ref, mag, 2.0 ** -11, 2.0 ** -14)


def test_attention_is_left_to_torch():
    h = _host()
    x = torch.randn(2, 8, 3 * 2 * 64, device="cuda").half()
    assert h.attention(x, 2) is not None
    assert h.attention(x.float(), 2) is None
    assert h.attention(x, 4) is None                                 # heads of 32
    assert h.attention(x, 5) is None
    assert h.attention(x.transpose(0, 1), 2) is None
    assert h.attention(x.clone().requires_grad_(), 2) is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert h.attention(x, 2) is None


# rows: one, the most; columns: less than a workgroup's, its edges, several; inputs: one piece, waves without work, more than one batch a wave
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,out_f,in_f", [(1, 4, 8), (16, 12, 24), (3, 16, 32), (5, 20, 136), (16, 6912, 1152), (2, 2304, 1160), (7, 68, 2600)])
def test_silu_linear(rows, out_f, in_f, dtype):
    say(f"[case] silu_linear {rows} x {in_f} -> {out_f} {dtype}")
    lin = nn.Linear(in_f, out_f, device="cuda", dtype=dtype)
    c = (torch.randn(rows, 2 * in_f, device="cuda") * 2).to(dtype)[:, :in_f]
    s = F.silu(c.float()).to(dtype).double()
    for bias in (lin.bias, None):
        with torch.no_grad():
            got = _host().silu_linear(c, lin.weight, bias).double()
        w = lin.weight.double()
        ref, mag = s @ w.t(), s.abs() @ w.abs().t()
        if bias is not None:
            ref = ref + bias.double()
        # the result's rounding; a silu that the kernel's exponential puts on the other side of a tie is off by a whole place, at worst
        # everywhere; fp16's smallest values
        assert ((got - ref).abs() <= HALF[dtype] * (ref.abs() + 2 * mag) + 2.0 ** -16 * mag + 2.0 ** -25).all()


def test_silu_linear_is_left_to_torch():
    from models import dit_xl as D
    h = _host()
    proj = nn.Sequential(nn.SiLU(), nn.Linear(64, 96)).cuda().half()
    lin, c = proj[1], torch.randn(4, 64, device="cuda").half()
    with torch.no_grad():
        assert h.silu_linear(c, lin.weight, lin.bias) is not None
        assert h.silu_linear(c.float(), lin.weight, lin.bias) is None
        assert h.silu_linear(torch.cat([c] * 5), lin.weight, lin.bias) is None              # 20 rows
        assert h.silu_linear(c, lin.weight.t().contiguous().t(), lin.bias) is None
        assert h.silu_linear(c.t().contiguous().t(), lin.weight, lin.bias) is None
        assert h.silu_linear(c, lin.weight, lin.bias.float()) is None
        assert torch.allclose(D._conditioned(proj, c).float(), proj(c).float(), atol=2e-2)
        seen = []
        hook = lin.register_forward_hook(lambda *a: seen.append(1))
        D._conditioned(proj, c)
        assert seen
        hook.remove()
    assert h.silu_linear(c, lin.weight, lin.bias) is None                                    # the weight wants a gradient
    D._conditioned(proj, c).sum().backward()
    assert lin.weight.grad is not None


def _layers():
    """The parts of a DiT that the library's kernels stand in for, with torch's own linears, and a call of each."""
    from models import dit_xl as D
    torch.manual_seed(1)
    x, c = torch.randn(2, 9, 128, device="cuda").half(), torch.randn(2, 128, device="cuda").half()
    return [(m.cuda().half().eval(), x, c) for m in (D.DiTBlock(128, 2), D.FinalLayer(128, 2, 4))]


def test_compiled_layers_are_left_to_torch():
    """One graph, as torch's operators give it: the library's entries are nothing that a compiler can trace."""
    for layer, x, c in _layers():
        say(f"[case] compiled {type(layer).__name__}")
        torch._dynamo.reset()
        with torch.no_grad():
            want = layer(x, c)
            got = torch.compile(layer, fullgraph=True, backend="eager")(x, c)
        assert torch.allclose(got.float(), want.float(), atol=2e-2, rtol=2e-2)


def test_compiled_block_of_structured_linears():
    from models import dit_xl as D
    from models.wrappers import BlastLinear
    layer, x, c = _layers()[0]
    for at, name, n, m in ((layer.attn, "qkv", 128, 384), (layer.attn, "proj", 128, 128), (layer.mlp, "fc1", 128, 512), (layer.mlp, "fc2", 512, 128)):
        setattr(at, name, BlastLinear(n, m, 4, 32, "triton_funcs.blast_kernels.triton_blast_bmm_fp16", "cuda", torch.float16))
    layer.mlp.fc1.fused_act = "gelu_tanh"
    torch._dynamo.reset()
    with torch.no_grad():
        want = layer(x, c)
        got = torch.compile(layer, backend="eager")(x, c)
    scale = want.float().abs().max().item()
    assert torch.allclose(got.float(), want.float(), atol=2e-2 * scale)


def test_function_modes_see_the_operators():
    from torch.overrides import TorchFunctionMode

    class Watch(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.seen = set()

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.add(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    for layer, x, c in _layers():
        with torch.no_grad(), Watch() as w:
            layer(x, c)
        assert {"layer_norm", "silu", "linear"} <= w.seen, w.seen


def test_attention_backend_of_the_caller():
    from torch.nn.attention import SDPBackend, sdpa_kernel
    h, x = _host(), torch.randn(2, 8, 3 * 2 * 64, device="cuda").half()
    with sdpa_kernel(SDPBackend.MATH):
        assert h.attention(x, 2) is None
    with sdpa_kernel(SDPBackend.EFFICIENT_ATTENTION):
        assert h.attention(x, 2) is None
    with sdpa_kernel([SDPBackend.MATH, SDPBackend.FLASH_ATTENTION]):
        assert h.attention(x, 2) is not None
    assert h.attention(x, 2) is not None
