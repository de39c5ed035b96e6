"""GPU parity of the small-tile GEMM kernels (products that do not fill the chip), each of the five tiles at the edges of its tiles, of
its stages of 64 k and of its groups of stages, and of reductions cut into slices.

Bound per element: one rounding of the result to its type, and fp32 accumulation in any order (K roundings of 2^-24 of
sum |x| |w|, K being generous)."""
import pytest
import torch

from gpu_util import say, ulp

pytestmark = pytest.mark.gpu


def _bound(ref, mag, k, dtype):
    return 0.5 * torch.from_numpy(ulp(ref.cpu().numpy(), dtype)).to(ref.device) * 1.01 + k * 2.0 ** -24 * mag


def _check(out, x, w, dtype, what):
    ref, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    err = (out.double().reshape(ref.shape) - ref).abs()
    assert torch.isfinite(out).all(), what
    bad = err > _bound(ref, mag, x.shape[-1], dtype)
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outside, worst {float(err[bad].max())}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [2, 3, 4, 5, 6])
# rows, columns, k: tiles are 32 or 64 rows by 64 or 128 columns, a wave group's stage is 64 k, up to four groups take turns
@pytest.mark.parametrize("m,n,k", [(17, 8, 8), (31, 72, 64), (65, 136, 72), (130, 64, 328), (33, 264, 1016), (200, 56, 2560), (64, 128, 192)])
def test_mid_tiles(m, n, k, tile, dtype):
    from triton_funcs import _lib as L, dense_kernels as D, blast_kernels as B
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    w = (torch.randn(k, n, device="cuda", generator=g) / k ** 0.5).to(dtype)
    say(f"[case] mid tile {tile} {dtype} m={m} n={n} k={k}")
    with L.options(BLR_GEMM_MID=tile):
        _check(D.triton_dense_fp16(x, w, {"algo": L.ALGO_TILED}), x, w, dtype, "dense (k, n)")
        # batched, both weight orders: BLAST's two products through the names that return the intermediates' arithmetic unfused
        b = 2
        V = (torch.randn(b, k // b if k % 16 == 0 else k, 16, device="cuda", generator=g) / k ** 0.5).to(dtype)
        xb = torch.randn(1, m, b * V.shape[1], device="cuda", generator=g).to(dtype)
        S = torch.zeros(16, b, b, device="cuda", dtype=dtype)
        S[:, 0, 0] = S[:, 1, 1] = 1.0                            # no mixing: out_i = (x_i V_i) U_i^T
        U = (torch.randn(b, n, 16, device="cuda", generator=g) / 4).to(dtype)
        with L.options(BLR_DECODE_ROWS=0, BLR_BLAST_ONE=0, BLR_BLAST_MIXU=0):
            out = B.triton_blast_bmm_fp16(xb, U, V, S, {"algo": L.ALGO_TILED})
        p = V.shape[1]
        for i in range(b):
            y = (xb[0, :, i * p:(i + 1) * p].double() @ V[i].double())
            mag = (xb[0, :, i * p:(i + 1) * p].double().abs() @ V[i].double().abs()) @ U[i].double().abs().t().contiguous()
            ref = y.to(dtype).double() @ U[i].double().t().contiguous()
            err = (out[0, :, i * n:(i + 1) * n].double() - ref).abs()
            # y and z are rounded to dtype on the way (each may fall on the other side of a tie: one unit of y)
            unit = torch.from_numpy(ulp(y.cpu().numpy(), dtype)).to(y.device) @ U[i].double().abs().t().contiguous()
            assert (err <= _bound(ref, mag, p + 16, dtype) + unit).all(), (i, float(err.max()))


@pytest.mark.parametrize("tile", [1, 3, 5])
# fp32 stages hold 32 k; the last two are cut into slices (only by the estimate, tile 1), 6 columns go to the kernel for unaligned operands
@pytest.mark.parametrize("m,n,k", [(1, 8, 4), (31, 72, 36), (65, 136, 100), (33, 6, 64), (100, 64, 1028), (35, 768, 3072), (64, 8, 5000)])
def test_fp32(m, n, k, tile):
    from triton_funcs import _lib as L, dense_kernels as D, monarch_kernels as Mo
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x, w = torch.randn(m, k, device="cuda", generator=g), torch.randn(k, n, device="cuda", generator=g) / k ** 0.5
    say(f"[case] fp32 tile {tile} m={m} n={n} k={k}")
    with L.options(BLR_GEMM_MID=tile):
        out = D.triton_dense_fp32(x, w)
        ref, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
        # fp32 sums in any order: k roundings of 2^-24 of sum |x| |w|, and one of the result
        assert ((out.double() - ref).abs() <= (k + 1) * 2.0 ** -24 * mag).all()
        # the scatter of Monarch's first product and its interleaved result
        w1, w2 = torch.randn(2, k, 8, device="cuda", generator=g) / k ** 0.5, torch.randn(2, n, 8, device="cuda", generator=g)
        xm = torch.randn(1, m, 2 * k, device="cuda", generator=g)
        got, out1, pre = Mo.triton_monarch_right_fp32(xm, w1, w2)
        p1 = torch.stack([xm[0, :, i * k:(i + 1) * k].double() @ w1[i].double() for i in range(2)])
        m1 = torch.stack([xm[0, :, i * k:(i + 1) * k].double().abs() @ w1[i].double().abs() for i in range(2)])
        assert ((pre.double() - p1).abs() <= (k + 1) * 2.0 ** -24 * m1).all()
        o2 = torch.stack([out1[i].double() @ w2[i].double().t().contiguous() for i in range(2)], dim=-1).reshape(m, -1)
        m2 = torch.stack([out1[i].double().abs() @ w2[i].double().abs().t().contiguous() for i in range(2)], dim=-1).reshape(m, -1)
        assert ((got[0].double() - o2).abs() <= 9 * 2.0 ** -24 * m2).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act", [None, "silu", "silu_mul"])
@pytest.mark.parametrize("m,n,k", [(130, 80, 8672), (257, 144, 4104), (150, 688, 10600), (279, 768, 768), (129, 3200, 9120)])
def test_long_reductions_by_estimate(m, n, k, act, dtype):
    """Shapes that the estimate cuts into slices (and two that it does not), plain and with an output stage."""
    from triton_funcs import _lib as L, dense_kernels as D
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    w = (torch.randn(k, n, device="cuda", generator=g) / k ** 0.5).to(dtype)
    bias = torch.randn(n, device="cuda", generator=g).to(dtype) if act else None
    say(f"[case] slices {dtype} m={m} n={n} k={k} act={act}")
    with L.fused_epilogue(bias, act):
        out = D.triton_dense_fp16(x, w)
    if act is None:
        return _check(out, x, w, dtype, "dense in slices")
    ref, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    pre = _bound(ref, mag, k, dtype)                              # what the rounded product may be off by
    v = ref + bias.double()
    silu = lambda t: t * torch.sigmoid(t)
    if act == "silu":
        want, slack = silu(v), 1.1 * pre                          # |silu'| <= 1.1
    else:
        h = n // 2
        want = silu(v[:, :h]) * v[:, h:]
        step = lambda t: torch.from_numpy(ulp(t.cpu().numpy(), dtype)).to(t.device)
        slack = (1.1 * pre[:, :h] + 0.5 * step(silu(v[:, :h]))) * v[:, h:].abs() * 1.1 + (pre[:, h:] + 0.5 * step(v[:, h:])) * silu(v[:, :h]).abs() * 1.1
    err = (out.double() - want).abs()
    # the activation's exponential and reciprocal are good to a few units of fp32
    lim = 0.51 * torch.from_numpy(ulp(want.cpu().numpy(), dtype)).to(want.device) + slack + 1e-5 * want.abs()
    assert (err <= lim).all(), float((err / lim).max())


@pytest.mark.parametrize("m,n,k", [(3, 768, 3072), (61, 136, 8672), (257, 144, 4104)])
def test_output_operands_of_any_alignment(m, n, k):
    """The same shapes with a bias, a gate and a residual that start two bytes past a 16-byte boundary: the sum of the slices reads eight
    columns at a time and leaves such calls to the kernels that take any address."""
    from triton_funcs import _lib as L, dense_kernels as D
    dtype = torch.float16
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    w = (torch.randn(k, n, device="cuda", generator=g) / k ** 0.5).to(dtype)
    odd = lambda rows: torch.randn(rows * n + 1, device="cuda", generator=g).to(dtype)[1:].view(rows, n)
    bias, gate, resid = odd(1).view(n), odd(1), odd(m)
    say(f"[case] unaligned output stage m={m} n={n} k={k}")
    with L.fused_epilogue(bias, None):
        out = D.triton_dense_fp16(x, w)
    ref, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    step = lambda t: 0.51 * torch.from_numpy(ulp(t.cpu().numpy(), dtype)).to(t.device)
    want, slack = ref + bias.double(), _bound(ref, mag, k, dtype)
    assert ((out.double() - want).abs() <= step(want) + slack + 2.0 ** -23 * want.abs()).all()
    with L.fused_epilogue(bias, None, gate, m, resid):
        out = D.triton_dense_fp16(x, w)
    full = want * gate.double() + resid.double()
    lim = step(full) + (step(want) + slack) * gate.double().abs() + 2.0 ** -22 * (want * gate.double()).abs() + 2.0 ** -22 * resid.double().abs()
    assert ((out.double() - full).abs() <= lim).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 16, 40, 100, 128, 200])
@pytest.mark.parametrize("n,k", [(64, 72), (136, 1048), (264, 200), (2304, 776)])
def test_infinite_weights(m, n, k, dtype):
    """A weight of infinity anywhere in a reduction that ends in a partial stage gives infinities of the right sign, not NaN: what
    stands in for the missing k of a stage meets zeros on both sides."""
    from triton_funcs import _lib as L, dense_kernels as D, blast_kernels as B
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = (torch.rand(m, k, device="cuda", generator=g) + 0.5).to(dtype)
    x[::2] *= -1
    w = (torch.randn(k, n, device="cuda", generator=g) / k ** 0.5).to(dtype)
    for col, row in enumerate((0, k - 1, k - 8, k - 5, k // 2)):
        w[row, col] = float("inf")
    say(f"[case] infinite weights {dtype} m={m} n={n} k={k}")
    f = D.triton_dense_fp32 if dtype == torch.float32 else D.triton_dense_fp16
    ref = x.double() @ w.double()
    outs = [f(x, w)]
    if dtype != torch.float32:
        outs.append(f(x, w, {"algo": L.ALGO_TILED}))
    if dtype != torch.float32 and m > 16:                            # (up to 16 rows BLAST streams its factors through other kernels)
        # the same product with the weights' k contiguous: BLAST's second one, U (b, q, r), behind a first that hands x through
        b = 2
        V, S = torch.eye(k, device="cuda").to(dtype).expand(b, k, k).contiguous(), torch.zeros(k, b, b, device="cuda").to(dtype)
        S[:, 0, 0] = S[:, 1, 1] = 1.0
        out = B.triton_blast_bmm_fp16(torch.cat([x, x], 1)[None], w.t().contiguous().expand(b, n, k).contiguous(), V, S)
        outs += [out[0, :, :n], out[0, :, n:]]
    for i, out in enumerate(outs):
        inf = torch.isinf(ref)
        assert inf[:, :5].all() and not inf[:, 5:].any()
        assert torch.equal(out[:, :5].double(), ref[:, :5]), i
        assert torch.isfinite(out[:, 5:]).all(), i
