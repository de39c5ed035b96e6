"""BLAST from 17 rows on as two products on small tiles with the mix between them, and the kernels it takes the place of."""
import numpy as np
import pytest
import torch

from gpu_util import assert_close, blast_inputs, dev, rounded, say
from oracle import blr_oracle as O

pytestmark = pytest.mark.gpu


# rows: the first, both sides of a tile of 32 and 64, the last of the rule for every rank, further by rows x rank; blocks: 16 (both mix
# kernels), others; widths that are not whole tiles
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", ["triton_blast_full_fp16", "triton_blast_bmm_fp16"])
@pytest.mark.parametrize("b,p,q,r", [(16, 72, 72, 64), (16, 136, 200, 136), (16, 16, 8, 32), (3, 40, 88, 24), (2, 1096, 24, 8)])
@pytest.mark.parametrize("M", [17, 32, 33, 65, 128, 129, 300])
def test_blast(M, b, p, q, r, name, dtype):
    from test_gpu_blast import _ref, _run_blast
    x, U, Vt, S = blast_inputs(b, p, q, r, (M,), seed=M + b)
    say(f"[case] few rows {name} b={b} p={p} q={q} r={r} M={M} {dtype}")
    out = _run_blast(name, x, U, Vt, S, dtype, "auto")
    assert_close(out, _ref(x, U, Vt, S, dtype)[0], dtype, f"{name} b={b} p={p} q={q} r={r} M={M}")


@pytest.mark.parametrize("M", [40, 100])
@pytest.mark.parametrize("b,p,q,r", [(16, 72, 72, 64), (16, 136, 72, 64), (16, 72, 200, 64)], ids=["one launch", "narrow out", "narrow in"])
def test_fused_kernels_at_few_rows(b, p, q, r, M):
    """BLR_DECODE_ROWS=0 leaves few rows to the kernels of many."""
    from test_gpu_blast import _ref, _run_blast
    from triton_funcs import _lib as L
    x, U, Vt, S = blast_inputs(b, p, q, r, (M,), seed=M)
    for name in ("triton_blast_full_fp16", "triton_blast_bmm_fp16"):
        say(f"[case] fused at few rows {name} b={b} p={p} q={q} r={r} M={M}")
        with L.options(BLR_DECODE_ROWS=0):
            out = _run_blast(name, x, U, Vt, S, torch.float16, "auto")
        assert_close(out, _ref(x, U, Vt, S, torch.float16)[0], torch.float16, f"{name} M={M}")


@pytest.mark.parametrize("act", ["gelu_tanh", "silu_mul"])
@pytest.mark.parametrize("M", [17, 100, 200])
def test_output_stage(M, act):
    """Bias, activation, gate and residual (or the gated halves) in the second product's output stage, rows of out wider than the result."""
    from triton_funcs import blast_kernels as K, _lib as L
    b, p, q, r, dtype = 4, 72, 80, 64, torch.float16
    x, U, Vt, S = blast_inputs(b, p, q, r, (M,), seed=M)
    Up, Vp, Sp = O.blast_to_partial_layout(U, Vt, S)
    rng = np.random.default_rng(M)
    bias = rng.standard_normal(b * q)
    say(f"[case] few rows output stage {act} M={M}")
    base = O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0] + rounded(bias, dtype)
    args = (dev(x, dtype), dev(Up, dtype), dev(Vp, dtype), dev(Sp, dtype))
    if act == "silu_mul":
        with L.fused_epilogue(dev(bias, dtype), act):
            out = K.triton_blast_full_fp16(*args)
        g, u = base[..., : b * q // 2], base[..., b * q // 2:]
        assert_close(out, g / (1 + np.exp(-g)) * u, dtype, f"silu_mul M={M}", scale=2.0)
        return
    gate, resid = rng.standard_normal((2, b * q)), rng.standard_normal((M, b * q))
    rows = (M + 1) // 2
    with L.fused_epilogue(dev(bias, dtype), act, dev(gate, dtype), rows, dev(resid, dtype)):
        out = K.triton_blast_full_fp16(*args)
    v = 0.5 * base * (1.0 + np.tanh(np.sqrt(2.0 / np.pi) * (base + 0.044715 * base ** 3)))
    assert_close(out, (rounded(resid, dtype) + rounded(gate, dtype)[np.arange(M) // rows] * v).reshape(out.shape), dtype, f"gate + residual M={M}", scale=2.0)


# low rank whose input has no equal slices of whole pieces (odd multiples of 8), two or four of them; the last slice from 8 rows up
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 5, 16])
@pytest.mark.parametrize("in_f,r,out_f", [(3736, 376, 1712), (3728, 72, 264), (8, 8, 8), (72, 16, 40), (1032, 200, 136), (776, 128, 3072), (4104, 1032, 520), (11000, 8, 72)])
def test_low_rank_unequal_slices(M, in_f, r, out_f, dtype):
    from triton_funcs import low_rank_kernels as LR
    g = torch.Generator("cuda").manual_seed(M + in_f)
    x = torch.randn(M, in_f, device="cuda", generator=g).to(dtype)
    a, b = (torch.randn(in_f, r, device="cuda", generator=g) / in_f ** 0.5).to(dtype), (torch.randn(r, out_f, device="cuda", generator=g) / r ** 0.5).to(dtype)
    say(f"[case] low rank {in_f} -> {out_f} r={r} M={M} {dtype}")
    ref = x.double().cpu() @ a.double().cpu() @ b.double().cpu()
    assert_close(LR.triton_low_rank_fp16(x, a, b), ref.numpy(), dtype, f"low rank {in_f} -> {out_f} M={M}", scale=2.0)


# a few rows and a long reduction: slices on tiles of 32 rows; a wide output: more tiles than compute units
@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (1, 4104, 136), (5, 72, 1032), (16, 11008, 72), (16, 512, 33024), (17, 4104, 136), (33, 11008, 72), (95, 2056, 1032), (17, 72, 33024), (64, 512, 65536)])
def test_dense(M, K, N):
    from triton_funcs import dense_kernels as D, _lib as L
    dtype = torch.float16
    g = torch.Generator("cuda").manual_seed(M)
    x, w = torch.randn(M, K, device="cuda", generator=g).half(), (torch.randn(K, N, device="cuda", generator=g) / K ** 0.5).half()
    say(f"[case] few rows dense {M} x {K} x {N}")
    ref = (x.float() @ w.float()).double().cpu().numpy()              # (fp32 on the GPU: 1e-5 against the bound's 1e-2)
    assert_close(D.triton_dense_fp16(x, w), ref, dtype, f"dense {M} x {K} x {N}")
    bias = torch.randn(N, device="cuda", generator=g).half()
    with L.fused_epilogue(bias, "silu"):
        out = D.triton_dense_fp16(x, w)
    v = ref + bias.double().cpu().numpy()
    assert_close(out, v / (1 + np.exp(-v)), dtype, f"dense {M} x {K} x {N} + bias + silu")


@pytest.mark.parametrize("M,in_f,r,out_f", [(2, 72, 8, 24), (7, 1536, 136, 200), (16, 768, 192, 2304), (16, 1544, 64, 72)])
def test_low_rank_of_a_small_layer(M, in_f, r, out_f):
    """Up to 16 rows, on either side of the rule; between a streaming call before and one after, whose workspace it shares."""
    from triton_funcs import blast_kernels as B, low_rank_kernels as K
    dtype = torch.float16
    rng = np.random.default_rng(M)
    x, a, bm = rng.standard_normal((M, in_f)), rng.standard_normal((in_f, r)) / np.sqrt(in_f), rng.standard_normal((r, out_f)) / np.sqrt(r)
    xb, U, Vt, S = blast_inputs(4, 64, 96, 128, (1,), seed=M)
    args = tuple(dev(t, dtype) for t in (xb,) + tuple(O.blast_to_partial_layout(U, Vt, S)))
    say(f"[case] few rows low rank M={M} {in_f} -> {r} -> {out_f}")
    before = B.triton_blast_full_fp16(*args)
    out = K.triton_low_rank_fp16(dev(x, dtype), dev(a, dtype), dev(bm, dtype))
    assert_close(out, rounded(rounded(x, dtype) @ rounded(a, dtype), dtype) @ rounded(bm, dtype), dtype, f"low rank M={M}", scale=2.0)
    assert torch.equal(B.triton_blast_full_fp16(*args), before)


@pytest.mark.parametrize("M", [1, 2, 16])
def test_long_reductions_stream(M):
    """Up to 16 rows, layers that the small tiles would cut into slices or feed too slowly from HBM: by default the bits of the streaming kernels."""
    from triton_funcs import dense_kernels as D, low_rank_kernels as K, _lib as L
    g = torch.Generator("cuda").manual_seed(M)
    t = lambda *s: (torch.randn(*s, device="cuda", generator=g) / s[0] ** 0.5).half()
    for i, o in ((1544, 768), (3072, 768), (2048, 2048), (4096, 4096)):
        say(f"[case] few rows dense {M} x {i} x {o} streams")
        x, w = t(M, i), t(i, o)
        assert torch.equal(D._dense("test", x, w, L.ALGO_AUTO)[0], D._dense("test", x, w, L.ALGO_STREAM)[0])
    for i, r, o in ((776, 128, 768), (1152, 256, 6912), (768, 256, 2304)):
        say(f"[case] few rows low rank {M} x {i} x {r} x {o} streams")
        x, a, b = t(M, i), t(i, r), t(r, o)
        assert torch.equal(K._low_rank("test", x, a, b, L.ALGO_AUTO, False)[0], K._low_rank("test", x, a, b, L.ALGO_STREAM, False)[0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,b,p,q,r,M", [("triton_blast_bmm_fp16", 12, 96, 104, 64, 129), ("triton_blast_bmm_fp16", 9, 128, 64, 32, 300),
                                            ("triton_blast_full_fp16", 12, 96, 104, 128, 1300)])
def test_nine_to_fifteen_blocks(name, b, p, q, r, M, dtype):
    """Above 128 rows, and with the rank contiguous beyond 5 * 2^15 rows x rank, narrow blocks without a fast mix of their own keep the
    kernels of many rows, bit for bit."""
    from test_gpu_blast import _ref, _run_blast
    from triton_funcs import _lib as L
    x, U, Vt, S = blast_inputs(b, p, q, r, (M,), seed=M + b)
    say(f"[case] {name} b={b} p={p} q={q} r={r} M={M} {dtype}")
    out = _run_blast(name, x, U, Vt, S, dtype, "auto")
    assert_close(out, _ref(x, U, Vt, S, dtype)[0], dtype, f"{name} b={b} M={M}")
    with L.options(BLR_DECODE_ROWS=0):
        assert torch.equal(_run_blast(name, x, U, Vt, S, dtype, "auto"), out)


@pytest.mark.parametrize("b,p,r,q,M", [(16, 32, 256, 128, 1100), (16, 32, 256, 96, 1500), (12, 32, 384, 128, 1409), (4, 32, 1032, 1000, 1000)])
def test_monarch_interleaved_columns(b, p, r, q, M):
    """Interleaved columns with work for half of the chip: the bits of the kernels that BLR_GEMM_MID=0 leaves (the first products fill the
    chip, which that option does not reach)."""
    from triton_funcs import monarch_kernels as K, _lib as L
    g = torch.Generator("cuda").manual_seed(M)
    t = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, w1, w2 = t(M, b * p).half(), (t(b, p, r) / p ** 0.5).half(), (t(b, r, q) / r ** 0.5).half()
    say(f"[case] monarch interleaved b={b} p={p} r={r} q={q} M={M}")
    out = K.triton_monarch_right_left_fp16(x, w1, w2)
    with L.options(BLR_GEMM_MID=0):
        assert torch.equal(K.triton_monarch_right_left_fp16(x, w1, w2), out)
    want = K.triton_monarch_right_left_fp32(x.float(), w1.float(), w2.float())[0]       # (fp32 throughout: only Z is not rounded on the way)
    assert_close(out, want.double().cpu().numpy(), torch.float16, f"monarch interleaved b={b} M={M}", scale=2.0)


def _small_integers(rng, *shape, top):
    return rng.integers(-top, top + 1, shape).astype(np.float64)


# w2 (l, s, r) with more than 256 groups of 64 output columns and ranks up to 1024 (one row: 2048): whole 16-byte pieces of the period and not, one to four
# steps of a round, two rounds, sliced input blocks (1104, 1040 and 2048 rows); w2 (l, r, s) with a period that is no multiple of 4, in column
# chunks of up to four pieces, whose lanes share the steps, and wider; low rank without equal slices
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("name,b,p,rank,s", [("triton_monarch_right_fp16", *c) for c in [(4, 512, 1024, 4200), (16, 88, 304, 1032), (16, 8, 16, 1040), (16, 1040, 48, 1032),
                                                                                         (12, 40, 744, 1416), (2, 1104, 176, 8200), (4, 8, 2048, 4104)]]
                         + [("triton_monarch_right_ideal_fp16", 4, 2048, 512, 4104)]
                         + [("triton_monarch_right_left_fp16", *c) for c in [(16, 88, 304, 224), (16, 8, 16, 8), (16, 1040, 48, 40), (8, 136, 1032, 72), (12, 40, 744, 136),
                                                                         (4, 1024, 1016, 72), (4, 64, 1032, 40), (4, 2752, 8, 8), (4, 64, 760, 1376), (4, 64, 1016, 2056), (4, 64, 232, 1032)]]
                         + [("low_rank", 1, *c) for c in [(3736, 376, 1712), (8, 8, 8), (72, 16, 40), (4088, 1032, 136), (11000, 2056, 72)]])
def test_intermediate_stays_in_fp32_up_to_four_rows(name, b, p, rank, s, M, dtype):
    """Whole numbers and halves of them down to 2^-k whose sums fp32 holds exactly in any order, the intermediate among them, which takes up to 14 bits:
    the result is the exact one, rounded once."""
    if M == 1 and "right_left" in name:
        pytest.skip("served by the single-row kernels")
    if M > 1 and rank == 2048:
        pytest.skip("the intermediate is rounded to the operand type")
    from triton_funcs import low_rank_kernels as LR, _lib as L
    from test_gpu_monarch_lowrank_dense import _blocked, _run_monarch
    rng = np.random.default_rng(rank + M)
    say(f"[case] exact intermediate {name} b={b} p={p} rank={rank} s={s} M={M} {dtype}")
    top = max(2, int((9000 / p ** 0.5) ** 0.5))                      # z of 3000 in the mean square, at most top^2 p
    x, w1 = _small_integers(rng, M, b * p, top=top), _small_integers(rng, b, rank, p, top=top)
    scale = 2.0 ** -round(np.log2(6 * (2 * rank / 3) ** 0.5))       # results of about 500
    w2 = _small_integers(rng, b, s, rank, top=1) * scale
    if name == "low_rank":
        z = x @ w1[0].T
        ref, size = z @ w2[0].T, np.abs(z) @ np.abs(w2[0].T)            # (size: no partial sum is larger)
        run = lambda: LR.triton_low_rank_fp16(*(torch.from_numpy(np.ascontiguousarray(t)).cuda().to(dtype) for t in (x, w1[0].T, w2[0].T)), {"algo": L.ALGO_STREAM})
    else:
        ref, _, z, _ = O.monarch_forward(x, w1, w2)
        size = np.abs(z) @ np.abs(w2).transpose(0, 2, 1)
        if "ideal" in name:
            ref = _blocked(ref, b)
        run = lambda: _run_monarch(name, x, w1, w2, dtype)
    assert p * top * top < 2 ** 24 and size.max() / scale < 2 ** 24
    want = torch.from_numpy(ref).float().to(dtype)
    assert torch.equal(run().cpu().reshape(want.shape), want)
    with L.options(BLR_DECODE_ROWS=0):                               # the kernels that take the call where the skinny products do not
        assert torch.equal(run().cpu().reshape(want.shape), want)
    bias = torch.from_numpy(_small_integers(rng, b * s, top=200)).to(dtype)
    with L.fused_epilogue(bias.cuda(), None):
        out = run().cpu().reshape(want.shape)
    assert torch.equal(out, (want.float() + bias.float()).to(dtype))
