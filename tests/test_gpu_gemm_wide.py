"""GPU parity of the GEMM on tiles of 256 rows x 96 .. 352 columns (csrc/blr_gemm_wide.hip) against the oracle.

BLR_GEMM_WIDE = 3 .. 11 asks for tiles of that many times 32 columns for every product that the kernels take, so the edges of every width are met
on small problems: one row or column more or less than a tile, reductions that end inside a stage of 64 k (with 8 .. 56 k left over),
more tiles than compute units (a workgroup walks several), the output stage, gated halves and Monarch's scatter.
"""
import numpy as np
import pytest
import torch

from oracle import blr_oracle as O
from gpu_util import assert_close, blast_call, blast_inputs, dev, launches, rounded, say, ulp

pytestmark = pytest.mark.gpu

TILED = {"algo": 2}
WIDTHS = list(range(3, 12))


def _product_close(out, x, w, dtype, what):
    """One rounding of a sum in fp32: half a unit of dtype, and K roundings of fp32 of the terms' absolute sum."""
    ref, mag = x @ w, np.abs(x) @ np.abs(w)
    err = np.abs(out.double().cpu().numpy() - ref)
    bound = 0.5 * ulp(ref, dtype) * (1 + 2.0 ** -9) + x.shape[1] * 2.0 ** -24 * mag
    assert (err <= bound).all(), f"{what}: {np.max(err / bound):.3f} of the bound"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tn", WIDTHS)
def test_dense_ragged_tiles(tn, dtype):
    from triton_funcs import dense_kernels as K, _lib as L
    w32 = 32 * tn
    for m, k, n in ((256, 128, w32), (257, 72, w32 + 8), (255, 136, w32 - 8), (31, 1000, 2 * w32 - 24), (513, 192, 8), (300, 120, 3 * w32 + 16), (40, 352, w32)):
        rng = np.random.default_rng(m + k + tn)
        x, w = rounded(rng.standard_normal((m, k)), dtype), rounded(rng.standard_normal((k, n)) / np.sqrt(k), dtype)
        say(f"[case] wide dense tn={tn} {m}x{n}x{k} {dtype}")
        with L.options(BLR_GEMM_WIDE=tn):
            out = K.triton_dense_fp16(dev(x, dtype), dev(w, dtype), TILED)
        _product_close(out, x, w, dtype, f"{m}x{n}x{k}")


@pytest.mark.parametrize("tn", WIDTHS)
def test_workgroups_that_walk_several_tiles(tn):
    """More than two tiles for most of 256 compute units, the last ones ragged in rows and columns; every kind of last stage."""
    from triton_funcs import dense_kernels as K, _lib as L
    dtype = torch.float16
    for k in (72, 128, 168):
        m, n = 256 * 8 + 19, 32 * tn * 66 + 24
        g = torch.Generator("cuda").manual_seed(tn + k)
        x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
        w = (torch.randn(k, n, device="cuda", generator=g) / k ** 0.5).to(dtype)
        say(f"[case] wide dense tn={tn} {m}x{n}x{k}, several tiles a workgroup")
        with L.options(BLR_GEMM_WIDE=tn):
            out = K.triton_dense_fp16(x, w, TILED)
        ref, mag = x.float() @ w.float(), x.float().abs() @ w.float().abs()        # (fp32 itself adds k roundings on this side)
        err = (out.float() - ref).abs()
        assert (err <= 2.0 ** -11 * 1.01 * ref.abs() + 2 * k * 2.0 ** -24 * mag + 2.0 ** -24).all(), f"tn={tn} k={k}: {float(err.max())}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tn", WIDTHS)
def test_blast_and_low_rank_through_wide_tiles(tn, dtype):
    """Batches, both orders of the second operand; two products of one matrix."""
    from triton_funcs import blast_kernels as K, low_rank_kernels as LR, _lib as L
    for b, p, q, r, m in ((4, 80, 40, 72, 300), (2, 176, 264, 136, 257)):
        x, U, Vt, S = blast_inputs(b, p, q, r, (m,), seed=b + m)
        ref = O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0]
        for name, lay in (("triton_blast_full_fp16", O.blast_to_partial_layout), ("triton_blast_bmm_fp16", O.blast_to_bmm_layout)):
            Uk, Vk, Sk = lay(U, Vt, S)
            say(f"[case] wide {name} tn={tn} b={b} p={p} q={q} r={r} m={m} {dtype}")
            with L.options(BLR_GEMM_WIDE=tn):
                out = getattr(K, name)(dev(x, dtype), dev(Uk, dtype), dev(Vk, dtype), dev(Sk, dtype), TILED)
            assert_close(out, ref, dtype, name)
    rng = np.random.default_rng(tn)
    x, A, B = rng.standard_normal((270, 200)), rng.standard_normal((200, 104)) / 104 ** 0.5, rng.standard_normal((104, 296)) / 104 ** 0.5
    say(f"[case] wide low rank tn={tn} {dtype}")
    with L.options(BLR_GEMM_WIDE=tn):
        out = LR.triton_low_rank_fp16(dev(x, dtype), dev(A, dtype), dev(B, dtype), TILED)
    assert_close(out, rounded(x, dtype) @ rounded(A, dtype) @ rounded(B, dtype), dtype, "low rank")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tn", WIDTHS)
def test_side_job_of_the_first_product(tn, dtype):
    """16 blocks of narrow outputs: workgroups of the first product's launch re-lay U and S for the kernel that does the rest, from both orders of either."""
    from triton_funcs import _lib as L
    for b, p, q, r, m in ((16, 136, 72, 96, 130), (16, 104, 8, 32, 300), (16, 200, 80, 160, 257)):
        x, U, Vt, S = blast_inputs(b, p, q, r, (m,), seed=p + m)
        ref = O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0]
        for name, lay in (("full", O.blast_to_partial_layout), ("bmm", O.blast_to_bmm_layout)):
            call, out = blast_call(name, *(dev(t, dtype) for t in (x,) + lay(U, Vt, S)), 2)
            say(f"[case] wide, side job {name} tn={tn} p={p} q={q} r={r} m={m} {dtype}")
            with L.options(BLR_GEMM_WIDE=tn, BLR_DECODE_ROWS=0):
                first, *rest = launches(call)
                side = -(-(16 * r // 8 * q + r * 64) // 512)
                assert len(rest) == 1 and first[2] == (512, 1, 1) and first[1][0] >= -(-side // 8) * 8 + 8
                call(L.stream_ptr(out.device))
            assert_close(out, ref, dtype, name)


# (rows, rank, columns per input block, the ring kernel's tile): 16 blocks of narrow outputs whose x V the rules give to a ring kernel
@pytest.mark.parametrize("m,r,p,ring", [(300, 768, 688, 128128), (1000, 320, 1024, 256128)])
def test_side_job_on_the_ring_kernels(m, r, p, ring):
    from triton_funcs import _lib as L
    b, q, dtype = 16, 72, torch.float16
    g = torch.Generator("cuda").manual_seed(m)
    rnd = lambda *sh: torch.randn(*sh, device="cuda", generator=g)
    x, U, V, S = rnd(m, b * p).to(dtype), (rnd(b, q, r) / r ** 0.5).to(dtype), (rnd(b, p, r) / p ** 0.5).to(dtype), rnd(r, b, b).to(dtype)
    call, out = blast_call("bmm", x, U, V, S, 2)
    say(f"[case] side job on the ring kernels m={m} r={r} p={p}")
    auto, by_name, on_wide = _three_ways(call, ring, 4)
    assert len(auto) == 2 and auto[0] == by_name[0] != on_wide[0]
    call(L.stream_ptr(out.device))
    Y = torch.bmm(x.double().view(m, b, p).transpose(0, 1).contiguous(), V.double())
    ref = torch.cat([(Y * S[:, i].double().t()[:, None]).sum(0) @ U[i].double().t().contiguous() for i in range(b)], 1)
    assert_close(out, ref.cpu().numpy(), dtype, "side job")


@pytest.mark.parametrize("tn", WIDTHS)
def test_output_stage_and_gated_halves(tn):
    from triton_funcs import dense_kernels as D, _lib as L
    dtype = torch.float16
    for m, k, n in ((300, 136, 32 * tn + 40), (256 * 5 + 3, 72, 32 * tn * 60 + 8)):
        g = torch.Generator("cuda").manual_seed(m + tn)
        rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
        x, w, bias, resid = rnd(m, k), rnd(k, 2 * n), rnd(2 * n), rnd(m, n)
        w = (w.float() / k ** 0.5).to(dtype)
        gate = rnd(-(-m // 7), n)
        say(f"[case] wide output stage tn={tn} {m}x{n}x{k}")
        y = (x.double() @ w.double()).half().double() + bias.double()               # the result is rounded before the bias is added
        h = torch.nn.functional.gelu(y[:, :n], approximate="tanh").half().double()
        ref = resid.double() + gate.double().repeat_interleave(7, 0)[:m] * h
        with L.options(BLR_GEMM_WIDE=tn), L.fused_epilogue(bias[:n].contiguous(), "gelu_tanh", gate=gate, gate_rows=7, residual=resid):
            out = D.triton_dense_fp16(x, w[:, :n].contiguous(), TILED)
        assert_close(out, ref.cpu().numpy(), dtype, "gate and residual")
        with L.options(BLR_GEMM_WIDE=tn), L.fused_epilogue(bias, "silu_mul"):
            out = D.triton_dense_fp16(x, w, TILED)
        ref = torch.nn.functional.silu(y[:, :n]).half().double() * y[:, n:].half().double()
        assert_close(out, ref.cpu().numpy(), dtype, "gated halves")


@pytest.mark.parametrize("tn", WIDTHS)
def test_monarch_scatter(tn):
    """A permutation writes every value where the other kernels write it."""
    from triton_funcs import monarch_kernels as K, _lib as L
    dtype = torch.float16
    for b, p, rank, s, m in ((4, 96, 160, 72, 300), (2, 80, 32 * tn, 40, 257), (16, 128, 384, 24, 270)):
        g = torch.Generator("cuda").manual_seed(b + tn)
        rnd = lambda *sh: torch.randn(*sh, device="cuda", generator=g).to(dtype)
        x, w1, w2 = rnd(1, m, b * p), (rnd(b, p, rank).float() / p ** 0.5).to(dtype), (rnd(b, rank, s).float() / rank ** 0.5).to(dtype)
        say(f"[case] wide monarch tn={tn} b={b} p={p} rank={rank} s={s} m={m}")
        with L.options(BLR_GEMM_WIDE=tn):
            out = K.triton_monarch_right_left_fp16(x, w1, w2, TILED)
        with L.options(BLR_GEMM_WIDE=0):
            ref = K.triton_monarch_right_left_fp16(x, w1, w2, TILED)
        assert_close(out, ref.double().cpu().numpy(), dtype, "monarch", scale=0.5)


@pytest.mark.parametrize("k", [72, 88, 120, 184])
def test_infinite_weights_stay_infinite(k):
    """The last stage of a reduction is read again from before its start: what it shares with the stage before counts once, infinities too."""
    from triton_funcs import dense_kernels as K, _lib as L
    x, w = np.ones((40, k)), np.ones((k, 96))
    w[k - 64, 3] = w[k - 1, 5] = w[0, 7] = w[63, 9] = np.inf
    with L.options(BLR_GEMM_WIDE=3):
        out = K.triton_dense_fp16(dev(x, torch.float16), dev(w, torch.float16), TILED).double().cpu().numpy()
    assert (out == x @ w).all()


def _three_ways(call, ring, wide):
    """What a call launches by the rules, with a ring kernel asked for by name, and with tiles of 32 wide columns."""
    from triton_funcs import _lib as L
    with L.options(BLR_GEMM_RING_TILE=ring, BLR_GEMM_RING_BK=64, BLR_GEMM_RING_WAVES=8, BLR_GEMM_RING_PER_CU=2 if ring == 128128 else 0):
        by_name = launches(call)
    with L.options(BLR_GEMM_WIDE=wide):
        on_wide = launches(call)
    return launches(call), by_name, on_wide


# (columns per input block, rank, rows, tile of the ring kernel, the wide tile that would be next): long reductions whose rows of x lie far apart
@pytest.mark.parametrize("p,rank,m,ring,wide", [(2752, 1024, 2048, 256128, 4), (1024, 1024, 2048, 256128, 4), (2752, 1024, 4096, 256256, 8)])
def test_monarch_of_long_blocks_stays_with_the_ring_kernels(p, rank, m, ring, wide):
    from triton_funcs import _lib as L
    b, s, dtype = 4, 64, torch.float16
    g = torch.Generator("cuda").manual_seed(p + m)
    rnd = lambda *sh: torch.randn(*sh, device="cuda", generator=g).to(dtype)
    x, w1, w2 = rnd(m, b * p), (rnd(b, p, rank).float() / p ** 0.5).to(dtype), rnd(b, rank, s)
    mid, out = torch.full((b, m, rank), float("nan"), device="cuda", dtype=dtype), torch.empty(m, b * s, device="cuda", dtype=dtype)

    def call(stream):
        L.check(L.lib().blr_monarch_fwd(x.data_ptr(), b * p, w1.data_ptr(), w2.data_ptr(), out.data_ptr(), b * s, mid.data_ptr(), m, b * p, b * s, b, rank, L.F16, L.W2_RS,
                                        L.OUT_BLOCKED, 2, None, 0, stream), "blr_monarch_fwd")

    say(f"[case] monarch, first product {m}x{rank}x{p} in {b}")
    auto, by_name, on_wide = _three_ways(call, ring, wide)
    assert auto[0] == by_name[0] != on_wide[0]
    call(L.stream_ptr(x.device))
    y = torch.stack([x[:, k * p:(k + 1) * p].float() @ w1[k].float() for k in range(b)])          # column c of block k -> block c / per, column k per + c % per
    per = rank // b
    ref = y.view(b, m, b, per).permute(2, 1, 0, 3).reshape(b, m, rank)
    assert_close(mid, ref.double().cpu().numpy(), dtype, "first product", scale=0.5)


@pytest.mark.parametrize("m,n,k,act,ring,wide", [(4096, 4096, 11008, "", 256256, 8), (1000, 6912, 1152, "gelu_tanh", 256128, 4), (2048, 2304, 2048, "gelu_tanh", 256128, 4),
                                                 (1043, 6328, 1992, "silu_mul", 256128, 4)])
def test_dense_products_that_the_ring_kernels_keep(m, n, k, act, ring, wide):
    """Plain, with bias and activation, and gated halves."""
    from triton_funcs import _lib as L
    dtype, h = torch.float16, 2 if act == "silu_mul" else 1
    g = torch.Generator("cuda").manual_seed(m)
    rnd = lambda *sh: torch.randn(*sh, device="cuda", generator=g).to(dtype)
    x, w, bias, out = rnd(m, k), (rnd(k, h * n).float() / k ** 0.5).to(dtype), rnd(h * n), torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
    code = {"": 0, "gelu_tanh": 1, "silu_mul": 3}[act]

    def call(stream):
        L.check(L.lib().blr_dense_fwd_ep(x.data_ptr(), k, w.data_ptr(), out.data_ptr(), n, m, k, h * n, L.F16, 2, None, 0, stream, bias.data_ptr() if act else None, code), "dense")

    say(f"[case] dense {m}x{n}x{k} {act}")
    auto, by_name, on_wide = _three_ways(call, ring, wide)
    assert auto == by_name and auto != on_wide
    call(L.stream_ptr(x.device))
    y = x.float() @ w.float()
    if act:
        y = y + bias.float()
        y = torch.nn.functional.gelu(y, approximate="tanh") if h == 1 else torch.nn.functional.silu(y[:, :n]) * y[:, n:]
    assert_close(out, y.double().cpu().numpy(), dtype, "dense")


@pytest.mark.parametrize("q,r,m,kept", [(1952, 120, 2833, True), (832, 192, 2600, True), (1952, 208, 2833, False), (1000, 120, 1900, False)])
def test_gated_halves_of_short_reductions(q, r, m, kept):
    """Eight blocks as four pairs, less than 200 k: with results for several rounds the ring kernels' rules, otherwise tiles of this kernel."""
    from triton_funcs import _lib as L
    b, p, dtype = 8, 40, torch.float16
    g = torch.Generator("cuda").manual_seed(q)
    rnd = lambda *sh: torch.randn(*sh, device="cuda", generator=g).to(dtype)
    x, U, V, S, bias = rnd(m, b * p), (rnd(b, q, r).float() / r ** 0.5).to(dtype), (rnd(b, p, r).float() / p ** 0.5).to(dtype), rnd(r, b, b), rnd(b * q)
    out = torch.full((m, b * q // 2), float("nan"), device="cuda", dtype=dtype)
    lib = L.lib()
    ws = torch.empty(lib.blr_blast_workspace_bytes(m, b * p, b * q, b, r, L.F16, 2), dtype=torch.uint8, device="cuda")

    def call(stream):
        L.check(lib.blr_blast_fwd_ep(x.data_ptr(), b * p, U.data_ptr(), V.data_ptr(), S.data_ptr(), out.data_ptr(), b * q // 2, m, b * p, b * q, b, r, L.F16, L.U_QR, L.S_RIJ, 2,
                                     ws.data_ptr(), ws.numel(), stream, bias.data_ptr(), 3), "blr_blast_fwd_ep")

    say(f"[case] gated halves q={q} r={r} m={m}")
    auto = launches(call)
    with L.options(BLR_GEMM_WIDE=0):
        ring = launches(call)
    assert (auto[-1] == ring[-1]) == kept
    call(L.stream_ptr(x.device))
    Y = torch.bmm(x.float().view(m, b, p).transpose(0, 1).contiguous(), V.float()).half().float()
    y = torch.cat([(Y * S[:, i].float().t()[:, None]).sum(0).half().float() @ U[i].float().t().contiguous() for i in range(b)], 1).half().float() + bias.float()
    h = b * q // 2
    assert_close(out, (torch.nn.functional.silu(y[:, :h]) * y[:, h:]).double().cpu().numpy(), dtype, "gated halves")
