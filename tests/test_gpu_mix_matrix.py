"""GPU parity of the mix on the matrix cores: Z_i = sum_j S(i, j, r) Y_j as a launch of its own (blast_mixm_kernel), which BLAST calls above 16 rows take
whose input blocks are too wide for a fused first half, and that first half (blast_ymix_kernel).  Edges: rows and ranks that end inside a tile of 32 x 64, 4 to 16 blocks, both
orders of S, workgroups that walk several tiles and change the rank tile on the way."""
import numpy as np
import pytest
import torch

from oracle import blr_oracle as O
from gpu_util import assert_close, blast_call, blast_inputs, dev, launches, rounded, say, ulp

pytestmark = pytest.mark.gpu
TILED = {"algo": 2}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", ["triton_blast_full_fp16", "triton_blast_bmm_fp16"])
@pytest.mark.parametrize("b,r,m", [(4, 8, 17), (4, 72, 33), (8, 64, 130), (8, 200, 300), (12, 136, 95), (12, 8, 17), (16, 8, 17), (16, 72, 33), (16, 8, 31), (16, 56, 257),
                                   (16, 192, 64), (16, 328, 1000)])
def test_mix_on_the_matrix_cores(b, r, m, name, dtype):
    from triton_funcs import _lib as L
    p, q = 200, 24                                    # (columns of a block that no fused first half takes)
    x, U, Vt, S = blast_inputs(b, p, q, r, (m,), seed=b + r + m)
    Uk, Vk, Sk = (O.blast_to_bmm_layout if "bmm" in name else O.blast_to_partial_layout)(U, Vt, S)
    say(f"[case] mix {name} b={b} r={r} m={m} {dtype}")
    call, out = blast_call(name, *(dev(t, dtype) for t in (x, Uk, Vk, Sk)), 2)
    with L.options(BLR_BLAST_MIXU=0, BLR_DECODE_ROWS=0):
        kernels = launches(call)
        assert len(kernels) == 3 and kernels[1][2:] == ((512, 1, 1), b * 4096)        # the mix of a tile of 32 x 64 in LDS
        call(L.stream_ptr(out.device))
    assert_close(out, O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0], dtype, name)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("order", ["rij", "jir", "ijr"])
@pytest.mark.parametrize("b", [4, 8, 12, 16])
def test_mix_element_by_element(b, order, dtype):
    """One rounding of sums in fp32, for a problem of more tiles than two per compute unit holds (rank tiles change inside a run)."""
    import ctypes
    from triton_funcs import _lib as L
    m, r, p, q = 40 * 32 + 5, 15 * 64 + 40, 16, 8
    dt = L.F16 if dtype == torch.float16 else L.BF16
    g = torch.Generator("cuda").manual_seed(b)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    x, V, U, Sc = rnd(m, b * p), rnd(b, p, r), rnd(b, r, q), rnd(b, b, r)
    S = {"rij": Sc.permute(2, 0, 1), "jir": Sc.permute(1, 0, 2), "ijr": Sc}[order].contiguous()
    z, y = (torch.full((b, m, r), float("nan"), device="cuda", dtype=dtype) for _ in range(2))
    out = torch.empty(m, b * q, device="cuda", dtype=dtype)
    lib = L.lib()
    lay = {"rij": L.S_RIJ, "jir": L.S_JIR, "ijr": L.S_IJR}[order]
    say(f"[case] mix elements b={b} S ({order}) {dtype}")
    ws = torch.empty(lib.blr_blast_workspace_bytes(m, b * p, b * q, b, r, dt, 2), dtype=torch.uint8, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.blr_blast_fwd(ptr(x), b * p, ptr(U), ptr(V), ptr(S), ptr(out), b * q, ptr(z), ptr(y), m, b * p, b * q, b, r, dt, L.U_RQ, lay, 2,
                           ptr(ws), ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.blr_last_error()
    yd, sd = y.double(), Sc.double()
    ref, mag = torch.zeros_like(yd), torch.zeros_like(yd)
    for i in range(b):
        for j in range(b):
            t = sd[i, j] * yd[j]
            ref[i] += t
            mag[i] += t.abs()
    err = (z.double() - ref).abs().cpu().numpy()
    bound = 0.5 * ulp(ref.cpu().numpy(), dtype) * (1 + 2.0 ** (-10 if dtype == torch.float16 else -7)) + 16 * 2.0 ** -24 * mag.cpu().numpy()
    assert (err <= bound).all(), f"{np.max(err / bound):.3f} of the bound"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", ["triton_blast_full_fp16", "triton_blast_bmm_fp16"])
@pytest.mark.parametrize("b,p,r,m", [(16, 192, 128, 1100), (16, 136, 64, 1300), (12, 208, 136, 300), (8, 200, 72, 131), (4, 200, 200, 2100)])
def test_s_off_its_boundary_mixes_to_the_same_bits(b, p, r, m, name, dtype):
    """S one element off the 16 bytes (or the 8 of (r, i, j)): the same kernel and sums, so the same bits; in fp16 the kernels that it went to otherwise sum in fp16."""
    from triton_funcs import blast_kernels as K, _lib as L
    x, U, Vt, S = blast_inputs(b, p, 24, r, (m,), seed=b + r)
    Uk, Vk, Sk = (O.blast_to_bmm_layout if "bmm" in name else O.blast_to_partial_layout)(U, Vt, S)
    xd, ud, vd, sd = dev(x, dtype), dev(Uk, dtype), dev(Vk, dtype), dev(Sk, dtype)
    off = torch.empty(sd.numel() + 1, device="cuda", dtype=dtype)[1:].view(sd.shape)
    off.copy_(sd)
    say(f"[case] mix {name} b={b} p={p} r={r} m={m} {dtype}, S one element off")
    with L.options(BLR_BLAST_MIXU=0, BLR_DECODE_ROWS=0):
        out, ref = (getattr(K, name)(xd, ud, vd, s, TILED) for s in (off, sd))
    assert torch.equal(out, ref)


def test_mix_past_two_gib_and_65536_tiles():
    """Y of more than 2 GiB (its offsets no longer fit 31 bits) in more than 65536 tiles of 32 x 64: sums in fp32 as at every other size, looked at in rows of the first
    tiles, about the middle, and of the last, ragged ones."""
    import ctypes
    from triton_funcs import _lib as L
    dtype, b, m, r, p, q = torch.float16, 16, 131072 + 4096 + 21, 1032, 8, 8
    g = torch.Generator("cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    x, V, U, S = rnd(m, b * p), rnd(b, p, r), rnd(b, r, q), rnd(b, b, r)
    z, y = (torch.empty(b, m, r, device="cuda", dtype=dtype) for _ in range(2))
    out = torch.empty(m, b * q, device="cuda", dtype=dtype)
    lib = L.lib()
    say(f"[case] mix of Y with {y.numel() * 2} bytes")
    ws = torch.empty(lib.blr_blast_workspace_bytes(m, b * p, b * q, b, r, L.F16, 2), dtype=torch.uint8, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.blr_blast_fwd(ptr(x), b * p, ptr(U), ptr(V), ptr(S), ptr(out), b * q, ptr(z), ptr(y), m, b * p, b * q, b, r, L.F16, L.U_RQ, L.S_IJR, 2,
                           ptr(ws), ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.blr_last_error()
    for rows in (slice(0, 70), slice(m // 2, m // 2 + 70), slice(m - 70, m)):
        yd, sd = y[:, rows].double(), S.double()
        assert torch.allclose(yd[3], x[rows, 3 * p:4 * p].double() @ V[3].double(), rtol=1e-3, atol=1e-2)
        ref = torch.stack([(sd[i][:, None] * yd).sum(0) for i in range(b)])
        mag = torch.stack([(sd[i][:, None] * yd).abs().sum(0) for i in range(b)])
        err = (z[:, rows].double() - ref).abs().cpu().numpy()
        bound = 0.5 * ulp(ref.cpu().numpy(), dtype) * (1 + 2.0 ** -10) + 16 * 2.0 ** -24 * mag.cpu().numpy()
        assert (err <= bound).all(), f"{np.max(err / bound):.3f} of the bound"


FUSED = {"algo": 3}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", ["triton_blast_full_fp16", "triton_blast_bmm_fp16"])
@pytest.mark.parametrize("b,p,r,m", [(16, 72, 288, 300), (16, 8, 8, 17), (16, 96, 72, 33), (12, 40, 136, 64), (8, 184, 200, 257), (4, 104, 72, 31),
                                     (4, 200, 64, 130), (8, 64, 328, 1500), (4, 24, 1000, 2100), (16, 136, 64, 95),
                                     (16, 72, 264, 1650), (12, 40, 520, 929), (16, 136, 1000, 545), (4, 72, 64, 128 * 32), (4, 72, 64, 256 * 32 + 1)])
def test_fused_first_half(b, p, r, m, name, dtype):
    """Blocks of one, two and three pieces of columns (the last one overlapping the one before), ranks and rows that end inside a tile of 16 rows
    (problems of at most 256 tiles of 32) and of 32, workgroups that walk several tiles."""
    from triton_funcs import blast_kernels as K, _lib as L
    q = 16
    x, U, Vt, S = blast_inputs(b, p, q, r, (m,), seed=b + r + m)
    Uk, Vk, Sk = (O.blast_to_bmm_layout if "bmm" in name else O.blast_to_partial_layout)(U, Vt, S)
    say(f"[case] fused {name} b={b} p={p} r={r} m={m} {dtype}")
    with L.options(BLR_BLAST_YMIXW=0):
        out = getattr(K, name)(dev(x, dtype), dev(Uk, dtype), dev(Vk, dtype), dev(Sk, dtype), FUSED)
    assert_close(out, O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0], dtype, name)


@pytest.mark.parametrize("name", ["triton_blast_full_fp16", "triton_blast_bmm_fp16"])
def test_fused_first_half_with_s_off_its_boundary(name):
    from triton_funcs import blast_kernels as K
    dtype, b, p, q, r, m = torch.float16, 8, 56, 24, 88, 150
    x, U, Vt, S = blast_inputs(b, p, q, r, (m,), seed=1)
    Uk, Vk, Sk = (O.blast_to_bmm_layout if "bmm" in name else O.blast_to_partial_layout)(U, Vt, S)
    flat = torch.empty(Sk.size + 1, device="cuda", dtype=dtype)
    s = flat[1:].view(Sk.shape)
    s.copy_(dev(Sk, dtype))
    say(f"[case] fused {name}, S one element off")
    out = getattr(K, name)(dev(x, dtype), dev(Uk, dtype), dev(Vk, dtype), s, FUSED)
    assert_close(out, O.blast_forward(rounded(x, dtype), rounded(U, dtype), rounded(Vt, dtype), rounded(S, dtype))[0], dtype, name)
