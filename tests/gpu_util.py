"""Shared helpers of the GPU parity tests (seeded inputs, oracle comparison, which kernels a call launches)."""
import ctypes
import sys

import numpy as np
import torch

TOL = {torch.float16: 1e-2, torch.bfloat16: 2e-2, torch.float32: 1e-4}


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype).contiguous()


def back(t):
    return t.detach().to(torch.float64).cpu().numpy()


def rounded(a, dtype):
    """Values as the kernel sees them: rounded to dtype, returned as float64 numpy."""
    return torch.from_numpy(np.ascontiguousarray(a)).to(dtype).to(torch.float64).numpy()


def assert_close(got, ref, dtype, what, scale=1.0):
    got = back(got) if isinstance(got, torch.Tensor) else np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    assert got.shape == ref.shape, f"{what}: shape {got.shape} != {ref.shape}"
    assert np.isfinite(got).all(), f"{what}: non-finite output"
    err = np.abs(got - ref).max()
    bound = TOL[dtype] * scale * max(np.abs(ref).max(), 1e-30)
    assert err <= bound, f"{what}: max abs err {err:.4g} > {bound:.4g} (max|ref| {np.abs(ref).max():.4g})"
    return err


def blast_inputs(b, p, q, r, lead, seed=0):
    """x ~ N(0,1); U, Vt ~ N(0, 1/r); S ~ N(0,1) in the reference's torch layouts (float64 numpy)."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(tuple(lead) + (b * p,))
    U = rng.standard_normal((b, q, r)) / np.sqrt(r)
    Vt = rng.standard_normal((b, r, p)) / np.sqrt(r)
    S = rng.standard_normal((b, b, r))
    return x, U, Vt, S


def ulp(ref, dtype):
    """Spacing of dtype's numbers at |ref| (float64 numpy): 2^(e - 10) for fp16, 2^(e - 7) for bf16, normal range."""
    a = np.maximum(np.abs(np.asarray(ref, dtype=np.float64)), 2.0 ** -14)
    return 2.0 ** (np.floor(np.log2(a)) - {torch.float16: 10, torch.bfloat16: 7}[dtype])


class _KernelNode(ctypes.Structure):                 # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3), ("params", ctypes.c_void_p),
                ("lds", ctypes.c_uint32)]


def launches(call):
    """(host function, grid, block, dynamic LDS) of every kernel that call(stream) launches on the stream that it is handed: captured into a graph that is looked at and
    not run.  call allocates nothing."""
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    stream, graph, n = torch.cuda.Stream(), ctypes.c_void_p(), ctypes.c_size_t()
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(ctypes.c_void_p(stream.cuda_stream), 2) == 0          # relaxed
    call(stream.cuda_stream)
    assert hip.hipStreamEndCapture(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind, k = ctypes.c_int(), _KernelNode()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0 and kind.value == 0, "a node that is no kernel"
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(k)) == 0
        out.append((k.func, tuple(k.grid), tuple(k.block), k.lds))
    assert hip.hipGraphDestroy(graph) == 0
    return out


def blast_call(name, x, U, V, S, algo):
    """A call of the C ABI with the layouts of name's functions, for launches() or a stream, and the tensor that it writes."""
    from triton_funcs import _lib as L
    bmm = "bmm" in name
    (b, p, r), m = V.shape, x.shape[0]
    q = U.shape[1] if bmm else U.shape[2]
    dt = L.F16 if x.dtype == torch.float16 else L.BF16
    out = torch.full((m, b * q), float("nan"), device="cuda", dtype=x.dtype)
    ws = torch.empty(L.lib().blr_blast_workspace_bytes(m, b * p, b * q, b, r, dt, algo), dtype=torch.uint8, device="cuda")

    def call(stream):
        L.check(L.lib().blr_blast_fwd(x.data_ptr(), b * p, U.data_ptr(), V.data_ptr(), S.data_ptr(), out.data_ptr(), b * q, None, None, m, b * p, b * q, b, r, dt,
                                      L.U_QR if bmm else L.U_RQ, L.S_RIJ if bmm else L.S_JIR, algo, ws.data_ptr(), ws.numel(), stream), "blr_blast_fwd")
    return call, out
