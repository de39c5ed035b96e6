"""The shims' workspaces under graphs and threads: replays go on where the capture left them, whatever the stream's calls have needed
since, and the launches of two threads' calls on one stream do not mix."""
import threading

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["native", "python"])
def path(request):
    from triton_funcs import _lib as L
    assert L.call_path(), "the native call path did not load"
    host = L._host
    L._host = host if request.param == "native" else False
    yield L
    L._host = host


def _problem(rows, b, p, q, r, seed=0):
    g = torch.Generator("cuda").manual_seed(seed)
    t = lambda *s: (torch.randn(*s, device="cuda", generator=g) / r ** 0.5).half()
    return t(1, rows, b * p), t(b, r, q), t(b, p, r), t(b, b, r)


def _beyond(L, rows):
    """What the current stream has for calls of `rows`, and a call that wants more."""
    from triton_funcs import blast_kernels as B, dense_kernels as D
    have = L.workspace(torch.device("cuda", 0), 1, L.ALGO_AUTO, rows, L.F16)
    if rows <= 16:
        n = 4096
        while L.lib().blr_dense_workspace_bytes(16, 2048, n, L.F16, L.ALGO_AUTO) <= have.numel():
            n *= 2
        assert n <= 1 << 17
        x, w = torch.randn(16, 2048, device="cuda").half(), (torch.randn(2048, n, device="cuda") / 45).half()
        return have, lambda: D.triton_dense_fp16(x, w)
    while L.lib().blr_blast_workspace_bytes(rows, 256, 256, 16, 512, L.F16, L.ALGO_AUTO) <= have.numel():
        rows *= 2
    args = _problem(rows, 16, 16, 16, 512)
    return have, lambda: B.triton_blast_full_fp16(*args)


# up to 16 rows: a streaming workspace, whose control words carry from call to call; more: plain scratch
@pytest.mark.parametrize("rows", [2, 40])
def test_growth_after_a_capture(path, rows):
    from triton_funcs import blast_kernels as B
    L = path
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        x, U, V, S = _problem(rows, 4, 64, 96, 128)
        want = B.triton_blast_full_fp16(x, U, V, S).clone()
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = B.triton_blast_full_fp16(x, U, V, S)
        old, larger = _beyond(L, rows)
        at, size = old.data_ptr(), old.numel()
        del old
        say(f"[case] workspace of {size} bytes outgrown, {rows} rows")
        first = larger().clone()
        assert L.workspace(x.device, 1, L.ALGO_AUTO, rows, L.F16).data_ptr() != at
        junk = [torch.full((size,), 90, dtype=torch.uint8, device="cuda") for _ in range(4)]
        assert all(t.data_ptr() != at for t in junk)
        for _ in range(3):
            out.zero_()
            g.replay()
            s.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(larger(), first)
            assert torch.equal(B.triton_blast_full_fp16(x, U, V, S), want)
        assert all(bool((t == 90).all()) for t in junk)
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows", [2, 40])
def test_growth_under_capture(path, rows):
    """Without a warm-up the workspace is the graph's: its zeros exist in replays only, so eager calls keep to their own."""
    L = path
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        old, larger = _beyond(L, rows)
        say(f"[case] workspace of {old.numel()} bytes too small under capture, {rows} rows")
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            outs = [larger(), larger()]
        want = larger().clone()                                     # before any replay
        for _ in range(3):
            for o in outs:
                o.zero_()
            g.replay()
            s.synchronize()
            assert all(torch.equal(o, want) for o in outs)
            assert torch.equal(larger(), want)
    torch.cuda.synchronize()


# one row and a few: streaming workspaces; 40: three launches over scratch; 300: products in tiles; gated: the full-width result behind it
@pytest.mark.parametrize("rows", [1, 4, 40, 300])
def test_threads_on_one_stream(path, rows):
    from triton_funcs import blast_kernels as B, dense_kernels as D
    L = path
    w = (torch.randn(1024, 512, device="cuda") / 32).half()
    xs = [torch.randn(rows, 1024, device="cuda").half() for _ in range(2)]
    args = [_problem(rows, 16, 64, 72, 128, seed) for seed in range(2)]

    def calls(i):
        def gated():
            with L.fused_epilogue(None, "silu_mul"):
                return D.triton_dense_fp16(xs[i], w)
        return (lambda: B.triton_blast_full_fp16(*args[i])), gated

    want = [[c() for c in calls(i)] for i in range(2)]
    torch.cuda.synchronize()
    say(f"[case] two threads on one stream, {rows} rows")
    start, got, errors = threading.Barrier(2), [[], []], []

    def work(i):
        try:
            cs = calls(i)
            start.wait()
            for n in range(100):
                got[i].append((n % 2, cs[n % 2]()))
        except Exception as e:                                      # noqa: BLE001 - shown by the test
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(2):
        assert len(got[i]) == 100 and all(torch.equal(o, want[i][k]) for k, o in got[i])
