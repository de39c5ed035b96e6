"""Benchmark of the structured-linear hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-table] [--no-cpu]

A step is one pass over the six BLAST linears of a Llama-7B decoder layer (q, k, v, o 4096->4096
r=512; gate_up 4096->22016 r=1024; down 11008->4096 r=1024; b=16, fp16) at M = 1 token, i.e. the
decode case the headline metric is quoted on.  Weights are synthetic (seed 0, std 1/sqrt(r)) and
already resident in HBM; the launches go through the C ABI of libblr.so and are replayed from a HIP
graph, rotating through enough weight copies that the 256 MB Infinity Cache cannot serve them.

The one JSON line printed last carries `value` = microseconds per layer-step (lower is better),
`roofline` for the dominant kernel (the gate_up streaming kernel), `cpu_baseline` (the CPU oracle's
torch port of the same step on the host cores), and `layers`: per-layer microseconds with the
fraction of HBM (M = 1, 16, 64) or fp16-MFMA (M = 2048) peak for BLAST, quantized BLAST, Monarch,
low-rank and dense.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(ROOT, "mem-efficient-blr_amd")
for _p in (ROOT, PKG):
    if _p not in sys.path:
        sys.path.insert(0, _p)

HBM_PEAK = 8.0e12            # B/s, MI355X HBM3E
MFMA_PEAK = 2.5e15           # FLOP/s, dense fp16/bf16
LAYERS = {"qkvo": (4096, 4096, 512), "gate_up": (4096, 22016, 1024), "down": (11008, 4096, 1024)}
B = 16

# HBM bytes per launch of the dominant kernel come from the committed counter summary (rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE,
# scaled by the same counters over a copy of known size): the line "traffic_bytes_per_launch: N" of this file.  No file, no figure.
DOMINANT_KERNEL = "decode3_kernel<f16,1,16>"
DOMINANT_PROFILE = os.path.join("profiles", "decode3_kernel_blast_llama7b_gate_up_m1.txt")
# the three launches of the BLAST gate_up call at M = 2048 (GEMM x V, mix, GEMM Z U): line "blast_traffic_bytes_per_call: N"
PREFILL_PROFILE = os.path.join("profiles", "gemm_mix_kernels_blast_llama7b_prefill_m2048.txt")


def traffic_from_profile(path, key="traffic_bytes_per_launch"):
    try:
        for line in open(os.path.join(ROOT, path)):
            if line.startswith(key + ":"):
                return float(line.split(":", 1)[1].split()[0])
    except OSError:
        pass
    return None


def blast_bytes_flops(n, i, r, o, b=B, elt=2):
    return (n * i + b * b * r + i * r + r * o + n * o) * elt, n * r * (i + o + b * b) * 2


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-table", action="store_true", help="skip the per-layer table")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--pmc", choices=["dominant", "calib", "prefill", "decode16"], default=None,
                    help="profiling helper: launch only the dominant decode kernel (dominant), only copy/probe kernels of "
                         "known size (calib), or only the BLAST gate_up prefill kernels at M=2048 (prefill), eagerly, and "
                         "print nothing but a note")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path (run with --gpus 1)", file=sys.stderr)
        sys.exit(2)

    import torch
    from triton_funcs import _lib as L
    lib = L.lib()
    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    torch.manual_seed(0)
    f16 = torch.float16

    def randn(*shape, std=1.0, dtype=f16):
        return (torch.randn(*shape, device=dev, dtype=torch.float32) * std).to(dtype)

    # ---- launch builders: each returns (callable(stream_ptr), keepalive) --------------------------
    def ws_for(nbytes):
        return torch.zeros(max(int(nbytes), 256), dtype=torch.uint8, device=dev)

    def mk_blast(M, in_f, out_f, r, u_layout, s_layout, algo=0):
        p, q = in_f // B, out_f // B
        x = randn(M, in_f)
        U = randn(B, r, q, std=r ** -0.5) if u_layout == L.U_RQ else randn(B, q, r, std=r ** -0.5)
        V = randn(B, p, r, std=r ** -0.5)
        S = randn(B, B, r) if s_layout == L.S_JIR else randn(r, B, B)
        out = torch.empty(M, out_f, device=dev, dtype=f16)
        ws = ws_for(lib.blr_blast_workspace_bytes(M, in_f, out_f, B, r, L.F16, algo))

        def go(st):
            L.check(lib.blr_blast_fwd(x.data_ptr(), in_f, U.data_ptr(), V.data_ptr(), S.data_ptr(), out.data_ptr(), out_f,
                                      None, None, M, in_f, out_f, B, r, L.F16, u_layout, s_layout, algo,
                                      ws.data_ptr(), ws.numel(), st), "blr_blast_fwd")
        return go, (x, U, V, S, out, ws)

    def mk_blast_q(M, in_f, out_f, r, bits):
        p, q = in_f // B, out_f // B
        x = randn(M, in_f)
        U = randn(B, r, q, std=r ** -0.5, dtype=torch.float32)          # (k, n)-ordered like V
        V = randn(B, p, r, std=r ** -0.5, dtype=torch.float32)
        S = randn(r, B, B)
        uc = torch.empty((B, r, q * bits // 8), dtype=torch.uint8, device=dev); us = torch.empty((B, q), dtype=f16, device=dev)
        vc = torch.empty((B, p, r * bits // 8), dtype=torch.uint8, device=dev); vs = torch.empty((B, r), dtype=f16, device=dev)
        L.check(lib.blr_quantize_sym(U.data_ptr(), L.F32, B, r, q, bits, uc.data_ptr(), us.data_ptr(), None), "quantize U")
        L.check(lib.blr_quantize_sym(V.data_ptr(), L.F32, B, p, r, bits, vc.data_ptr(), vs.data_ptr(), None), "quantize V")
        torch.cuda.synchronize()
        del U, V
        out = torch.empty(M, out_f, device=dev, dtype=f16)
        ws = ws_for(lib.blr_blast_q_workspace_bytes(M, in_f, out_f, B, r, bits))

        def go(st):
            L.check(lib.blr_blast_q_fwd(x.data_ptr(), in_f, uc.data_ptr(), us.data_ptr(), vc.data_ptr(), vs.data_ptr(), S.data_ptr(),
                                        out.data_ptr(), out_f, M, in_f, out_f, B, r, L.F16, bits, 0, ws.data_ptr(), ws.numel(), st),
                    "blr_blast_q_fwd")
        return go, (x, uc, us, vc, vs, S, out, ws)

    def mk_dense(M, in_f, out_f):
        x = randn(M, in_f); W = randn(in_f, out_f, std=in_f ** -0.5)
        out = torch.empty(M, out_f, device=dev, dtype=f16)
        ws = ws_for(lib.blr_dense_workspace_bytes(M, in_f, out_f, L.F16, 0))

        def go(st):
            L.check(lib.blr_dense_fwd(x.data_ptr(), in_f, W.data_ptr(), out.data_ptr(), out_f, M, in_f, out_f, L.F16, 0,
                                      ws.data_ptr(), ws.numel(), st), "blr_dense_fwd")
        return go, (x, W, out, ws)

    def mk_low_rank(M, in_f, out_f, r=1024):
        x = randn(M, in_f); A = randn(in_f, r, std=r ** -0.5); Bm = randn(r, out_f, std=r ** -0.5)
        out = torch.empty(M, out_f, device=dev, dtype=f16)
        ws = ws_for(lib.blr_low_rank_workspace_bytes(M, in_f, out_f, r, L.F16, 0))

        def go(st):
            L.check(lib.blr_low_rank_fwd(x.data_ptr(), in_f, A.data_ptr(), Bm.data_ptr(), out.data_ptr(), out_f, None,
                                         M, in_f, out_f, r, L.F16, 0, ws.data_ptr(), ws.numel(), st), "blr_low_rank_fwd")
        return go, (x, A, Bm, out, ws)

    def mk_monarch(M, in_f, out_f, b=4, rank=1024):
        x = randn(M, in_f)
        w1 = randn(b, in_f // b, rank, std=(in_f // b) ** -0.5); w2 = randn(b, rank, out_f // b, std=rank ** -0.5)
        out = torch.empty(M, out_f, device=dev, dtype=f16)
        ws = ws_for(lib.blr_monarch_workspace_bytes(M, in_f, out_f, b, rank, L.F16, 0))

        def go(st):
            L.check(lib.blr_monarch_fwd(x.data_ptr(), in_f, w1.data_ptr(), w2.data_ptr(), out.data_ptr(), out_f, None,
                                        M, in_f, out_f, b, rank, L.F16, L.W2_RS, L.OUT_INTERLEAVED, 0,
                                        ws.data_ptr(), ws.numel(), st), "blr_monarch_fwd")
        return go, (x, w1, w2, out, ws)

    # ---- timing: HIP events on the launch stream around a graph that replays `launches` -----------
    def graph_of(launches):
        for go in launches:                       # eager once: populates one-time caches, checks errors
            go(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            st = torch.cuda.current_stream().cuda_stream
            for go in launches:
                go(st)
        return g

    def time_graph(g, n_launches, reps=5, warm_ms=60.0):
        # replays for at least warm_ms before the timed ones: from idle the card needs some tens of milliseconds of work to settle
        # on its clocks, and a matrix-bound call timed right after a pause read up to 10 % slower than in steady state (the dense
        # 4096 -> 4096 GEMM at 2048 rows: 75.6 us as the first thing measured, 67.5 after 60 ms of replays); decode rows do not move
        g.replay(); torch.cuda.synchronize()
        t_w = time.perf_counter()
        while (time.perf_counter() - t_w) * 1e3 < warm_ms:
            g.replay(); torch.cuda.synchronize()
        best = []
        for _ in range(reps):
            e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
            e0.record(); g.replay(); e1.record(); torch.cuda.synchronize()
            best.append(e0.elapsed_time(e1) * 1e3 / n_launches)      # us per launch
        best.sort()
        return best[len(best) // 2]

    def copies_for(weight_bytes, lo=2, target=600e6, hi=80):
        # enough copies that one pass over them is more than twice the 256 MB Infinity Cache (a ring only just larger than the
        # cache still gets hits: the gate_up kernel measured 14.6 us over 270 MB of copies and 15.2 - 15.4 us over 650 MB)
        return int(max(lo, min(hi, -(-target // max(weight_bytes, 1)))))

    def measure(mk, weight_bytes, launches_per_graph=48):
        n = copies_for(weight_bytes)
        built = [mk() for _ in range(n)]
        launches = [built[i % n][0] for i in range(max(launches_per_graph, n))]
        g = graph_of(launches)
        us = time_graph(g, len(launches))
        del g, built
        torch.cuda.empty_cache()
        return us

    # ---- counter-collection helper (run under rocprofv3 --pmc) ---------------------------------------
    if args.pmc == "calib":
        nbytes = 256 << 20
        src = torch.empty(nbytes, dtype=torch.uint8, device=dev).random_(0, 255)
        dst = torch.empty_like(src)
        words = torch.zeros(lib.blr_probe_dst_words(), dtype=torch.int32, device=dev)
        for _ in range(4):
            dst.copy_(src)                                                   # reads 256 MiB, writes 256 MiB
            L.check(lib.blr_stream_probe(src.data_ptr(), nbytes, words.data_ptr(), torch.cuda.current_stream().cuda_stream), "probe")
        torch.cuda.synchronize()
        print(json.dumps({"pmc": "calib", "copy_bytes_read": nbytes, "copy_bytes_written": nbytes, "probe_bytes_read": nbytes}))
        return
    if args.pmc == "prefill":
        pf = [mk_blast(2048, *LAYERS["gate_up"][:2], LAYERS["gate_up"][2], L.U_RQ, L.S_JIR) for _ in range(4)]
        st = torch.cuda.current_stream().cuda_stream
        for i in range(24):
            pf[i % 4][0](st)
        dn = [mk_dense(2048, *LAYERS["gate_up"][:2]) for _ in range(2)]
        for i in range(8):
            dn[i % 2][0](st)
        torch.cuda.synchronize()
        print(json.dumps({"pmc": "prefill", "launches": 24, "flops": blast_bytes_flops(2048, 4096, 1024, 22016)[1],
                          "dense_launches": 8, "dense_flops": 2.0 * 2048 * 4096 * 22016}))
        return
    if args.pmc == "decode16":
        # the other decode kernels at full shape, eager launches over rotating weight copies: dense gate_up at M = 1 and 16
        # (slab kernel + sum of the k-slices), BLAST gate_up at M = 16 (matrix-core decode kernel), int8 BLAST gate_up at M = 16
        st = torch.cuda.current_stream().cuda_stream
        i_f, o_f, r = LAYERS["gate_up"]
        for mk in (lambda: mk_dense(1, i_f, o_f), lambda: mk_dense(16, i_f, o_f),
                   lambda: mk_blast(16, i_f, o_f, r, L.U_RQ, L.S_JIR), lambda: mk_blast_q(16, i_f, o_f, r, 8)):
            built = [mk() for _ in range(4)]
            for i in range(12):
                built[i % 4][0](st)
            torch.cuda.synchronize()
            del built
            torch.cuda.empty_cache()
        print(json.dumps({"pmc": "decode16", "launches_each": 12, "dense_bytes_m1": 2 * (i_f + i_f * o_f + o_f),
                          "dense_bytes_m16": 2 * (16 * i_f + i_f * o_f + 16 * o_f),
                          "blast_bytes_m16": blast_bytes_flops(16, i_f, r, o_f)[0]}))
        return
    if args.pmc == "dominant":
        gu = [mk_blast(1, *LAYERS["gate_up"][:2], LAYERS["gate_up"][2], L.U_RQ, L.S_JIR) for _ in range(12)]
        st = torch.cuda.current_stream().cuda_stream
        for i in range(36):
            gu[i % 12][0](st)
        torch.cuda.synchronize()
        print(json.dumps({"pmc": "dominant", "launches": 36, "algorithmic_bytes": blast_bytes_flops(1, 4096, 1024, 22016)[0]}))
        return

    # ---- headline: one decoder layer's six BLAST linears at M = 1 ---------------------------------
    M = 1
    step_bytes = 4 * blast_bytes_flops(M, *LAYERS["qkvo"][:1], LAYERS["qkvo"][2], LAYERS["qkvo"][1])[0] \
        + blast_bytes_flops(M, LAYERS["gate_up"][0], LAYERS["gate_up"][2], LAYERS["gate_up"][1])[0] \
        + blast_bytes_flops(M, LAYERS["down"][0], LAYERS["down"][2], LAYERS["down"][1])[0]
    ncopies = copies_for(step_bytes, lo=3)
    sets = []
    for _ in range(ncopies):
        one = [mk_blast(M, *LAYERS["qkvo"][:2], LAYERS["qkvo"][2], L.U_RQ, L.S_JIR) for _ in range(4)]
        one.append(mk_blast(M, *LAYERS["gate_up"][:2], LAYERS["gate_up"][2], L.U_RQ, L.S_JIR))
        one.append(mk_blast(M, *LAYERS["down"][:2], LAYERS["down"][2], L.U_RQ, L.S_JIR))
        sets.append(one)
    # One graph per weight copy (one step each) and one graph that runs a step on every copy in turn: the timed region
    # replays the long graph steps // ncopies times and finishes the remainder with single-step graphs - exactly `steps`
    # steps, with the host out of the way between most of them.
    step_graphs = [graph_of([go for go, _ in one]) for one in sets]
    round_graph = graph_of([go for one in sets for go, _ in one])
    for s in range(args.warmup):
        step_graphs[s % ncopies].replay()
    round_graph.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps // ncopies):
        round_graph.replay()
    for s in range(args.steps % ncopies):
        step_graphs[s].replay()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    ms_per_step = (t1 - t0) * 1e3 / max(args.steps, 1)

    # dominant kernel: gate_up streaming kernel, event-timed on its launch stream over the same copies
    gu_bytes_one = blast_bytes_flops(M, LAYERS["gate_up"][0], LAYERS["gate_up"][2], LAYERS["gate_up"][1])[0]
    gu_built = [one[4] for one in sets]
    while len(gu_built) < copies_for(gu_bytes_one):             # the step's copies of this layer alone are barely past the cache
        gu_built.append(mk_blast(M, *LAYERS["gate_up"][:2], LAYERS["gate_up"][2], L.U_RQ, L.S_JIR))
    gu = [one[0] for one in gu_built]
    n_l = max(48, len(gu))
    g_gu = graph_of([gu[i % len(gu)] for i in range(n_l)])
    gu_us = time_graph(g_gu, n_l)
    gu_bytes, gu_flops = blast_bytes_flops(M, LAYERS["gate_up"][0], LAYERS["gate_up"][2], LAYERS["gate_up"][1])
    achieved = gu_bytes / (gu_us * 1e-6) / 1e9
    roofline = {"bound": "hbm", "kernel": DOMINANT_KERNEL + " (BLAST gate_up 4096->22016 r=1024 b=16, M=1: one launch, all of V, S and U)",
                "achieved": round(achieved, 1), "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": round(achieved * 1e9 / HBM_PEAK, 4),
                "us_per_launch": round(gu_us, 3), "algorithmic_bytes": gu_bytes, "traffic": traffic_from_profile(DOMINANT_PROFILE),
                "traffic_source": DOMINANT_PROFILE}
    del g_gu, step_graphs, round_graph, sets, gu_built, gu
    torch.cuda.empty_cache()

    # second roofline object: the dominant kernel at M = 2048, the GEMM (one launch = the dense gate_up layer), MFMA bound
    i_f, o_f, _ = LAYERS["gate_up"]
    # (48 launches per replay over four copies, as in the layer table: the card takes some milliseconds of matrix work to settle
    # on the clock its power limit allows, and a replay of a dozen launches read 6 % slower than the table's row of the same kernel)
    dn = [mk_dense(2048, i_f, o_f) for _ in range(4)]
    g_dn = graph_of([dn[i % 4][0] for i in range(48)])
    dn_us = time_graph(g_dn, 48)
    dn_flops = 2.0 * 2048 * i_f * o_f
    roofline_prefill = {"bound": "mfma", "kernel": "gemm_wide_kernel<f16, 256x352, 8 waves, stages of 64 k> (dense gate_up 4096->22016, M=2048: one launch)",
                        "achieved": round(dn_flops / (dn_us * 1e-6) / 1e12, 1), "peak": MFMA_PEAK / 1e12, "unit": "TFLOP/s",
                        "frac": round(dn_flops / (dn_us * 1e-6) / MFMA_PEAK, 4), "us_per_launch": round(dn_us, 2),
                        "algorithmic_flops": dn_flops, "algorithmic_bytes": 2 * (2048 * i_f + i_f * o_f + 2048 * o_f),
                        "traffic": traffic_from_profile(PREFILL_PROFILE, "dense_traffic_bytes_per_launch"), "traffic_source": PREFILL_PROFILE}
    del g_dn, dn
    torch.cuda.empty_cache()

    # third roofline object: what the metric names for M = 2048 - the BLAST gate_up layer itself (three launches: GEMM x V, the
    # rank-space mix, GEMM Z U), its algorithmic flops over the event time of the whole call; traffic = HBM bytes of the three
    # launches from the committed counter summary, against the algorithmic bytes of the call
    i_f, o_f, r_gu = LAYERS["gate_up"]
    bp = [mk_blast(2048, i_f, o_f, r_gu, L.U_RQ, L.S_JIR) for _ in range(4)]
    g_bp = graph_of([bp[i % 4][0] for i in range(48)])
    bp_us = time_graph(g_bp, 48)
    bp_bytes, bp_flops = blast_bytes_flops(2048, i_f, r_gu, o_f)
    roofline_blast_prefill = {"bound": "mfma", "kernel": "BLAST gate_up 4096->22016 r=1024 b=16, M=2048: gemm_wide_kernel (x V), blast_mixm_kernel (the mix), gemm_wide_kernel (Z U)",
                              "achieved": round(bp_flops / (bp_us * 1e-6) / 1e12, 1), "peak": MFMA_PEAK / 1e12, "unit": "TFLOP/s",
                              "frac": round(bp_flops / (bp_us * 1e-6) / MFMA_PEAK, 4), "us_per_call": round(bp_us, 2),
                              "algorithmic_flops": bp_flops, "algorithmic_bytes": bp_bytes,
                              "traffic": traffic_from_profile(PREFILL_PROFILE, "blast_traffic_bytes_per_call"), "traffic_source": PREFILL_PROFILE}
    del g_bp, bp
    torch.cuda.empty_cache()

    # what the matrix cores sustain on this card with nothing in their way (blr_mfma_probe: operands in registers, about a
    # quarter of a second per variant): the practical ceiling next to the published peak that `frac` is quoted against
    sink = torch.zeros(16, dtype=torch.int32, device=dev)
    mfma_sustained = {}
    for key, rnd, reads in (("ones", 0, 0), ("random", 1, 0), ("random_with_lds_fragment_reads", 1, 6)):
        iters = 600000
        st = torch.cuda.current_stream().cuda_stream
        L.check(lib.blr_mfma_probe(2000, rnd, reads, sink.data_ptr(), st), "mfma_probe")
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        L.check(lib.blr_mfma_probe(iters, rnd, reads, sink.data_ptr(), st), "mfma_probe")
        e1.record(); torch.cuda.synchronize()
        tf = lib.blr_mfma_probe_flops(iters) / (e0.elapsed_time(e1) * 1e-3) / 1e12
        mfma_sustained[key] = {"TFLOP/s": round(tf, 1), "frac_of_peak": round(tf * 1e12 / MFMA_PEAK, 3)}
    roofline_prefill["sustained_mfma_probe"] = mfma_sustained

    # ---- per-layer table ----------------------------------------------------------------------------
    table = {}
    if not args.no_table:
        def row(name, us, by, fl, m):
            hbm = by / (us * 1e-6) / HBM_PEAK
            mf = fl / (us * 1e-6) / MFMA_PEAK
            table[name] = {"us": round(us, 2), "pct_hbm": round(100 * hbm, 1), "pct_mfma": round(100 * mf, 1),
                           "bound": "hbm" if m <= 128 else "mfma"}
        for lname, (i_f, o_f, r) in LAYERS.items():
            for m in (1, 16, 64, 2048):
                by, fl = blast_bytes_flops(m, i_f, r, o_f)
                wbytes = 2 * r * (i_f + o_f + B * B)
                row(f"blast_full/{lname}/M{m}", measure(lambda: mk_blast(m, i_f, o_f, r, L.U_RQ, L.S_JIR), wbytes), by, fl, m)
                row(f"blast_bmm/{lname}/M{m}", measure(lambda: mk_blast(m, i_f, o_f, r, L.U_QR, L.S_RIJ), wbytes), by, fl, m)
                dby, dfl = 2 * (m * i_f + i_f * o_f + m * o_f), 2 * m * i_f * o_f
                row(f"dense/{lname}/M{m}", measure(lambda: mk_dense(m, i_f, o_f), 2 * i_f * o_f), dby, dfl, m)
                lby, lfl = 2 * (1024 * (i_f + o_f) + m * (i_f + o_f)), 2 * m * 1024 * (i_f + o_f)
                row(f"low_rank/{lname}/M{m}", measure(lambda: mk_low_rank(m, i_f, o_f), 2 * 1024 * (i_f + o_f)), lby, lfl, m)
                row(f"monarch_b4/{lname}/M{m}", measure(lambda: mk_monarch(m, i_f, o_f), 2 * 1024 * (i_f + o_f)), lby, lfl, m)
        for lname in ("gate_up", "down"):
            i_f, o_f, r = LAYERS[lname]
            for bits in (8, 4):
                for m in (1, 4, 16, 64):
                    by = r * (i_f + o_f) * bits // 8 + 2 * B * B * r + 2 * (o_f + B * r) + 2 * m * (i_f + o_f)
                    fl = 2 * m * r * (i_f + o_f + B * B)
                    row(f"blast_int{bits}/{lname}/M{m}", measure(lambda: mk_blast_q(m, i_f, o_f, r, bits), by), by, fl, m)

    # ---- DiT-XL/2 end to end: 16 latents [4,32,32], every qkv/proj/fc1/fc2 linear replaced ----
    dit = None
    if not args.no_table:
        try:
            import yaml
            from models import dit_xl
            ncfg = yaml.safe_load(open(os.path.join(PKG, "configs", "networks", "dit_xl.yaml")))
            dit = {"batch": 16, "tokens_per_image": 256, "dtype": "f16"}
            import contextlib
            with contextlib.redirect_stdout(sys.stderr):          # the harness reports what it replaced; stdout carries the one JSON line only
                # The methods are within a few per cent of each other and the card drifts by as much between one measurement and
                # the next: every method is measured the same number of times, in interleaved order; every pass is reported
                # and the figure of a method is the median of its passes.  nn_linear: stock nn.Linear (hipBLASLt), for scale.
                passes = {m: [] for m in ("blast", "dense", "low_rank", "nn_linear")}
                for _ in range(3):
                    for method in passes:
                        if method == "nn_linear":
                            ms = dit_xl.benchmark(None, None, None, 256, 10, dev, f16, batch=16)
                        else:
                            lc = {k: {"rank": v.get("rank"), "b": v.get("b"), "func": v["triton"]["func"]} for k, v in ncfg[method].items()}
                            ms = dit_xl.benchmark(method, "triton", lc, 256, 10, dev, f16, batch=16)
                        passes[method].append(round(ms, 3))
                        torch.cuda.empty_cache()
                for method, lst in passes.items():
                    ms = sorted(lst)[len(lst) // 2]
                    dit[f"{method}_img_per_s"] = round(16 / (ms * 1e-3), 1)
                    dit[f"{method}_ms"] = ms
                dit["passes_ms"] = passes
                dit["reported"] = "median of 3 interleaved passes per method"
        except Exception as e:                       # the headline must still be printed
            dit = {"error": str(e)}

    # ---- CPU baseline: the oracle's torch port of the same step, fp32, all host cores -----------------
    cpu = None
    if not args.no_cpu:
        from oracle import torch_port as T
        torch.set_num_threads(os.cpu_count() or 1)
        cores = torch.get_num_threads()
        g = torch.Generator().manual_seed(0)
        ops = []
        for lname, cnt in (("qkvo", 4), ("gate_up", 1), ("down", 1)):
            i_f, o_f, r = LAYERS[lname]
            for _ in range(cnt):
                ops.append((torch.randn(1, 1, i_f, generator=g), torch.randn(B, o_f // B, r, generator=g) * r ** -0.5,
                            torch.randn(B, r, i_f // B, generator=g) * r ** -0.5, torch.randn(B, B, r, generator=g)))
        for _ in range(3):
            for x, U, Vt, S in ops:
                T.blast(x, U, Vt, S)
        reps, t_used, times = 0, 0.0, []
        while t_used < 12.0 and reps < 100000:
            c0 = time.perf_counter()
            for x, U, Vt, S in ops:
                T.blast(x, U, Vt, S)
            dt = time.perf_counter() - c0
            times.append(dt); t_used += dt; reps += 1
        times.sort()
        cpu = {"value": round(times[len(times) // 2] * 1e6, 1), "unit": "us/layer-step", "cores": cores, "kind": "port",
               "sample": f"{reps} repetitions (~{t_used:.0f} s) of the full M=1 step (6 BLAST linears) in fp32 with oracle/torch_port.blast"}

    # ---- the reference's own CPU-runnable case (GPT-2-small c_fc, fp32) on the host and on the GPU ---------
    cpu1 = None
    if not args.no_cpu:
        from oracle import torch_port as T
        g = torch.Generator().manual_seed(0)
        b1, r1, i1, o1 = 4, 128, 768, 3072
        x1 = torch.randn(1, 128, i1, generator=g)
        U1 = torch.randn(b1, o1 // b1, r1, generator=g) * r1 ** -0.5
        V1 = torch.randn(b1, r1, i1 // b1, generator=g) * r1 ** -0.5
        S1 = torch.randn(b1, b1, r1, generator=g)
        for _ in range(5):
            T.blast(x1, U1, V1, S1)
        reps, t_used, times = 0, 0.0, []
        while t_used < 5.0 and reps < 20000:
            c0 = time.perf_counter()
            T.blast(x1, U1, V1, S1)
            dt = time.perf_counter() - c0
            times.append(dt); t_used += dt; reps += 1
        times.sort()
        from triton_funcs import blast_kernels as K
        xg = x1.to(dev)
        Ug, Vg, Sg = (U1.permute(0, 2, 1).contiguous().to(dev), V1.permute(0, 2, 1).contiguous().to(dev), S1.permute(1, 0, 2).contiguous().to(dev))
        for _ in range(3):
            K.triton_blast_full_fp32(xg, Ug, Vg, Sg)
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(50):
            K.triton_blast_full_fp32(xg, Ug, Vg, Sg)
        e1.record(); torch.cuda.synchronize()
        cpu1 = {"value": round(times[len(times) // 2] * 1e6, 1), "unit": "us/forward", "cores": torch.get_num_threads(), "kind": "port",
                "sample": f"{reps} repetitions (~{t_used:.0f} s) of BLAST c_fc x[1,128,768] -> 3072, b=4, r=128, fp32, oracle/torch_port.blast",
                "gpu_us": round(e0.elapsed_time(e1) * 1e3 / 50, 1), "gpu_path": "triton_blast_full_fp32 (eager calls, intermediates returned)"}

    result = {
        "metric": "Llama-7B layer us + %HBM/%MFMA roofline at M=1 and 2048; DiT-XL/2 img/s",
        "value": round(ms_per_step * 1e3, 2), "unit": "us/layer-step (6 BLAST linears, M=1)",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "f16", "data": "synthetic",
        "config": {"workload": "BASELINE configs[2]: BLAST Llama-7B linears fp16 b=16 (4x qkvo r=512, gate_up r=1024, down r=1024), M=1 decode, "
                               "triton_blast_full_fp16 layouts, HIP-graph replay, weight copies rotated past the Infinity Cache",
                   "weight_copies": ncopies, "algorithmic_bytes_per_step": step_bytes,
                   "pct_hbm_step": round(100 * step_bytes / (ms_per_step * 1e-3) / HBM_PEAK, 1)},
        "roofline": roofline, "roofline_prefill": roofline_prefill, "roofline_blast_prefill": roofline_blast_prefill, "cpu_baseline": cpu, "cpu_baseline_config1": cpu1,
        "layers": table, "dit_xl": dit,
    }
    print(json.dumps(result))


if __name__ == "__main__":
    main()
