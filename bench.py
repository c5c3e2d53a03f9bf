"""Headline benchmark: fused residual add + RMSNorm + MXFP8 at 16384 x 7168 on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--ops]

A step is one launch of ``k3h_residual_rms_mxfp8`` over the whole [16384, 7168]
chunk with inputs resident in HBM.  Timing: W untimed
warm-up steps (continued in batches of 100 until --warm-s seconds of launches
have run, so the clocks are at steady state), then K steps between two HIP
events on the launch stream, with a device synchronisation on both sides.  ``value`` is the effective HBM bandwidth
(algorithmic bytes per step / mean step time).  Algorithmic bytes: x and the
residual read once, gamma once, residual_out + e4m3 payload + E8M0 scales
written once = 825,767,936 B.

``roofline`` gives the achieved rate against MI355X's 8 TB/s HBM peak and, when
``profiles/traffic.json`` holds rocprofv3 FETCH_SIZE/WRITE_SIZE counts for the
kernel, the measured HBM bytes per launch (``traffic_source`` says so: they come
from those profiling runs, not from this one).  ``flushed`` times the same launch
one at a time with a 512 MB clean-read cache flush before each (median, p10,
p90), the per-op protocol of the --ops table, beside the back-to-back value.  ``cpu_baseline`` times the C oracle
(OpenMP over the host cores) on the same inputs -- the checker run as a
reported baseline, never the measured path.  One JSON line goes to stdout;
progress goes to stderr.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "kern-k3_amd"))

METRIC = "effective HBM GB/s (% of peak) for residual+RMSNorm+MXFP8 at 16384x7168"
H = 7168
T = 16384
PEAK_GBS = 8000.0
# MI355X dense MFMA peak for e4m3 operands (TFLOP/s); e4m3 x e2m1 issues at the
# e4m3 rate (4.95 PFLOP/s measured register-to-register).
PEAK_MX_TFLOPS = 5000.0


def algo_bytes(rows: int) -> int:
    n = rows * H
    return 2 * n * 2 + H * 2 + n * 2 + n + n // 32


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


DATA = ("synthetic: k3h_synth_normal, one xoshiro256** stream per tensor seeded "
        "24301 ^ fnv1a64('<config>/<tensor>'), Box-Muller normals; x with 0.1% outliers x50")


def syn(name: str, shape, mean: float = 0.0, std: float = 1.0, outlier_p: float = 0.0,
        dtype=None):
    """A BASELINE-config input from the seeded host generator, copied to the GPU."""
    import torch
    import k3h
    return k3h.synth_normal(name, shape, mean, std, outlier_p, 50.0,
                            dtype or torch.bfloat16).cuda()


def make_inputs(rows: int):
    """Config 2: x ~N(0,1) with 0.1% outliers x50, residual ~N(0,1), gamma ~N(1,0.1)."""
    return (syn("2/x", (rows, H), outlier_p=0.001), syn("2/residual", (rows, H)),
            syn("2/gamma", (H,), 1.0, 0.1))


def native_oracle() -> str:
    """Builds the C oracle with -march=native for the host this runs on, into a
    directory of its own, and points oracle.py at it (K3_ORACLE_LIB) for the CPU
    baseline; the in-tree portable build (x86-64-v3) stays the tests' checker.
    Returns a note for the JSON line."""
    import subprocess
    import tempfile
    path = os.path.join(tempfile.mkdtemp(prefix="k3oracle_"), "libk3oracle_native.so")
    r = subprocess.run(["make", "-s", "-C", os.path.join(REPO, "oracle"), "ARCH=native", f"LIB={path}"],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode == 0 and os.path.exists(path):
        os.environ["K3_ORACLE_LIB"] = path
        return "gcc -O3 -march=native -fopenmp build of oracle/ on this host"
    log(f"native oracle build failed, timing the portable build: {r.stdout[-300:]}")
    return "portable (x86-64-v3) build of oracle/ (the native build failed on this host)"


def cpu_baseline(x, res, gamma, gpu_out, budget_s: float = 10.0, build_note: str = "") -> dict:
    """Times the C oracle (the checker) on the same inputs: inputs copied into
    buffers that the OpenMP threads touch first, outputs allocated once outside
    the timed calls (first touched by the threads in the warm-up call), one
    warm-up, then the median of 5 calls (fewer if they exceed ~budget_s)."""
    import numpy as np
    import torch
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import oracle as O

    def h(t):
        return t.cpu().view(torch.int16).numpy().view(np.uint16)

    xh, rh, gh = O.par_copy(h(x)), O.par_copy(h(res)), O.par_copy(h(gamma))
    rows = xh.shape[0]
    outs = (np.empty((rows, H), np.uint16), np.empty((rows, H), np.uint8),
            np.empty((rows, H // 32), np.uint8), None)
    O.residual_rms_mxfp8(xh, rh, gh, rows, 1e-6, want_normed=False, out=outs)  # warm-up
    times = []
    t_start = time.perf_counter()
    while len(times) < 5 and (not times or time.perf_counter() - t_start < budget_s):
        t0 = time.perf_counter()
        O.residual_rms_mxfp8(xh, rh, gh, rows, 1e-6, want_normed=False, out=outs)
        times.append(time.perf_counter() - t0)
    med = sorted(times)[len(times) // 2]
    ro, q, sf = (t.cpu().numpy() if t.dtype != torch.bfloat16 else h(t) for t in gpu_out)
    match = bool((outs[0] == ro).all() and (outs[1] == q).all() and (outs[2] == sf).all())
    return {
        "value": round(algo_bytes(rows) / med / 1e9, 2),
        "unit": "GB/s",
        "cores": O.num_threads(),
        "kind": "port",
        "sample": f"full {rows}x{H} workload: 1 warm-up, median of {len(times)} timed oracle passes "
                  f"({med * 1e3:.0f} ms each), inputs first touched by the threads, outputs "
                  f"allocated outside the timed calls; {O.num_threads()} OpenMP threads "
                  f"(omp_get_max_threads) of {os.cpu_count()} hardware threads; {build_note}; "
                  f"bit-exact vs GPU: {match}",
    }


def copy_ceiling(ctx, rows: int, reps: int) -> float:
    """Rate of the plain 16-byte streaming copy over one [rows, 7168] bf16 tensor."""
    import torch
    src = torch.empty(rows * H, dtype=torch.bfloat16, device="cuda").fill_(1.0)
    dst = torch.empty_like(src)
    s = torch.cuda.current_stream()
    for _ in range(3):
        ctx.stream_copy(src, dst, stream=s)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(s)
    for _ in range(reps):
        ctx.stream_copy(src, dst, stream=s)
    e1.record(s)
    torch.cuda.synchronize()
    us = e0.elapsed_time(e1) * 1e3 / reps
    gbs = 2 * src.numel() * 2 / (us * 1e-6) / 1e9
    log(f"copy ceiling: {us:.1f} us per {2 * src.numel() * 2 / 1e6:.0f} MB -> {gbs:.0f} GB/s")
    del src, dst
    return gbs


def cpu_timer(budget_s: float):
    """Times one oracle call (the checker, run as a reported baseline): one untimed
    warm-up call, then up to 5 timed calls within `budget_s`; returns the median
    in s.  These per-op calls allocate their outputs inside the call."""
    def run(fn):
        t0 = time.perf_counter()
        fn()
        first = time.perf_counter() - t0
        times = []
        while len(times) < 5 and (not times or sum(times) + first < budget_s):
            t0 = time.perf_counter()
            fn()
            times.append(time.perf_counter() - t0)
        return sorted(times)[len(times) // 2]
    return run


def bench_ops(ctx, reps: int, out_path: str | None, cpu_budget: float = 0.0, graph: bool = False) -> list:
    """Runs _bench_ops on a stream of its own (a HIP graph is captured from a
    non-default stream); see _bench_ops."""
    import torch
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        return _bench_ops(ctx, reps, out_path, cpu_budget, graph)


def _bench_ops(ctx, reps: int, out_path: str | None, cpu_budget: float = 0.0, graph: bool = False) -> list:
    """Every op at its BASELINE config shape: 5 warm-up launches, then `reps`
    launches each between two HIP events on the launch stream, with the caches
    flushed before each launch (outside the events); median, p10, p90.  Two
    flushes, each over all reps: "clean" reads a 512 MB buffer (the L2s and the
    256 MB MALL then hold only clean lines, so the op starts cold and owes no
    write-back), "dirty" writes a 512 MB buffer (the op then also pays for
    writing back the dirty lines its own traffic evicts).  The clean figures
    are the table's; the dirty ones are reported beside them.
    With graph, each op's time inside a HIP graph is measured too (graph_time
    below: rounds of a clean 512 MB read and the op, against the reads alone):
    the reference times its prefill as graph replays, and for the short ops
    (config 1, rms) the eager per-launch figure carries the launch.
    With cpu_budget > 0, the rows of BASELINE configs 1-5 also time the C oracle
    (OpenMP over the host cores) on host copies of the same inputs."""
    import numpy as np
    import torch
    O = None
    if cpu_budget > 0:
        sys.path.insert(0, os.path.join(REPO, "oracle"))
        import oracle as O
        cpu_run = cpu_timer(cpu_budget)
        log(f"CPU oracle column: {O.num_threads()} OpenMP threads of {os.cpu_count()} hardware threads")

    def h(t):
        """Host copy: bf16 tensors as uint16 bit patterns, others as their numpy dtype."""
        if t.dtype == torch.bfloat16:
            return np.ascontiguousarray(t.cpu().view(torch.int16).numpy().view(np.uint16))
        return np.ascontiguousarray(t.cpu().numpy())
    import ctypes
    import k3h
    s = torch.cuda.current_stream()
    flush = torch.empty(512 << 20, dtype=torch.uint8, device="cuda")
    flush_rd = torch.ones(128 << 20, dtype=torch.float32, device="cuda")
    rd_sink = torch.zeros(256, dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(24301)

    def bf(*shape, mean=0.0, std=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(torch.bfloat16)

    def timed(fn):
        for _ in range(5):
            fn()
        out = []
        for clean in (True, False):
            ts = []
            for _ in range(reps):
                if clean:
                    flush_rd.sum()
                else:
                    flush.fill_(1)
                e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                e0.record(s)
                fn()
                e1.record(s)
                e1.synchronize()
                ts.append(e0.elapsed_time(e1) * 1e3)
            ts.sort()
            pick = lambda f: ts[min(len(ts) - 1, int(f * len(ts)))]
            out += [pick(0.5), pick(0.1), pick(0.9)]
        if graph:
            out.append(graph_time(fn))
        return tuple(out)

    # in-graph time of one op: a graph of GR rounds of (clean 512 MB read, op) against
    # a graph of GR clean reads alone, each replayed `reps` times; the difference of
    # the median replay times over GR is the op's incremental time inside a graph
    # (its kernels' dispatch inside the graph included, the graph launch excluded)
    GR = 20
    rd_fn = ctx.function("k3h_probe", "k3h_probe_read_u4")
    rd_n16 = flush_rd.numel() * 4 // 16
    rd_buf = k3h.pack_args(["in buffer<u8>", "i64", "out buffer<u32>"], [flush_rd, rd_n16, rd_sink])
    rd_c = ctypes.create_string_buffer(rd_buf, len(rd_buf))
    rd_g, rd_b = (ctypes.c_uint32 * 3)(rd_n16 // 1024, 1, 1), (ctypes.c_uint32 * 3)(256, 1, 1)

    def clean_read():
        rc = ctx.L.k3h_launch(rd_fn, rd_g, rd_b, 0, s.cuda_stream, ctypes.cast(rd_c, ctypes.c_void_p), len(rd_buf))
        if rc:
            raise k3h.K3HError(rc, "k3h_probe_read_u4")

    def replay_med(body):
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr, stream=s):
            for _ in range(GR):
                body()
        for _ in range(2):
            gr.replay()
        ts = []
        for _ in range(max(5, reps // 2)):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(s)
            gr.replay()
            e1.record(s)
            e1.synchronize()
            ts.append(e0.elapsed_time(e1) * 1e3)
        del gr
        return sorted(ts)[len(ts) // 2]

    def graph_time(fn):
        try:
            with_op = replay_med(lambda: (clean_read(), fn()))
            base = replay_med(clean_read)
        except Exception as exc:  # an op whose launches cannot be captured
            log(f"graph capture failed: {exc}")
            return None
        return (with_op - base) / GR

    rows = []

    def add(op, kernel, shape, nbytes, t, note="", cpu=None):
        us, p10, p90, us_d = t[:4]
        gbs = nbytes / (us * 1e-6) / 1e9
        row = {"op": op, "kernel": kernel, "shape": shape, "bytes": int(nbytes),
               "launches": 5 + 2 * reps,
               "us": round(us, 2), "us_p10": round(p10, 2), "us_p90": round(p90, 2),
               "gbs": round(gbs, 1), "pct_peak": round(100 * gbs / PEAK_GBS, 1),
               "us_dirty": round(us_d, 2), "gbs_dirty": round(nbytes / (us_d * 1e-6) / 1e9, 1),
               "note": note}
        if len(t) > 6 and t[6] is not None:
            row.update({"us_graph": round(t[6], 2), "gbs_graph": round(nbytes / (t[6] * 1e-6) / 1e9, 1)})
        cpu_txt = ""
        if cpu is not None and O is not None:
            sec = cpu_run(cpu)
            row.update({"cpu_ms": round(sec * 1e3, 2), "cpu_gbs": round(nbytes / sec / 1e9, 2),
                        "cpu_threads": O.num_threads()})
            cpu_txt = f" | CPU {sec * 1e3:8.1f} ms {nbytes / sec / 1e9:6.2f} GB/s"
        rows.append(row)
        gtxt = f" | graph {row['us_graph']:8.2f} us" if "us_graph" in row else ""
        log(f"{op:42s} {us:8.2f} us (p10 {p10:7.2f}, p90 {p90:7.2f}) {gbs:7.0f} GB/s "
            f"{100 * gbs / PEAK_GBS:5.1f}% | dirty {us_d:8.2f} us{gtxt}{cpu_txt}  {note}")

    T = 16384
    # copy ceiling
    a = torch.empty(T * H, dtype=torch.bfloat16, device="cuda").fill_(1)
    b = torch.empty_like(a)
    add("stream copy (ceiling)", "k3h_stream_copy", f"{T}x{H} bf16", 4 * T * H,
        timed(lambda: ctx.stream_copy(a, b, stream=s)))
    del a, b
    # config 1: K1b nb = 0 at 1024 x 7168, eps 1e-6
    B1 = 1024
    p1, r1, g1 = syn("1/x", (B1, H)), syn("1/residual", (B1, H)), syn("1/gamma", (H,), 1.0, 0.1)
    o1, n1 = torch.empty_like(p1), torch.empty_like(p1)
    sw = torch.zeros(H, dtype=torch.float32, device="cuda")
    add("residual add + RMSNorm (cfg 1)", "kern_k3_land_add_attnres_rms", f"{B1}x{H}",
        4 * B1 * H * 2 + H * 2,
        timed(lambda: ctx.land_add_attnres_rms(p1, r1, None, sw, g1, o1, n1, 0, 0, B1, eps=1e-6, stream=s)),
        cpu=O and (lambda a=(h(p1), h(r1), h(sw), h(g1)):
                   O.land_add_attnres_rms(a[0], a[1], None, a[2], a[3], 0, 0, B1, eps=1e-6)))
    # config 2: fused, and the standalone quantisers at the same shape
    x, res, gm = make_inputs(T)
    ro = torch.empty_like(x)
    q = torch.empty((T, H), dtype=torch.uint8, device="cuda")
    sf = torch.empty((T, H // 32), dtype=torch.uint8, device="cuda")
    add("residual+RMSNorm+MXFP8 (cfg 2)", "k3h_residual_rms_mxfp8", f"{T}x{H}", algo_bytes(T),
        timed(lambda: ctx.residual_rms_mxfp8(x, res, gm, ro, q, sf, None, eps=1e-6, B=T, stream=s)),
        cpu=O and (lambda a=(h(x), h(res), h(gm)):
                   O.residual_rms_mxfp8(a[0], a[1], a[2], T, 1e-6, want_normed=False)))
    xh = h(x) if O else None
    add("MXFP8 quant alone", "kern_k3_moe_quant", f"{T}x{H}", T * H * 2 + T * H + T * H // 32,
        timed(lambda: ctx.moe_quant(x, q, sf, T, H, stream=s)), cpu=O and (lambda: O.moe_quant(xh, T, H)))
    sc = torch.empty(1, dtype=torch.float32, device="cuda")
    parts = torch.empty(2048, dtype=torch.float32, device="cuda")
    add("per-tensor fp8 pair (amax+apply)", "k3h_quant_fp8_{mark,once}", f"{T}x{H}",
        T * H * 2 + T * H, timed(lambda: ctx.quant_fp8_tensor(x, q, sc, parts, T * H, stream=s)),
        note="x counted once; one launch keeps 100.7 MB of it on the chip and reads the rest again from the MALL",
        cpu=O and (lambda: O.quant_fp8_apply(xh, T * H, O.quant_fp8_amax(xh, T * H, 2048), 2048)))
    del xh
    del ro, q, sf
    # config 3: KDA span gather + output gate (24 heads x 128)
    inner = 3072
    part = syn("3/partial", (T, 4 * inner))
    cw = syn("3/conv_w", (3, 4, inner), std=0.5).float()
    state = torch.zeros(2 * 1628160, dtype=torch.uint8, device="cuda")
    line = torch.zeros(T, dtype=torch.int32, device="cuda")
    wsm = syn("3/wsm", (T, 256), dtype=torch.float32)
    sq, sk, sv = (torch.empty((T, inner), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    beta = torch.empty(24 * T, dtype=torch.bfloat16, device="cuda")
    flow = torch.empty((T, 128), dtype=torch.bfloat16, device="cuda")
    at0 = torch.zeros(1, dtype=torch.int32, device="cuda")
    add("KDA span gather (cfg 3a)", "kern_k3_span_gather", f"T={T} 24x128",
        3 * T * inner * 2 * 2 + 3 * 4 * inner * 4 + 2 * 3 * 3 * inner * 2 + T * (24 + 128) * 4 + T * 24 * 2 + T * 128 * 2,
        timed(lambda: ctx.span_gather(part, cw, state, line, 1628160, wsm, sq, sk, sv, beta, flow, at0, T, stream=s)),
        cpu=O and (lambda a=(h(part), h(cw), np.zeros((3, 3, inner), np.uint16), h(wsm)):
                   O.span_gather(a[0], a[1], a[2], a[3], 0, T)))
    attn = syn("3/attn", (T, inner))
    gam = torch.ones(128, dtype=torch.float32, device="cuda")
    gated = torch.empty((T, inner), dtype=torch.bfloat16, device="cuda")
    add("KDA output gate (cfg 3b, eps 1e-6)", "kern_k3_kda_out_gate", f"T={T} 24x128",
        3 * T * inner * 2 + 512,
        timed(lambda: ctx.kda_out_gate(attn, part, gam, gated, at0, T, stream=s, eps=1e-6)),
        cpu=O and (lambda a=(h(attn), h(part), h(gam), np.zeros((T, inner), np.uint16)):
                   O.kda_out_gate(a[0], a[1], a[2], a[3], 0, T, eps=1e-6)))
    del part, sq, sk, sv, attn, gated, wsm
    # config 4: MLA prep (reference form, bf16 partial) and the RoPE + pack form
    mp = syn("4/partial", (T, 5184))
    gq, gk = syn("4/gamma_q", (1536,), 1.0, 0.1), syn("4/gamma_kv", (512,), 1.0, 0.1)
    slots = torch.arange(T, dtype=torch.int64, device="cuda")
    slab = torch.empty((T // 64) * 64 * 576, dtype=torch.bfloat16, device="cuda")
    qn = torch.empty((T, 1536), dtype=torch.bfloat16, device="cuda")
    mg = torch.empty((T, 3072), dtype=torch.bfloat16, device="cuda")
    add("MLA prep (cfg 4, reference form)", "k3h_mla_prep_fused", f"T={T} [T,5184] bf16",
        T * 5184 * 2 + T * (1536 + 576 + 3072) * 2 + 4096,
        timed(lambda: ctx.mla_prep(mp, gq, gk, slots, slab, 0, qn, mg, T, page_stride=64 * 576, stream=s)),
        cpu=O and (lambda a=(h(mp), h(gq), h(gk), h(slots), h(slab)):
                   O.mla_prep(a[0], a[1], a[2], a[3], a[4], 0, 64 * 576, T)))
    del mp, qn, mg
    lat, kr, qq = syn("4/latent", (T, 512)), syn("4/k_rope", (T, 64)), syn("4/q", (T, 16, 192))
    lo = torch.empty((T, 576), dtype=torch.bfloat16, device="cuda")
    qo = torch.empty_like(qq)
    add("MLA latent norm + RoPE + q pack", "k3h_mla_rope_pack", f"T={T} H=16",
        T * (512 + 64 + 16 * 192) * 2 + T * (576 + 16 * 192) * 2,
        timed(lambda: ctx.mla_rope_pack(lat, kr, qq, gk, slots, lo, qo, T, 16, stream=s)),
        cpu=O and (lambda a=(h(lat), h(kr), h(qq), h(gk), h(slots)):
                   O.mla_rope_pack(a[0], a[1], a[2], a[3], a[4], T, 16)))
    del lat, kr, qq, lo, qo, slab
    # config 5: MoE routing + EP dispatch / finalize (top-8 of 224, EP rank 0 of 4)
    Sx = syn("5/logits", (T, 224), dtype=torch.float32)
    bias = syn("5/bias", (224,), std=0.01, dtype=torch.float32)
    rs = torch.full((1,), 2.5, dtype=torch.bfloat16, device="cuda")
    idx = torch.empty((T, 8), dtype=torch.int32, device="cuda")
    wts = torch.empty((T, 8), dtype=torch.float32, device="cuda")
    add("router top-8 (cfg 5a)", "k3h_router_topk_pairs", f"[{T},224]", T * 224 * 4 + 896 + 2 * T * 8 * 4,
        timed(lambda: ctx.router_topk(Sx, bias, rs, idx, wts, T, topk=8, stream=s)),
        "latency-bound (sequential picks)",
        cpu=O and (lambda a=(h(Sx), h(bias), int(h(rs)[0])): O.router_topk(a[0], a[1], a[2], T, 8)))
    E, nblk = 56, T // 256
    cap = T * 8 + E * 128
    bc = torch.empty(nblk * E, dtype=torch.int32, device="cuda")
    bo = torch.empty_like(bc)
    cb = torch.empty(cap // 128 + 1, dtype=torch.int32, device="cuda")
    cl = torch.empty_like(cb)
    nne = torch.zeros(1, dtype=torch.int32, device="cuda")
    tp = torch.zeros(1, dtype=torch.int32, device="cuda")
    rmap = torch.zeros(cap, dtype=torch.int32, device="cuda")
    e2p = torch.empty(T * 8, dtype=torch.int32, device="cuda")

    def route():
        ctx.moe_route_count(idx, T, 0, E, bc, topk=8, stream=s)
        ctx.moe_route_tables(bc, nblk, E, 128, bo, cb, cl, nne, tp, rmap, stream=s, T=T, topk=8)
        ctx.moe_route_scatter(idx, bo, T, 0, E, rmap, e2p, topk=8, stream=s)
    t_route = timed(route)
    torch.cuda.synchronize()
    tpad = int(tp.item())
    live = int((e2p >= 0).sum().item())
    add("EP routing tables (count+tables+scatter)", "kern_k3_moe_route_{count,tables,scatter}",
        f"T={T} top-8 E=56", 2 * T * 8 * 4 + 3 * nblk * E * 4 + tpad * 4, t_route,
        "latency-bound (three launches, one single-workgroup scan)",
        cpu=O and (lambda a=h(idx): cpu_route(O, a, T, nblk, E, cap)))
    sync = torch.zeros(2, dtype=torch.int32, device="cuda")
    add("EP routing, one launch (k3h_moe_route)", "k3h_moe_route_fused", f"T={T} top-8 E=56",
        2 * T * 8 * 4 + 3 * nblk * E * 4 + tpad * 4,
        timed(lambda: ctx.moe_route(idx, T, 0, E, bc, bo, cb, cl, nne, tp, rmap, e2p, sync, topk=8,
                                    stream=s)),
        "latency-bound (one launch, one grid barrier)",
        cpu=O and (lambda a=h(idx): cpu_route(O, a, T, nblk, E, cap)))
    x8 = torch.randint(0, 256, (T, H), dtype=torch.uint8, device="cuda", generator=g)
    sf8 = torch.randint(0, 256, (T, H // 32), dtype=torch.uint8, device="cuda", generator=g)
    pq = torch.empty((tpad, H), dtype=torch.uint8, device="cuda")
    psf = torch.empty((tpad, H // 32), dtype=torch.uint8, device="cuda")
    add("MXFP8 permute (cfg 5c)", "k3h_moe_permute_mx", f"{tpad} rows x {H}", 2 * tpad * (H + H // 32),
        timed(lambda: ctx.moe_permute_mx(x8, sf8, rmap, tp, H, pq, psf, stream=s)),
        note="a token's repeated rows read from the MALL",
        cpu=O and (lambda a=(h(x8), h(sf8), h(rmap)): O.moe_permute_mx(a[0], a[1], a[2], tpad, H)))
    del pq, psf, x8, sf8
    fc2 = syn("5/fc2", (tpad, H))
    out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    add("weighted finalize (cfg 5d)", "k3h_moe_finalize_rows", f"T={T} cols={H}",
        live * H * 2 + 2 * T * 8 * 4 + T * H * 2,
        timed(lambda: ctx.moe_finalize(fc2, e2p, wts, out, T, H, topk=8, stream=s)),
        cpu=O and (lambda a=(h(fc2), h(e2p), h(wts)): O.moe_finalize(a[0], a[1], a[2], T, 8, H)))
    del fc2, out
    bench_push_land(ctx, add, timed, bf, g, s, O, h)

    def add_flop(op, kernel, shape, flops, nbytes, t, note=""):
        us, p10, p90, us_d = t[:4]
        tf = flops / (us * 1e-6) / 1e12
        rows.append({"op": op, "kernel": kernel, "shape": shape, "bytes": int(nbytes),
                     "flops": int(flops), "bound": "mfma", "launches": 5 + 2 * reps,
                     "us_dirty": round(us_d, 2),
                     "us": round(us, 2), "us_p10": round(p10, 2), "us_p90": round(p90, 2),
                     "tflops": round(tf, 1), "pct_peak": round(100 * tf / PEAK_MX_TFLOPS, 1),
                     "gbs": round(nbytes / (us * 1e-6) / 1e9, 1), "note": note})
        log(f"{op:42s} {us:8.2f} us (p10 {p10:7.2f}, p90 {p90:7.2f}) {tf:7.0f} TFLOP/s "
            f"{100 * tf / PEAK_MX_TFLOPS:5.1f}% of MFMA  {note}")

    bench_gemm(ctx, add_flop, timed, g, s, rmap, cb, nne, tpad, T, E)
    if out_path:
        with open(out_path, "w") as f:
            json.dump(rows, f, indent=1)
    return rows


def bench_ceilings(ctx, out_path: str | None, reps: int = 100, flushed_reps: int = 30,
                   only: str | None = None) -> list:
    """Ceilings of this GPU (module k3h_probe): HBM rates of read-only, write-only,
    copy and the fused op's 2-read : 1.5-write byte shape, over 235 MB streams,
    with 1 or 4 coalesced 16-byte loads in flight per lane (flat grids), 4 or 8
    (persistent grids, 8 workgroups per CU), non-temporal or cacheable; each
    timed back to back (`reps` launches between two events, mean) and one launch
    at a time after a 512 MB clean-read flush (median of `flushed_reps`).  Then
    the register-to-register issue rate of v_mfma_scale_f32_32x32x64_f8f6f4 for
    e4m3 x e2m1 (the MoE GEMMs' operands), e4m3 x e4m3 and e2m1 x e2m1.  The
    fused op and the operators' stream copy run in the same process.  `only`: a
    regular expression; only the rows whose probe names match run (for counter
    runs of a few shapes)."""
    import ctypes
    import re
    want = (lambda name: re.search(only, name) is not None) if only else (lambda name: True)
    import torch
    import k3h
    L = ctx.L
    s = torch.cuda.current_stream()
    n16 = T * H * 2 // 16
    mk = lambda n: torch.empty(n, dtype=torch.uint8, device="cuda").fill_(1)
    a, b, c, d = mk(16 * n16), mk(16 * n16), mk(16 * n16), mk(8 * n16)
    sink = torch.zeros(256, dtype=torch.int32, device="cuda")
    flush_rd = torch.ones(128 << 20, dtype=torch.float32, device="cuda")
    keep = []

    def launcher(entry, grid, kinds, vals, block=256):
        fn = ctx.function("k3h_probe", entry)
        buf = k3h.pack_args(kinds, vals)
        cbuf = ctypes.create_string_buffer(buf, len(buf))
        g, bl = (ctypes.c_uint32 * 3)(grid, 1, 1), (ctypes.c_uint32 * 3)(block, 1, 1)
        keep.append((cbuf, g, bl))

        def go():
            rc = L.k3h_launch(fn, g, bl, 0, s.cuda_stream, ctypes.cast(cbuf, ctypes.c_void_p), len(buf))
            if rc:
                raise k3h.K3HError(rc, entry)
        return go

    def time_it(fn, nrep, nflush):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(s)
        for _ in range(nrep):
            fn()
        e1.record(s)
        torch.cuda.synchronize()
        b2b = e0.elapsed_time(e1) * 1e3 / nrep
        ts = []
        for _ in range(nflush):
            flush_rd.sum()
            e0.record(s)
            fn()
            e1.record(s)
            e1.synchronize()
            ts.append(e0.elapsed_time(e1) * 1e3)
        ts.sort()
        return b2b, ts[len(ts) // 2]

    rows = []
    P = "in buffer<u8>", "out buffer<u8>", "i64", "i32"
    shapes = {  # op -> (bytes moved, kinds, values)
        "read": (16 * n16, [P[0], P[2], P[1]], [a, n16, sink]),
        "write": (16 * n16, [P[1], P[2], P[3]], [c, n16, 0x01010101]),
        "copy": (32 * n16, [P[0], P[1], P[2]], [a, c, n16]),
        "shape": (56 * n16, [P[0], P[0], P[1], P[1], P[2]], [a, b, c, d, n16]),
    }
    variants = [("u1", 1, None), ("u2", 2, None), ("u4", 4, None), ("u7", 7, None), ("u8", 8, None),
                ("u4p", 4, 2048), ("u8p", 8, 2048), ("u4_c", 4, None)]
    for op, (nbytes, kinds, vals) in shapes.items():
        for suf, U, pgrid in variants:
            if not want(f"{op}_{suf}"):
                continue
            grid = pgrid or n16 // (256 * U)
            b2b, fl = time_it(launcher(f"k3h_probe_{op}_{suf}", grid, kinds, vals), reps, flushed_reps)
            row = {"probe": f"{op}_{suf}", "op": op, "loads_in_flight": U,
                   "grid": "persistent 2048" if pgrid else f"flat {grid}",
                   "cache": "cacheable" if suf.endswith("_c") else "non-temporal",
                   "bytes": nbytes, "us_b2b": round(b2b, 2), "gbs_b2b": round(nbytes / b2b / 1e3, 1),
                   "us_flushed": round(fl, 2), "gbs_flushed": round(nbytes / fl / 1e3, 1)}
            rows.append(row)
            log(f"{row['probe']:12s} {b2b:8.2f} us {row['gbs_b2b']:7.0f} GB/s back to back | "
                f"{fl:8.2f} us {row['gbs_flushed']:7.0f} GB/s flushed")
    # the operators' copy and the fused op, same process
    ta = a.view(torch.bfloat16)
    tc = c.view(torch.bfloat16)
    if want("k3h_stream_copy"):
        b2b, fl = time_it(lambda: ctx.stream_copy(ta, tc, stream=s), reps, flushed_reps)
        rows.append({"probe": "k3h_stream_copy (operators' module)", "op": "copy", "loads_in_flight": 1,
                     "grid": f"flat {n16 // 256}", "cache": "non-temporal", "bytes": 32 * n16,
                     "us_b2b": round(b2b, 2), "gbs_b2b": round(32 * n16 / b2b / 1e3, 1),
                     "us_flushed": round(fl, 2), "gbs_flushed": round(32 * n16 / fl / 1e3, 1)})
    del a, b, c, d
    x, res, gm = make_inputs(T)
    ro = torch.empty_like(x)
    q = torch.empty((T, H), dtype=torch.uint8, device="cuda")
    sf = torch.empty((T, H // 32), dtype=torch.uint8, device="cuda")
    nb = algo_bytes(T)
    if want("k3h_residual_rms_mxfp8"):
        b2b, fl = time_it(lambda: ctx.residual_rms_mxfp8(x, res, gm, ro, q, sf, None, eps=1e-6, B=T,
                                                         stream=s), reps, flushed_reps)
        rows.append({"probe": "k3h_residual_rms_mxfp8 (the fused op)", "op": "shape", "loads_in_flight": 14,
                     "grid": f"flat {T // 2}", "cache": "non-temporal", "bytes": nb,
                     "us_b2b": round(b2b, 2), "gbs_b2b": round(nb / b2b / 1e3, 1),
                     "us_flushed": round(fl, 2), "gbs_flushed": round(nb / fl / 1e3, 1)})
    del x, res, gm, ro, q, sf
    if only:  # the operator-shape and MFMA rows are not filtered: a filtered run stops here
        if out_path:
            with open(out_path, "w") as f:
                json.dump(rows, f, indent=1)
        return rows
    rows += bench_op_shapes(ctx, launcher, time_it, reps, flushed_reps)
    # MFMA issue rate, register operands
    n_wg, iters = 256 * 2, 2000
    mout = torch.empty(n_wg * 256, dtype=torch.float32, device="cuda")
    for fmt in ("f8f4", "f8f8", "f4f4"):
        fn = launcher(f"k3h_probe_mfma_{fmt}", n_wg, ["out buffer<f32>", "i32"], [mout, iters])
        b2b, _ = time_it(fn, 20, 1)
        flops = n_wg * 4 * iters * 4 * 131072
        rows.append({"probe": f"mfma_{fmt}", "op": "mfma", "grid": f"{n_wg} x 256",
                     "flops": flops, "us_b2b": round(b2b, 2),
                     "tflops": round(flops / b2b / 1e6, 1)})
        log(f"mfma {fmt}: {b2b:.1f} us, {flops / b2b / 1e6:.0f} TFLOP/s")
    if out_path:
        with open(out_path, "w") as f:
            json.dump(rows, f, indent=1)
    return rows


def bench_op_shapes(ctx, launcher, time_it, reps: int, flushed_reps: int) -> list:
    """The operator-shape probes of k3h_probe next to the operators they mirror,
    in one process on the same inputs' shapes: the KDA span gather (cfg 3a: 3-row
    re-read per 16 or per 32 rows, or none), the weighted finalize (cfg 5d: rows
    gathered through the config-5 routing's exp2perm, one row written per token),
    the MXFP8 permute's payload (cfg 5c: one row gathered per padded row), the MLA
    RoPE pack (cfg 4: one wave per token) and the residual push v3 at nb 0 (one row read, five written, at 128 or 896 threads
    per row).  Each probe's bytes are its own algorithmic bytes (re-reads not counted);
    the operator rows carry the operators' algorithmic bytes."""
    import torch
    s = torch.cuda.current_stream()
    out = []

    def row(name, op, nbytes, fn, grid, note):
        b2b, fl = time_it(fn, reps, flushed_reps)
        r = {"probe": name, "op": op, "loads_in_flight": "-", "grid": grid, "cache": note,
             "bytes": nbytes, "us_b2b": round(b2b, 2), "gbs_b2b": round(nbytes / b2b / 1e3, 1),
             "us_flushed": round(fl, 2), "gbs_flushed": round(nbytes / fl / 1e3, 1)}
        out.append(r)
        log(f"{name:40s} {b2b:8.2f} us {r['gbs_b2b']:7.0f} GB/s back to back | "
            f"{fl:8.2f} us {r['gbs_flushed']:7.0f} GB/s flushed")

    # span gather: [T, 4 * 3072] bf16 -> 3 x [T, 3072]
    inner = 3072
    part = syn("3/partial", (T, 4 * inner))
    d = [torch.empty((T, inner), dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    P5 = ["in buffer<bf16>"] + ["out buffer<bf16>"] * 3 + ["i32"]
    span_bytes = 2 * 3 * T * inner * 2
    for S, blk, note in ((0, 128, "no tap rows"), (1, 128, "3 tap rows per 16"), (2, 256, "3 tap rows per 32")):
        grid = 18 * -(-T // (16 * max(S, 1)))
        row(f"span_s{S}", "span gather shape", span_bytes,
            launcher(f"k3h_probe_span_s{S}", grid, P5, [part, *d, T], block=blk), f"flat {grid} x {blk}",
            f"non-temporal, {note}")
    cw = syn("3/conv_w", (3, 4, inner), std=0.5).float()
    state = torch.zeros(2 * 1628160, dtype=torch.uint8, device="cuda")
    line = torch.zeros(T, dtype=torch.int32, device="cuda")
    wsm = syn("3/wsm", (T, 256), dtype=torch.float32)
    beta = torch.empty(24 * T, dtype=torch.bfloat16, device="cuda")
    flow = torch.empty((T, 128), dtype=torch.bfloat16, device="cuda")
    at0 = torch.zeros(1, dtype=torch.int32, device="cuda")
    row("kern_k3_span_gather (the operator, cfg 3a)", "span gather", 619180032,
        lambda: ctx.span_gather(part, cw, state, line, 1628160, wsm, *d, beta, flow, at0, T, stream=s),
        "typed call", "non-temporal, 3 tap rows per 32")
    del part, d, cw, state, line, wsm, beta, flow
    # config-5 routing (the per-op table's inputs)
    Sx = syn("5/logits", (T, 224), dtype=torch.float32)
    bias = syn("5/bias", (224,), std=0.01, dtype=torch.float32)
    rs = torch.full((1,), 2.5, dtype=torch.bfloat16, device="cuda")
    idx = torch.empty((T, 8), dtype=torch.int32, device="cuda")
    wts = torch.empty((T, 8), dtype=torch.float32, device="cuda")
    ctx.router_topk(Sx, bias, rs, idx, wts, T, topk=8, stream=s)
    E, nblk = 56, T // 256
    cap = T * 8 + E * 128
    i32 = lambda n: torch.zeros(n, dtype=torch.int32, device="cuda")
    bc, bo, cb, cl, nne, tp = i32(nblk * E), i32(nblk * E), i32(cap // 128 + 1), i32(cap // 128 + 1), i32(1), i32(1)
    rmap, e2p, sync = i32(cap), i32(T * 8), i32(2)
    ctx.moe_route(idx, T, 0, E, bc, bo, cb, cl, nne, tp, rmap, e2p, sync, topk=8, stream=s)
    torch.cuda.synchronize()
    tpad, live = int(tp.item()), int((e2p >= 0).sum().item())
    fc2 = syn("5/fc2", (tpad, H))
    fo = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    fin_bytes = live * H * 2 + 2 * T * 8 * 4 + T * H * 2
    row("gather", "finalize shape", live * H * 2 + T * 8 * 4 + T * H * 2,
        launcher("k3h_probe_gather", T, ["in buffer<bf16>", "in buffer<i32>", "out buffer<bf16>", "i32", "i32"],
                 [fc2, e2p, fo, T, H], block=448), f"flat {T} x 448", "non-temporal, rows through exp2perm")
    row("k3h_moe_finalize_rows (the operator, cfg 5d)", "finalize", fin_bytes,
        lambda: ctx.moe_finalize(fc2, e2p, wts, fo, T, H, topk=8, stream=s), "typed call", "non-temporal")
    del fc2, fo
    x8 = torch.ones((T, H), dtype=torch.uint8, device="cuda")
    sf8 = torch.ones((T, H // 32), dtype=torch.uint8, device="cuda")
    pq = torch.empty((tpad, H), dtype=torch.uint8, device="cuda")
    psf = torch.empty((tpad, H // 32), dtype=torch.uint8, device="cuda")
    row("rowgather", "permute shape (payload)", 2 * tpad * H,
        launcher("k3h_probe_rowgather", -(-tpad // 4), ["in buffer<u8>", "in buffer<i32>", "out buffer<u8>", "i32", "i32"],
                 [x8, rmap, pq, tpad, H]), f"flat {-(-tpad // 4)} x 256", "non-temporal, one row per wave")
    row("k3h_moe_permute_mx (the operator, cfg 5c)", "permute", 2 * tpad * (H + H // 32),
        lambda: ctx.moe_permute_mx(x8, sf8, rmap, tp, H, pq, psf, stream=s), "typed call", "non-temporal")
    del x8, sf8, pq, psf
    # MLA latent norm + RoPE + q pack (cfg 4): one wave per token
    lat, kr, qq = syn("4/latent", (T, 512)), syn("4/k_rope", (T, 64)), syn("4/q", (T, 16, 192))
    gk = syn("4/gamma_kv", (512,), 1.0, 0.1)
    pos = torch.arange(T, dtype=torch.int64, device="cuda")
    lo = torch.empty((T, 576), dtype=torch.bfloat16, device="cuda")
    qo = torch.empty_like(qq)
    rope_bytes = T * (512 + 64 + 16 * 192) * 2 + T * (576 + 16 * 192) * 2
    row("rope", "RoPE pack shape", rope_bytes,
        launcher("k3h_probe_rope", -(-T // 4), ["in buffer<bf16>"] * 3 + ["out buffer<bf16>"] * 2 + ["i32", "i32"],
                 [lat, kr, qq, lo, qo, T, 16]), f"flat {-(-T // 4)} x 256",
        "non-temporal, one wave per token, q in batches of 8 vectors per lane")
    row("k3h_mla_rope_pack (the operator, cfg 4)", "RoPE pack", rope_bytes,
        lambda: ctx.mla_rope_pack(lat, kr, qq, gk, pos, lo, qo, T, 16, stream=s), "typed call", "non-temporal")
    del lat, kr, qq, lo, qo
    # residual push v3 at nb 0, 4 ranks (the per-op table's (f)1 row): one row
    # read, the snapshot slot and four normed copies written
    B = T // 4
    prefix = syn("f1/prefix", (B, H))
    blocks = torch.empty((B, 8, H), dtype=torch.bfloat16, device="cuda")
    normed = [torch.empty((4 * B, H), dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    peer = torch.tensor([t.data_ptr() for t in normed], dtype=torch.int64, device="cuda")
    gm = syn("f1/gamma", (H,), mean=1.0, std=0.1)
    sw = torch.zeros(H, dtype=torch.float32, device="cuda")
    P7 = ["in buffer<bf16>"] + ["out buffer<bf16>"] * 5 + ["i32"]
    for nt in (128, 896):
        row(f"push_t{nt}", "push shape", 6 * B * H * 2,
            launcher(f"k3h_probe_push_t{nt}", B, P7, [prefix, blocks, *normed, B], block=nt),
            f"flat {B} x {nt}", f"non-temporal, {7168 // 8 // nt} vector{'s' if nt < 896 else ''} per lane, 1 row read : 5 written")
    row("k3h_attnres_rms_push_nb0w896 (the operator, push v3 nb 0)", "push", 6 * B * H * 2 + H * 2,
        lambda: ctx.attnres_rms_push(prefix, blocks, sw, gm, normed[1], peer, 0, 1, B, 1, 4, version=3,
                                     stream=s), "typed call", "non-temporal")
    return out


def ceilings_markdown(rows: list) -> str:
    out = ["| probe | access | loads in flight per lane | grid | bytes | back to back us | GB/s | % of 8 TB/s "
           "| flushed us | GB/s | % of 8 TB/s |",
           "|---|---|---:|---|---:|---:|---:|---:|---:|---:|---:|"]
    for r in rows:
        if r["op"] == "mfma":
            continue
        out.append(f"| {r['probe']} | {r['op']}, {r['cache']} | {r['loads_in_flight']} | {r['grid']} | "
                   f"{r['bytes']:,} | {r['us_b2b']:.2f} | {r['gbs_b2b']:.0f} | "
                   f"{100 * r['gbs_b2b'] / PEAK_GBS:.1f} | {r['us_flushed']:.2f} | {r['gbs_flushed']:.0f} | "
                   f"{100 * r['gbs_flushed'] / PEAK_GBS:.1f} |")
    out += ["", "| MFMA probe | operands (A x B) | grid | FLOPs per launch | us | TFLOP/s |",
            "|---|---|---|---:|---:|---:|"]
    names = {"mfma_f8f4": "e4m3 x e2m1", "mfma_f8f8": "e4m3 x e4m3", "mfma_f4f4": "e2m1 x e2m1"}
    for r in rows:
        if r["op"] == "mfma":
            out.append(f"| {r['probe']} | {names[r['probe']]} | {r['grid']} | {r['flops']:,} | "
                       f"{r['us_b2b']:.1f} | {r['tflops']:.0f} |")
    return "\n".join(out)


def cpu_route(O, ids, T, nblk, E, cap) -> None:
    """The oracle's count -> tables -> scatter chain for EP rank 0 (CPU baseline)."""
    bc = O.route_count(ids, T, 8, 0, E)
    tb = O.route_tables(bc, nblk, E, 128, cap)
    O.route_scatter(ids, tb["blockoff"], T, 8, 0, E, tb["route_map"])


def bench_push_land(ctx, add, timed, bf, g, s, O=None, h=None) -> None:
    """The residual push family and the landing kernels at one TP rank's share of
    the 16k prefill (B = tokens / 4 = 4096 rows; manifest shapes).  On one GPU
    the four ranks' normed_all buffers are local, so every normed copy is an HBM
    write here (three of the four cross xGMI on a 4-GPU node).  With the oracle
    module O (and the host-copy helper h) the single-rank rows also time the C
    oracle; the push rows have no CPU counterpart of their multi-rank stores."""
    import torch
    B, HH = 4096, H
    row = B * HH * 2
    gm = bf(HH, mean=1.0, std=0.1)
    sw = torch.randn(HH, generator=g, device="cuda") * 0.05
    sw_mlp = torch.randn(HH, generator=g, device="cuda") * 0.05
    prefix = bf(B, HH)
    blocks = bf(B, 8, HH)
    normed = [torch.empty((4 * B, HH), dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    peer = torch.tensor([t.data_ptr() for t in normed], dtype=torch.int64, device="cuda")
    add("residual push v3 (res_in, nb 0, 4 ranks)", "k3h_attnres_rms_push_nb0w896", f"B={B} nb=0",
        row + HH * 2 + row + 4 * row,
        timed(lambda: ctx.attnres_rms_push(prefix, blocks, sw, gm, normed[1], peer, 0, 1, B, 1, 4,
                                           version=3, stream=s)))
    nb = 4
    p1, p2, prefix2 = bf(B, HH), bf(B, HH), bf(B, HH)
    hidden = torch.empty_like(p1)
    stats = torch.empty((B, 8, 2), dtype=torch.float32, device="cuda")
    add("residual push_add2 (res_in, nb 4, 4 ranks)", "k3h_attnres_rms_push_nb4s",
        f"B={B} nb={nb} two=1", 3 * row + nb * row + 2 * HH * 4 + HH * 2 + row + row + 4 * row + B * nb * 8,
        timed(lambda: ctx.attnres_rms_push_add2(blocks, sw, gm, normed[0], peer, nb, 1, B, 0, 4,
                                                sw_mlp, stats, p1, p2, prefix2, hidden, 1, stream=s)))
    # normed_sync: the arrival barrier after the push, every peer already arrived
    # (their slot counters at the top of the 32-bit range, so every call passes)
    flags = [torch.zeros(372, dtype=torch.int64, device="cuda") for _ in range(4)]
    for q in (0, 2, 3):
        flags[q][1] = 0xFFFFFFFF
    fpeer = torch.tensor([f.data_ptr() for f in flags], dtype=torch.int64, device="cuda")
    ctx.epoch_bump(flags[1], 896, stream=s)
    add("arrival barrier (normed_sync, peers arrived)", "kern_k3_rs_arrive1", "1 wave, 4 ranks", 0,
        timed(lambda: ctx.rs_arrive(flags[1], fpeer, 896, 1, 4, stream=s)),
        "fence, add, 4 polls, fence")
    part = bf(B, HH)
    pre2, nrm = torch.empty_like(part), torch.empty_like(part)
    for k, kern in ((1, "k3h_land_add_attnres_rms_nb1s"), (4, "k3h_land_add_attnres_rms_nb4s"),
                    (8, "k3h_land_add_attnres_rms_nb8s")):
        add(f"K1b nb {k} (res_mlp, typed call)", kern, f"B={B} nb={k}",
            2 * row + k * row + HH * 4 + HH * 2 + 2 * row,
            timed(lambda k=k: ctx.land_add_attnres_rms_nb(part, prefix, blocks, sw, gm, pre2, nrm, k,
                                                          0, B, stream=s)),
            "vector-split row body" + (" (reference on GB300: 155 us)" if k == 8 else ""),
            cpu=O and (lambda a=(h(part), h(prefix), h(blocks), h(sw), h(gm)), k=k:
                       O.land_add_attnres_rms(a[0], a[1], a[2], a[3], a[4], k, 0, B)))
    add("res_mlp nb 5 with res_in statistics (nb_stats 4)", "k3h_land_add_attnres_rms_nb5s",
        f"B={B} nb=5", 2 * row + 5 * row + HH * 4 + HH * 2 + 2 * row + B * 4 * 8,
        timed(lambda: ctx.land_add_attnres_rms_nb_stats(part, prefix, blocks, sw_mlp, gm, pre2, nrm,
                                                        5, 0, B, stats, 4, stream=s)),
        cpu=O and (lambda a=(h(part), h(prefix), h(blocks), h(sw_mlp), h(gm), h(stats)):
                   O.land_add_attnres_rms_stats(a[0], a[1], a[2], a[3], a[4], 5, 0, B, a[5], 4)))
    del normed, peer, p1, p2, prefix2, hidden, part, pre2, nrm, blocks, prefix
    # landing kernels (k3_land / k3_situ_bf16 / k3_land_fused)
    hd = 3584
    lat = bf(B, hd)
    gl = bf(hd, mean=1.0, std=0.1)
    ln = torch.empty_like(lat)
    add("rms (l0, h 3584)", "kern_k3_rms", f"B={B} h={hd}", 2 * B * hd * 2 + hd * 2,
        timed(lambda: ctx.rms(lat, gl, ln, hd, B, stream=s)),
        cpu=O and (lambda a=(h(lat), h(gl)): O.rms(a[0], a[1], hd, B)))
    pf = torch.randn((B, hd), generator=g, device="cuda")
    lo = torch.empty((B, hd), dtype=torch.bfloat16, device="cuda")
    add("land (l0, n 3584)", "kern_k3_land", f"B={B} n={hd}", B * hd * 4 + B * hd * 2,
        timed(lambda: ctx.land(pf, lo, hd, 0, hd, B, stream=s)),
        cpu=O and (lambda a=h(pf): O.land(a, hd, 0, hd, B)))
    del pf, lo
    for n, kind in ((33792, "f32"), (6144, "f32"), (33792, "situ_bf16")):
        if kind == "f32":
            p = torch.randn((B, 2 * n), generator=g, device="cuda") * 3.0
            nm, ker, ib = f"SiTU landing f32 (n {n})", "kern_k3_land_situ", 4
        else:
            p = bf(B, 2 * n, std=3.0)
            nm, ker, ib = f"SiTU landing bf16 (l0, n {n})", "kern_k3_situ_bf16", 2
        act = torch.empty((B, n), dtype=torch.bfloat16, device="cuda")
        add(nm, ker, f"B={B} n={n}", B * 2 * n * ib + B * n * 2,
            timed(lambda: ctx.land_situ(p, act, n, B, variant="situ_bf16" if kind != "f32" else None,
                                        stream=s)),
            cpu=O and (lambda a=h(p): O.land_situ(a, n, B)))
        del p, act
    n = 6144
    sp = bf(B, 2 * n, std=2.0)
    act = torch.empty((B, n), dtype=torch.bfloat16, device="cuda")
    add("SiTU landing + latent rms (fused)", "kern_k3_situ_rms_bf16", f"B=L={B} n={n} h={hd}",
        B * 2 * n * 2 + B * n * 2 + 2 * B * hd * 2 + hd * 2,
        timed(lambda: ctx.situ_rms(sp, act, lat, gl, ln, n, B, hd, B, 4 * B, stream=s)),
        cpu=O and (lambda a=(h(sp), h(lat), h(gl)): O.situ_rms(a[0], a[1], a[2], n, B, hd, B, 4 * B)))


def bench_gemm(ctx, add_flop, timed, g, s, rmap, cta_batch, num_tiles, tpad, T, E) -> None:
    """The MoE expert GEMMs at the reference's shapes (latent 3584, intermediate 3072,
    56 local experts, e2m1 weights), over the routing tables of the top-8 router run:
    fc1 gathers its rows through route_map (SiTU-GLU + MXFP8 epilogue), fc2 reads fc1's
    output (bf16 out).  FLOPs count the padded rows the tiles compute."""
    import torch
    KL, INTER, COLS = 3584, 3072, 3584
    max_tiles = rmap.numel() // 128
    lat = (torch.randn((T, KL), generator=g, device="cuda")).to(torch.bfloat16)
    aq = torch.empty((T, KL), dtype=torch.uint8, device="cuda")
    asf = torch.empty((T, KL // 32), dtype=torch.uint8, device="cuda")
    ctx.moe_quant(lat, aq, asf, T, KL, stream=s)
    del lat

    def weights(n, k, gated):
        w = torch.randint(0, 256, (E * n * k // 2,), generator=g, device="cuda", dtype=torch.uint8)
        sc = torch.randint(121, 126, (E * n * k // 32,), generator=g, device="cuda",
                           dtype=torch.uint8)
        wt, st = torch.empty_like(w), torch.empty_like(sc)
        ctx.moe_w_tile(w, wt, E, n, k, gated, stream=s)
        ctx.moe_sf_tile(sc, st, E, n, k, gated, stream=s)
        return wt, st
    w13, s13 = weights(2 * INTER, KL, 1)
    w2, s2 = weights(COLS, INTER, 0)
    alpha = torch.full((E,), 4.0, device="cuda")
    beta = torch.full((E,), 25.0, device="cuda")
    o1 = torch.empty((max_tiles * 128, INTER), dtype=torch.uint8, device="cuda")
    o1sf = torch.empty((max_tiles * 128, INTER // 32), dtype=torch.uint8, device="cuda")
    o2 = torch.empty((max_tiles * 128, COLS), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    add_flop("MoE fc1 (MX GEMM + SiTU-GLU + MXFP8)", "kern_k3h_moe_gemm3_situ_mx",
             f"{tpad} rows x {KL} -> 2x{INTER}, E={E}", 2 * tpad * KL * 2 * INTER,
             E * 2 * INTER * (KL // 2 + KL // 32) + tpad * (KL + KL // 32) + tpad * (INTER + INTER // 32),
             timed(lambda: ctx.moe_gemm_mx(ctx.GEMM_SITU_MX, aq, asf, rmap, w13, s13, num_tiles,
                                           cta_batch, max_tiles, E, 2 * INTER, KL, o1, o1sf, alpha,
                                           beta, stream=s)),
             "e4m3 x e2m1 MFMA; gathers rows through route_map")
    add_flop("MoE fc2 (MX GEMM, bf16 out)", "kern_k3h_moe_gemm2_bf16",
             f"{tpad} rows x {INTER} -> {COLS}, E={E}", 2 * tpad * INTER * COLS,
             E * COLS * (INTER // 2 + INTER // 32) + tpad * (INTER + INTER // 32) + tpad * COLS * 2,
             timed(lambda: ctx.moe_gemm_mx(ctx.GEMM_BF16, o1, o1sf, None, w2, s2, num_tiles,
                                           cta_batch, max_tiles, E, COLS, INTER, o2, stream=s)),
             "e4m3 x e2m1 MFMA")
    del w13, s13, w2, s2, o1, o1sf, o2, aq, asf


# Per-op kernels, in launch order, for the counter table (kernel names as the
# rocprofv3 CSV output prints them).
OP_KERNELS = {
    "stream copy (ceiling)": ["k3h_stream_copy"],
    "residual add + RMSNorm (cfg 1)": ["kern_k3_land_add_attnres_rms"],
    "residual+RMSNorm+MXFP8 (cfg 2)": ["k3h_residual_rms_mxfp8"],
    "MXFP8 quant alone": ["kern_k3_moe_quant"],
    "per-tensor fp8 pair (amax+apply)": ["k3h_quant_fp8_mark", "k3h_quant_fp8_once"],
    "KDA span gather (cfg 3a)": ["kern_k3_span_gather"],
    "KDA output gate (cfg 3b, eps 1e-6)": ["kern_k3_kda_out_gate"],
    "MLA prep (cfg 4, reference form)": ["k3h_mla_prep_fused"],
    "MLA latent norm + RoPE + q pack": ["k3h_mla_rope_pack"],
    "router top-8 (cfg 5a)": ["k3h_router_topk_pairs"],
    "EP routing tables (count+tables+scatter)": ["kern_k3_moe_route_count", "kern_k3_moe_route_tables",
                                                 "kern_k3_moe_route_scatter"],
    "EP routing, one launch (k3h_moe_route)": ["k3h_moe_route_fused"],
    "MXFP8 permute (cfg 5c)": ["k3h_moe_permute_mx"],
    "weighted finalize (cfg 5d)": ["k3h_moe_finalize_rows"],
    "residual push v3 (res_in, nb 0, 4 ranks)": ["k3h_attnres_rms_push_nb0w896"],
    "residual push_add2 (res_in, nb 4, 4 ranks)": ["k3h_attnres_rms_push_nb4s"],
    "arrival barrier (normed_sync, peers arrived)": ["kern_k3_rs_arrive1"],
    "K1b nb 1 (res_mlp, typed call)": ["k3h_land_add_attnres_rms_nb1s"],
    "K1b nb 4 (res_mlp, typed call)": ["k3h_land_add_attnres_rms_nb4s"],
    "K1b nb 8 (res_mlp, typed call)": ["k3h_land_add_attnres_rms_nb8s"],
    "res_mlp nb 5 with res_in statistics (nb_stats 4)": ["k3h_land_add_attnres_rms_nb5s"],
    "rms (l0, h 3584)": ["kern_k3_rms"],
    "land (l0, n 3584)": ["kern_k3_land"],
    "SiTU landing f32 (n 33792)": ["kern_k3_land_situ"],
    "SiTU landing f32 (n 6144)": ["kern_k3_land_situ"],
    "SiTU landing bf16 (l0, n 33792)": ["kern_k3_situ_bf16"],
    "SiTU landing + latent rms (fused)": ["kern_k3_situ_rms_bf16"],
    "MoE fc1 (MX GEMM + SiTU-GLU + MXFP8)": ["kern_k3h_moe_gemm3_situ_mx"],
    "MoE fc2 (MX GEMM, bf16 out)": ["kern_k3h_moe_gemm2_bf16"],
}


def _csv_rows(path: str):
    import csv
    with open(path, newline="") as f:
        yield from csv.DictReader(f)


def _col(row: dict, *names: str) -> str:
    low = {k.lower(): v for k, v in row.items()}
    for n in names:
        if n.lower() in low:
            return low[n.lower()]
    raise KeyError(f"none of {names} in {sorted(row)}")


def counter_values(csv_path: str, counter: str) -> dict:
    """Per kernel name: `counter` (KiB per dispatch) of every dispatch, in
    dispatch order, from a rocprofv3 --pmc CSV (counter_collection.csv)."""
    per = {}
    for r in _csv_rows(csv_path):
        if _col(r, "Counter_Name") != counter:
            continue
        name = _col(r, "Kernel_Name").split("(")[0].strip()
        per.setdefault(name, []).append((int(_col(r, "Dispatch_Id")), float(_col(r, "Counter_Value"))))
    return {k: [v for _, v in sorted(d)] for k, d in per.items()}


class _Dispatches:
    """Hands out each op's dispatches of a kernel in launch order (ops that share
    an entry name, e.g. the push modules, take consecutive runs)."""

    def __init__(self, values: dict):
        self.values, self.pos = values, {k: 0 for k in values}

    def median(self, kernel: str, n: int):
        if kernel not in self.values:
            return None
        i = self.pos[kernel]
        run = self.values[kernel][i:i + n]
        self.pos[kernel] = i + n
        return sorted(run)[len(run) // 2] if run else None


def traffic_table(fetch_csv: str, write_csv: str, ops_json: str) -> str:
    """Markdown table of measured HBM bytes per op call: FETCH_SIZE and WRITE_SIZE
    (KiB per dispatch, median), each scaled by the factor that maps the same
    counter of k3h_stream_copy onto its known byte count, against the op's
    algorithmic bytes (from a bench.py --ops-out JSON of the same shapes)."""
    fv, wv = counter_values(fetch_csv, "FETCH_SIZE"), counter_values(write_csv, "WRITE_SIZE")
    fetch, write = _Dispatches(fv), _Dispatches(wv)
    ops = {r["op"]: r for r in json.load(open(ops_json))}
    copy_bytes = ops["stream copy (ceiling)"]["bytes"] // 2  # read once, written once
    n_copy = ops["stream copy (ceiling)"].get("launches", len(fv["k3h_stream_copy"]))
    kf = copy_bytes / (fetch.median("k3h_stream_copy", n_copy) * 1024)
    kw = copy_bytes / (write.median("k3h_stream_copy", n_copy) * 1024)
    fetch, write = _Dispatches(fv), _Dispatches(wv)
    out = [f"Scale factors from k3h_stream_copy ({copy_bytes:,} B read and written): "
           f"FETCH_SIZE x {kf:.5f}, WRITE_SIZE x {kw:.5f}", "",
           "| op | kernels | read B | written B | measured B | algorithmic B | measured / algorithmic |",
           "|---|---|---:|---:|---:|---:|---:|"]
    for op, kernels in OP_KERNELS.items():
        if op not in ops:
            continue
        n = ops[op].get("launches", 0)
        f = [fetch.median(k, n) for k in kernels]
        w = [write.median(k, n) for k in kernels]
        if None in f or None in w:
            continue
        rd = sum(f) * 1024 * kf
        wr = sum(w) * 1024 * kw
        alg = ops[op]["bytes"]
        if not alg:  # latency rows (the arrival barrier) move no payload
            continue
        out.append(f"| {op} | {', '.join('`%s`' % k for k in kernels)} | {rd:,.0f} | {wr:,.0f} | "
                   f"{rd + wr:,.0f} | {alg:,} | {(rd + wr) / alg:.3f} |")
    return "\n".join(out)


def trace_table(trace_csv: str, ops_json: str) -> str:
    """Markdown table of kernel-trace durations per op: from a rocprofv3
    --kernel-trace CSV of a bench.py --ops-only run and that run's --ops-out JSON,
    each op's dispatches are taken in launch order (5 warm-ups, then `reps` after
    the clean-read flush, then `reps` after the dirty flush); an op's time per
    launch is the sum of its kernels' spans; the median over the clean-flush
    launches is set beside the HIP-event median of the same launches (which also
    holds the launch itself)."""
    per = {}
    for r in _csv_rows(trace_csv):
        name = _col(r, "Kernel_Name").split("(")[0].strip()
        span = (int(_col(r, "End_Timestamp")) - int(_col(r, "Start_Timestamp"))) / 1e3
        per.setdefault(name, []).append((int(_col(r, "Dispatch_Id")), span))
    per = {k: [d for _, d in sorted(v)] for k, v in per.items()}
    pos = {k: 0 for k in per}
    ops = {r["op"]: r for r in json.load(open(ops_json))}
    out = ["| op | kernels | HIP-event median us | kernel median us | GB/s (kernel time) | % of 8 TB/s "
           "| TFLOP/s (kernel time) |", "|---|---|---:|---:|---:|---:|---:|"]
    for op, kernels in OP_KERNELS.items():
        if op not in ops:
            continue
        r = ops[op]
        n = r.get("launches", 0)
        reps = (n - 5) // 2
        runs = []
        for k in kernels:
            if k not in per:
                runs = None
                break
            runs.append(per[k][pos[k]:pos[k] + n])
            pos[k] += n
        if not runs or any(len(x) < n for x in runs):
            continue
        clean = sorted(sum(x[i] for x in runs) for i in range(5, 5 + reps))
        us = clean[len(clean) // 2]
        if r.get("bound") == "mfma":
            rate = f" | | | {r['flops'] / (us * 1e-6) / 1e12:.1f}"
        elif not r["bytes"]:  # latency rows (the arrival barrier) move no payload
            rate = " | | | "
        else:
            gbs = r["bytes"] / (us * 1e-6) / 1e9
            rate = f" | {gbs:.1f} | {100 * gbs / PEAK_GBS:.1f} | "
        out.append(f"| {op} | {', '.join('`%s`' % k for k in kernels)} | {r['us']:.2f} | {us:.2f}{rate} |")
    return "\n".join(out)


def ops_markdown(ops_json: str) -> str:
    """Markdown tables of a bench.py --ops-out JSON: the HBM-bound ops (GB/s, % of
    8 TB/s, % of the run's copy ceiling, CPU oracle column where timed) and the
    MFMA-bound ops (TFLOP/s, % of the 5.0 PFLOP/s e4m3 peak)."""
    ops = json.load(open(ops_json))
    copy = next((r["gbs"] for r in ops if r["kernel"] == "k3h_stream_copy"), None)
    thr = next((r["cpu_threads"] for r in ops if "cpu_threads" in r), None)
    gr = any("us_graph" in r for r in ops)
    gh, gs = ("| us, graph replay | GB/s, graph replay ", "---:|---:|") if gr else ("", "")
    out = ["| op | kernel | shape | algorithmic bytes | median us | p10 us | p90 us | GB/s | % of 8 TB/s "
           f"| % of copy | us, dirty flush | GB/s, dirty flush {gh}"
           f"| CPU ms{f' ({thr} threads)' if thr else ''} | CPU GB/s | GPU / CPU | note |",
           f"|---|---|---|---:|---:|---:|---:|---:|---:|---:|---:|---:|{gs}---:|---:|---:|---|"]
    for r in ops:
        if r.get("bound") == "mfma":
            continue
        c = (f"{r['cpu_ms']:.1f} | {r['cpu_gbs']:.2f} | {r['gbs'] / r['cpu_gbs']:.0f}x"
             if "cpu_ms" in r else " | | ")
        pc = f"{100 * r['gbs'] / copy:.0f}" if copy else ""
        d = f"{r['us_dirty']:.2f} | {r['gbs_dirty']:.1f}" if "us_dirty" in r else " | "
        if gr:
            d += (f" | {r['us_graph']:.2f} | {r['gbs_graph']:.1f}" if "us_graph" in r else " | | ")
        out.append(f"| {r['op']} | `{r['kernel']}` | {r['shape']} | {r['bytes']:,} | {r['us']:.2f} | "
                   f"{r['us_p10']:.2f} | {r['us_p90']:.2f} | {r['gbs']:.1f} | {r['pct_peak']:.1f} | {pc} | "
                   f"{d} | {c} | {r['note']} |")
    mf = [r for r in ops if r.get("bound") == "mfma"]
    if mf:
        out += ["", "| op | kernel | shape | FLOPs | bytes | median us | p10 us | p90 us | TFLOP/s "
                "| % of 5.0 PFLOP/s | us, dirty flush | note |",
                "|---|---|---|---:|---:|---:|---:|---:|---:|---:|---:|---|"]
        for r in mf:
            out.append(f"| {r['op']} | `{r['kernel']}` | {r['shape']} | {r['flops']:,} | {r['bytes']:,} | "
                       f"{r['us']:.2f} | {r['us_p10']:.2f} | {r['us_p90']:.2f} | {r['tflops']:.1f} | "
                       f"{r['pct_peak']:.1f} | {r.get('us_dirty', float('nan')):.2f} | {r['note']} |")
    return "\n".join(out)


TRAFFIC_JSON = "profiles/traffic.json"


def flushed_timing(step, stream, nbytes: int, reps: int) -> dict:
    """The same launch timed one at a time, each between two HIP events on its
    stream, with a 512 MB clean read before each (outside the events), so it
    starts with cold L2s and MALL and owes no write-back: median, p10, p90."""
    import torch
    flush_rd = torch.ones(128 << 20, dtype=torch.float32, device="cuda")
    ts = []
    for _ in range(reps):
        flush_rd.sum()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        step()
        e1.record(stream)
        e1.synchronize()
        ts.append(e0.elapsed_time(e1) * 1e3)
    del flush_rd
    ts.sort()
    pick = lambda f: ts[min(len(ts) - 1, int(f * len(ts)))]
    us = pick(0.5)
    return {"protocol": "512 MB clean-read flush before each launch, per-launch HIP events",
            "reps": reps, "us": round(us, 2), "us_p10": round(pick(0.1), 2),
            "us_p90": round(pick(0.9), 2), "gbs": round(nbytes / (us * 1e-6) / 1e9, 1),
            "frac": round(nbytes / (us * 1e-6) / 1e9 / PEAK_GBS, 4)}


def load_traffic(kernel: str, workload: str):
    p = os.path.join(REPO, TRAFFIC_JSON)
    try:
        d = json.load(open(p))
        return d[kernel][workload]["hbm_bytes_per_launch"]
    except (OSError, KeyError, ValueError):
        return None


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--warm-s", type=float, default=0.3,
                    help="keep warming up (batches of 100 steps) until this many seconds have run")
    ap.add_argument("--rows", type=int, default=T)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-budget", type=float, default=10.0)
    ap.add_argument("--flushed-reps", type=int, default=50,
                    help="launches timed one by one after a cache flush (the 'flushed' record)")
    ap.add_argument("--op", choices=["fused", "copy", "ceilings"], default="fused",
                    help="copy: only the 16-byte streaming copy (counter calibration); "
                         "ceilings: HBM access-shape and MFMA-rate probes (markdown on stdout)")
    ap.add_argument("--ceilings-out", default=None, help="write the ceilings rows as JSON")
    ap.add_argument("--probe-filter", default=None,
                    help="--op ceilings: a regular expression; only the probes whose names match run")
    ap.add_argument("--ceilings-table", metavar="CEILINGS_JSON",
                    help="print the markdown table of a --ceilings-out JSON; no GPU")
    ap.add_argument("--ops", action="store_true",
                    help="also time every op at its config shape (table on stderr)")
    ap.add_argument("--ops-only", action="store_true", help="only the per-op table")
    ap.add_argument("--graph", action="store_true",
                    help="per-op table: also time each op as a captured HIP graph replay")
    ap.add_argument("--ops-out", default=None, help="write the per-op table as JSON")
    ap.add_argument("--ops-table", metavar="OPS_JSON",
                    help="print the per-op markdown table of an --ops-out JSON; no GPU")
    ap.add_argument("--trace-table", nargs=2, metavar=("TRACE_CSV", "OPS_JSON"),
                    help="print per-op kernel-trace medians (clean-flush launches) from a rocprofv3 "
                         "--kernel-trace CSV of --ops-only and its --ops-out JSON; no GPU")
    ap.add_argument("--traffic-table", nargs=3, metavar=("FETCH_CSV", "WRITE_CSV", "OPS_JSON"),
                    help="print the per-op HBM byte table from two rocprofv3 --pmc CSVs "
                         "(FETCH_SIZE, WRITE_SIZE runs of --ops-only) and an --ops-out JSON; no GPU")
    a = ap.parse_args()
    if a.traffic_table:
        print(traffic_table(*a.traffic_table))
        return 0
    if a.trace_table:
        print(trace_table(*a.trace_table))
        return 0
    if a.ops_table:
        print(ops_markdown(a.ops_table))
        return 0
    if a.ceilings_table:
        print(ceilings_markdown(json.load(open(a.ceilings_table))))
        return 0
    if a.gpus != 1:
        print(f"bench.py measures one GPU only (asked for {a.gpus}); the op family shards "
              "by rows / heads / experts with no exchange on the measured path.", file=sys.stderr)
        return 2

    build_note = ""
    if not a.no_cpu and a.op == "fused":
        build_note = native_oracle()  # before any import of oracle.py in this process
    import torch
    import k3h

    ctx = k3h.Ctx()
    rows = a.rows
    if a.op == "ceilings":
        print(ceilings_markdown(bench_ceilings(ctx, a.ceilings_out, only=a.probe_filter)), flush=True)
        return 0
    if a.ops_only:
        bench_ops(ctx, max(5, a.steps), a.ops_out, 0.0 if a.no_cpu else 3.0, a.graph)
        return 0
    copy_gbs = copy_ceiling(ctx, rows, a.steps if a.op == "copy" else 20)
    if a.op == "copy":
        print(json.dumps({"op": "k3h_stream_copy", "bytes_per_launch": 2 * rows * H * 2,
                          "gbs": round(copy_gbs, 1)}), flush=True)
        return 0
    log(f"inputs {rows}x{H} bf16 on {torch.cuda.get_device_name(0)}")
    x, res, gamma = make_inputs(rows)
    ro = torch.empty_like(x)
    q = torch.empty((rows, H), dtype=torch.uint8, device="cuda")
    sf = torch.empty((rows, H // 32), dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream()

    def step():
        ctx.residual_rms_mxfp8(x, res, gamma, ro, q, sf, None, eps=1e-6, B=rows, stream=stream)

    # W warm-up steps, continued in batches of 100 until at least --warm-s seconds
    # of launches have run: the first ~0.1 s of a burst runs below steady clocks.
    t_warm = time.perf_counter()
    n_warm = 0
    for _ in range(a.warmup):
        step()
    torch.cuda.synchronize()
    n_warm += a.warmup
    while time.perf_counter() - t_warm < a.warm_s:
        for _ in range(100):
            step()
        torch.cuda.synchronize()
        n_warm += 100
    log(f"warm-up: {n_warm} launches in {time.perf_counter() - t_warm:.2f} s")
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(a.steps):
        step()
    e1.record(stream)
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / a.steps
    nbytes = algo_bytes(rows)
    gbs = nbytes / (ms * 1e-3) / 1e9
    log(f"{ms * 1e3:.1f} us/step, {gbs:.0f} GB/s ({100 * gbs / PEAK_GBS:.1f}% of 8 TB/s)")

    flushed = flushed_timing(step, stream, nbytes, a.flushed_reps)
    log(f"flushed (512 MB clean read before each launch): median {flushed['us']} us "
        f"(p10 {flushed['us_p10']}, p90 {flushed['us_p90']}) = {flushed['gbs']} GB/s")

    traffic = load_traffic("k3h_residual_rms_mxfp8", f"{rows}x{H}")
    roof = {"bound": "hbm", "achieved": round(gbs, 1), "peak": PEAK_GBS, "unit": "GB/s",
            "frac": round(gbs / PEAK_GBS, 4), "traffic": traffic,
            "traffic_source": (f"{TRAFFIC_JSON} (rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE runs of "
                               "this kernel at this shape, each scaled by the same counter's reading "
                               "for k3h_stream_copy; not measured in this run)")
            if traffic is not None else None,
            "kernel": "k3h_residual_rms_mxfp8", "algorithmic_bytes": nbytes,
            "avg_launch_us": round(ms * 1e3, 2), "copy_ceiling_gbs": round(copy_gbs, 1)}
    ops = None
    if a.ops:
        ops = bench_ops(ctx, 50, a.ops_out, 0.0 if a.no_cpu else 3.0, a.graph)
    cpu = None
    if not a.no_cpu:
        log("CPU baseline: C oracle on the same inputs")
        cpu = cpu_baseline(x, res, gamma, (ro, q, sf), a.cpu_budget, build_note)
        log(f"CPU {cpu['value']} GB/s on {cpu['cores']} threads; {cpu['sample']}")
    line = {
        "metric": METRIC, "value": round(gbs, 1), "unit": "GB/s", "n_gpus": 1,
        "steps": a.steps, "warmup": a.warmup, "warmup_launches": n_warm, "ms_per_step": round(ms, 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
        "data": DATA,
        "config": {"workload": "fused residual add + RMSNorm + MXFP8 (BASELINE config 2)",
                   "tokens": rows, "hidden": H, "eps": 1e-6, "block": 32,
                   "payload": "e4m3 (OCP)", "scale": "E8M0"},
        "pct_of_peak": round(100 * gbs / PEAK_GBS, 2),
        "roofline": roof, "cpu_baseline": cpu, "flushed": flushed,
    }
    if ops:
        line["ops"] = {r["op"]: {"us": r["us"], "gbs": r["gbs"], "pct_peak": r["pct_peak"]} for r in ops}
    print(json.dumps(line), flush=True)
    ctx.close()
    return 0


if __name__ == "__main__":
    sys.exit(main())
