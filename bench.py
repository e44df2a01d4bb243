"""Benchmark of the mapstencil hot path on one MI355X.

Default workload: Game of Life on an 8192 x 8192 UInt8 grid (Bernoulli(0.3),
seed 2), Moore(1), Wrap, Halo padding, B3/S23, as a device-resident
SwitchingStencilArray.  One step is one generation (one `mapstencil!` call);
the timed steps run as replays of a captured hipGraph.  Prints one JSON line.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]
"""
import argparse
import ctypes
import json
import os
import re
import sys
import time
from pathlib import Path

import numpy as np

REPO = Path(__file__).resolve().parent
sys.path.insert(0, str(REPO / "stencils.jl_amd"))
sys.path.insert(0, str(REPO / "oracle"))

METRIC = "cells/s + % HBM roofline, batched/served vs plain mapstencil; p99 latency"
HBM_PEAK_GBS = 8000.0


def life_grid(n: int, seed: int = 2, p: float = 0.3) -> np.ndarray:
    rng = np.random.Generator(np.random.PCG64(seed))
    return (rng.random((n, n)) < p).astype(np.uint8)


def device_switching(A: np.ndarray, sh, torch):
    dev = torch.device("cuda", torch.cuda.current_device())
    t = sh.colmajor_empty(A.shape, torch.uint8, dev)
    t.copy_(torch.from_numpy(np.ascontiguousarray(A)).to(dev))
    return sh.SwitchingStencilArray(t, sh.Moore(1), boundary=sh.Wrap(), padding=sh.Halo())


def time_steps(sh, torch, S, rule, steps: int, graph: bool, flags: int = 0):
    """Wall time and HIP-event time of `steps` generations (inputs resident)."""
    stream = torch.cuda.current_stream()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    start.record(stream)
    S = sh.mapstencil_steps(rule, S, steps, graph=graph, flags=sh._abi.ASYNC | flags)
    end.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    return S, wall, start.elapsed_time(end) / 1e3


def kernel_launch_us(sh, torch, S, rule, launches: int = 200):
    """Average duration of the single-generation kernel: graph-replayed steps
    without temporal blocking, between HIP events on the launch stream."""
    stream = torch.cuda.current_stream()
    for _ in range(1 if launches % 2 == 0 else 2):  # capture this schedule's graphs before timing
        S = sh.mapstencil_steps(rule, S, launches, graph=True, flags=sh._abi.ASYNC | sh._abi.NO_FUSE)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    e0.record(stream)
    S = sh.mapstencil_steps(rule, S, launches, graph=True, flags=sh._abi.ASYNC | sh._abi.NO_FUSE)
    e1.record(stream)
    torch.cuda.synchronize()
    return S, e0.elapsed_time(e1) / launches * 1e3


# Generations whose time and traffic the headline's roofline gives, and the
# generations of the launch that profiles/lifep_kernel_gol_8192.md measured.
LIFE_GENS = 8
LIFE_PROFILED_GENS = 32


def fused_launch_us(sh, torch, S, rule, gens: int, m1: int = 1, m2: int = 5):
    """Average duration of `gens` generations of the multi-generation Life
    kernel, without the ends of a call: the difference of two calls of
    3 + 32 gens m generations, timed between HIP events on the launch stream,
    is (m2 - m1) x 32 times as many.  Both calls' graphs are captured before
    timing."""
    stream = torch.cuda.current_stream()
    steps = lambda m: 3 + 32 * gens * m  # noqa: E731
    for m in (m1, m2, m1, m2):  # capture both keys at both buffer parities
        S = sh.mapstencil_steps(rule, S, steps(m), graph=True, flags=sh._abi.ASYNC)
    t = {}
    for m in (m1, m2):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record(stream)
        S = sh.mapstencil_steps(rule, S, steps(m), graph=True, flags=sh._abi.ASYNC)
        e1.record(stream)
        torch.cuda.synchronize()
        t[m] = e0.elapsed_time(e1) * 1e3  # us
    return S, (t[m2] - t[m1]) / ((m2 - m1) * 32)


def profiled_traffic(name: str):
    """HBM bytes per launch from the committed rocprofv3 counter summary
    (FETCH_SIZE and WRITE_SIZE runs, calibrated against a copy kernel)."""
    p = REPO / "profiles" / name
    if not p.exists():
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*(\d+)", p.read_text(), re.M)
    return int(m.group(1)) if m else None


def cpu_baseline(A: np.ndarray, target_s: float = 10.0):
    """The oracle (plain-C restatement of the reference) on all host cores,
    on a bounded number of generations of the same grid."""
    import oracle
    import stencils_hip as sh
    cores = oracle.host_cores()
    S = sh.SwitchingStencilArray(np.asfortranarray(A), sh.Moore(1), boundary=sh.Wrap(),
                                 padding=sh.Halo())
    t0 = time.perf_counter()
    S = oracle.mapstencil_steps(sh.LifeRule(), S, 1, nthreads=cores)
    t1 = time.perf_counter() - t0
    steps = int(max(2, min(200, target_s / max(t1, 1e-3))))
    t0 = time.perf_counter()
    oracle.mapstencil_steps(sh.LifeRule(), S, steps, nthreads=cores)
    dt = time.perf_counter() - t0
    cells = A.size * steps
    return {"value": cells / dt, "unit": "cells/s", "cores": cores, "kind": "port",
            "sample": f"{steps} generations of the same {A.shape[0]}x{A.shape[1]} grid "
                      f"({dt:.1f} s, oracle/stencil_oracle.c on {cores} threads)"}


def graph_time(torch, fn, reps: int, inner: int = 10):
    """GPU time per call of `fn` (which only enqueues work on the current
    stream), from a captured torch CUDA graph of `inner` calls replayed
    `reps` times; returns seconds per call."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()  # warm the library's kernel selection outside capture
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(inner):
            fn()
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        g.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / 1e3 / (reps * inner)


def bench_mean_blur(sh, torch, oracle_ok: bool):
    """mapstencil(mean, StencilArray(A, Window(1); Remove(0.0), Conditional)),
    A 1000x1000 Float64 uniform[0,1) (PCG64 seed 1): the README benchmark."""
    rng = np.random.Generator(np.random.PCG64(1))
    A = rng.random((1000, 1000))
    dev = torch.device("cuda", torch.cuda.current_device())
    t = sh.colmajor_empty(A.shape, torch.float64, dev)
    t.copy_(torch.from_numpy(np.ascontiguousarray(A)).to(dev))
    sa = sh.StencilArray(t, sh.Window(1), boundary=sh.Remove(0.0))
    dest = sh.colmajor_empty(A.shape, torch.float64, dev)
    per_call = graph_time(torch, lambda: sh.mapstencil_(sh.mean, dest, sa, flags=sh._abi.ASYNC), 20)
    # end-to-end call from Python (descriptor build, launch, synchronise)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    n = 200
    for _ in range(n):
        sh.mapstencil(sh.mean, sa)
    torch.cuda.synchronize()
    e2e = (time.perf_counter() - t0) / n
    cells = A.size
    out = {"workload": "mean blur 1000x1000 Float64, Window(1), Remove(0.0), Conditional",
           "kernel_us": per_call * 1e6, "cells_per_s": cells / per_call,
           "gbs": 16 * cells / per_call / 1e9, "call_us_python": e2e * 1e6,
           "reference_published_ms": 2.755}
    # the same call at 16384^2 (PCG64 seed 11), where bandwidth, not launch
    # latency, bounds it
    big = 16384
    tb = sh.colmajor_empty((big, big), torch.float64, dev)
    tb.copy_(torch.from_numpy(np.random.Generator(np.random.PCG64(11)).random((big, big))).to(dev).T)
    sb = sh.StencilArray(tb, sh.Window(1), boundary=sh.Remove(0.0))
    db = sh.colmajor_empty((big, big), torch.float64, dev)
    big_call = graph_time(torch, lambda: sh.mapstencil_(sh.mean, db, sb, flags=sh._abi.ASYNC), 5)
    out["large"] = {"workload": f"mean blur {big}x{big} Float64, Window(1), Remove(0.0), Conditional",
                    "kernel_us": big_call * 1e6, "cells_per_s": big * big / big_call,
                    "gbs": 16 * big * big / big_call / 1e9,
                    "frac_of_peak": 16 * big * big / big_call / 1e9 / HBM_PEAK_GBS}
    del tb, sb, db
    if oracle_ok:
        import oracle
        B = np.asfortranarray(A)
        t0 = time.perf_counter()
        reps = 20
        for _ in range(reps):
            oracle.mapstencil(sh.mean, sh.StencilArray(B, sh.Window(1), boundary=sh.Remove(0.0)),
                              nthreads=oracle.host_cores())
        out["cpu_oracle_ms"] = (time.perf_counter() - t0) / reps * 1e3
    return out


def bench_multi(sh, torch, n: int = 8192):
    """Multi-array gather (sth_map_multi) on n x n Float32 fields, uniform
    [0,1) (PCG64 seed 6): heat with a source, one step of
    mapstencil!(Terms(Laplacian(0.2), Scaled(0.05, center)), S, Q) with S a
    SwitchingStencilArray (VonNeumann(1), Wrap, Conditional) and Q a plain
    array (12 B/cell: two reads, one write); and three StencilArrays
    (Window(1) mean, Moore(1) maximum, VonNeumann(2) sum; Remove(0f0)) summed
    (16 B/cell)."""
    rng = np.random.Generator(np.random.PCG64(6))
    dev = torch.device("cuda", torch.cuda.current_device())

    def field():
        t = sh.colmajor_empty((n, n), torch.float32, dev)
        t.copy_(torch.from_numpy(rng.random((n, n), dtype=np.float32)).to(dev).T)
        return t

    def timed(fn, reps=20):
        fn()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / 1e3 / reps

    U, Q = field(), field()
    S = [sh.SwitchingStencilArray(U, sh.VonNeumann(1), boundary=sh.Wrap())]
    f = sh.Terms(sh.Laplacian(0.2), sh.Scaled(float(np.float32(0.05)), sh.center))

    def step():
        S[0] = sh.mapstencil_(f, S[0], Q, flags=sh._abi.ASYNC)
    t_heat = timed(step)
    A, B, C = field(), field(), field()
    z = sh.Remove(np.float32(0))
    args = (sh.StencilArray(A, sh.Window(1), boundary=z), sh.StencilArray(B, sh.Moore(1), boundary=z),
            sh.StencilArray(C, sh.VonNeumann(2), boundary=z))
    g = sh.Terms(sh.mean, sh.maximum, sh.sum)
    out = sh.colmajor_empty((n, n), torch.float32, dev)
    t_three = timed(lambda: sh.mapstencil_(g, out, *args, flags=sh._abi.ASYNC))
    t_passes = timed(lambda: sh.mapstencil_(g, out, *args, flags=sh._abi.ASYNC | sh._abi.NO_FUSE))
    cells = n * n
    return {"workload": f"coupled fields {n}x{n} Float32: heat with a source (Laplacian(0.2) + 0.05 * source), "
                        "and three StencilArrays (mean + maximum + sum)",
            "heat_source_us": t_heat * 1e6, "heat_source_gbs": 12 * cells / t_heat / 1e9,
            "three_arrays_us": t_three * 1e6, "three_arrays_gbs": 16 * cells / t_three / 1e9,
            "three_arrays_one_pass_per_argument_us": t_passes * 1e6,
            "three_arrays_fused_speedup": t_passes / t_three}


def bench_scatter(sh, torch, n: int = 8192, oracle_ok: bool = False):
    """scatterstencil! (sth_scatter) on n x n Float64 fields (PCG64 seed 7):
    water flowing downhill, Scatter.downhill_flow(0.1) with + over Moore(1),
    Remove(0.0) (and the same under Wrap and Reflect), the elevation a second
    StencilArray; dest accumulates (it is read and written).  Algorithmic
    bytes: water, elevation and dest read, dest written (32 B/cell)."""
    rng = np.random.Generator(np.random.PCG64(7))
    dev = torch.device("cuda", torch.cuda.current_device())

    def field(scale):
        t = sh.colmajor_empty((n, n), torch.float64, dev)
        t.copy_(torch.from_numpy(rng.random((n, n)) * scale).to(dev).T)
        return t

    water, dem, dest = field(1.0), field(10.0), field(0.0)
    f = sh.Scatter.downhill_flow(0.1)

    def timed(bc, reps=10):
        w = sh.StencilArray(water, sh.Moore(1), boundary=bc)
        z = sh.StencilArray(dem, sh.Moore(1), boundary=bc)

        def run():
            sh.scatterstencil_(f, "+", dest, w, z, flags=sh._abi.ASYNC)
        run()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            run()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / 1e3 / reps

    cells = n * n
    t = timed(sh.Remove(0.0))
    out = {"workload": f"scatter {n}x{n} Float64: downhill flow 0.1, +, Moore(1), Remove(0.0), elevation field",
           "kernel_us": t * 1e6, "cells_per_s": cells / t, "gbs": 32 * cells / t / 1e9}
    for name, bc in (("wrap", sh.Wrap()), ("reflect", sh.Reflect())):
        tb = timed(bc)
        out[f"{name}_kernel_us"] = tb * 1e6
    if oracle_ok:
        import oracle
        m = 1024  # a bounded sample: the reference's loop on one thread
        A = np.asfortranarray(rng.random((m, m)))
        B = np.asfortranarray(rng.random((m, m)) * 10)
        D = np.zeros((m, m), order="F")
        t0 = time.perf_counter()
        oracle.scatterstencil(f, "+", D, sh.StencilArray(A, sh.Moore(1), boundary=sh.Remove(0.0)),
                              sh.StencilArray(B, sh.Moore(1), boundary=sh.Remove(0.0)))
        out["cpu_oracle_cells_per_s_1_thread"] = m * m / (time.perf_counter() - t0)
    return out


def bench_runtime(sh, torch, n: int = 8192):
    """The runtime-offset tile kernel (user offset lists and integer folds) on
    n x n arrays (PCG64 seed 9), one gatherstencil! per call, against the
    catalogue streaming kernel on the same size: Float32 sum over a
    six-offset Positional stencil (Wrap), Int64 sum over Moore(1)
    (Remove(0)), UInt8 maximum over Moore(2) (Wrap), and the catalogue
    Float32 sum over Moore(1) (Wrap).  Algorithmic bytes: one read and one
    write of the element type per cell."""
    rng = np.random.Generator(np.random.PCG64(9))
    dev = torch.device("cuda", torch.cuda.current_device())
    cases = [
        ("f32 sum Positional((-2,0),(0,-1),(0,0),(1,1),(2,-2),(-1,2)) Wrap", torch.float32,
         sh.Positional((-2, 0), (0, -1), (0, 0), (1, 1), (2, -2), (-1, 2)), sh.Wrap(), sh.sum),
        ("i64 sum Moore(1) Remove(0)", torch.int64, sh.Moore(1), sh.Remove(np.int64(0)), sh.sum),
        ("u8 maximum Moore(2) Wrap", torch.uint8, sh.Moore(2), sh.Wrap(), sh.maximum),
        ("f32 sum Moore(1) Wrap (catalogue streaming kernel)", torch.float32, sh.Moore(1), sh.Wrap(), sh.sum),
    ]
    out = {"workload": f"runtime-offset tile kernel, {n}x{n}", "cases": {}}
    for name, dt, st, bc, fold in cases:
        t = sh.colmajor_empty((n, n), dt, dev)
        if dt.is_floating_point:
            t.copy_(torch.from_numpy(rng.random((n, n), dtype=np.float32)).to(dev).T)
        else:
            t.copy_(torch.from_numpy(rng.integers(0, 100, (n, n))).to(dt).to(dev).T)
        sa = sh.StencilArray(t, st, boundary=bc)
        dest = sh.colmajor_empty((n, n), dt, dev)
        per_call = graph_time(torch, lambda: sh.mapstencil_(fold, dest, sa, flags=sh._abi.ASYNC), 10)
        es = torch.empty((), dtype=dt).element_size()
        out["cases"][name] = {"kernel_us": per_call * 1e6, "gbs": 2 * es * n * n / per_call / 1e9}
        del t, dest, sa
    out["tuning"] = sh._lib.tuning_table()
    return out


def bench_iterate_batch(sh, torch, n: int = 64, seed: int = 8):
    """Many iterations with uneven step counts: n Float32 SwitchingStencilArrays
    (sides log-uniform 64..1024, aspect 0.5..2, PCG64 seed 8) of 2-D heat,
    Laplacian(0.2) over VonNeumann(1) under Wrap, each iterated U{10..200}
    steps.  Three ways: the reference's loop (one mapstencil! per array and
    step), one sth_iterate per array (its steps graph-replayed), and one
    sth_iterate_batch call (all arrays advance together, one launch per round;
    its schedule graph-replayed).  Wall time with synchronisation, inputs
    resident; the graphs are captured in a warm-up call."""
    rng = np.random.Generator(np.random.PCG64(seed))
    dev = torch.device("cuda", torch.cuda.current_device())
    f = sh.Laplacian(0.2)
    arrays, steps, cells = [], [], 0
    for _ in range(n):
        side = float(np.exp(rng.uniform(np.log(64), np.log(1024))))
        asp = rng.uniform(0.5, 2.0)
        shape = (max(8, int(side * np.sqrt(asp))), max(8, int(side / np.sqrt(asp))))
        t = sh.colmajor_empty(shape, torch.float32, dev)
        t.copy_(torch.from_numpy(rng.random(shape, dtype=np.float32)).to(dev))
        arrays.append(sh.SwitchingStencilArray(t, sh.VonNeumann(1), boundary=sh.Wrap()))
        k = int(rng.integers(10, 201))
        steps.append(k)
        cells += shape[0] * shape[1] * k

    def wall(fn, reps=3):
        fn()
        torch.cuda.synchronize()
        best = float("inf")
        for _ in range(reps):
            t0 = time.perf_counter()
            fn()
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best

    def loop_steps():
        for i, A in enumerate(arrays):
            for _ in range(steps[i]):
                A = sh.mapstencil_(f, A, flags=sh._abi.ASYNC)
            arrays[i] = A

    def loop_iterate():
        for i, A in enumerate(arrays):
            arrays[i] = sh.mapstencil_steps(f, A, steps[i], graph=True, flags=sh._abi.ASYNC)

    def batched():
        res = sh.mapstencil_steps_batch([(f, A, k) for A, k in zip(arrays, steps)], graph=True,
                                        flags=sh._abi.ASYNC)
        arrays[:] = res

    t_loop = wall(loop_steps, reps=1)
    t_iter = wall(loop_iterate)
    t_batch = wall(batched)
    return {"workload": f"{n} uneven Float32 2-D heat arrays (sides 64..1024), Laplacian(0.2), VonNeumann(1), "
                        "Wrap, U{10..200} steps each",
            "cell_steps": cells, "max_steps": max(steps),
            "reference_loop_ms": t_loop * 1e3, "per_array_iterate_ms": t_iter * 1e3,
            "iterate_batch_ms": t_batch * 1e3, "cell_steps_per_s": cells / t_batch,
            "speedup_vs_reference_loop": t_loop / t_batch, "speedup_vs_per_array_iterate": t_iter / t_batch}


def gaussian_weights(sigma: float = 1.5, R: int = 3) -> np.ndarray:
    a = np.arange(-R, R + 1)
    W = np.exp(-(a[:, None] ** 2 + a[None, :] ** 2) / (2 * sigma ** 2))
    return W / W.sum()


def bench_gaussian(sh, torch, n: int = 16384):
    """Kernel(Window(3)) 7x7 Gaussian (sigma 1.5) over n x n uniform[0,1)
    (PCG64 seed 3), Reflect, Halo: Float32, then BF16 storage with f32
    accumulation; errors against an FP64 evaluation on two 512x512 crops."""
    import scipy.ndimage as ndi
    rng = np.random.Generator(np.random.PCG64(3))
    A = rng.random((n, n), dtype=np.float32)
    W = gaussian_weights()
    dev = torch.device("cuda", torch.cuda.current_device())
    res = {"workload": f"gaussian 7x7 sigma=1.5 {n}x{n}, Reflect, Halo"}
    crops = [(slice(4000, 4512), slice(9000, 9512)), (slice(0, 509), slice(0, 509))]
    ref = []
    A64 = A.astype(np.float64)
    for cx, cy in crops:
        lo0, lo1 = max(cx.start - 3, 0), max(cy.start - 3, 0)
        sub = A64[lo0:cx.stop + 3, lo1:cy.stop + 3]
        full = ndi.correlate(sub, W, mode="mirror")
        ref.append(full[cx.start - lo0:cx.start - lo0 + (cx.stop - cx.start),
                        cy.start - lo1:cy.start - lo1 + (cy.stop - cy.start)])
    for name, tdt in (("f32", torch.float32), ("bf16", torch.bfloat16)):
        src = sh.colmajor_empty((n, n), tdt, dev)
        src.copy_(torch.from_numpy(A).to(dev).to(tdt))
        K = sh.Kernel(sh.Window(3), W.astype(np.float32))
        sa = sh.StencilArray(src, K, boundary=sh.Reflect(), padding=sh.Halo())
        del src
        dest = sh.colmajor_empty((n, n), tdt, dev)
        per = graph_time(torch, lambda: sh.mapstencil_(sh.kernelproduct, dest, sa, flags=sh._abi.ASYNC),
                         3, inner=5)
        esz = 4 if name == "f32" else 2
        errs = []
        for (cx, cy), r in zip(crops, ref):
            g = dest[cx, cy].float().cpu().numpy().astype(np.float64)
            errs.append((np.abs(g - r).max(), (np.abs(g - r) / np.abs(r)).max()))
        res[name] = {"kernel_us": per * 1e6, "cells_per_s": n * n / per,
                     "gbs": 2 * esz * n * n / per / 1e9,
                     "max_abs_err_vs_fp64": max(e[0] for e in errs),
                     "max_rel_err_vs_fp64": max(e[1] for e in errs)}
        del sa, dest
        torch.cuda.empty_cache()
    return res


def batched_workload(sh, torch, n: int = 512, seed: int = 4):
    """512 Float32 arrays, side s log-uniform in [64, 4096], aspect a in
    [0.5, 2] (shape (s, round(s a))), each with a uniform choice of
    {Window(1), Circle(3), VonNeumann(2)} x {sum, maximum, mean},
    Remove(0f0), Conditional; data uniform[0,1) from a seeded device RNG."""
    rng = np.random.Generator(np.random.PCG64(seed))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dev = torch.device("cuda", torch.cuda.current_device())
    shapes = [sh.Window(1), sh.Circle(3), sh.VonNeumann(2)]
    fs = [sh.sum, sh.maximum, sh.mean]
    calls = []
    for _ in range(n):
        s = int(round(np.exp(rng.uniform(np.log(64), np.log(4096)))))
        a = rng.uniform(0.5, 2.0)
        shape = (s, max(8, int(round(s * a))))
        st = shapes[int(rng.integers(3))]
        f = fs[int(rng.integers(3))]
        t = sh.colmajor_empty(shape, torch.float32, dev)
        t.copy_(torch.rand(shape[::-1], generator=gen, device=dev).T)
        sa = sh.StencilArray(t, st, boundary=sh.Remove(np.float32(0)))
        calls.append((f, sh.colmajor_empty(shape, torch.float32, dev), sa))
    return calls


def bench_batched(sh, torch):
    """Config 4: sth_map_batch (one launch per type, shape and op) against one
    launch per array: asynchronous from C, asynchronous from Python, and one
    blocking call per array."""
    calls = batched_workload(sh, torch)
    plan = sh.BatchPlan(calls)
    cells = plan.cells

    def timed(fn, reps):
        fn()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0 = time.perf_counter()
        e0.record()
        for _ in range(reps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / reps, e0.elapsed_time(e1) / 1e3 / reps

    wall_b, gpu_b = timed(lambda: plan.run(flags=sh._abi.ASYNC), 5)
    wall_s, gpu_s = timed(lambda: plan.run(serial=True, flags=sh._abi.ASYNC), 5)

    def python_loop():
        for f, d, sa in calls:
            sh.mapstencil_(f, d, sa, flags=sh._abi.ASYNC)
    wall_p, gpu_p = timed(python_loop, 2)

    # One blocking sth_map call per array, descriptors prebuilt: the
    # reference's per-array mapstencil loop, where every call synchronises
    # (src/gatherstencil.jl:100), without Python-side descriptor building.
    L = sh._lib.lib()
    ctx = sh._lib.context(torch.cuda.current_device())
    strm = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def blocking_loop():
        for i in range(plan.n):
            j = plan.jobs[i]
            sh._lib.check(L.sth_map(ctx, ctypes.byref(j.src), ctypes.byref(j.dst), ctypes.byref(j.stencil),
                                    j.boundary, j.padval, j.padding, ctypes.byref(j.op), 0, strm))
    wall_k, _ = timed(blocking_loop, 2)
    # spot check: the batched results equal single calls
    plan.run()
    for f, d, sa in calls[:8]:
        assert torch.equal(d, sh.mapstencil(f, sa)), "batched result differs from a single call"
    return {"workload": "512 uneven Float32 arrays (sides log-uniform 64..4096, aspect 0.5..2), "
                        "Window(1)/Circle(3)/VonNeumann(2) x sum/maximum/mean, Remove(0f0), Conditional",
            "cells": cells, "bytes": 8 * cells,
            "batched": {"ms": wall_b * 1e3, "gpu_ms": gpu_b * 1e3, "cells_per_s": cells / wall_b,
                        "gbs": 8 * cells / gpu_b / 1e9},
            "per_array_launches_c": {"ms": wall_s * 1e3, "gpu_ms": gpu_s * 1e3,
                                     "cells_per_s": cells / wall_s},
            "per_array_python_loop": {"ms": wall_p * 1e3, "cells_per_s": cells / wall_p},
            "per_array_blocking_calls": {"ms": wall_k * 1e3, "cells_per_s": cells / wall_k},
            "speedup_vs_c_loop": wall_s / wall_b, "speedup_vs_python_loop": wall_p / wall_b,
            "speedup_vs_blocking_calls": wall_k / wall_b}


def served_requests(sh, torch, n: int, tdt, seed: int = 5, rate: float = 200.0):
    """Poisson stream (rate/s) of 3-D heat solves: Float32 cube, side uniform
    in {32..256}, steps uniform in {10..1000}, uniform[0,1) state,
    VonNeumann(1,3) Laplacian(0.15), Wrap, Conditional (seed 5)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    dev = torch.device("cuda", torch.cuda.current_device())
    t = 0.0
    out = []
    for _ in range(n):
        t += float(rng.exponential(1.0 / rate))
        side = int(rng.integers(32, 257))
        steps = int(rng.integers(10, 1001))
        g = torch.Generator(device=dev).manual_seed(int(rng.integers(1 << 31)))
        A = sh.colmajor_empty((side,) * 3, tdt, dev)
        A.copy_(torch.rand((side,) * 3, generator=g, device=dev).to(tdt))
        out.append((sh.SwitchingStencilArray(A, sh.VonNeumann(1, 3), boundary=sh.Wrap()), steps, t))
    return out


def bench_served(sh, torch, n: int = 120, budget: int = 2 << 30):
    """Config 5: the request stream through the continuous-batching server
    (FP32 and BF16 storage) and through the one-request-at-a-time path with
    one plain launch per step; latency p50/p99, throughput, and each
    result's error against the same request run in Float64."""
    f = sh.Laplacian(0.15)
    res = {"workload": f"Poisson 200 req/s x {n} requests, 3-D heat VonNeumann(1,3) Laplacian(0.15), "
                       f"Wrap, cube side U{{32..256}}, steps U{{10..1000}}; HBM budget {budget >> 20} MiB"}

    def run(reqs, serial):
        srv = sh.Server(hbm_budget=budget, round_steps=8, serial=serial)
        tags = {}
        for S, steps, arr in reqs:
            tags[srv.submit(f, S, steps, arrival=arr)] = (S, steps)
        torch.cuda.synchronize()
        srv.start()
        srv.drain(timeout=600)
        done = srv.completions()
        st = srv.stats()
        srv.close()
        summ = sh.serve_latency_summary(done)
        summ.update({"hbm_peak_mib": st["hbm_peak"] / 2**20, "rounds": st["rounds"],
                     "launches": st["launches"], "gbs": summ["cell_steps_per_s"] * 8 / 1e9})
        return done, tags, summ

    for name, tdt in (("f32", torch.float32), ("bf16", torch.bfloat16)):
        reqs = served_requests(sh, torch, n, tdt)
        done, tags, summ = run(reqs, False)
        if name == "bf16":
            summ["gbs"] = summ["cell_steps_per_s"] * 4 / 1e9
        # FP64 reference of every request: the same steps from the same initial values
        errs = []
        for c in done:
            S, steps = tags[c.tag]
            a = sh.colmajor_empty(S.size(), torch.float64, S.source.device)
            a.copy_(S.source.to(torch.float64))
            b = sh.colmajor_empty(S.size(), torch.float64, S.source.device)
            R = sh.mapstencil_steps(f, sh.SwitchingStencilArray(
                stencil=S.stencil, boundary=S.boundary, padding=S.padding, _buffers=(a, b)), steps)
            d = (c.result.to(torch.float64) - R.source).abs()
            errs.append((float(d.max()), float((d / R.source.abs().clamp_min(1e-300)).max())))
            del a, b, R, d
        summ["max_abs_err_vs_fp64"] = max(e[0] for e in errs)
        summ["max_rel_err_vs_fp64"] = max(e[1] for e in errs)
        summ["median_abs_err_vs_fp64"] = float(np.median([e[0] for e in errs]))
        res[name] = summ
        if name == "f32":
            _, _, ser = run(reqs, True)
            res["f32_serial_plain_launches"] = ser
            res["served_vs_serial"] = {"throughput": summ["cell_steps_per_s"] / ser["cell_steps_per_s"],
                                       "p50_latency": ser["p50_s"] / summ["p50_s"],
                                       "p99_latency": ser["p99_s"] / summ["p99_s"]}
            # capacity: the same requests all arriving at t = 0, so both paths
            # are saturated and throughput measures the device, not the arrivals
            burst = [(S, steps, 0.0) for S, steps, _ in reqs]
            _, _, cap = run(burst, False)
            _, _, cap_ser = run(burst, True)
            res["f32_burst_capacity"] = {
                "served_cell_steps_per_s": cap["cell_steps_per_s"],
                "serial_plain_cell_steps_per_s": cap_ser["cell_steps_per_s"],
                "throughput_ratio": cap["cell_steps_per_s"] / cap_ser["cell_steps_per_s"],
                "served_span_s": cap["span_s"], "serial_span_s": cap_ser["span_s"]}
        del reqs, done, tags
        torch.cuda.empty_cache()
    return res


def bench_heat_iterate(sh, torch, n: int = 512, steps: int = 200):
    """3-D heat iteration (VonNeumann(1,3) Laplacian(0.15), Wrap, n^3) as
    `steps` hipGraph-replayed steps: several steps per launch (zmarch_kernel or zmarch2_kernel)
    against one streaming step per launch (STH_NO_FUSE).  The achieved rates
    count every step's algorithmic bytes."""
    f = sh.Laplacian(0.15)
    dev = torch.device("cuda", torch.cuda.current_device())
    stream = torch.cuda.current_stream()
    res = {"workload": f"heat {n}^3 VonNeumann(1,3) Laplacian(0.15) Wrap, {steps} steps, hipGraph"}
    for name, tdt in (("f32", torch.float32), ("bf16", torch.bfloat16), ("f64", torch.float64)):
        A = sh.colmajor_empty((n,) * 3, tdt, dev)
        A.copy_(torch.rand((n,) * 3, device=dev).to(tdt))
        S = sh.SwitchingStencilArray(A, sh.VonNeumann(1, 3), boundary=sh.Wrap())
        t = {}
        for key, fl in (("multi_step", 0), ("one_step", sh._abi.NO_FUSE)):
            S = sh.mapstencil_steps(f, S, 8, flags=sh._abi.ASYNC | fl)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            e0.record(stream)
            S = sh.mapstencil_steps(f, S, steps, flags=sh._abi.ASYNC | fl)
            e1.record(stream)
            torch.cuda.synchronize()
            t[key] = e0.elapsed_time(e1) / steps * 1e3  # us per step
        es = A.element_size()
        cells = n ** 3
        res[name] = {"multi_step_us_per_step": t["multi_step"], "one_step_us_per_step": t["one_step"],
                     "speedup": t["one_step"] / t["multi_step"],
                     "cell_steps_per_s": cells / (t["multi_step"] * 1e-6),
                     "multi_step_achieved_gbs": 2 * es * cells / (t["multi_step"] * 1e-6) / 1e9,
                     "one_step_achieved_gbs": 2 * es * cells / (t["one_step"] * 1e-6) / 1e9}
        if name == "f32" and n == 512:
            # (the profile is of a launch of four steps)
            traffic = profiled_traffic("zmarch_kernel_heat_512.md")
            res[name]["multi_step_traffic_per_step"] = traffic and traffic // 4
            res[name]["one_step_traffic"] = profiled_traffic("zmarch1_kernel_heat_512.md")
        del A, S
        torch.cuda.empty_cache()
    return res


def bench_life_only(sh, torch, steps: int, n: int = 8192):
    """The headline Game of Life leg alone (for profiling): `steps`
    graph-replayed generations after an untimed pass that captures the
    graphs, then one 256 MiB device-to-device copy whose HBM counters
    calibrate FETCH_SIZE / WRITE_SIZE."""
    A = life_grid(n)
    rule = sh.LifeRule()
    S = device_switching(A, sh, torch)
    S, _, _ = time_steps(sh, torch, S, rule, steps, graph=True)
    S, wall, ev = time_steps(sh, torch, S, rule, steps, graph=True)
    src = torch.empty(256 << 20, dtype=torch.uint8, device="cuda").fill_(1)
    dst = torch.empty_like(src)
    dst.copy_(src)
    torch.cuda.synchronize()
    return {"workload": f"game-of-life {n}x{n}, {steps} generations, hipGraph", "gens_per_launch": LIFE_GENS,
            "us_per_generation": ev / steps * 1e6, "cells_per_s": n * n * steps / wall,
            "calibration_copy_bytes": 256 << 20}


def bench_heat3d_step(sh, torch, n: int = 512, reps: int = 10):
    """One step of the 3-D heat stencil (VonNeumann(1,3) Laplacian(0.15),
    Wrap) on n^3, Float32, BF16 and Float64, as `reps` single
    gatherstencil! calls with the tuned kernel (for profiling the one-step
    body)."""
    f = sh.Laplacian(0.15)
    dev = torch.device("cuda", torch.cuda.current_device())
    res = {"workload": f"heat {n}^3 one step, VonNeumann(1,3) Laplacian(0.15) Wrap"}
    for name, tdt in (("f32", torch.float32), ("bf16", torch.bfloat16), ("f64", torch.float64)):
        A = sh.colmajor_empty((n,) * 3, tdt, dev)
        A.copy_(torch.rand((n,) * 3, device=dev).to(tdt))
        sa = sh.StencilArray(A, sh.VonNeumann(1, 3), boundary=sh.Wrap())
        dest = sh.colmajor_empty((n,) * 3, tdt, dev)
        kernel = sh.autotune(f, dest, sa)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for _ in range(reps):
            sh.mapstencil_(f, dest, sa, flags=sh._abi.ASYNC)
        e1.record()
        torch.cuda.synchronize()
        us = e0.elapsed_time(e1) / reps * 1e3
        es = A.element_size()
        res[name] = {"kernel": kernel, "us": us, "achieved_gbs": 2 * es * n ** 3 / (us * 1e-6) / 1e9}
        del A, dest, sa
        torch.cuda.empty_cache()
    return res


def bench_heat_iterate_2d(sh, torch, steps: int = 100):
    """2-D heat iteration (VonNeumann(1) Laplacian(0.2), Wrap) as `steps`
    hipGraph-replayed steps: several steps per launch (ymarch_kernel) against one
    streaming step per launch (STH_NO_FUSE); f32 and bf16 on 16384^2, f64 on
    8192^2 (a 16384^2 f64 grid is past the multi-step kernel's 2 GiB offsets)."""
    f = sh.Laplacian(0.2)
    dev = torch.device("cuda", torch.cuda.current_device())
    stream = torch.cuda.current_stream()
    res = {"workload": f"heat 2-D VonNeumann(1) Laplacian(0.2) Wrap, {steps} steps, hipGraph"}
    for name, tdt, n in (("f32", torch.float32, 16384), ("bf16", torch.bfloat16, 16384),
                         ("f64", torch.float64, 8192)):
        A = sh.colmajor_empty((n, n), tdt, dev)
        A.copy_(torch.rand((n, n), device=dev).to(tdt))
        S = sh.SwitchingStencilArray(A, sh.VonNeumann(1), boundary=sh.Wrap())
        t = {}
        for key, fl in (("multi_step", 0), ("one_step", sh._abi.NO_FUSE)):
            S = sh.mapstencil_steps(f, S, 8, flags=sh._abi.ASYNC | fl)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            e0.record(stream)
            S = sh.mapstencil_steps(f, S, steps, flags=sh._abi.ASYNC | fl)
            e1.record(stream)
            torch.cuda.synchronize()
            t[key] = e0.elapsed_time(e1) / steps * 1e3
        es = A.element_size()
        res[name] = {"n": n, "multi_step_us_per_step": t["multi_step"], "one_step_us_per_step": t["one_step"],
                     "speedup": t["one_step"] / t["multi_step"],
                     "multi_step_achieved_gbs": 2 * es * n * n / (t["multi_step"] * 1e-6) / 1e9,
                     "one_step_achieved_gbs": 2 * es * n * n / (t["one_step"] * 1e-6) / 1e9}
        if name == "f32":
            # (the profile is of a launch of eight steps)
            traffic = profiled_traffic("ymarch_kernel_heat2d_16384.md")
            res[name]["multi_step_traffic_per_step"] = traffic and traffic // 8
        del A, S
        torch.cuda.empty_cache()
    return res


def result_line(out: dict) -> dict:
    """The headline with its roofline, the plain paths beside it, and the
    batched and served workloads' figures."""
    line = {k: v for k, v in out.items() if k not in ("cpu_baseline", "configs", "single_generation_kernel")}
    line["config"] = {"workload": "game-of-life 8192x8192 UInt8, Moore(1), Wrap, Halo, B3/S23, all steps in one "
                                  "sth_iterate call", "cells": out["config"]["cells"], "step": "one generation"}
    line["roofline"] = {k: out["roofline"][k] for k in ("bound", "achieved", "peak", "unit", "frac", "traffic",
                                                        "bytes_per_launch", "avg_launch_us", "stream_copy_gbs")}
    line["roofline"]["note"] = "algorithmic bytes; several generations per launch, so frac may exceed 1"
    line["plain_per_step"] = {"value": out["plain_per_step"]["value"], "unit": "cells/s"}
    if "cpu_baseline" in out:
        line["cpu_baseline"] = {k: v for k, v in out["cpu_baseline"].items() if isinstance(v, (int, float))}
    if "configs" in out:
        b, v = out["configs"]["batched_uneven"], out["configs"]["served_heat_3d"]
        line["batched"] = {"cells_per_s": b["batched"]["cells_per_s"], "vs_c_loop": b["speedup_vs_c_loop"],
                           "vs_blocking_calls": b["speedup_vs_blocking_calls"]}
        line["served"] = {"cell_steps_per_s": v["f32"]["cell_steps_per_s"], "p50_ms": v["f32"]["p50_s"] * 1e3,
                          "p99_ms": v["f32"]["p99_s"] * 1e3,
                          "vs_plain": {k: v["served_vs_serial"][k] for k in ("throughput", "p99_latency")}}
    return line


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=1000)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--n", type=int, default=8192)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=10.0)
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the secondary workloads (mean blur, Gaussian)")
    ap.add_argument("--only", choices=["life", "heat3d-step", "heat3d", "heat2d", "served", "batched", "gaussian",
                                       "meanblur", "multi", "scatter", "runtime", "iterbatch"],
                    help="run one secondary workload alone and print its JSON (for profiling)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: --gpus {args.gpus} is not supported "
              "(the batched and served workloads shard without exchange; see DESIGN.md)",
              file=sys.stderr)
        sys.exit(2)

    import torch
    import stencils_hip as sh
    sh.load_library()
    torch.cuda.set_device(int(os.environ.get("LOCAL_RANK", 0)))
    if args.only:
        run_one = {"life": lambda: bench_life_only(sh, torch, args.steps),
                   "heat3d-step": lambda: bench_heat3d_step(sh, torch),
                   "heat3d": lambda: bench_heat_iterate(sh, torch, steps=args.steps),
                   "heat2d": lambda: bench_heat_iterate_2d(sh, torch),
                   "served": lambda: bench_served(sh, torch),
                   "batched": lambda: bench_batched(sh, torch),
                   "gaussian": lambda: bench_gaussian(sh, torch),
                   "meanblur": lambda: bench_mean_blur(sh, torch, False),
                   "multi": lambda: bench_multi(sh, torch),
                   "scatter": lambda: bench_scatter(sh, torch, oracle_ok=True),
                   "runtime": lambda: bench_runtime(sh, torch),
                   "iterbatch": lambda: bench_iterate_batch(sh, torch)}[args.only]
        print(json.dumps({args.only: run_one()}), flush=True)
        return

    n = args.n
    A = life_grid(n)
    rule = sh.LifeRule()
    cells = n * n

    S = device_switching(A, sh, torch)
    S, _, _ = time_steps(sh, torch, S, rule, args.warmup, graph=True)
    # The iteration engine captures a hipGraph per schedule the first time it
    # sees it; run the timed call's schedule once untimed (at both buffer
    # parities when the step count is odd) so the timed steps only replay.
    for _ in range(1 if args.steps % 2 == 0 else 2):
        S, _, _ = time_steps(sh, torch, S, rule, args.steps, graph=True)
    S, wall, ev = time_steps(sh, torch, S, rule, args.steps, graph=True)
    bytes_per_step = 2 * cells  # 1 B read + 1 B written per interior cell and generation
    gen_us = ev / args.steps * 1e6
    # The steady steps run lifep_kernel on packed bits (temporal blocking); the
    # roofline is that of LIFE_GENS generations, timed on their own.
    S, launch_us = fused_launch_us(sh, torch, S, rule, LIFE_GENS)
    bytes_per_launch = LIFE_GENS * bytes_per_step
    life_traffic = profiled_traffic("lifep_kernel_gol_8192.md")
    achieved = bytes_per_launch / (launch_us * 1e-6) / 1e9
    S, plain_launch_us = kernel_launch_us(sh, torch, S, rule)
    # measured stream-copy bandwidth on the same bytes (one read + one write)
    src_t = torch.empty(cells, dtype=torch.uint8, device="cuda").fill_(1)
    dst_t = torch.empty_like(src_t)
    for _ in range(5):
        dst_t.copy_(src_t)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(50):
        dst_t.copy_(src_t)
    e1.record()
    torch.cuda.synchronize()
    copy_gbs = 2 * cells / (e0.elapsed_time(e1) / 1e3 / 50) / 1e9
    del src_t, dst_t

    # the same steps as plain per-step launches (no graph, one generation each)
    S, _, _ = time_steps(sh, torch, S, rule, 10, graph=False, flags=sh._abi.NO_FUSE)
    S, wall_plain, _ = time_steps(sh, torch, S, rule, args.steps, graph=False, flags=sh._abi.NO_FUSE)

    out = {
        "metric": METRIC,
        "value": cells * args.steps / wall,
        "unit": "cells/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": wall / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u8",
        "data": "synthetic",
        "config": {"workload": f"game-of-life {n}x{n} UInt8 Bernoulli(0.3) seed 2, Moore(1), Wrap, "
                               "Halo, B3/S23; SwitchingStencilArray resident in HBM; all steps in one "
                               "sth_iterate call with STH_GRAPH (replayed as hipGraphs from 17 launches, "
                               "launched directly below)", "cells": cells, "step": "one generation"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS,
                     "traffic": life_traffic and life_traffic * LIFE_GENS // LIFE_PROFILED_GENS,
                     "kernel": f"lifep_kernel: {LIFE_GENS} generations of it (a launch runs up to 32), one bit "
                               "per cell",
                     "bytes_per_launch": bytes_per_launch, "avg_launch_us": launch_us,
                     "per_generation_us": gen_us,
                     "note": "algorithmic bytes count 2 B per cell and generation (temporal-blocking "
                             "savings excluded), so frac may exceed 1; traffic is the HBM bytes they move "
                             "(rocprofv3 FETCH_SIZE x2 + WRITE_SIZE, a quarter of a 32-generation launch)",
                     "stream_copy_gbs": copy_gbs},
        "single_generation_kernel": {
            "kernel": "life_kernel<KY tuned, B3/S23>: one generation per launch (graph steps without temporal blocking)",
            "avg_launch_us": plain_launch_us,
            "achieved_gbs": bytes_per_step / (plain_launch_us * 1e-6) / 1e9,
            "traffic": profiled_traffic("life_kernel_gol_8192.md")},
        "plain_per_step": {"value": cells * args.steps / wall_plain, "unit": "cells/s",
                           "ms_per_step": wall_plain / args.steps * 1e3,
                           "graph_speedup": wall_plain / wall},
    }
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline(A, args.cpu_seconds)
    if not args.no_configs:
        out["configs"] = {"mean_blur_f64": bench_mean_blur(sh, torch, not args.no_cpu_baseline),
                          "gaussian_7x7": bench_gaussian(sh, torch),
                          "batched_uneven": bench_batched(sh, torch),
                          "heat_3d_iterate": bench_heat_iterate(sh, torch),
                          "heat_2d_iterate": bench_heat_iterate_2d(sh, torch),
                          "served_heat_3d": bench_served(sh, torch),
                          "coupled_fields": bench_multi(sh, torch),
                          "scatter_downhill": bench_scatter(sh, torch),
                          "runtime_offsets": bench_runtime(sh, torch),
                          "iterate_batch_uneven": bench_iterate_batch(sh, torch)}
    # the measured workloads in full go to stderr; the result line stays short
    # enough to be read back from the end of a log
    print(json.dumps(out), file=sys.stderr, flush=True)
    print(json.dumps(result_line(out)), flush=True)


if __name__ == "__main__":
    main()
