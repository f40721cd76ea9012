"""Benchmark: QuickSampling nodes/s at 1000^2 TI, n=80, k=1.5 (continuous).

One step = one full QS realisation of the 1000x1000 simulation grid from the
1000x1000 log-normal GRF training image (1,000,000 path nodes), i.e. the
reference's timed path loop (src/qs.cpp:2153,2229-2235): neighbour search,
path waves on the MI355X scan, draws and writes. The TI spectra are built
before the timed region (inputs resident in HBM).

Prints one JSON line (rank 0). Single GPU only.
"""
import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
PROFILES = {"k_pencil1024": "profiles/k_pencil1024__qs_2d_continuous_1000.md",
            "k_flow_direct": "profiles/k_flow_direct__qs_2d_continuous_1000.md"}


def measured_bytes_per_node(kernel):
    """HBM bytes per node of `kernel` (calibrated FETCH_SIZE + WRITE_SIZE)
    from the committed rocprofv3 counter summary, or None."""
    try:
        with open(os.path.join(ROOT, PROFILES[kernel])) as fh:
            for line in fh:
                if line.startswith(f"hbm_bytes_per_node {kernel}:"):
                    f, w = line.split(":", 1)[1].split()
                    return float(f) + float(w)
    except OSError:
        pass
    return None


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--workload", type=int, default=2, choices=(1, 2, 3, 4),
                    help="2: the benchmark (1000^2 continuous); 1, 3, 4: the other parity workloads, timed "
                         "alone (path loop, loop roofline; no learned form, calibration or CPU leg)")
    ap.add_argument("--steps", type=int, default=1)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--size", type=int, default=1000, help="TI and simulation extent (default 1000)")
    ap.add_argument("--sim-size", type=int, default=0, help="simulation extent when smaller than the TI (profiling)")
    ap.add_argument("--copy-calib", action="store_true",
                    help="also run a plain 256 MiB device copy (HBM counter calibration under rocprofv3 --pmc)")
    ap.add_argument("--wave", type=int, default=256,
                    help="max path nodes per wave: the workload batches 256 path nodes per launch")
    ap.add_argument("--stage-every", type=int, default=32,
                    help="wave loop: HIP events around the stages of every k-th wave of the timed steps (1: every wave; "
                         "events cost ~1.5%% of the loop when recorded for every wave)")
    ap.add_argument("--graph-steps", type=int, default=1,
                    help="also time the step with each wave replayed as a captured HIP graph (0: skip)")
    ap.add_argument("--alt-wave", type=int, default=512,
                    help="also time one realisation with waves of at most this many nodes (0: skip)")
    ap.add_argument("--tune", action="append", default=[], metavar="KEY=VALUE",
                    help="scan-kernel launch parameter for the TIs of the run (qsmi_set_default_tuning)")
    ap.add_argument("--cpu-sample", type=int, default=-1,
                    help="path nodes of the CPU baseline sample (-1: four per thread, 0: skip)")
    ap.add_argument("--cpu-threads", type=int, default=0, help="CPU baseline threads (0: nproc)")
    ap.add_argument("--learned", type=int, default=1,
                    help="also measure the learned-proposal form (1) or not (0)")
    ap.add_argument("--lp-train-sets", type=int, default=8,
                    help="GRF TIs (seeds 200..) whose plain QS runs give training pairs")
    ap.add_argument("--lp-record", type=int, default=500,
                    help="simulation extent of each recording run (8 x 500^2 = 2M pairs)")
    ap.add_argument("--lp-steps", type=int, default=1000, help="Adam steps per TI per epoch")
    ap.add_argument("--lp-epochs", type=int, default=4)
    ap.add_argument("--lp-min-cover", type=float, default=0.35,
                    help="exact scan for nodes with a smaller fraction of neighbours on the key stencil")
    ap.add_argument("--calib-iters", type=int, default=4,
                    help="auto_qs calibration iterations on the same TI (0: skip the calibration leg)")
    ap.add_argument("--lp-audit", type=int, default=1,
                    help="1: audited 300x300 learned realisation for the recall figures (0: skip, for profiling)")
    return ap.parse_args()


def field_stats(a, b, dims):
    """How a realisation b reproduces a (same grid, dims in G2S order): the
    two-sample KS distance of the values, the variogram gamma(h) = mean((z(x
    + h) - z(x))^2) / 2 of log values at lags 1..32 along both axes (largest
    relative difference), and the connectivity of the cells above a's 90th
    percentile (4-connected clusters of scipy.ndimage.label): the share of
    those cells in the largest cluster and tau(h), the probability that two
    such cells h apart along either axis share a cluster."""
    from scipy import ndimage

    za = a.reshape(dims[1], dims[0]).astype(np.float64)
    zb = b.reshape(dims[1], dims[0]).astype(np.float64)
    sa, sb = np.sort(za.ravel()), np.sort(zb.ravel())
    grid = np.concatenate([sa, sb])
    ks = float(np.max(np.abs(np.searchsorted(sa, grid, side="right") / sa.size
                             - np.searchsorted(sb, grid, side="right") / sb.size)))
    lags = (1, 2, 4, 8, 16, 32)

    def vario(z):
        lz = np.log(np.maximum(z, 1e-30))
        return np.array([[0.5 * np.mean((lz[:, h:] - lz[:, :-h]) ** 2) for h in lags],
                         [0.5 * np.mean((lz[h:, :] - lz[:-h, :]) ** 2) for h in lags]])

    va, vb = vario(za), vario(zb)
    thr = np.quantile(za, 0.9)

    def conn(z):
        lab, nlab = ndimage.label(z > thr)
        sizes = np.bincount(lab.ravel())[1:]
        largest = float(sizes.max() / sizes.sum()) if nlab else 0.0
        tau = []
        for h in lags:
            same = both = 0
            for x0, x1 in ((lab[:, h:], lab[:, :-h]), (lab[h:, :], lab[:-h, :])):
                m = (x0 > 0) & (x1 > 0)
                both += int(m.sum())
                same += int((m & (x0 == x1)).sum())
            tau.append(same / max(both, 1))
        return largest, np.array(tau)

    la, ta = conn(za)
    lb, tb = conn(zb)
    return dict(ks=ks, variogram_lags=list(lags),
                variogram_max_rel_diff=float(np.max(np.abs(vb - va) / va)),
                connectivity_threshold="exact realisation's 90th percentile",
                largest_cluster_share=[la, lb], tau=[ta.round(4).tolist(), tb.round(4).tolist()],
                tau_max_abs_diff=float(np.max(np.abs(tb - ta))))


def learned_form(cfg, args, exact_ms, exact_sim=None):
    """Learned-proposal QS on the same workload: pairs recorded by plain QS on
    other seeded GRF TIs (range 20, exp), the encoders trained on the GPU,
    keys built for this TI, then one timed realisation (every 64th node and
    every node the encoders cannot see on the exact scan) and an audited
    300x300 realisation for the k-best recall of the proposals."""
    import g2s_amd
    from g2s_amd import lp as L
    from g2s_amd import synth

    t0 = time.time()
    sets = []
    for s in range(args.lp_train_sets):
        g = synth.grf(tuple(cfg["ti_dims"][::-1]), 20.0, seed=200 + s)
        ti_s, dims_s = synth.to_g2s(np.exp(g))
        ti_s = np.ascontiguousarray(ti_s[:, 0])
        r = args.lp_record
        _, _, st = g2s_amd.qs(ti_s, dims_s, np.full(r * r, np.nan, np.float32), (r, r), [0], cfg["n"], cfg["k"],
                              seed=300 + s, record=r * r)
        sets.append((ti_s, dims_s, st["pairs"]))
    t_rec = time.time() - t0
    net = L.LearnedProposal(seed=1)
    t0 = time.time()
    losses = []
    for e in range(args.lp_epochs):
        for i, (ti_s, dims_s, pairs) in enumerate(sets):
            losses.append(net.train(ti_s, dims_s, pairs, steps=args.lp_steps,
                                    lr=(1e-3, 3e-4, 1e-4, 5e-5)[min(e, 3)], seed=100 * e + i))
    t_train = time.time() - t0
    print(f"[bench] learned: {len(sets)} x {args.lp_record}^2 pair sets in {t_rec:.1f}s, training {t_train:.1f}s, "
          f"loss {losses[0][0]:.3f} -> {losses[-1][-1]:.3f}", file=sys.stderr, flush=True)
    ti = np.ascontiguousarray(cfg["ti"][:, 0])
    dims, sdims = cfg["ti_dims"], cfg["sim_dims"]
    net.build_keys(ti, dims)
    kw = dict(lp=net, lp_shortlist=4096, lp_fallback_every=64, lp_fallback_mse=0.5, lp_min_cover=args.lp_min_cover)
    di = np.full(int(np.prod(sdims)), np.nan, np.float32)
    lsim, _, st = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], cfg["n"], cfg["k"], seed=cfg["seed"], **kw)
    stats = field_stats(exact_sim, lsim, sdims) if exact_sim is not None else None
    a = 300
    au = dict(lp_audit_nodes=0, lp_audit_hits=0, lp_audit_best_hits=0)
    if args.lp_audit:
        _, _, au = g2s_amd.qs(ti, dims, np.full(a * a, np.nan, np.float32), (a, a), cfg["types"], cfg["n"], cfg["k"],
                              seed=cfg["seed"], lp_audit=True, **kw)
    n_a = max(1, au["lp_audit_nodes"])
    nodes = st["nodes"]
    out = dict(value=nodes / (st["path_loop_ms"] / 1e3), unit="nodes/s", ms_per_step=st["path_loop_ms"],
               speedup_vs_exact=exact_ms / st["path_loop_ms"],
               proposed_frac=st["lp_proposed"] / max(1, nodes), fallback_frac=st["lp_fallbacks"] / max(1, nodes),
               mean_shortlist=st["lp_shortlist_sum"] / max(1, st["lp_proposed"]),
               recall_best_proposed=au["lp_audit_best_hits"] / n_a,
               recall_kbest_proposed=au["lp_audit_hits"] / (n_a * int(np.ceil(cfg["k"]))),
               recall_audit_sample=f"{a}x{a} realisation on the same TI, {au['lp_audit_nodes']} proposed nodes",
               training=dict(pairs=int(sum(len(p[2]) for _, _, p in sets)), steps=args.lp_steps * args.lp_epochs *
                             len(sets), seconds=t_rec + t_train, final_loss=float(losses[-1][-1])),
               vs_exact_realisation=stats,
               rules=f"exact scan for every 64th node, nodes with < {args.lp_min_cover:.0%} of neighbours on the key "
                     "stencil, best proposed mismatch > 0.5 sigma^2 per neighbour, shortlist overflow")
    net.close()
    return out


def host_threads():
    """What nproc prints: the CPUs this process may run on, capped by
    OMP_NUM_THREADS / OMP_THREAD_LIMIT when set."""
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    for var in ("OMP_NUM_THREADS", "OMP_THREAD_LIMIT"):
        try:
            v = int(os.environ.get(var, "").split(",")[0])
            if v > 0:
                n = min(n, v) if var == "OMP_THREAD_LIMIT" else v
        except ValueError:
            pass
    return max(1, n)


def cpu_model():
    """The host CPU as lscpu names it (model name, sockets x cores x threads)."""
    info = {}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            info[k.strip()] = v.strip()
    except (OSError, subprocess.SubprocessError):
        pass
    name = info.get("Model name")
    if not name:
        try:
            with open("/proc/cpuinfo") as fh:
                name = next((l.split(":", 1)[1].strip() for l in fh if l.startswith("model name")), "unknown")
        except OSError:
            name = "unknown"
    return dict(model=name, sockets=info.get("Socket(s)"), cores_per_socket=info.get("Core(s) per socket"),
                threads_per_core=info.get("Thread(s) per core"), online=info.get("On-line CPU(s) list"),
                affinity_cpus=len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else None)


def cpu_baseline(cfg, sim, threads, sample):
    """The oracle in reference-dataflow mode (FP32 FFT scan + fKst select,
    src/CPUThreadDevice.cpp:349-490 restated) timed on this host for a
    contiguous slice of the same path, one node per thread at a time."""
    from concurrent.futures import ThreadPoolExecutor

    import g2s_amd
    import oracle

    oracle.build()
    ti, dims = cfg["ti"], cfg["ti_dims"]
    kd = [d // 2 + 1 for d in dims]
    offs = oracle.offsets(kd)
    kern = np.ones(int(np.prod(kd)), np.float32)
    informed = np.zeros(int(np.prod(cfg["sim_dims"])), np.uint8)
    p, s, b = oracle.path(informed, cfg["seed"])
    t0 = time.time()
    orc = oracle.Sim(ti, dims, cfg["types"], [], [], cfg["sim_dims"], kd, kern, offs, cfg["n"], cfg["k"], p, s, b,
                     mode=1)
    setup = time.time() - t0
    start = len(p) // 10  # a slice 10% into the path
    nodes = list(range(start, start + sample))
    di = np.ascontiguousarray(sim, np.float32)

    def one(i):
        return orc.node(di, i)

    with ThreadPoolExecutor(max_workers=threads) as ex:
        list(ex.map(one, nodes[:threads]))  # warm (FFT plans, caches)
        t0 = time.time()
        res = list(ex.map(one, nodes))
        dt = time.time() - t0
    return dict(value=len(nodes) / dt, unit="nodes/s", cores=threads, kind="port", host=cpu_model(),
                sample=(f"{len(nodes)} path nodes {start}..{start + len(nodes) - 1} of the same 1000^2 "
                        f"realisation, oracle reference-dataflow FP32 FFT + fKst, {threads} threads, "
                        f"own mixed-radix CPU FFT (no FFTW on the host); spectra setup {setup:.1f}s untimed"))


def calibration_leg(cfg, iters, cpu_sample):
    """auto_qs calibration on the benchmark TI with auto_qs's defaults
    (neighbour counts 1..79, the seven densities, maxK 1, power 2, minIter
    1000) and a uniform 201x201 kernel: samples scored per second. The CPU
    baseline is the oracle (FP64 brute-force maps, OpenMP) on a bounded
    subset of the settings, one iteration."""
    import g2s_amd

    ti, dims = cfg["ti"], cfg["ti_dims"]
    kd = (201, 201)
    ker = np.ones(kd[0] * kd[1], np.float32)
    nb = g2s_amd.default_neighbour_configs((80,))
    g2s_amd.calibration([ti], dims, [0], [ker], [kd], nb_configs=nb[:4], max_iter=1, seed=4)  # warm
    r = g2s_amd.calibration([ti], dims, [0], [ker], [kd], nb_configs=nb, max_iter=iters, seed=5, stage_timing=True)
    # the dominant kernel is the exact scan's spectrum stage (k_taps1024 + k_pencil1024):
    # the same algorithmic bytes per scanned sample as per path node
    V, S, N = 2, (dims[0] // 2 + 1) * dims[1], dims[0] * dims[1]
    a_node = V * S * 8 + 2 * N * 4
    roof = None
    if r["spectrum_ms"] > 0:
        achieved = a_node * r["distributions"] / (r["spectrum_ms"] / 1e3) / 1e9
        roof = dict(bound="hbm", achieved=achieved, peak=HBM_PEAK_GBS, unit="GB/s", frac=achieved / HBM_PEAK_GBS,
                    traffic=None, kernel="k_pencil1024", avg_launch_us=r["spectrum_ms"] * 1e3 / max(1, r["waves"]),
                    samples_per_launch=r["distributions"] / max(1, r["waves"]), algorithmic_bytes_per_sample=a_node)
    out = dict(value=r["distributions"] / (r["ms"] / 1e3), unit="samples/s", samples=r["distributions"],
               iterations=r["iterations"], waves=r["waves"], ms=r["ms"], scan_ms=r["scan_ms"],
               draw_ms=r["draw_ms"], setup_ms=r["setup_ms"], spectrum_ms=r["spectrum_ms"], rows_ms=r["rows_ms"],
               roofline=roof,
               config=(f"auto_qs calibration, TI {dims[0]}x{dims[1]} exp(GRF), uniform kernel {kd[0]}x{kd[1]}, "
                       f"{nb.shape[0]} neighbour counts x 7 densities, maxK 1, power 2, {iters} iterations, "
                       f"exclusion radius {(dims[0] * dims[1] * 0.005) ** 0.5:.1f}"))
    if cpu_sample != 0:
        import oracle

        oracle.build()
        sub = nb[[9, 39, 78]]
        t0 = time.perf_counter()
        c = oracle.calibration([ti], dims, [0], [ker], [kd], sub, g2s_amd.DEFAULT_DENSITIES, 1, 2.0, 1, 1000, 0.0, 5)
        dt = time.perf_counter() - t0
        out["cpu_baseline"] = dict(value=c["distributions"] / dt, unit="samples/s",
                                   cores=host_threads(), kind="port",
                                   sample=(f"{c['distributions']} samples: one iteration over neighbour counts "
                                           f"10, 40, 79 x 7 densities, oracle FP64 brute-force maps (OpenMP)"))
    return out


# The other parity workloads: (synth constructor, tie quantum, per-variable
# kernel weights, algorithmic bytes per node V*S*8 + 2*N*4 with V active
# spectra, S the half spectrum and N the FFT grid of the TI)
OTHER_WORKLOADS = {
    1: ("config1_categorical_2d", "auto", None, 2 * 126 * 250 * 8 + 2 * 250 * 250 * 4),
    3: ("config3_categorical_3d", "auto", None, 3 * 91 * 150 * 120 * 8 + 2 * 180 * 150 * 120 * 4),
    4: ("config4_multivariate_2d", 0.0, (0.5, 0.5), 6 * 251 * 500 * 8 + 2 * 500 * 500 * 4),
}


def other_workload(args):
    """One parity workload at its full simulation grid (--sim-size shrinks
    it): warmup, timed realisations, nodes/s and the loop's fraction of the
    A_node roofline."""
    import g2s_amd
    from g2s_amd import synth

    name, quantum, weights, a_node = OTHER_WORKLOADS[args.workload]
    cfg = getattr(synth, name)()
    ti, dims, sdims = cfg["ti"], cfg["ti_dims"], tuple(cfg["sim_dims"])
    if args.sim_size:
        sdims = tuple([args.sim_size] * len(sdims))
    nvar = len(cfg["types"])
    di = cfg.get("di")
    if di is None or args.sim_size:
        di = np.full(int(np.prod(sdims)) * nvar, np.nan, np.float32)
    q = -1.0 if quantum == "auto" else quantum
    kw = {}
    if weights is not None:
        kd = [d // 2 + 1 for d in dims]
        kw = dict(kernel=np.tile(np.asarray(weights, np.float32), int(np.prod(kd))), kernel_dims=kd)
    print(f"[bench] workload {args.workload}: TI {dims} sim {sdims} n={cfg['n']} k={cfg['k']}", file=sys.stderr,
          flush=True)
    for w in range(args.warmup):
        g2s_amd.qs(ti, dims, di, sdims, cfg["types"], cfg["n"], cfg["k"], seed=1000 + w, wave_size=args.wave,
                   tie_quantum=q, **kw)
    times, st = [], None
    for s in range(args.steps):
        _, _, st = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], cfg["n"], cfg["k"], seed=cfg["seed"] + s,
                              wave_size=args.wave, tie_quantum=q, stage_timing=args.stage_every, progress=30, **kw)
        times.append(st["path_loop_ms"])
        print(f"[bench] step {s}: {st}", file=sys.stderr, flush=True)
    ms = float(np.mean(times))
    value = st["nodes"] / (ms / 1e3)
    return {
        "metric": f"QS nodes/sec, parity workload {args.workload}",
        "value": value,
        "unit": "nodes/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "config": {"workload": f"{name}: TI {dims}, sim {sdims}, n={cfg['n']}, k={cfg['k']}, waves<={args.wave}",
                   "nodes_per_step": st["nodes"]},
        "algorithmic_bytes_per_node": a_node,
        "hbm_roofline_frac_whole_loop": a_node * value / (HBM_PEAK_GBS * 1e9),
        "stats": st,
    }


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; --gpus above 1 is not supported"}))
        sys.exit(2)
    import g2s_amd
    from g2s_amd import synth

    for kv in args.tune:
        key, val = kv.split("=")
        g2s_amd.set_default_tuning(key, int(val))
    if args.workload != 2:
        print(json.dumps(other_workload(args)))
        return
    cfg = synth.config2_continuous_2d(args.size)
    if args.sim_size:
        cfg["sim_dims"] = (args.sim_size, args.sim_size)
    ti, dims, sdims = cfg["ti"], cfg["ti_dims"], cfg["sim_dims"]
    if args.copy_calib:
        import torch

        a = torch.empty(64 * 1024 * 1024, dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        a.fill_(1.0)
        torch.cuda.synchronize()
        b.copy_(a)  # reads 256 MiB, writes 256 MiB
        torch.cuda.synchronize()
        print("[bench] copy calibration: 268435456 B read + 268435456 B written", file=sys.stderr, flush=True)
    di = np.full(int(np.prod(sdims)), np.nan, np.float32)
    n, k = cfg["n"], cfg["k"]
    print(f"[bench] workload TI {dims} sim {sdims} n={n} k={k}", file=sys.stderr, flush=True)

    # warmup: full realisations with other seeds (kernel load, allocations)
    for w in range(args.warmup):
        _, _, st = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], n, k, seed=1000 + w, wave_size=args.wave)
        print(f"[bench] warmup {w}: {st}", file=sys.stderr, flush=True)

    times, stats = [], []
    sim = None
    for s in range(args.steps):
        t0 = time.perf_counter()
        sim, idx, st = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], n, k, seed=cfg["seed"] + s, wave_size=args.wave,
                                  stage_timing=args.stage_every)
        wall = time.perf_counter() - t0
        times.append(st["path_loop_ms"])
        stats.append(st)
        print(f"[bench] step {s}: wall {wall:.2f}s {st}", file=sys.stderr, flush=True)

    nodes = stats[-1]["nodes"]
    ms = float(np.mean(times))
    value = nodes / (ms / 1e3)
    # roofline of the dominant kernel: algorithmic bytes per node
    # A = V*S*8 + 2*N*4 (V=2 spectra of S=501*1000 complex64, N=10^6 map
    # floats written and read: a scan by transforms) over its event-timed
    # duration. The data-flow loop (no gather stage of its own) is one kernel,
    # launched for 64 waves of nodes at a time (for fewer where its rate is
    # judged against the waves': figures per launch are per 64 waves); the wave
    # loop's dominant kernel is the spectrum stage, launched once a wave.
    V, S, N = 2, (dims[0] // 2 + 1) * dims[1], dims[0] * dims[1]
    a_node = V * S * 8 + 2 * N * 4
    st = stats[-1]
    kernel_ms = st.get("spectrum_ms", 0.0)
    roof = None
    if kernel_ms > 0:
        flow = st["gather_ms"] == 0.0
        kernel = "k_flow_direct" if flow else "k_pencil1024"
        launches = max(1, -(-st["scanned_nodes"] // min(65536, 64 * args.wave)) if flow else st["waves"])
        achieved = a_node * st["scanned_nodes"] / (kernel_ms / 1e3) / 1e9
        nodes_per_launch = st["scanned_nodes"] / launches
        per_node = measured_bytes_per_node(kernel) if dims == (1000, 1000) else None
        if flow:
            timing = "HIP events around every launch of the timed step"
            note = ("the algorithmic bytes are those of a scan by transforms; the kernel sums the map's terms "
                    "directly and drops positions by a running bound, from the TI in the caches: it is bound by "
                    "VALU and scalar issue and L1, and traffic is its measured HBM bytes per launch")
        else:
            timing = (f"HIP events on the stream of every {args.stage_every}-th wave of the timed "
                      "step (k_taps work included with the gather)")
            note = ("the algorithmic bytes count a 4-byte map per TI cell written and read once; the "
                    "pencil and rows kernels never materialise that map (column transforms pass between "
                    "them), so achieved may exceed the HBM peak: the pencil is bound by VALU issue, and "
                    "traffic is its measured HBM bytes per launch. Consecutive waves of one dependency level "
                    "run on two streams, so a launch's duration includes time shared with the other "
                    "stream's kernels")
        roof = dict(bound="hbm", achieved=achieved, peak=HBM_PEAK_GBS, unit="GB/s", frac=achieved / HBM_PEAK_GBS,
                    traffic=(per_node * nodes_per_launch if per_node else None),
                    kernel=kernel, avg_launch_us=kernel_ms * 1e3 / launches,
                    nodes_per_launch=nodes_per_launch, algorithmic_bytes_per_node=a_node,
                    traffic_source=(PROFILES[kernel] if per_node else None), launch_timing=timing, note=note)
    alt = None
    if args.alt_wave > 0 and args.alt_wave != args.wave:
        _, _, sa = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], n, k, seed=cfg["seed"], wave_size=args.alt_wave,
                              stage_timing=args.stage_every)
        alt = dict(wave=args.alt_wave, value=sa["nodes"] / (sa["path_loop_ms"] / 1e3), ms_per_step=sa["path_loop_ms"],
                   waves=sa["waves"], spectrum_ms=sa["spectrum_ms"], rows_ms=sa["rows_ms"], merge_ms=sa["merge_ms"])
        print(f"[bench] waves <= {args.alt_wave}: {alt}", file=sys.stderr, flush=True)
    graph = None
    if args.graph_steps:
        # the same step with each wave's kernels replayed as one captured HIP
        # graph per stream (tuning key loop.graph; identical realisation)
        g2s_amd.set_default_tuning("loop.graph", 1)
        try:
            sg, _, sgs = g2s_amd.qs(ti, dims, di, sdims, cfg["types"], n, k, seed=cfg["seed"] + args.steps - 1,
                                    wave_size=args.wave)
        finally:
            g2s_amd.set_default_tuning("loop.graph", 0)
        graph = dict(value=sgs["nodes"] / (sgs["path_loop_ms"] / 1e3), ms_per_step=sgs["path_loop_ms"],
                     waves=sgs["waves"], identical_realisation=bool(np.array_equal(sg, sim)))
        print(f"[bench] captured wave steps: {graph}", file=sys.stderr, flush=True)
    learned = learned_form(cfg, args, ms, sim) if args.learned else None
    calib = calibration_leg(cfg, args.calib_iters, args.cpu_sample) if args.calib_iters > 0 else None
    if calib:
        print(f"[bench] calibration: {calib}", file=sys.stderr, flush=True)
    threads = args.cpu_threads or host_threads()
    cpu = None
    if args.cpu_sample != 0:
        cpu = cpu_baseline(cfg, sim, threads, args.cpu_sample if args.cpu_sample > 0 else 4 * threads)
    out = {
        "metric": "QS nodes/sec at 1000^2 TI n=80 k=1.5",
        "value": value,
        "unit": "nodes/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": f"QS unconditional 2D continuous, TI {dims[0]}x{dims[1]} exp(GRF range 20), "
                               f"sim {sdims[0]}x{sdims[1]}, n={n}, k={k}, waves<={args.wave}",
                   "nodes_per_step": nodes},
        "hbm_roofline_frac_whole_loop": a_node * value / (HBM_PEAK_GBS * 1e9),
        "roofline": roof,
        "cpu_baseline": cpu,
        "learned_proposal": learned,
        "calibration": calib,
        "alt_wave": alt,
        "graph_steps": graph,
        "stats": st,
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
