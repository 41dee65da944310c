"""Benchmark: Poisson apply on the MI355X (order 7, prec 1e-6, 16 Gaussians).

One step = one full apply(prec, out, P, f) on a fresh output tree: every
breadth-first level's screening, generated band nodes, band sums and
reductions, then the top-down/bottom-up transforms and norms.  Inputs (the
projected source tree and the operator with its device band tables) are
resident in HBM before the timed region.  Prints one JSON line.

    python bench.py [--gpus 1] [--steps 5] [--warmup 2] [--workload gauss16_k7] [--no-cpu-baseline]
    python bench.py --copy-probe     (three 256 MiB device copies: HBM counter calibration)

roofline.traffic (HBM bytes per band-kernel launch) comes from the rocprofv3
FETCH_SIZE / WRITE_SIZE summary committed under profiles/ for the same
workload, scaled by the copy-probe calibration; it is null when absent.
"""
import argparse
import json
import os
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

FP64_PEAK_TFLOPS = 78.6   # MI355X dense FP64 (vector and matrix)
HBM_PEAK_GBS = 8000.0
METRIC = "Poisson apply s/tree + GFLOP/s (order 7, \u03b5=1e-6), chosen vs plain FP64 GPU"


def band_kernel(precision, order=7):
    """Family of the band kernel that a single tree runs: the one-wave-per-item
    kernels for FP64 at every order and FP32 at order 7 (unless the tile layout is
    selected there), the tile-shared one otherwise."""
    import mrcpp_amd as mr
    if (precision == "fp64" and order != 7) or (order == 7 and precision in ("fp64", "fp32") and mr.band_layout() != "tiles"):
        return "k_band_waves"
    return "k_band_mfma"
COPY_PROBE_BYTES = 256 << 20


def copy_probe():
    """Three device-to-device copies of COPY_PROBE_BYTES through the library:
    the known traffic against which FETCH_SIZE / WRITE_SIZE are scaled."""
    import ctypes
    import mrcpp_amd as mr
    L = mr.lib()
    L.mwg_init.argtypes = [ctypes.c_int]
    L.mwg_malloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    L.mwg_copy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    assert L.mwg_init(0) == 0
    a, b = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.mwg_malloc(ctypes.byref(a), COPY_PROBE_BYTES) == 0
    assert L.mwg_malloc(ctypes.byref(b), COPY_PROBE_BYTES) == 0
    for _ in range(3):
        assert L.mwg_copy(b, a, COPY_PROBE_BYTES) == 0
    L.mwg_synchronize()
    print("copied %d bytes x3" % COPY_PROBE_BYTES, flush=True)


def measured_traffic(workload, precision="fp64"):
    """HBM bytes per band-kernel launch from the committed counter summary
    (lines 'workload: <name>' and 'traffic_bytes_per_launch_<precision>: <int>')."""
    path = os.path.join(HERE, "profiles", "%s_%s_traffic.md" % (band_kernel(precision), workload))
    if not os.path.exists(path):
        return None, None
    kv = {}
    for line in open(path):
        if ":" in line and not line.startswith(("#", "`", " ")):
            k, v = line.split(":", 1)
            kv[k.strip()] = v.strip()
    key = "traffic_bytes_per_launch_" + precision
    if kv.get("workload") != workload or key not in kv:
        return None, None
    return int(float(kv[key])), os.path.relpath(path, HERE)


def flops_per_tuple(order):
    """Algorithmic FLOP of one applied (f, ft, gt, term) tuple: three
    [(k+1)^2 x (k+1)] x [(k+1) x (k+1)] sweeps = 6 (k+1)^4."""
    return 6 * (order + 1) ** 4


def setup(workload):
    import mrcpp_amd as mr
    from mrcpp_amd import workloads as W
    w = W.WORKLOADS[workload]
    src = w["sources"]()
    mra = mr.MultiResolutionAnalysis((-w["box"], w["box"]), w["order"])
    f = mr.FunctionTree(mra)
    g = mr.GaussExp.from_sources(src)
    mr.build_grid(f, g)
    mr.project(w["prec"], f, g)
    if w["mu"] is None:
        P = mr.PoissonOperator(mra, w["prec"])
    else:
        P = mr.HelmholtzOperator(mra, w["mu"], w["prec"])
    return mr, w, src, mra, f, P


def time_projection(mr, w, src, mra, reps=3):
    """build_grid + project of the workload's input on the GPU (median of reps)
    and on the host cores (one run), with the node counts."""
    import time
    g = mr.GaussExp.from_sources(src)
    out = {}
    for target, n in (("device", reps), ("host", 1)):
        mr.set_projection_target(target)
        ts, nodes = [], 0
        for _ in range(n):
            f = mr.FunctionTree(mra)
            mr.device_synchronize()
            t0 = time.perf_counter()
            mr.build_grid(f, g)
            mr.project(w["prec"], f, g)
            mr.device_synchronize()
            ts.append(time.perf_counter() - t0)
            nodes = f.getNNodes()
        out[target] = {"s": sorted(ts)[len(ts) // 2], "nodes": int(nodes)}
    mr.set_projection_target("auto")
    return {"gpu_s": round(out["device"]["s"], 6), "host_s": round(out["host"]["s"], 4), "nodes": out["device"]["nodes"],
            "nodes_host": out["host"]["nodes"], "speedup": round(out["host"]["s"] / out["device"]["s"], 1),
            "what": "build_grid + project of the input tree (ProjectionCalculator levels on the GPU vs the host cores)"}


def time_operator_build(mr, w, mra):
    """Construction of the workload's operator with its 2D operator trees formed
    on the GPU (second of two builds) and on the host cores; the trees are
    bit-identical."""
    out = {}
    for target, n in (("device", 2), ("host", 1)):
        mr.set_operator_target(target)
        for _ in range(n):
            P = mr.PoissonOperator(mra, w["prec"]) if w["mu"] is None else mr.HelmholtzOperator(mra, w["mu"], w["prec"])
        out[target] = P.build_seconds()
        if target == "device":
            phases = P.build_phases()
    mr.set_operator_target("auto")
    return {"gpu_s": round(out["device"], 5), "host_s": round(out["host"], 5), "speedup": round(out["host"] / out["device"], 1),
            "terms": P.size(), "gpu_phases_s": {k: round(v, 5) for k, v in phases.items()},
            "what": "operator construction (kernel expansion, 1D kernel trees, 2D operator trees, transforms, caches)"}


def time_tree_io(g, box):
    """Writing and reading the apply result (its coefficients in HBM) as a
    binary tree file and as MADNESS-convention text (the text format needs a
    world cube [-2^m, 2^m], as MRCPP's reader does)."""
    import shutil
    import tempfile
    text_ok = box > 0 and (box & (box - 1)) == 0
    d = tempfile.mkdtemp()
    try:
        base, txt = os.path.join(d, "g"), os.path.join(d, "g.txt")
        out = {}
        for name, arg, path in (("binary", base, base + ".tree"), ("text", txt, txt)):
            if name == "text" and not text_ok:
                out[name] = "not applicable: the world is not a cube [-2^m, 2^m]"
                continue
            t0 = time.perf_counter()
            (g.saveTree if name == "binary" else g.saveTreeTXT)(arg)
            t1 = time.perf_counter()
            h = type(g)(g.mra)
            (h.loadTree if name == "binary" else h.loadTreeTXT)(arg)
            t2 = time.perf_counter()
            size = os.path.getsize(path)
            out[name] = {"save_s": round(t1 - t0, 4), "load_s": round(t2 - t1, 4), "bytes": size,
                         "save_MB_s": round(size / (t1 - t0) / 1e6, 1), "load_MB_s": round(size / (t2 - t1) / 1e6, 1)}
        out["nodes"] = g.getNNodes()
        out["what"] = "saveTree/loadTree and saveTreeTXT/loadTreeTXT of the output tree (host cores; the save includes the copy from HBM)"
        return out
    finally:
        shutil.rmtree(d, ignore_errors=True)


def time_arithmetic(mr, w, f, P):
    """add, multiply and dot of the input f and a fresh apply result V = P f
    (held in HBM only), each the median of three, with the output sizes."""
    V = mr.FunctionTree(f.mra)
    mr.apply(w["prec"], V, P, f)
    def med(fn):
        ts = []
        for _ in range(3):
            mr.device_synchronize()
            t0 = time.perf_counter()
            r = fn()
            mr.device_synchronize()
            ts.append(time.perf_counter() - t0)
        return sorted(ts)[1], r
    def add_once():
        h = mr.FunctionTree(f.mra)
        mr.add(w["prec"], h, 1.0, f, -1.0, V)
        return h
    def mul_once():
        p = mr.FunctionTree(f.mra)
        mr.multiply(w["prec"], p, 1.0, f, V)
        return p
    t_add, h = med(add_once)
    t_mul, p = med(mul_once)
    t_dot, d = med(lambda: mr.dot(f, V))
    return {"add_s": round(t_add, 5), "add_nodes": h.getNNodes(), "multiply_s": round(t_mul, 5), "multiply_nodes": p.getNNodes(),
            "dot_s": round(t_dot, 6), "dot": d, "what": "add(f - V), multiply(f V), dot(f, V) of the input and the Poisson result, on the GPU"}


def time_batch_operator_build(mr, mra, specs):
    """Construction of the batch's distinct operators: all together with their
    2D trees formed on the GPU (second of two builds) against one by one on
    the host cores."""
    keys = sorted({(sp["mu"], sp["prec"]) for sp in specs}, key=lambda k: (k[0] is not None, k[0] or 0.0, k[1]))
    out = {}
    for target, n in (("device", 2), ("host", 1)):
        for _ in range(n):
            ops = mr.build_operators(mra, keys, target)
        out[target] = ops[0].build_seconds()
        if target == "device":
            phases = ops[0].build_phases()
            terms = sum(op.size() for op in ops)
    return {"gpu_s": round(out["device"], 5), "host_s": round(out["host"], 5), "speedup": round(out["host"] / out["device"], 2),
            "operators": len(keys), "terms": terms, "gpu_phases_s": {k: round(v, 5) for k, v in phases.items()},
            "what": "construction of the batch's distinct Poisson/Helmholtz operators (one device pass vs one by one on the host cores)"}


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def cpu_baseline(workload, w, src, repeats=5):
    """The CPU oracle's apply on the same workload (one full tree per run),
    timed on this host's cores: one warm-up, then the median of `repeats`
    runs with every OpenMP thread, then one run on a single thread."""
    import oracle as O
    omra = O.OracleMRA((-w["box"], w["box"]), w["order"])
    of = O.OracleTree(omra)
    of.project_gaussians(w["prec"], src.coefs, src.exponents, src.centers)
    op = O.OracleOperator(omra, w["prec"], mu=w["mu"])
    cores = O.Oracle.max_threads()

    def one():
        og = O.OracleTree(omra)
        return O.apply(w["prec"], og, op, of)

    one()  # warm-up
    runs = [one() for _ in range(repeats)]
    secs = sorted(r["seconds"] for r in runs)
    med = secs[len(secs) // 2]
    st = runs[0]
    O.Oracle.set_threads(1)
    try:
        s1 = one()["seconds"]
    finally:
        O.Oracle.set_threads(cores)
    gflop = st["n_applied"] * flops_per_tuple(w["order"]) / 1e9
    return {
        "value": gflop / med,
        "unit": "GFLOP/s",
        "cores": cores,
        "kind": "port",
        "sample": "full applies of %s on the host (OpenMP over output nodes): 1 warm-up, median of %d at %d threads %.3f s/tree, "
                  "1 thread %.3f s/tree, %d applied tuples" % (workload, repeats, cores, med, s1, st["n_applied"]),
        "s_per_tree": med,
        "s_per_tree_runs": [round(s, 4) for s in secs],
        "s_per_tree_1_thread": s1,
        "value_1_thread": gflop / s1,
        "cpu_model": cpu_model(),
        "n_applied": st["n_applied"],
        "n_output_nodes": st["n_g"],
    }


def precision_error(mr, w, mra, f, P, precision):
    """Relative L2 error of one reduced-precision apply against the FP64 apply
    (itself equal to the FP64 CPU oracle to ~1e-15), and whether the output
    trees have the same node set."""
    import numpy as np
    out = {}
    for name in ("fp64", precision):
        mr.set_sweep_precision(name)
        g = mr.FunctionTree(mra)
        mr.apply(w["prec"], g, P, f)
        out[name] = g.export()
    mr.set_sweep_precision(precision)
    (i0, c0, _), (i1, c1, _) = out["fp64"], out[precision]
    same = bool(np.array_equal(i0, i1))
    if same:
        rel = float(np.linalg.norm(c1 - c0) / np.linalg.norm(c0))
    else:
        k0 = {tuple(x): j for j, x in enumerate(i0)}
        pairs = [(k0[tuple(x)], j) for j, x in enumerate(i1) if tuple(x) in k0]
        a = np.array([c0[j] for j, _ in pairs])
        b = np.array([c1[j] for _, j in pairs])
        rel = float(np.linalg.norm(b - a) / np.linalg.norm(a))
    return {"rel_l2": rel, "same_node_set": same, "nodes_fp64": int(len(i0)), "nodes": int(len(i1))}


def setup_batch(mr, W):
    """The 64-tree batch: uneven Gaussian sums, precisions 1e-5..1e-7, half
    Poisson and half Helmholtz (one operator per distinct (mu, prec))."""
    specs = W.batch_sources()
    mra = mr.MultiResolutionAnalysis((-32, 32), 7)
    ops, trees = {}, []
    for sp in specs:
        f = mr.FunctionTree(mra)
        g = mr.GaussExp.from_sources(sp["sources"])
        mr.build_grid(f, g)
        mr.project(sp["prec"], f, g)
        key = (sp["mu"], sp["prec"])
        if key not in ops:
            ops[key] = mr.PoissonOperator(mra, sp["prec"]) if sp["mu"] is None else mr.HelmholtzOperator(mra, sp["mu"], sp["prec"])
        trees.append((sp["prec"], ops[key], f))
    return mra, trees, specs


def run_batch_bench(args):
    print(json.dumps(batch_bench(args, args.steps, args.warmup)))


def batch_bench(args, steps, warmup):
    """Chosen form (one apply_batch of all trees at --precision) against the
    plain form (one FP64 apply per tree), same trees; one step = all trees."""
    import numpy as np
    import mrcpp_amd as mr
    from mrcpp_amd import workloads as W
    mra, trees, specs = setup_batch(mr, W)
    n = len(trees)

    def plain_step():
        mr.set_sweep_precision("fp64")
        outs, sts = [], []
        for prec, P, f in trees:
            g = mr.FunctionTree(mra)
            sts.append(mr.apply(prec, g, P, f))
            outs.append(g)
        mr.device_synchronize()
        return outs, sts

    pred = load_predictor(mr, 7)
    centers = [np.asarray(sp["sources"].centers) for sp in specs]

    def chosen_step(predictor=None, precision=None):
        mr.set_sweep_precision(precision or args.precision)
        outs = [mr.FunctionTree(mra) for _ in trees]
        sts = mr.apply_predicted([(prec, g, P, f) for (prec, P, f), g in zip(trees, outs)], predictor=predictor, centers=centers)
        mr.device_synchronize()
        return outs, sts

    def timed(step):
        for _ in range(max(warmup, 1)):
            step()
        times = []
        for _ in range(steps):
            t0 = time.perf_counter()
            outs, sts = step()
            times.append(time.perf_counter() - t0)
        return outs, sts, times

    p_outs, p_sts, p_times = timed(plain_step)
    # the batching gain alone: one apply_batch in plain FP64 (bit-identical
    # trees to the applies one by one)
    b_outs, b_sts, b_times = timed(lambda: chosen_step(precision="fp64"))
    b_ident = sum(1 for a, b in zip(p_outs, b_outs) if all(np.array_equal(x, y) for x, y in zip(a.export(), b.export())))
    fp64_batch = {"form": "one apply_batch of all trees, fp64 sweeps", "ms_per_step": round(float(np.mean(b_times)) * 1e3, 4),
                  "speedup_vs_plain": round(float(np.mean(p_times)) / float(np.mean(b_times)), 3), "bit_identical_trees": b_ident}
    with_pred = None
    if pred is not None and not args.no_predictor:
        w_outs, w_sts, w_times = timed(lambda: chosen_step(pred))
        wnum = wden = 0.0
        wsame = 0
        for a, b in zip(p_outs, w_outs):
            ai, ac, _ = a.export()
            bi, bc, _ = b.export()
            if np.array_equal(ai, bi):
                wsame += 1
                wnum += float(np.sum((bc - ac) ** 2))
                wden += float(np.sum(ac ** 2))
        with_pred = {"form": "one apply_batch of all trees, %s sweeps + refinement predictor" % args.precision,
                     "ms_per_step": round(float(np.mean(w_times)) * 1e3, 4),
                     "speedup_vs_plain": round(float(np.mean(p_times)) / float(np.mean(w_times)), 3),
                     "passes": int(max(st["n_levels"] for st in w_sts)),
                     "n_applied": int(sum(st["n_applied"] for st in w_sts)),
                     "same_node_set_trees": wsame, "rel_l2_same_trees": (wnum / wden) ** 0.5 if wden > 0 else None}
    mr.profile(True, kinds=("band",))  # events around the band kernel only while timing
    c_outs, c_sts, c_times = timed(chosen_step)
    prof = mr.profile_read()
    mr.profile(False)
    mr.profile(True)  # one untimed pass with events around every kernel: the breakdown
    chosen_step()
    every = mr.profile_read()
    mr.profile(False)
    flop = sum(st["n_applied"] for st in p_sts) * flops_per_tuple(7)
    c_s = float(np.mean(c_times))
    p_s = float(np.mean(p_times))
    # error of the chosen form against the plain FP64 trees, and node-set identity
    num = den = 0.0
    same = 0
    for a, b in zip(p_outs, c_outs):
        ai, ac, _ = a.export()
        bi, bc, _ = b.export()
        if np.array_equal(ai, bi):
            same += 1
            num += float(np.sum((bc - ac) ** 2))
            den += float(np.sum(ac ** 2))
    band_ms, band_launches = prof["band"]
    band_ms_per_step = band_ms / (steps + max(warmup, 1))
    c_flop = sum(st["n_applied"] for st in c_sts) * flops_per_tuple(7)
    res = {
        "metric": METRIC, "value": round(flop / c_s / 1e9, 3), "unit": "GFLOP/s", "n_gpus": 1, "steps": steps, "warmup": warmup,
        "ms_per_step": round(c_s * 1e3, 4), "s_per_tree": c_s / n, "higher_is_better": True, "scaling": "strong", "vs_baseline": None,
        "dtype": DTYPES[args.precision],
        "precision": args.precision, "form": "one apply_batch of all trees, %s sweeps" % args.precision,
        "with_refinement_predictor": with_pred, "fp64_batch": fp64_batch, "data": "synthetic seeded Gaussian sources",
        "passes_chosen": int(max(st["n_levels"] for st in c_sts)), "passes_plain": int(max(st["n_levels"] for st in p_sts)),
        "config": {"workload": "batch64_k7", "trees": n, "order": 7, "box": [-32, 32], "precs": sorted({sp["prec"] for sp in specs}),
                   "n_gaussians": [len(sp["sources"]) for sp in specs], "operators": "Poisson (even) / Helmholtz mu~U[0.5,3] (odd)",
                   "n_applied": int(sum(st["n_applied"] for st in p_sts)), "parallelism": "single GPU"},
        "plain_fp64_sequential": {"ms_per_step": round(p_s * 1e3, 4), "s_per_tree": p_s / n, "gflops": round(flop / p_s / 1e9, 3)},
        "speedup_vs_plain": round(p_s / c_s, 3),
        "error_vs_plain_fp64": {"rel_l2_same_trees": (num / den) ** 0.5 if den > 0 else None, "same_node_set_trees": same, "trees": n,
                                "applied_chosen": int(sum(st["n_applied"] for st in c_sts))},
        # a batch's long levels take the kernel by rows
        "roofline": {"bound": "mfma", "kernel": band_kernel(args.precision).replace("waves", "rows, k_band_waves"), "achieved": round(c_flop / (band_ms_per_step / 1e3) / 1e12, 4),
                     "peak": FP64_PEAK_TFLOPS if args.precision in ("fp64", "fp64_vector") else 157.3, "unit": "TFLOP/s",
                     "launches_per_step": band_launches / (steps + max(warmup, 1))},
        "kernel_ms_per_step": {k: round(v[0], 4) for k, v in every.items()},
        "host_breakdown_s": {k: c_sts[0][k] for k in ("seconds", "t_setup", "t_screen", "t_generate", "t_band", "t_transform", "t_host",
                                                      "t_cleanup")},
        "step_times_s": [round(t, 6) for t in c_times],
    }
    res["roofline"]["frac"] = round(res["roofline"]["achieved"] / res["roofline"]["peak"], 5)
    res["operator_build"] = time_batch_operator_build(mr, mra, specs)
    mr.set_sweep_precision("fp64")
    return res


PEAKS = {"fp64": FP64_PEAK_TFLOPS, "fp64_vector": FP64_PEAK_TFLOPS, "fp32": 157.3, "bf16x3": 2500.0}
DTYPES = {"fp64": "f64", "fp64_vector": "f64", "fp32": "f32 sweeps, f64 band sum", "bf16x3": "bf16x3 sweeps, f64 band sum"}
PREDICTOR_PARAMS = os.path.join(HERE, "mrcpp_amd", "share", "predictor_k7.npy")


def load_predictor(mr, order):
    """The trained refinement predictor (order 7 only), or None."""
    import numpy as np
    if order != 7 or not os.path.exists(PREDICTOR_PARAMS):
        return None
    return mr.RefinePredictor(params=np.load(PREDICTOR_PARAMS), threshold=0.5)


def time_form(mr, run_one, steps, warmup):
    """warmup untimed runs, then steps timed runs with HIP events around the
    band kernel only (Python's cyclic garbage collector paused while timing),
    then up to 5 untimed runs with events around every kernel for the
    per-kernel breakdown."""
    import gc
    for _ in range(max(warmup, 1)):
        run_one()
    mr.device_synchronize()
    mr.profile(True, kinds=("band",))
    mr.device_synchronize()
    times, stats = [], []
    out = None
    gc.collect()
    gc.disable()
    try:
        t0 = time.perf_counter()
        for _ in range(steps):
            ts = time.perf_counter()
            out, st = run_one()
            mr.device_synchronize()
            times.append(time.perf_counter() - ts)
            stats.append(st)
        mr.device_synchronize()
        elapsed = time.perf_counter() - t0
    finally:
        gc.enable()
    prof = mr.profile_read()
    mr.profile(False)
    nb = min(steps, 5)
    mr.profile(True)
    for _ in range(nb):
        run_one()
    every = mr.profile_read()
    mr.profile(False)
    breakdown = {k: v[0] / nb for k, v in every.items()}  # ms per apply
    return dict(s=elapsed / steps, times=times, stats=stats, prof=prof, out=out, breakdown=breakdown)


def roofline(prof, flop, steps, precision, workload):
    band_ms, launches = prof["band"]
    achieved = flop / (band_ms / steps / 1e3) / 1e12  # algorithmic TFLOP/s while the band kernel runs
    peak = PEAKS[precision]
    traffic, src = measured_traffic(workload, precision)
    return {"bound": "mfma", "kernel": band_kernel(precision), "precision": precision, "achieved": round(achieved, 4), "peak": peak,
            "unit": "TFLOP/s", "frac": round(achieved / peak, 5), "traffic": traffic, "traffic_source": src,
            "launches_per_step": launches / steps, "avg_launch_ms": band_ms / max(launches, 1), "flop_per_launch": flop / max(launches / steps, 1)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="gauss16_k7")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--copy-probe", action="store_true")
    ap.add_argument("--precision", default="fp32", choices=["fp64", "fp32", "bf16x3", "fp64_vector"],
                    help="band sweep precision of the chosen form (the plain form is always fp64)")
    ap.add_argument("--predictor", action="store_true", help="chosen form with the refinement predictor")
    ap.add_argument("--no-predictor", action="store_true", help="do not time the refinement-predictor variant beside the chosen form")
    ap.add_argument("--no-batch", action="store_true", help="leave out the 64-tree batch comparison (profiling runs of the single tree)")
    ap.add_argument("--no-autotune", action="store_true", help="leave out the launch-shape autotuner run")
    ap.add_argument("--no-ahead", action="store_true", help="leave out the plain FP64 apply with levels formed ahead on the GPU")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one MI355X: the apply path runs on a single GPU "
              "(sharding across GPUs is not launched); use --gpus 1", file=sys.stderr)
        sys.exit(2)
    if args.copy_probe:
        copy_probe()
        return
    if args.workload == "batch64_k7":
        run_batch_bench(args)
        return

    import numpy as np
    mr, w, src, mra, f, P = setup(args.workload)
    order, prec = w["order"], w["prec"]
    # the chosen form: FP32 sweeps (the fastest form within 1e-6 of plain
    # FP64); the refinement predictor is timed beside it (or chosen with --predictor)
    trained = load_predictor(mr, order)
    pred = trained if args.predictor else None

    def plain_one():
        mr.set_sweep_precision("fp64")
        g = mr.FunctionTree(mra)
        return g, mr.apply(prec, g, P, f)

    def form_one(predictor):
        def one():
            mr.set_sweep_precision(args.precision)
            g = mr.FunctionTree(mra)
            st = mr.apply_predicted([(prec, g, P, f)], predictor=predictor, centers=[src.centers])[0]
            return g, st
        return one

    plain = time_form(mr, plain_one, args.steps, args.warmup)
    chosen = time_form(mr, form_one(pred), args.steps, args.warmup)
    variant = None
    if not args.predictor and not args.no_predictor:
        variant = time_form(mr, form_one(trained), args.steps, args.warmup)
    mr.set_sweep_precision("fp64")
    pst, cst = plain["stats"][-1], chosen["stats"][-1]
    n_applied = pst["n_applied"]
    flop = n_applied * flops_per_tuple(order)  # algorithmic work: tuples under the plain screening
    i0, c0, _ = plain["out"].export()
    i1, c1, _ = chosen["out"].export()
    same = bool(np.array_equal(i0, i1))
    rel = float(np.linalg.norm(c1 - c0) / np.linalg.norm(c0)) if same else None
    res = {
        "metric": METRIC,
        # the headline is the FP64 drop-in (the reference's arithmetic); the
        # chosen reduced-precision form is reported beside it with its error
        "value": round(flop / plain["s"] / 1e9, 3),
        "unit": "GFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(plain["s"] * 1e3, 4),
        "s_per_tree": plain["s"],
        "higher_is_better": True,
        "scaling": "strong",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic seeded Gaussian sources",
        "config": {"workload": args.workload, "order": order, "prec": prec, "box": [-w["box"], w["box"]],
                   "n_gaussians": len(src), "operator": "Poisson" if w["mu"] is None else "Helmholtz mu=%g" % w["mu"],
                   "separation_rank": P.size(), "n_applied": int(n_applied),
                   "n_candidate_pairs": int(pst["n_pairs"]), "n_generated_nodes": int(pst["n_generated"]),
                   "n_output_nodes": int(pst["n_output_nodes"]), "parallelism": "single GPU"},
        "plain_fp64": {"form": "FP64 sweeps (drop-in)", "ms_per_step": round(plain["s"] * 1e3, 4), "s_per_tree": plain["s"],
                       "gflops": round(flop / plain["s"] / 1e9, 3),
                       "passes": int(pst["n_levels"]), "step_times_s": [round(t, 6) for t in plain["times"]],
                       "kernel_ms_per_step": {k: round(v, 4) for k, v in plain["breakdown"].items()},
                       "host_breakdown_s": {k: pst[k] for k in ("seconds", "t_setup", "t_screen", "t_generate", "t_band", "t_transform",
                                                                "t_host", "t_cleanup")}},
        "roofline": roofline(plain["prof"], flop, args.steps, "fp64", args.workload),
        "chosen": {"form": "%s sweeps%s" % (args.precision, " + refinement predictor" if pred is not None else ""),
                   "dtype": DTYPES[args.precision], "ms_per_step": round(chosen["s"] * 1e3, 4), "s_per_tree": chosen["s"],
                   "gflops": round(flop / chosen["s"] / 1e9, 3), "speedup_vs_plain": round(plain["s"] / chosen["s"], 3),
                   "error_vs_plain_fp64": {"same_node_set": same, "rel_l2": rel, "nodes_plain": int(len(i0)), "nodes_chosen": int(len(i1))},
                   "roofline": roofline(chosen["prof"], flop, args.steps, args.precision, args.workload),
                   "passes": int(cst["n_levels"]), "n_predicted": int(cst.get("n_predicted", 0)),
                   "n_cropped": int(cst.get("n_cropped", 0)), "n_fallback": int(cst.get("n_fallback", 0)),
                   "n_applied": int(cst["n_applied"]), "step_times_s": [round(t, 6) for t in chosen["times"]],
                   "kernel_ms_per_step": {k: round(v, 4) for k, v in chosen["breakdown"].items()}},
    }
    if variant is not None:
        vst = variant["stats"][-1]
        i2, c2, _ = variant["out"].export()
        vsame = bool(np.array_equal(i0, i2))
        res["with_refinement_predictor"] = {
            "form": "%s sweeps + refinement predictor" % args.precision, "ms_per_step": round(variant["s"] * 1e3, 4),
            "speedup_vs_plain": round(plain["s"] / variant["s"], 3), "passes": int(vst["n_levels"]),
            "n_predicted": int(vst.get("n_predicted", 0)), "n_cropped": int(vst.get("n_cropped", 0)),
            "n_fallback": int(vst.get("n_fallback", 0)), "same_node_set": vsame,
            "rel_l2": float(np.linalg.norm(c2 - c0) / np.linalg.norm(c0)) if vsame else None,
            "step_times_s": [round(t, 6) for t in variant["times"]],
            "kernel_ms_per_step": {k: round(v, 4) for k, v in variant["breakdown"].items()}}
    res["projection"] = time_projection(mr, w, src, mra)
    res["arithmetic"] = time_arithmetic(mr, w, f, P)
    res["tree_io"] = time_tree_io(plain["out"], w["box"])
    res["operator_build"] = time_operator_build(mr, w, mra)
    # the comparison on the 64-tree batch: one apply_batch of all
    # trees in the chosen form (with and without the refinement predictor)
    # against the plain FP64 apply of each tree in turn
    if not args.no_batch:
        b = batch_bench(args, 3, 1)
        res["batch64_k7"] = {k: b[k] for k in ("form", "ms_per_step", "s_per_tree", "plain_fp64_sequential", "speedup_vs_plain",
                                               "error_vs_plain_fp64", "with_refinement_predictor", "fp64_batch", "passes_chosen", "passes_plain",
                                               "roofline", "kernel_ms_per_step", "host_breakdown_s", "config")}
    if not args.no_autotune:
        # launch-shape autotuner on one plain FP64 apply (reported beside the
        # headline, which keeps the default shape); defaults restored after
        t = mr.autotune_band(lambda: plain_one(), repeats=3)
        default = [c for c in t["candidates"] if c["layout"] == "rows" and c["unit_groups"] == 32 and c["workgroups_per_cu"] == 0]
        res["autotuned"] = {"what": "band launch shape timed on one plain FP64 apply (median of 3 per candidate)",
                            "best": t["best"], "default_seconds": default[0]["seconds"] if default else None,
                            "candidates": t["candidates"]}
        mr.set_band_layout("auto")
        mr.set_band_launch(32, 0)
    if not args.no_ahead:
        # the plain FP64 apply with each next level formed and screened on the
        # GPU before the host's split (opt-in; the same tree bit for bit)
        mr.set_level_ahead(True)
        try:
            ah = time_form(mr, plain_one, args.steps, args.warmup)
        finally:
            mr.set_level_ahead(False)
        ia, ca, _ = ah["out"].export()
        ast = ah["stats"][-1]
        res["level_ahead"] = {"form": "FP64 sweeps, next level formed and screened on the GPU (set_level_ahead)",
                              "ms_per_step": round(ah["s"] * 1e3, 4), "speedup_vs_plain": round(plain["s"] / ah["s"], 3),
                              "steps_formed_ahead": int(ast["n_ahead"]), "passes": int(ast["n_levels"]),
                              "identical_to_plain": bool(np.array_equal(ia, i0) and np.array_equal(ca, c0)),
                              "kernel_ms_per_step": {k: round(v, 4) for k, v in ah["breakdown"].items()}}
    if not args.no_cpu_baseline:
        res["cpu_baseline"] = cpu_baseline(args.workload, w, src)
        res["gpu_vs_cpu"] = res["cpu_baseline"]["s_per_tree"] / plain["s"]
        res["chosen_gpu_vs_cpu"] = res["cpu_baseline"]["s_per_tree"] / chosen["s"]
    print(json.dumps(res))


if __name__ == "__main__":
    main()
