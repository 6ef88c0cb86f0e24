#!/usr/bin/env python3
"""Benchmark of the pawpyseed projection hot path on one MI355X.

Workload (216-atom defect supercell): diamond-lattice cubic cell a = 16.29 A
with one vacancy and its 4 neighbours moved 0.15 A inward (S, 215 sites)
projected onto the bulk cell (R, 216 sites); 520 eV cutoff (116,329 plane
waves per k), 108^3 FFT grid, 2x2x1 Monkhorst-Pack (4 k), 512 bands per k,
18 projectors per site (l = 0,1,2 x 2 radial channels, rmax 1.6 A).
Synthetic seeded inputs (no VASP data can be shipped).

One step = the full projection of S onto R:
  (1) setup_projections of S: sphere tables, then scatter -> 3D FFT ->
      sphere sums for all 512 x 4 (band, k);      -> band-projections/s
  (2) band-overlap matrix <R b,k | S b',k> of all pairs as one GEMM per k
                                                    -> overlap TFLOP/s
  (3) O_M augmentation of all pairs (FP64).
The basis R is set up once before timing (one basis serves many projected
structures).  Paths: "fp32" (FFT, sphere sums and overlap GEMM in FP32 on
MFMA, FP64 reductions and augmentation) is the headline `value`; "fp64" is
the plain FP64 path.  The overlap GEMM is re-run as split-plane products on
MFMA: "fp16x3" (two power-of-two-scaled fp16 planes per operand, 3
products: the headline overlap TFLOP/s), "bf16x3" and "bf16x6".

Prints one JSON line.  --gpus N > 1 exits: this build runs on one GPU.
"""

from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM = 8.0e12
PEAK = {"fp64": 78.6e12, "fp32": 157.3e12, "bf16": 2.5e15, "fp16": 2.5e15}
# split-plane overlap modes: MFMA arithmetic and products per complex term
SPLIT_MODES = {"fp16x3": ("fp16", 3), "bf16x3": ("bf16", 3), "bf16x6": ("bf16", 6)}


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def make_coefficients(torch, wl, Gs, seed, nband, ldc):
    """c_G ~ CN(0,1) exp(-|k+G|^2 / (2 (Gcut/2)^2)), normalised per band,
    generated on the GPU with a seeded generator."""
    from pawpyseed_amd import synthetic
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rec = synthetic.reciprocal_lattice(wl.lattice)
    gcut = math.sqrt(synthetic.C_EV * wl.encut)
    C = torch.zeros((len(Gs), nband, ldc), dtype=torch.complex64, device="cuda")
    for k, (kp, G) in enumerate(zip(wl.kpts, Gs)):
        kg = (G.astype(np.float64) + kp[None, :]) @ rec
        env = np.exp(-np.einsum("ij,ij->i", kg, kg) / (2.0 * (0.5 * gcut) ** 2)).astype(np.float32)
        envt = torch.from_numpy(env).cuda()
        re = torch.randn((nband, len(G)), generator=gen, device="cuda")
        im = torch.randn((nband, len(G)), generator=gen, device="cuda")
        c = torch.complex(re * envt, im * envt)
        c /= torch.linalg.vector_norm(c, dim=1, keepdim=True)
        C[k, :, : len(G)] = c
        del re, im, c
    return C


def apply_settings(ctx, spec):
    """Tuning parameters "name=value,..." onto a context."""
    for kv in [t for t in spec.split(",") if t]:
        name, value = kv.split("=")
        ctx.set_param(name.strip(), int(value))


def cpu_cores():
    try:
        n = len(os.sched_getaffinity(0))
    except Exception:
        n = os.cpu_count() or 1
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit():
        n = min(n, int(env))
    return max(1, n)


def cpu_fft(orc):
    """The 3D FFT the CPU baseline runs: MKL's (the reference's library),
    loaded from libmkl_rt through its FFTW3 entry points, where the host has
    it; else the oracle's own mixed-radix transform."""
    if orc.fft_use_mkl(True):
        return "MKL (libmkl_rt, FFTW3 interface over DFTI, sequential inside each OpenMP thread)"
    return "the oracle's own mixed-radix FFT (libmkl_rt not loadable)"


def cpu_model():
    """The host CPU's model name (/proc/cpuinfo), for the CPU baseline."""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "pmc_traffic_216atom.md")
RS_TRAFFIC_FILE = os.path.join(ROOT, "profiles", "realspace_aedensity_216atom.md")


def read_traffic_file(path):
    """{path: {class: HBM bytes per launch}} from the json block of a
    rocprofv3 --pmc summary kept with the profiles ({} when absent)."""
    try:
        txt = open(path).read()
        blk = txt.split("```json", 1)[1].split("```", 1)[0]
        return {p: {k: float(v) for k, v in d.items()} for p, d in json.loads(blk)["traffic_bytes_per_launch"].items()}
    except Exception:
        return {}


def read_traffic(path_name, settings):
    """HBM bytes per launch of each kernel class, from the rocprofv3 --pmc
    summary kept with the profiles (FETCH_SIZE and WRITE_SIZE per dispatch,
    scaled by the factors a plain 1 GiB device copy reads on the same
    counters), for the path and the settings that change what a launch
    moves (fft_xmask: the x pass writes only covered points; sphere_parts:
    the sphere sums' partial rows; gemm_planes: whether the split-plane
    GEMMs read materialised planes).  The summary keys its entries
    "<path>/fft_xmask=<x>,sphere_parts=<p>,gemm_planes=<g>".  Empty when
    there is no entry for those settings."""
    try:
        txt = open(TRAFFIC_FILE).read()
        blk = txt.split("```json", 1)[1].split("```", 1)[0]
        d = json.loads(blk)
    except Exception:
        return {}
    key = (f"{path_name}/fft_xmask={int(settings.get('fft_xmask', 0))},"
           f"sphere_parts={int(settings.get('sphere_parts', 0))},gemm_planes={int(settings.get('gemm_planes', 3))}")
    return {k: float(v) for k, v in d.get("traffic_bytes_per_launch", {}).get(key, {}).items()}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--nband", type=int, default=512)
    ap.add_argument("--cpu-seconds", type=float, default=20.0, help="target CPU-baseline work (seconds)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline and oracle checks")
    ap.add_argument("--paths", default="fp32,fp64", help="comma list of fp32, fp64 setup/overlap paths")
    ap.add_argument("--workload", default="216atom", choices=["216atom", "spinor512", "aedensity216", "cfg3"],
                    help="216atom: the headline workload; spinor512: the 512-atom noncollinear case; "
                         "aedensity216: all-electron density of the 216-atom cell on the doubled grid; "
                         "cfg3: three perturbed 216-atom structures onto one reference over 64 wedge k-points "
                         "with uneven plane-wave and band counts (separate lines)")
    ap.add_argument("--nk", type=int, default=64, help="k-points of the cfg3 workload")
    ap.add_argument("--no-graph", action="store_true", help="skip the graph-replay timing")
    ap.add_argument("--no-tune", action="store_true",
                    help="skip the autotuner (library defaults for the setup path)")
    ap.add_argument("--no-fused", action="store_true",
                    help="run the x pass and the sphere sums as separate kernels (comparison)")
    ap.add_argument("--profile-step", action="store_true",
                    help="for rocprofv3 --pmc: a 1 GiB device copy (counter calibration) and one fp32 setup step")
    ap.add_argument("--set", default="",
                    help="comma list name=value of tuning parameters applied before anything runs (e.g. the "
                         "settings of a timed run, for a profile of the same configuration)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the projection path shards by k-point, see the design notes)", file=sys.stderr)
        sys.exit(2)

    import torch

    from pawpyseed_amd import synthetic
    from pawpyseed_amd.core import batched as B

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    if args.workload == "spinor512":
        bench_spinor512(args, torch, B)
        return
    if args.workload == "aedensity216":
        bench_aedensity(args, torch, B)
        return
    if args.workload == "cfg3":
        bench_cfg3(args, torch, B)
        return
    wl = synthetic.config1(nband=args.nband)
    Gs = wl.ensure_gvecs()
    nk = len(Gs)
    nb = args.nband
    nw = np.array([len(g) for g in Gs], np.int32)
    ldc = int(-(-nw.max() // 64) * 64)
    gofs = np.concatenate([[0], np.cumsum(nw)]).astype(np.int32)
    Gdev = torch.from_numpy(np.ascontiguousarray(np.concatenate(Gs), np.int32)).cuda()
    log(f"workload: {len(wl.frac_R)}/{len(wl.frac_S)} sites, W={nw.tolist()}, grid={wl.fftg.tolist()}, "
        f"nk={nk}, nband={nb}")
    CR = make_coefficients(torch, wl, Gs, 1001, nb, ldc)
    CS = make_coefficients(torch, wl, Gs, 2002, nb, ldc)
    torch.cuda.synchronize()

    stream = torch.cuda.Stream()
    ctx = B.Context(0, stream=stream)
    apply_settings(ctx, args.set)
    if args.no_fused:
        ctx.set_param("fused", 0)
    labels_R = np.zeros(len(wl.frac_R), np.int32)
    labels_S = np.zeros(len(wl.frac_S), np.int32)
    paths = [p for p in args.paths.split(",") if p]
    plans, projR, projS, Om = {}, {}, {}, {}
    for p in paths:
        plans[p] = (B.SpherePlan(ctx, wl.lattice, wl.fftg, wl.frac_R, labels_R, [wl.species], p),
                    B.SpherePlan(ctx, wl.lattice, wl.fftg, wl.frac_S, labels_S, [wl.species], p))
        pR, pS = plans[p]
        projR[p] = torch.zeros((nk, nb, pR.ptot), dtype=torch.complex128, device="cuda")
        projS[p] = torch.zeros((nk, nb, pS.ptot), dtype=torch.complex128, device="cuda")
        Om[p] = torch.zeros((nk, nb, nb), dtype=torch.complex128, device="cuda")
        with torch.cuda.stream(stream):
            B.setup_projections(ctx, pR, wl.kpts, gofs, Gdev, CR, projR[p], p)  # basis, once
    ptotS = plans[paths[0]][1].ptot
    ptotR = plans[paths[0]][0].ptot

    def step(p, ev):
        pR, pS = plans[p]
        with torch.cuda.stream(stream):
            ev[0].record(stream)
            pS.rebuild(wl.frac_S)
            B.setup_projections(ctx, pS, wl.kpts, gofs, Gdev, CS, projS[p], p, sync=False)
            ev[1].record(stream)
            B.overlap_gemm(ctx, nk, 1, False, nw, CR, CS, Om[p], p, sync=False)
            ev[2].record(stream)
            B.augmentation(ctx, nk, 1, False, projR[p], pR.proj_off, labels_R, projS[p], pS.proj_off, labels_S,
                           wl.M_R, wl.M_S, [wl.species], [wl.delta_o], Om[p], sync=False)
            ev[3].record(stream)

    if args.profile_step:
        a = torch.empty(1 << 28, dtype=torch.float32, device="cuda")  # 1 GiB
        b = torch.empty_like(a)
        a.fill_(1.0)
        torch.cuda.synchronize()
        b.copy_(a)  # calibration: reads and writes exactly 1 GiB
        torch.cuda.synchronize()
        log("profile step settings", json.dumps({n: ctx.get_param(n) for n in B.TUNED}))
        evs = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        step(paths[0], evs)
        # the overlap GEMM of every other arithmetic once (their MFMA counters)
        ob = torch.zeros((nk, nb, nb), dtype=torch.complex128, device="cuda")
        for prec in ("fp64", "fp16x3", "bf16x3", "bf16x6"):
            with torch.cuda.stream(stream):
                B.overlap_gemm(ctx, nk, 1, False, nw, CR, CS, ob, prec)
        torch.cuda.synchronize()
        log("profile step done")
        return

    results = {}
    for p in paths:
        tuned, trials = None, []
        if not args.no_tune:
            # the project's autotuner on this workload's own inputs (untimed)
            pR, pS = plans[p]
            with torch.cuda.stream(stream):
                tuned, trials = B.autotune(ctx, pS, wl.kpts, gofs, Gdev, CS, projS[p], p, repeats=2)
            torch.cuda.synchronize()
            log(p, "autotune", json.dumps(tuned))
        for _ in range(args.warmup):
            evs = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
            step(p, evs)
        torch.cuda.synchronize()
        # timed steps: the library's default two-stream chunk pipeline, no
        # per-launch events
        rec = []
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            evs = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
            step(p, evs)
            rec.append(evs)
        torch.cuda.synchronize()
        wall = (time.perf_counter() - t0) / args.steps
        ts = np.mean([e[0].elapsed_time(e[1]) for e in rec]) / 1e3
        to = np.mean([e[1].elapsed_time(e[2]) for e in rec]) / 1e3
        ta = np.mean([e[2].elapsed_time(e[3]) for e in rec]) / 1e3
        # breakdown step: one chunk in flight (serialised), HIP events
        # around every launch on its stream -> per-kernel durations
        ctx.set_param("streams", 1)
        ctx.set_timing(True)
        ctx.timing_reset()
        evs = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        step(p, evs)
        torch.cuda.synchronize()
        kt = ctx.timing()
        ctx.set_timing(False)
        ctx.set_param("streams", tuned["streams"] if tuned else 2)
        ts_serial = evs[0].elapsed_time(evs[1]) / 1e3
        # the same setup (tables as built by the last step) replayed as one
        # HIP graph
        pR, pS = plans[p]
        ts_graph = None
        if not args.no_graph:
            with torch.cuda.stream(stream):
                graph = B.SetupGraph(ctx, pS, wl.kpts, gofs, Gdev, CS, projS[p], p)
                g0, g1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                g0.record(stream)
                for _ in range(args.steps):
                    graph.replay(sync=False)
                g1.record(stream)
            torch.cuda.synchronize()
            ts_graph = g0.elapsed_time(g1) / 1e3 / args.steps
            graph.close()
        nproj = nb * nk * ptotS
        ovl_flops = 8.0 * nb * nb * float(nw.sum())
        results[p] = dict(setup_s=ts, overlap_s=to, aug_s=ta, step_wall_s=wall,
                          band_projections_per_s=nproj / ts, overlap_tflops=ovl_flops / to / 1e12,
                          setup_s_one_chunk_in_flight=ts_serial,
                          setup_s_graph_replay=ts_graph,
                          band_projections_per_s_graph_replay=nproj / ts_graph if ts_graph else None,
                          autotune=tuned, autotune_trials=[list(t) for t in trials],
                          kernels={k: {"ms_total": v[0], "launches": v[1]} for k, v in kt.items()})
        log(p, json.dumps({k: v for k, v in results[p].items() if k != "kernels"}))
        log(p, "kernels (breakdown step)", json.dumps(results[p]["kernels"]))

    # the overlap as split-plane products on MFMA (same inputs): fp16x3 (two
    # scaled fp16 planes, 3 products), bf16x3 and bf16x6; timed over
    # args.steps calls of all k, then one call with per-launch events for
    # the split / GEMM / reduction breakdown
    ob = {}
    ovl_flops = 8.0 * nb * nb * float(nw.sum())
    for mode in SPLIT_MODES:
        ob[mode] = torch.zeros((nk, nb, nb), dtype=torch.complex128, device="cuda")
        with torch.cuda.stream(stream):
            B.overlap_gemm(ctx, nk, 1, False, nw, CR, CS, ob[mode], mode)  # warm
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                B.overlap_gemm(ctx, nk, 1, False, nw, CR, CS, ob[mode], mode, sync=False)
            e1.record(stream)
        torch.cuda.synchronize()
        t_m = e0.elapsed_time(e1) / 1e3 / args.steps
        ctx.set_timing(True)
        ctx.timing_reset()
        with torch.cuda.stream(stream):
            B.overlap_gemm(ctx, nk, 1, False, nw, CR, CS, ob[mode], mode)
        torch.cuda.synchronize()
        kt = ctx.timing()
        ctx.set_timing(False)
        results[mode] = dict(overlap_s=t_m, overlap_tflops=ovl_flops / t_m / 1e12,
                             kernels={k: {"ms_total": v[0], "launches": v[1]} for k, v in kt.items()})
        log(mode, "overlap", json.dumps(results[mode]))

    head = "fp32" if "fp32" in results else paths[0]
    R = results[head]
    # dominant kernel of the headline path and its roofline.  Algorithmic
    # bytes per launch (one 64-band chunk of one k-point):
    #   fft_x (last 1D pass): read the populated x-slab of the grid
    #     (the plane-wave sphere spans xs_k planes), write the grid points
    #     the projector spheres hold (fft_xmask; else the whole grid):
    #     NB prec (N1 N2 xs_k + covered), averaged over k;
    #   fft_y: read xs_k planes restricted to the populated y-rows ys_k(x),
    #     write the xs_k planes in full;
    #   fft_z: read the plane-wave coefficients in place (W_k points), write
    #     every populated (x, y) z-line in full;
    #   sphere_sum: gather NB values per sphere point, one real table row,
    #     one phase and one grid index per point;  gemm: 8 M N K flop;
    #   fft_x_sphere (the x pass fused with the sphere sums): read the
    #     populated x-slab, one real table row and one phase per sphere
    #     point, write one FP32 partial row (P x NB) per (work item, site).
    prec_bytes = 8 if head != "fp64" else 16
    n0, n1, n2 = (int(v) for v in wl.fftg)
    NB = 64
    bx, by, bz = [], [], []
    xmask_on = bool((R.get("autotune") or {}).get("fft_xmask", ctx.get_param("fft_xmask")))
    covered = plans[head][1].coverage()
    for G in Gs:
        gx, gy = G[:, 0].astype(np.int64), G[:, 1].astype(np.int64)
        xs = int(gx.max() - gx.min() + 1)
        rows = np.unique(gx * 4096 + gy).size  # populated (x, y) z-lines
        yrow = 0
        for x in np.unique(gx):
            sel = gy[gx == x]
            yrow += int(sel.max() - sel.min() + 1)
        # written: the whole grid, or with fft_xmask only the points the
        # projector spheres hold (their union)
        bx.append(n1 * n2 * NB * prec_bytes * xs + (covered if xmask_on else n0 * n1 * n2) * NB * prec_bytes)
        by.append(NB * prec_bytes * n2 * (yrow + xs * n1))
        bz.append(NB * prec_bytes * (len(G) + rows * n2))
    planS = plans[head][1]
    # grid gather (NB complex), real table row (P reals), phase (complex), index (int32) per point
    sphere_bytes = planS.npts * (NB * prec_bytes + (ptotS // len(wl.frac_S)) * prec_bytes // 2 + prec_bytes + 4)
    alg = {"fft_x": float(np.mean(bx)), "fft_y": float(np.mean(by)), "fft_z": float(np.mean(bz)),
           "sphere_sum": float(sphere_bytes)}
    usable, _, nrows, _, _ = planS.fused_info()
    if usable:
        P = ptotS // len(wl.frac_S)
        xs_read = float(np.mean([n1 * n2 * NB * prec_bytes * (b / (n1 * n2 * NB * prec_bytes) - n0) for b in bx]))
        alg["fft_x_sphere"] = xs_read + planS.npts * (P * prec_bytes // 2 + prec_bytes) + nrows * P * NB * 8
    gemm_flops = 8.0 * nb * nb * float(nw.mean())
    timed_settings = dict(R.get("autotune") or {n: ctx.get_param(n) for n in B.TUNED})
    timed_settings["gemm_planes"] = ctx.get_param("gemm_planes")
    timed_settings["fft_xmask"] = int(xmask_on)
    traffic = read_traffic(head, timed_settings)
    rl = {}
    for c, b in alg.items():
        kc = R["kernels"].get(c)
        if not kc or not kc["launches"]:
            continue
        ms = kc["ms_total"] / kc["launches"]
        rl[c] = {"bound": "hbm", "achieved": b / (ms * 1e-3) / 1e9, "peak": PEAK_HBM / 1e9, "unit": "GB/s",
                 "alg_bytes": b, "avg_launch_ms": ms, "ms_per_step": kc["ms_total"],
                 "traffic": traffic.get(c)}
    # augmentation (O_M of all pairs): dO applied to S's matched projector
    # rows (read once, written once), then one FP64 GEMM over the KM matched
    # projectors of every k, which gathers R's rows itself
    KM = int(sum(plans[head][1].proj_off[s + 1] - plans[head][1].proj_off[s] for s in wl.M_S))
    aug_bytes = 32.0 * KM * nb
    kc = R["kernels"].get("aug_prep")
    if kc and kc["launches"]:
        ms = kc["ms_total"] / kc["launches"]  # one launch covers all k
        rl["aug_prep"] = {"bound": "hbm", "achieved": aug_bytes * nk / (ms * 1e-3) / 1e9, "peak": PEAK_HBM / 1e9,
                          "unit": "GB/s", "alg_bytes": aug_bytes * nk, "avg_launch_ms": ms,
                          "ms_per_step": kc["ms_total"], "traffic": traffic.get("aug_prep"),
                          "what": "k_aug_apply of one call (all k): 16 B per applied value, read and written"}
    kc = R["kernels"].get("aug_gemm")
    if kc and kc["launches"]:
        ms = kc["ms_total"] / kc["launches"]
        aug_flops = 8.0 * nb * nb * KM * nk / kc["launches"]  # a launch covers several k
        rl["aug_gemm"] = {"bound": "mfma", "achieved": aug_flops / (ms * 1e-3) / 1e12,
                          "peak": PEAK["fp64"] / 1e12, "unit": "TFLOP/s", "alg_flops": aug_flops,
                          "avg_launch_ms": ms, "ms_per_step": kc["ms_total"], "traffic": traffic.get("aug_gemm"),
                          "what": "FP64 MFMA conj(X_R) Y^T of all k-points over the matched projectors"}
    kc = R["kernels"].get("gemm")
    if kc and kc["launches"]:
        ms = kc["ms_total"] / kc["launches"]
        per_launch = gemm_flops * nk / kc["launches"]  # FP32: one k-point; FP64: several
        rl["gemm"] = {"bound": "mfma", "achieved": per_launch / (ms * 1e-3) / 1e12,
                      "peak": PEAK["fp32" if head != "fp64" else "fp64"] / 1e12, "unit": "TFLOP/s",
                      "alg_flops": per_launch, "avg_launch_ms": ms, "ms_per_step": kc["ms_total"],
                      "traffic": traffic.get("gemm")}
    # split-plane overlap GEMMs: the plane GEMM on the MFMA peak of its
    # 16-bit arithmetic (products x 8 M N K flop per k-point), and the split
    # of both operands (read 8 B, write 2 B per plane per real of each c64)
    for mode, (arith, nprod) in SPLIT_MODES.items():
        kt = results.get(mode, {}).get("kernels", {})
        kc, ks = kt.get("gemm"), kt.get("gemm_split")
        if kc and kc["launches"]:
            ms = kc["ms_total"] / kc["launches"]
            rl[f"gemm_{mode}"] = {"bound": "mfma", "achieved": nprod * gemm_flops / (ms * 1e-3) / 1e12,
                                  "peak": PEAK[arith] / 1e12, "unit": "TFLOP/s", "alg_flops": nprod * gemm_flops,
                                  "tflops_equivalent": gemm_flops / (ms * 1e-3) / 1e12, "avg_launch_ms": ms,
                                  "ms_per_step": kc["ms_total"], "traffic": traffic.get(f"gemm_{mode}"),
                                  "what": f"plane GEMM of one k-point ({nprod} {arith} products per complex term)"}
        if ks and ks["launches"]:
            ms = ks["ms_total"] / ks["launches"]
            nplanes = 3 if mode == "bf16x6" else 2
            # gemm_planes 3: the two-plane GEMMs split their operands
            # themselves; fp16x3 first reads both operands for the chunk
            # exponents (and bf16x3 has no pass at all)
            cvt = timed_settings["gemm_planes"] == 3 and nplanes == 2
            sb = (2.0 * nb) * float(nw.mean()) * (8.0 if cvt else 8.0 + 4.0 * nplanes)
            rl[f"gemm_split_{mode}"] = {"bound": "hbm", "achieved": sb / (ms * 1e-3) / 1e9, "peak": PEAK_HBM / 1e9,
                                        "unit": "GB/s", "alg_bytes": sb, "avg_launch_ms": ms,
                                        "ms_per_step": ks["ms_total"], "traffic": traffic.get(f"gemm_split_{mode}"),
                                        "what": "exponent pass over both operands of one k-point (reads only)"
                                        if cvt else "plane split of both operands of one k-point"}
    for v in rl.values():
        v["frac"] = v["achieved"] / v["peak"]
    # the (a) stage against its unit of 8 W + 16 N^3 bytes per (band, k):
    # scatter and the three FFT passes of a step over their summed time
    stage_a = [c for c in ("scatter", "fft_z", "fft_y", "fft_x") if c in R["kernels"]]
    if stage_a:
        t_a = sum(R["kernels"][c]["ms_total"] for c in stage_a) * 1e-3
        unit_a = 8.0 * float(nw.mean()) + 16.0 * n0 * n1 * n2
        rl_stage_a = {"bound": "hbm", "unit": "GB/s", "peak": PEAK_HBM / 1e9,
                      "achieved": unit_a * nb * nk / t_a / 1e9, "alg_bytes_per_band_k": unit_a,
                      "ms_per_step": t_a * 1e3,
                      "what": "scatter + z/y/x passes of a step (breakdown timing) against 8 W + 16 N^3 bytes per "
                              "(band, k)"}
        rl_stage_a["frac"] = rl_stage_a["achieved"] / rl_stage_a["peak"]
    dom = max((c for c in rl if not c.startswith("gemm_")), key=lambda c: rl[c]["ms_per_step"])
    roof = {k: rl[dom][k] for k in ("bound", "achieved", "peak", "unit", "frac", "traffic")}
    roof["kernel"] = dom
    roof["avg_launch_ms"] = rl[dom]["avg_launch_ms"]
    roof["timing"] = "breakdown step after the timed steps: one band chunk in flight, HIP events per launch"
    roof["settings"] = {k: timed_settings.get(k) for k in ("fft_xmask", "fft_nt", "fft_tile", "sphere_parts", "gemm_planes")}
    # whole setup: algorithmic bytes of all its kernels over the pipelined time
    setup_bytes = sum(b for c, b in alg.items() if c in rl) * nk * -(-nb // NB)
    pipe = {"achieved": setup_bytes / R["setup_s"] / 1e9, "unit": "GB/s", "peak": PEAK_HBM / 1e9,
            "frac": setup_bytes / R["setup_s"] / PEAK_HBM,
            "what": "algorithmic bytes of the FFT passes and sphere sums (or the fused x pass) of one step / "
                    "timed setup time"}

    out = {
        "metric": "band_projections_per_sec",
        "value": R["band_projections_per_s"],
        "unit": "band-projections/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": (R["setup_s"] + R["overlap_s"] + R["aug_s"]) * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32 (FFT, sphere sums, overlap GEMM on MFMA; fp64 reductions and augmentation)"
        if head == "fp32" else head,
        "data": "synthetic (seeded)",
        "config": {"workload": "216-atom diamond defect supercell, a=16.29 A, 520 eV (W=116329/k), 108^3 grid, "
                               "2x2x1 MP (4 k), 512 bands/k, 18 projectors/site, S (215 sites) onto R (216)",
                   "nband": nb, "nk": nk, "fftg": wl.fftg.tolist(), "plane_waves": nw.tolist(),
                   "projectors_S": ptotS, "projectors_R": ptotR},
        "overlap_tflops": results["fp16x3"]["overlap_tflops"],
        "overlap_precision": "fp16x3 (two power-of-two-scaled fp16 planes per operand, 3 products, FP32 "
                             "accumulation over 512 terms, FP64 across chunks)",
        "overlap_tflops_by_precision": {m: results[m]["overlap_tflops"] for m in ("fp32", "fp64", *SPLIT_MODES)
                                        if m in results},
        "paths": {p: {k: v for k, v in r.items() if k != "kernels"} for p, r in results.items()},
        "kernels": rl,
        "stage_a": rl_stage_a if stage_a else None,
        "roofline": roof,
        "setup_pipeline_bandwidth": pipe,
    }
    if "fp64" in results:
        out["speedup_vs_fp64_gpu"] = R["band_projections_per_s"] / results["fp64"]["band_projections_per_s"]

    if not args.no_cpu:
        out.update(cpu_and_errors(args, torch, wl, Gs, CR, CS, projR, projS, Om, ob, plans, results, head))
    print(json.dumps(out), flush=True)


def bench_spinor512(args, torch, B):
    """The large noncollinear case: 512 sites, a = 21.72 A, 192^3 grid, 2
    k-points, W = 275,953 per spinor component, 2048 spinor bands, 18
    projectors per site.  One step projects both components of every band
    (B.setup_projections_spinor); errors on sampled bands against the FP64
    oracle.  Prints its own JSON line."""
    from oracle import pyoracle as orc
    from pawpyseed_amd import synthetic
    nb = 2048 if args.nband == 512 else args.nband
    wl = synthetic.config4(nband=nb)
    Gs = wl.ensure_gvecs()
    nk = len(Gs)
    W = [len(g) for g in Gs]
    ldc2 = -(-2 * max(W) // 64) * 64
    C2 = make_coefficients(torch, wl, Gs, 3003, nb, ldc2)  # up components in [0, W)
    dn = make_coefficients(torch, wl, Gs, 4004, nb, max(W))
    for k in range(nk):
        C2[k, :, W[k]:2 * W[k]] = dn[k, :, :W[k]]
    del dn
    gofs = np.concatenate([[0], np.cumsum(W)]).astype(np.int32)
    Gdev = torch.from_numpy(np.ascontiguousarray(np.concatenate(Gs), np.int32)).cuda()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    ctx = B.Context(0, stream=stream)
    apply_settings(ctx, args.set)
    labels = np.zeros(len(wl.frac_S), np.int32)
    log(f"spinor workload: {len(wl.frac_S)} sites, W={W} per component, grid={wl.fftg.tolist()}, nk={nk}, "
        f"nband={nb}")
    res, outs = {}, {}
    for p in [q for q in args.paths.split(",") if q]:
        plan = B.SpherePlan(ctx, wl.lattice, wl.fftg, wl.frac_S, labels, [wl.species], p)
        up = torch.zeros((nk, nb, plan.ptot), dtype=torch.complex128, device="cuda")
        down = torch.zeros_like(up)
        with torch.cuda.stream(stream):
            for _ in range(args.warmup):
                B.setup_projections_spinor(ctx, plan, wl.kpts, gofs, Gdev, C2, up, down, p)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                plan.rebuild(wl.frac_S)
                B.setup_projections_spinor(ctx, plan, wl.kpts, gofs, Gdev, C2, up, down, p, sync=False)
            e1.record(stream)
        torch.cuda.synchronize()
        t = e0.elapsed_time(e1) / 1e3 / args.steps
        nproj = 2 * nb * nk * plan.ptot
        res[p] = {"setup_s": t, "band_projections_per_s": nproj / t}
        sample = [0, nb - 1]
        outs[p] = (up[:, sample].cpu().numpy(), down[:, sample].cpu().numpy())
        log(p, json.dumps(res[p]))
        plan.close()
        del up, down
    # the band overlap of the spinor bands with those of a second structure
    # (2 W-long vectors, pseudoprojector.c:85 with num_waves = 2 W)
    CR2 = make_coefficients(torch, wl, Gs, 5005, nb, ldc2)
    dn = make_coefficients(torch, wl, Gs, 6006, nb, max(W))
    for k in range(nk):
        CR2[k, :, W[k]:2 * W[k]] = dn[k, :, :W[k]]
    del dn
    nw2 = np.array([2 * w for w in W], np.int32)
    ovl, ovl_out = {}, {}
    ob = torch.zeros((nk, nb, nb), dtype=torch.complex128, device="cuda")
    for p in [q for q in args.paths.split(",") if q] + ["fp16x3", "bf16x6"]:
        with torch.cuda.stream(stream):
            B.overlap_gemm(ctx, nk, 1, False, nw2, CR2, C2, ob, p)  # warm
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                B.overlap_gemm(ctx, nk, 1, False, nw2, CR2, C2, ob, p, sync=False)
            e1.record(stream)
        torch.cuda.synchronize()
        t = e0.elapsed_time(e1) / 1e3 / args.steps
        ovl[p] = {"overlap_s": t, "overlap_tflops": 8.0 * nb * nb * float(nw2.sum()) / t / 1e12}
        ovl_out[p] = ob[:, :4, :4].cpu().numpy()
        log(p, "spinor overlap", json.dumps(ovl[p]))
    del ob
    errs = {}
    if not args.no_cpu:
        # FP64 sums of the stored coefficients for the sampled 4 x 4 blocks
        for p, o in ovl_out.items():
            e = 0.0
            for k in range(nk):
                a = CR2[k, :4, : 2 * W[k]].cpu().numpy().astype(np.complex128)
                b = C2[k, :4, : 2 * W[k]].cpu().numpy().astype(np.complex128)
                ref = a.conj() @ b.T
                e = max(e, float(np.abs(o[k] - ref).max() / np.abs(ref).max()))
            errs[f"overlap_{p}"] = e
    if not args.no_cpu:
        sample = [0, nb - 1]
        Cs = C2[:, sample].cpu().numpy()
        T = orc.site_tables(wl.lattice, wl.fftg, wl.frac_S, [wl.species], labels)
        want_up = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts, Gs, [Cs[k, :, :W[k]] for k in range(nk)], T)
        want_dn = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts, Gs,
                                        [Cs[k, :, W[k]:2 * W[k]] for k in range(nk)], T)
        for p, (gu, gd) in outs.items():
            errs[f"projections_{p}"] = max(float(np.abs(gu - want_up).max() / np.abs(want_up).max()),
                                           float(np.abs(gd - want_dn).max() / np.abs(want_dn).max()))
        log("errors (sampled bands", sample, "both k and components):", json.dumps(errs))
    head = "fp32" if "fp32" in res else next(iter(res))
    out = {"metric": "band_projections_per_sec", "value": res[head]["band_projections_per_s"],
           "unit": "band-projections/s (each spinor component counted)", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "higher_is_better": True, "dtype": head, "data": "synthetic (seeded)",
           "config": {"workload": "512-atom diamond cell, a=21.72 A, 520 eV (W=275953 per spinor component), 192^3 "
                                  "grid, 2 k, 2048 spinor bands, 18 projectors/site", "nband": nb, "nk": nk},
           "paths": res, "spinor_overlap": ovl, "max_err_vs_fp64_oracle": errs}
    print(json.dumps(out), flush=True)


def bench_aedensity(args, torch, B):
    """All-electron charge density of the 216-atom S structure on the doubled
    grid 216^3 (get_realspace_density's default, density.c:158-179): per
    k-point and 64-band chunk, scatter + FP64/FP32 FFT, the partial-wave
    differences of the 215 sites (spheres of radius 1.6 A) weighted by the
    projections, and sum_b w_b |psi_b|^2; 512 bands x 4 k per step (all
    weighted 2 w_k).  Prints its own JSON line."""
    import time

    from oracle import pyoracle as orc
    from pawpyseed_amd import synthetic
    wl = synthetic.config1(nband=args.nband)
    Gs = wl.ensure_gvecs()
    nk, nb = len(Gs), args.nband
    nw = np.array([len(g) for g in Gs], np.int32)
    ldc = int(-(-nw.max() // 64) * 64)
    gofs = np.concatenate([[0], np.cumsum(nw)]).astype(np.int32)
    Gdev = torch.from_numpy(np.ascontiguousarray(np.concatenate(Gs), np.int32)).cuda()
    CS = make_coefficients(torch, wl, Gs, 2002, nb, ldc)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    ctx = B.Context(0, stream=stream)
    apply_settings(ctx, args.set)
    labels = np.zeros(len(wl.frac_S), np.int32)
    plan = B.SpherePlan(ctx, wl.lattice, wl.fftg, wl.frac_S, labels, [wl.species], "fp64")
    proj = torch.zeros((nk, nb, plan.ptot), dtype=torch.complex128, device="cuda")
    with torch.cuda.stream(stream):
        B.setup_projections(ctx, plan, wl.kpts, gofs, Gdev, CS, proj, "fp64")
    fine = tuple(int(2 * n) for n in wl.fftg)
    t0 = time.perf_counter()
    rs = B.RealspacePlan(ctx, wl.lattice, fine, wl.frac_S, labels, [wl.species])
    plan_s = time.perf_counter() - t0
    log(f"aedensity: grid {fine}, {rs.npts} sphere points, {rs.ncolors} colours, atomic {rs.atomic}, "
        f"plan {plan_s:.3f} s")
    dens = torch.zeros(fine, dtype=torch.float64, device="cuda")
    wk = [np.full(nb, 2.0 * wl.kws[k]) for k in range(nk)]

    def step(p, ks=range(nk)):
        for k in ks:
            B.realspace_states(ctx, rs, wl.kpts[k], Gdev[gofs[k]:gofs[k + 1]], CS[k], proj[k], density_out=dens,
                               weights=wk[k], precision=p, sync=False)

    if args.profile_step:
        # for rocprofv3 --pmc: the 1 GiB copy of the counter calibration and
        # one k-point (8 band chunks) of the first path
        a = torch.empty(1 << 28, dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        a.fill_(1.0)
        torch.cuda.synchronize()
        b.copy_(a)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            step([q for q in args.paths.split(",") if q][0], ks=[1])
        torch.cuda.synchronize()
        log("profile step done")
        return

    res = {}
    for p in [q for q in args.paths.split(",") if q]:
        with torch.cuda.stream(stream):
            for _ in range(args.warmup):
                step(p)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                step(p)
            e1.record(stream)
        torch.cuda.synchronize()
        t = e0.elapsed_time(e1) / 1e3 / args.steps
        # breakdown step: one chunk in flight, HIP events around every launch
        nstreams = ctx.get_param("streams")
        ctx.set_param("streams", 1)
        ctx.set_timing(True)
        ctx.timing_reset()
        with torch.cuda.stream(stream):
            step(p)
        torch.cuda.synchronize()
        kern = ctx.timing()
        ctx.set_timing(False)
        ctx.set_param("streams", nstreams)
        res[p] = {"step_s": t, "band_states_per_s": nb * nk / t, "kernels": kern}
        log(p, json.dumps({k: v for k, v in res[p].items() if k != "kernels"}))
        log(p, "kernels", json.dumps(kern))
    # algorithmic bytes per 64-band chunk (averaged over k): the FFT passes
    # restricted to the plane-wave sphere as in the projection path (z:
    # coefficients in, populated z-lines out; y: populated rows of the
    # x-slab in, the slab out; x: the slab in, the whole grid out),
    # augmentation and density in one pass: the chunk in, the density read
    # and written, the table (8 P per sphere point)
    npts = int(np.prod(fine))
    n0, n1, n2 = fine
    NBc = 64
    nchunks = nk * -(-nb // NBc)
    P = 18
    prune = bool(ctx.get_param("rs_prune"))
    rs_traffic = read_traffic_file(RS_TRAFFIC_FILE)
    roof = {}
    for p, r in res.items():
        pb = 16 if p == "fp64" else 8
        bx, by, bz = [], [], []
        for G in Gs:
            gx, gy = G[:, 0].astype(np.int64), G[:, 1].astype(np.int64)
            xs = int(gx.max() - gx.min() + 1) if prune else n0
            rows = np.unique(gx * 4096 + gy).size if prune else n0 * n1
            yrow = sum(int(gy[gx == x].max() - gy[gx == x].min() + 1) for x in np.unique(gx)) if prune else n0 * n1
            bx.append(NBc * pb * (n1 * n2 * xs + npts))
            by.append(NBc * pb * n2 * (yrow + xs * n1))
            bz.append(NBc * pb * ((len(G) if prune else npts) + rows * n2))
        alg = {"fft_z": float(np.mean(bz)), "fft_y": float(np.mean(by)), "fft_x": float(np.mean(bx)),
               "rs_augment": npts * (NBc * pb + 16) + rs.npts * 8 * P}
        kr = {}
        for c, b in alg.items():
            kc = r["kernels"].get(c)
            if not kc:
                continue
            ms = kc[0] / nchunks  # per chunk
            kr[c] = {"bound": "hbm", "achieved": b / (ms * 1e-3) / 1e9, "peak": PEAK_HBM / 1e9, "unit": "GB/s",
                     "alg_bytes_per_chunk": b, "ms_per_chunk": ms, "ms_per_step": kc[0], "launches": kc[1]}
            kr[c]["frac"] = kr[c]["achieved"] / kr[c]["peak"]
            kr[c]["traffic"] = rs_traffic.get(p, {}).get(c)
        roof[p] = kr
    # oracle check and CPU baseline on one state (band 0, k 1)
    errs, cpu = {}, None
    if not args.no_cpu:
        k, b = 1, 0
        W = orc.WaveData([wl.species])
        pr = proj[k, b].cpu().numpy()
        C0 = CS[k, b, :nw[k]].cpu().numpy()
        t0 = time.perf_counter()
        want = orc.realspace_state(wl.lattice, fine, wl.kpts[k], Gs[k], C0, W, labels, wl.frac_S, pr)
        tc = time.perf_counter() - t0
        cpu = {"value": 1.0 / tc, "unit": "band-states/s", "cores": 1, "kind": "port", "cpu_model": cpu_model(),
               "sample": f"oracle realspace_state of one state (band {b}, k {k}) on {fine}: {tc:.1f} s"}
        for p in res:
            one = torch.zeros((1,) + fine, dtype=torch.complex128, device="cuda")
            with torch.cuda.stream(stream):
                B.realspace_states(ctx, rs, wl.kpts[k], Gdev[gofs[k]:gofs[k + 1]], CS[k, b:b + 1], proj[k, b:b + 1],
                                   states_out=one, precision=p)
            got = one[0].cpu().numpy()
            errs[f"state_{p}"] = float(np.abs(got - want).max() / np.abs(want).max())
            del one
        log("errors vs the FP64 oracle:", json.dumps(errs), "cpu", json.dumps(cpu))
    head = "fp64" if "fp64" in res else next(iter(res))
    out = {"metric": "ae_density_band_states_per_sec", "value": res[head]["band_states_per_s"],
           "unit": "band-states/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
           "ms_per_step": res[head]["step_s"] * 1e3, "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": head, "data": "synthetic (seeded)",
           "config": {"workload": "all-electron density of the 216-atom S cell (215 sites, partial-wave spheres "
                                  "1.6 A) on the doubled grid 216^3, 4 k x 512 bands", "grid": list(fine),
                      "sphere_points": rs.npts, "colours": rs.ncolors, "plan_s": plan_s},
           "paths": {p: {k: v for k, v in r.items() if k != "kernels"} for p, r in res.items()},
           "kernels": roof, "max_err_vs_fp64_oracle": errs, "cpu_baseline": cpu}
    print(json.dumps(out), flush=True)
    rs.close()
    plan.close()


def pass_bytes(G, fftg, nb, prec_bytes, covered=None):
    """Algorithmic bytes of the three pruned FFT passes of one chunk of nb
    bands at one k-point (G its plane waves): z reads the coefficients in
    place and writes every populated z-line, y reads the populated rows of
    the x-slab and writes the slab, x reads the slab and writes the grid
    (or only the `covered` points)."""
    n0, n1, n2 = (int(v) for v in fftg)
    gx, gy = G[:, 0].astype(np.int64), G[:, 1].astype(np.int64)
    xs = int(gx.max() - gx.min() + 1)
    rows = np.unique(gx * 4096 + gy).size
    yrow = sum(int(gy[gx == x].max() - gy[gx == x].min() + 1) for x in np.unique(gx))
    bz = nb * prec_bytes * (len(G) + rows * n2)
    by = nb * prec_bytes * n2 * (yrow + xs * n1)
    bx = nb * prec_bytes * (n1 * n2 * xs + (covered if covered is not None else n0 * n1 * n2))
    return bx, by, bz


def bench_cfg3(args, torch, B):
    """The batched uneven workload: three perturbed copies of the 216-atom
    cell (the vacancy cell, a 0.05 A jitter, 8 sites moved 0.1 A) projected
    onto the bulk reference over `--nk` random k-points of the irreducible
    wedge whose plane-wave counts spread +-10%, with 384-640 bands per
    (structure, k).  One step = the setup of the three structures as one
    work list (pp_setup_projections_multi), the overlap of every structure
    with the reference at every k (one GEMM per (structure, k)) and O_M of
    all those pairs.  The reference is set up once.  The setup is also
    captured as one HIP graph and replayed.  Prints its own JSON line."""
    from oracle import pyoracle as orc
    from pawpyseed_amd import synthetic
    nk = args.nk
    wl = synthetic.config3(nk=nk)
    Gs = wl.ensure_gvecs()
    nw = np.array([len(g) for g in Gs], np.int32)
    gofs = np.concatenate([[0], np.cumsum(nw)]).astype(np.int32)
    Gd = torch.from_numpy(np.ascontiguousarray(np.concatenate(Gs), np.int32)).cuda()
    rec = synthetic.reciprocal_lattice(wl.lattice)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5005)
    # per (structure, k) coefficients of exactly nbands x ldc_k (structure 0 = the reference)
    C = [[None] * nk for _ in range(4)]
    for k in range(nk):
        kg = (Gs[k].astype(np.float64) + wl.kpts[k][None, :]) @ rec
        gcut = math.sqrt(synthetic.C_EV * wl.encuts[k])
        env = torch.from_numpy(np.exp(-np.einsum("ij,ij->i", kg, kg) / (2.0 * (0.5 * gcut) ** 2))
                               .astype(np.float32)).cuda()
        ldk = int(-(-nw[k] // 64) * 64)
        for s in range(4):
            nb = int(wl.nbands[s][k])
            c = torch.zeros((nb, ldk), dtype=torch.complex64, device="cuda")
            re = torch.randn((nb, int(nw[k])), generator=gen, device="cuda") * env
            im = torch.randn((nb, int(nw[k])), generator=gen, device="cuda") * env
            v = torch.complex(re, im)
            v /= torch.linalg.vector_norm(v, dim=1, keepdim=True)
            c[:, : nw[k]] = v
            C[s][k] = c
            del re, im, v
    torch.cuda.synchronize()
    log(f"cfg3: {nk} k, W {int(nw.min())}..{int(nw.max())}, bands {int(wl.nbands.min())}..{int(wl.nbands.max())}, "
        f"{torch.cuda.memory_allocated() / 2**30:.1f} GiB of coefficients")
    stream = torch.cuda.Stream()
    ctx = B.Context(0, stream=stream)
    apply_settings(ctx, args.set)
    paths = [p for p in args.paths.split(",") if p]
    res, kernels = {}, {}
    keep_out = {}
    for p in paths:
        plans = [B.SpherePlan(ctx, wl.lattice, wl.fftg, wl.frac[s], np.zeros(len(wl.frac[s]), np.int32),
                              [wl.species], p) for s in range(4)]
        P = [[torch.zeros((int(wl.nbands[s][k]), plans[s].ptot), dtype=torch.complex128, device="cuda")
              for k in range(nk)] for s in range(4)]
        O = [[torch.zeros((1, int(wl.nbands[0][k]), int(wl.nbands[s][k])), dtype=torch.complex128, device="cuda")
              for k in range(nk)] for s in range(4)]
        with torch.cuda.stream(stream):
            B.setup_projections_multi(ctx, plans[:1], wl.kpts, gofs, Gd, C[:1], P[:1], p)  # reference, once
            tuned, trials = None, []
            if not args.no_tune:
                ks = min(nk, 8)
                tuned, trials = B.autotune_multi(ctx, plans[1:], wl.kpts[:ks], gofs[: ks + 1], Gd,
                                                 [C[s][:ks] for s in range(1, 4)], [P[s][:ks] for s in range(1, 4)],
                                                 p, repeats=1)
                log(p, "autotune (first", ks, "k)", json.dumps(tuned))

        def step(ev):
            with torch.cuda.stream(stream):
                ev[0].record(stream)
                for s in range(1, 4):
                    plans[s].rebuild(wl.frac[s])
                B.setup_projections_multi(ctx, plans[1:], wl.kpts, gofs, Gd, C[1:], P[1:], p, sync=False)
                ev[1].record(stream)
                for s in range(1, 4):
                    for k in range(nk):
                        B.overlap_gemm(ctx, 1, 1, False, nw[k:k + 1], C[0][k].unsqueeze(0), C[s][k].unsqueeze(0),
                                       O[s][k], p, sync=False)
                ev[2].record(stream)
                for s in range(1, 4):
                    M_R, M_S = wl.M[s - 1]
                    for k in range(nk):
                        B.augmentation(ctx, 1, 1, False, P[0][k].unsqueeze(0), plans[0].proj_off,
                                       np.zeros(len(wl.frac[0]), np.int32), P[s][k].unsqueeze(0),
                                       plans[s].proj_off, np.zeros(len(wl.frac[s]), np.int32), M_R, M_S,
                                       [wl.species], [wl.delta_o], O[s][k], sync=False)
                ev[3].record(stream)

        for _ in range(args.warmup):
            step([torch.cuda.Event(enable_timing=True) for _ in range(4)])
        torch.cuda.synchronize()
        rec_ev = []
        t0 = time.perf_counter()
        for _ in range(args.steps):
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
            step(ev)
            rec_ev.append(ev)
        torch.cuda.synchronize()
        wall = (time.perf_counter() - t0) / args.steps
        ts = np.mean([e[0].elapsed_time(e[1]) for e in rec_ev]) / 1e3
        to = np.mean([e[1].elapsed_time(e[2]) for e in rec_ev]) / 1e3
        ta = np.mean([e[2].elapsed_time(e[3]) for e in rec_ev]) / 1e3
        # breakdown: one batch in flight, HIP events around every launch
        nstreams = ctx.get_param("streams")
        ctx.set_param("streams", 1)
        ctx.set_timing(True)
        ctx.timing_reset()
        step([torch.cuda.Event(enable_timing=True) for _ in range(4)])
        torch.cuda.synchronize()
        kt = ctx.timing()
        ctx.set_timing(False)
        ctx.set_param("streams", nstreams)
        # the setup replayed as one graph
        ts_graph = None
        if not args.no_graph:
            with torch.cuda.stream(stream):
                g = B.MultiGraph(ctx, plans[1:], wl.kpts, gofs, Gd, C[1:], P[1:], p)
                g0, g1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                g0.record(stream)
                for _ in range(args.steps):
                    g.replay(sync=False)
                g1.record(stream)
            torch.cuda.synchronize()
            ts_graph = g0.elapsed_time(g1) / 1e3 / args.steps
            g.close()
        nproj = sum(int(wl.nbands[s][k]) * plans[s].ptot for s in range(1, 4) for k in range(nk))
        flops = sum(8.0 * int(wl.nbands[0][k]) * int(wl.nbands[s][k]) * int(nw[k]) for s in range(1, 4)
                    for k in range(nk))
        res[p] = dict(setup_s=ts, overlap_s=to, aug_s=ta, step_wall_s=wall, band_projections_per_s=nproj / ts,
                      overlap_tflops=flops / to / 1e12, setup_s_graph_replay=ts_graph,
                      band_projections_per_s_graph_replay=nproj / ts_graph if ts_graph else None,
                      autotune=tuned, autotune_trials=[list(t) for t in trials])
        log(p, json.dumps(res[p]))
        log(p, "kernels (breakdown step)", json.dumps(kt))
        # algorithmic bytes of the setup's kernel classes over all items of a step
        pb = 8 if p != "fp64" else 16
        alg = {"fft_x": 0.0, "fft_y": 0.0, "fft_z": 0.0, "sphere_sum": 0.0, "scatter": 0.0}
        # with fft_xmask the x pass writes only the points a structure's
        # projector spheres hold
        xmask_on = bool((tuned or {}).get("fft_xmask", ctx.get_param("fft_xmask")))
        covered = {s: plans[s].coverage() for s in range(1, 4)} if xmask_on else {}
        for k in range(nk):
            for s in range(1, 4):
                bx, by, bz = pass_bytes(Gs[k], wl.fftg, 1, pb, covered.get(s))
                nb = int(wl.nbands[s][k])
                alg["fft_x"] += bx * nb
                alg["fft_y"] += by * nb
                alg["fft_z"] += bz * nb
                alg["scatter"] += (8 + pb) * int(nw[k]) * nb
                P_site = plans[s].ptot // len(wl.frac[s])
                alg["sphere_sum"] += plans[s].npts * (nb * pb + P_site * pb // 2 + pb + 4)
        kr = {}
        for c, b in alg.items():
            if c not in kt:
                continue
            ms, n = kt[c]
            kr[c] = {"bound": "hbm", "achieved": b / (ms * 1e-3) / 1e9, "peak": PEAK_HBM / 1e9, "unit": "GB/s",
                     "alg_bytes_per_step": b, "ms_per_step": ms, "launches": n, "avg_launch_ms": ms / max(1, n)}
            kr[c]["frac"] = kr[c]["achieved"] / kr[c]["peak"]
        kernels[p] = kr
        keep_out[p] = ({(s, k): P[s][k][[0, -1]].cpu().numpy() for s in range(1, 4) for k in (0, nk - 1)},
                       {(s, k): O[s][k][0, :4, :4].cpu().numpy() for s in range(1, 4) for k in (0, nk - 1)})
        for s in range(4):
            plans[s].close()
        del P, O
        torch.cuda.empty_cache()
    # oracle: sampled bands of every structure at the first and last k-point
    errs, cpu = {}, None
    if not args.no_cpu:
        cores = cpu_cores()
        fft_lib = cpu_fft(orc)
        tsum, npairs = 0.0, 0
        want_P = {}
        for s in range(1, 4):
            labels = np.zeros(len(wl.frac[s]), np.int32)
            T = orc.site_tables(wl.lattice, wl.fftg, wl.frac[s], [wl.species], labels)
            for k in (0, nk - 1):
                Ch = C[s][k][[0, -1], : nw[k]].cpu().numpy()
                t0 = time.perf_counter()
                want_P[(s, k)] = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts[k:k + 1], [Gs[k]], [Ch], T,
                                                       nthreads=cores)[0]
                tsum += time.perf_counter() - t0
                npairs += 2
        per_pair = tsum / npairs
        total_pairs = sum(int(wl.nbands[s][k]) for s in range(1, 4) for k in range(nk))
        nproj_all = sum(int(wl.nbands[s][k]) * (3888 if len(wl.frac[s]) == 216 else 3870) for s in range(1, 4)
                        for k in range(nk))
        cpu = {"value": nproj_all / (per_pair * total_pairs), "unit": "band-projections/s", "cores": cores,
               "kind": "port", "cpu_model": cpu_model(), "fft": fft_lib,
               "sample": f"oracle scatter/FFT/sphere sums of {npairs} (structure, k, band) samples in {tsum:.1f} s "
                         f"on {cores} threads ({per_pair * 1e3:.1f} ms each), extrapolated to all {total_pairs}"}
        for p, (gp, go) in keep_out.items():
            e = 0.0
            for key, w in want_P.items():
                e = max(e, float(np.abs(gp[key] - w).max() / np.abs(w).max()))
            errs[f"projections_{p}"] = e
        # overlap + O_M of the sampled 4 x 4 blocks: FP64 sums of the stored
        # coefficients and the oracle's O_M on its own projections
        labels0 = np.zeros(len(wl.frac[0]), np.int32)
        T0 = orc.site_tables(wl.lattice, wl.fftg, wl.frac[0], [wl.species], labels0)
        refs = {}
        for s in range(1, 4):
            Ts = orc.site_tables(wl.lattice, wl.fftg, wl.frac[s], [wl.species], np.zeros(len(wl.frac[s]), np.int32))
            M_R, M_S = wl.M[s - 1]
            for k in (0, nk - 1):
                a = C[0][k][:4, : nw[k]].cpu().numpy()
                b = C[s][k][:4, : nw[k]].cpu().numpy()
                ref = a.astype(np.complex128).conj() @ b.astype(np.complex128).T
                PR = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts[k:k + 1], [Gs[k]], [a], T0, nthreads=cores)
                PS = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts[k:k + 1], [Gs[k]], [b], Ts, nthreads=cores)
                for j in range(4):
                    ref[:, j] += orc.compensation_terms_m(np.zeros(4, complex), 0, 1, 1, PR, T0, labels0,
                                                          PS[:, j], Ts, M_R, M_S, [wl.delta_o], [wl.species.ls])
                refs[(s, k)] = ref
        for p, (gp, go) in keep_out.items():
            errs[f"overlap_total_{p}"] = max(float(np.abs(o - refs[key]).max() / np.abs(refs[key]).max())
                                             for key, o in go.items())
        log("errors vs the FP64 oracle:", json.dumps(errs), "cpu", json.dumps(cpu))
    head = "fp32" if "fp32" in res else paths[0]
    R = res[head]
    kr = kernels[head]
    dom = max(kr, key=lambda c: kr[c]["ms_per_step"]) if kr else None
    roof = None
    if dom:
        roof = {k: kr[dom][k] for k in ("bound", "achieved", "peak", "unit", "frac")}
        roof.update(kernel=dom, traffic=None, avg_launch_ms=kr[dom]["avg_launch_ms"],
                    timing="breakdown step: one batch of work items in flight, HIP events per launch; achieved = "
                           "algorithmic bytes of the class over the step / its launch time")
    out = {"metric": "band_projections_per_sec", "value": R["band_projections_per_s"], "unit": "band-projections/s",
           "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
           "ms_per_step": (R["setup_s"] + R["overlap_s"] + R["aug_s"]) * 1e3, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None,
           "dtype": "fp32 (FFT, sphere sums, overlap GEMM on MFMA; fp64 reductions and augmentation)"
           if head == "fp32" else head, "data": "synthetic (seeded)",
           "config": {"workload": f"3 perturbed 216-atom structures onto one reference, {nk} wedge k-points, "
                                  f"W {int(nw.min())}..{int(nw.max())} (+-10%), 384-640 bands per (structure, k), "
                                  "108^3 grid, 18 projectors/site", "nk": nk,
                      "plane_waves": nw.tolist(), "bands": wl.nbands.tolist()},
           "overlap_tflops": R["overlap_tflops"], "paths": res, "kernels": kernels, "roofline": roof,
           "max_err_vs_fp64_oracle": errs, "cpu_baseline": cpu}
    if "fp64" in res and head != "fp64":
        out["speedup_vs_fp64_gpu"] = R["band_projections_per_s"] / res["fp64"]["band_projections_per_s"]
    print(json.dumps(out), flush=True)


def cpu_and_errors(args, torch, wl, Gs, CR, CS, projR, projS, Om, ob, plans, results, head):
    """CPU baseline (the oracle on the host cores, a bounded sample) and
    errors of every path against the FP64 oracle on sampled entries."""
    from oracle import pyoracle as orc
    nk = len(Gs)
    nb = CR.shape[1]
    cores = cpu_cores()
    fft_lib = cpu_fft(orc)
    # S sphere tables (the per-structure setup of the CPU path)
    t0 = time.perf_counter()
    TS = orc.site_tables(wl.lattice, wl.fftg, wl.frac_S, wl.species)
    t_tab = time.perf_counter() - t0
    SB = sorted({0, 1, nb // 2, nb - 1})
    RB = sorted({0, 7, nb // 3})
    CSh = [CS[k, :, : len(Gs[k])].cpu().numpy() for k in range(nk)]
    # calibrate, then run a sample of (k, band) pairs sized to ~cpu-seconds
    pairs = [(k, b) for b in SB for k in range(nk)]
    t0 = time.perf_counter()
    P_or = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts, Gs, CSh, TS, pairs=np.array(pairs, np.int32),
                                 nthreads=cores)
    t_first = time.perf_counter() - t0
    per_pair = t_first / len(pairs)
    extra = int(max(0, (args.cpu_seconds - t_first - t_tab) / max(per_pair, 1e-3)))
    extra = min(extra, nk * nb - len(pairs))
    rng = np.random.default_rng(5)
    done = set(pairs)
    more = [p for p in ((int(rng.integers(nk)), int(rng.integers(nb))) for _ in range(4 * extra + 8))
            if p not in done][:extra]
    # the sample in five timed batches; the median per-pair time of the
    # batches (the first, calibration batch also warms up the thread pool)
    t_more, per_pair_batches = 0.0, []
    for batch in (np.array_split(np.array(more, np.int32), 5) if len(more) >= 5 else []):
        t0 = time.perf_counter()
        orc.setup_projections(wl.lattice, wl.fftg, wl.kpts, Gs, CSh, TS, pairs=batch, nthreads=cores)
        dt = time.perf_counter() - t0
        t_more += dt
        per_pair_batches.append(dt / len(batch))
    npairs = len(pairs) + len(more)
    t_pairs = t_first + t_more
    per_pair_med = float(np.median(per_pair_batches)) if per_pair_batches else t_first / len(pairs)
    t_cpu_all = t_tab + per_pair_med * nk * nb
    cpu_value = nb * nk * TS.ptot / t_cpu_all
    log(f"cpu: tables {t_tab:.2f}s, {npairs} pairs in {t_pairs:.2f}s on {cores} threads "
        f"(median of {len(per_pair_batches)} batches: {per_pair_med * 1e3:.2f} ms per pair) -> "
        f"{cpu_value:.4g} band-projections/s")

    # CPU overlap: the reference's FP32-accumulating cdotc, one projected band
    CRh = [CR[k, :, : len(Gs[k])].cpu().numpy() for k in range(nk)]
    t0 = time.perf_counter()
    ov_or = orc.pseudoprojection(CRh, CSh, SB[1], nk, 1, fp32acc=True)
    t_ov = time.perf_counter() - t0
    cpu_ov_tflops = 8.0 * nb * float(sum(len(g) for g in Gs)) / t_ov / 1e12

    # errors vs the FP64 oracle
    errs = {}
    for p in projS:
        g = projS[p].cpu().numpy()
        e = {}
        for k in range(nk):
            ref = P_or[k, SB]
            d = g[k, SB] - ref
            e[k] = dict(max_rel=float(np.abs(d).max() / np.abs(ref).max()),
                        rms_rel=float(np.sqrt(np.mean(np.abs(d) ** 2)) / np.sqrt(np.mean(np.abs(ref) ** 2))))
        errs[f"projections_{p}"] = e
    # overlap: FP64 oracle on sampled rows/columns
    CRs = [c[RB] for c in CRh]
    CSs = [c[SB] for c in CSh]
    ovref = np.zeros((nk, len(RB), len(SB)), np.complex128)
    for j in range(len(SB)):
        ovref[:, :, j] = orc.pseudoprojection(CRs, CSs, j, nk, 1).reshape(len(RB), nk).T
    # augmentation of the sampled pairs by the oracle, on FP64 oracle projections
    TR = orc.site_tables(wl.lattice, wl.fftg, wl.frac_R, wl.species)
    prR = orc.setup_projections(wl.lattice, wl.fftg, wl.kpts, Gs, [c[RB] for c in CRh], TR, nthreads=cores)
    prS = P_or[:, SB]
    aug = np.zeros((nk, len(RB), len(SB)), np.complex128)
    for j in range(len(SB)):
        a = orc.compensation_terms_m(np.zeros(len(RB) * nk, complex), 0, nk, 1, prR, TR,
                                     np.zeros(len(wl.frac_R), np.int32), prS[:, j], TS, wl.M_R, wl.M_S,
                                     [wl.delta_o], [wl.species.ls])
        aug[:, :, j] = a.reshape(len(RB), nk).T
    total_ref = ovref + aug
    for mode, o in ob.items():
        obh = o.cpu().numpy()[:, RB][:, :, SB]
        errs[f"overlap_{mode}_pseudo"] = {k: float(np.abs(obh[k] - ovref[k]).max() / np.abs(ovref[k]).max())
                                          for k in range(nk)}
    for p in Om:
        o = Om[p].cpu().numpy()[:, RB][:, :, SB]
        errs[f"overlap_total_{p}"] = {
            k: dict(max_rel=float(np.abs(o[k] - total_ref[k]).max() / np.abs(total_ref[k]).max()),
                    rms_rel=float(np.sqrt(np.mean(np.abs(o[k] - total_ref[k]) ** 2))
                                  / np.sqrt(np.mean(np.abs(total_ref[k]) ** 2))))
            for k in range(nk)}
    worst = {name: max((v["max_rel"] if isinstance(v, dict) else v) for v in e.values()) for name, e in errs.items()}
    log("errors (max over k of max|d|/max|ref|):", json.dumps(worst))
    return {
        "cpu_baseline": {"value": cpu_value, "unit": "band-projections/s", "cores": cores, "kind": "port",
                         "fft": fft_lib,
                         "sample": f"oracle on the host: S sphere tables (215 sites, {t_tab:.1f}s) + scatter/FFT/"
                                   f"sphere sums of {npairs} of {nk * nb} (band,k) pairs in {t_pairs:.1f}s "
                                   f"(median per-pair time of {len(per_pair_batches)} timed batches), "
                                   f"extrapolated to all pairs",
                         "cpu_model": cpu_model(),
                         "overlap_tflops": cpu_ov_tflops,
                         "overlap_sample": f"FP32-accumulated dots of 1 projected band vs {nb}x{nk} basis bands"},
        "max_err_vs_fp64_oracle": worst,
        "errors_per_k": errs,
        "speedup_vs_cpu": results[head]["band_projections_per_s"] / cpu_value,
    }


if __name__ == "__main__":
    main()
