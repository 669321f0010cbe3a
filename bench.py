#!/usr/bin/env python3
"""Benchmark: Mpaths/s of plain wavefront PT (pt2 semantics) on one MI355X.

Workload (the at-scale configuration): seeded procedural scene of 1,008,288
triangles (displaced 512x512 heightfield + 200 geodesic icospheres), GGX
metal / glass / mirror / Lambert materials, procedural 1024x512 HDR sky with a
sun disc, pinhole 1920x1080, max depth 16, 4 wavelengths per path, FP32
tracing/shading, FP64 framebuffer.  One step = one pass of 8 samples per pixel
over the full frame (16,588,800 camera paths through the regenerating wavefront);
the default 32 steps render the 256-spp frame.  Prints ONE JSON line.
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

METRIC = "Mpaths/s plain PT, and relMSE at equal time (plain vs learned guiding), 1 MI355X"
HBM_PEAK_GBS = 8000.0
TRACE_BYTES_PER_RAY = 48     # ray origin+direction read (32 B) + hit record written (16 B)
SHADE_BYTES_PER_PATH = 224   # hit 16 + path state 48 + material 32 read; state 48 + ray 32 + shadow 48 written
SHADOW_BYTES_PER_RAY = 36 + 32  # shadow ray 32 + contribution 16 + flags, radiance read/write


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=32)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--spp-per-step", type=int, default=8,
                    help="samples per pixel of one step (one pass over the frame); 32 steps x 8 = the 256-spp frame")
    ap.add_argument("--width", type=int, default=1920)
    ap.add_argument("--height", type=int, default=1080)
    ap.add_argument("--depth", type=int, default=16)
    ap.add_argument("--cpu-baseline", type=int, default=1, help="time the oracle on the host (0 = skip)")
    ap.add_argument("--cpu-sample-rows", type=int, default=0, help="rows of the frame the CPU sample renders (0 = auto)")
    ap.add_argument("--wavefront", type=int, default=0)
    ap.add_argument("--copy-calibration-mib", type=int, default=0,
                    help="only run device-to-device copies of this size (PMC byte-counter calibration) and exit")
    ap.add_argument("--relmse-budget", type=float, default=1.0,
                    help="seconds per method for the equal-time relMSE comparison (0 = skip)")
    ap.add_argument("--relmse-size", type=int, default=256)
    ap.add_argument("--media", type=int, default=1,
                    help="also measure the participating-media workload (pt2 Mpaths/s, guided relMSE at equal time)")
    ap.add_argument("--guide-max-spp", type=int, default=16)
    ap.add_argument("--nn-size", type=int, default=2048, help="frame side of the learned-guide inference roofline")
    ap.add_argument("--nn-guide-max-spp", type=int, default=4, help="training passes of the inference roofline's guide")
    ap.add_argument("--leg", default="all", choices=["all", "nn", "media", "guided", "cornell"],
                    help="run one leg alone and print its JSON (for profiling): the learned guide's inference "
                         "roofline, the media throughput, or the equal-time relMSE comparison")
    ap.add_argument("--pmc-program", default="bench", help="output name of the --pmc runs --summarize-pmc reads")
    ap.add_argument("--summarize-counters", default="",
                    help="print the markdown table of every counter of a directory of rocprofv3 --pmc CSV runs and exit")
    ap.add_argument("--summarize-pmc", default="",
                    help="print the markdown traffic summary of a directory of rocprofv3 --pmc CSV runs and exit")
    return ap.parse_args()


TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "traffic_terrain_1080p.md")
COPY_MIB = 256


def _demangle_nested(m):
    """Qualified name of an Itanium-mangled nested function name (_ZN <len><id>... [I<args>E] E),
    with integer / bool template arguments; the anonymous namespace is left out.  (The binutils
    demangler does not know the bf16 parameter types these kernels take.)"""
    i, parts = 3, []
    while i < len(m) and m[i].isdigit():
        j = i
        while m[j].isdigit():
            j += 1
        n = int(m[i:j])
        ident = m[j:j + n]
        i = j + n
        if i < len(m) and m[i] == "I":
            args, i = [], i + 1
            while i < len(m) and m[i] == "L":
                k = m.index("E", i)
                lit = m[i + 2:k]
                args.append({"b0": "false", "b1": "true"}.get(m[i + 1:k], lit))
                i = k + 1
            i += 1  # the E closing the template arguments
            ident += "<" + ", ".join(args) + ">"
        if not ident.startswith("_GLOBAL__N"):
            parts.append(ident)
    return "::".join(parts) if parts else m


def _kernel_name(raw):
    """Short kernel name: demangled where the trace kept the mangled one, without the return type
    ("void ttgpu::k_shade<false>(...)"), the anonymous namespace and the parameter list."""
    name = _demangle_nested(raw) if raw.startswith("_ZN") else raw
    name = name.replace("(anonymous namespace)::", "")
    if name.startswith("void "):
        name = name[len("void "):]
    return name.split("(")[0]


def _pmc_means(csv_path):
    import csv
    import collections
    acc = collections.defaultdict(list)
    for row in csv.DictReader(open(csv_path)):
        acc[_kernel_name(row["Kernel_Name"])].append(float(row["Counter_Value"]))
    return {k: (sum(v) / len(v), len(v)) for k, v in acc.items()}


def _pmc_table(csv_path):
    """{kernel: {counter: (mean value per dispatch, dispatches)}} of one rocprofv3 --pmc CSV."""
    import csv
    import collections
    acc = collections.defaultdict(lambda: collections.defaultdict(list))
    names = {}
    for row in csv.DictReader(open(csv_path)):
        raw = row["Kernel_Name"]
        if raw not in names:
            names[raw] = _kernel_name(raw)
        acc[names[raw]][row["Counter_Name"]].append(float(row["Counter_Value"]))
    return {k: {c: (sum(v) / len(v), len(v)) for c, v in cs.items()} for k, cs in acc.items()}


SIMDS = 1024  # 256 CUs x 4 SIMDs
XCDS = 8      # GRBM_GUI_ACTIVE is summed over the 8 XCDs: cycles of the dispatch = value / 8


def summarize_counters(d):
    """Markdown table of every counter found in the --pmc runs under d (one sub-directory per run),
    mean per dispatch for each ttgpu kernel, with the ratios derived from them: VALU lane use
    (SQ_THREAD_CYCLES_VALU / SQ_ACTIVE_INST_VALU / 64), VALU busy (the share of SIMD cycles issuing
    VALU work: SQ_ACTIVE_INST_VALU x 4 cycles / (SIMDs x GRBM_GUI_ACTIVE / XCDs)), L2 hit rate
    (TCC_HIT / (TCC_HIT + TCC_MISS)), MFMA busy (SQ_VALU_MFMA_BUSY_CYCLES / (SIMDs x
    GRBM_GUI_ACTIVE / XCDs)) and the bf16 MFMA operations counted by the hardware
    (SQ_INSTS_VALU_MFMA_MOPS_BF16 x 512)."""
    import glob
    merged = {}
    for f in sorted(glob.glob(os.path.join(d, "*", "*_counter_collection.csv"))):
        for k, cs in _pmc_table(f).items():
            merged.setdefault(k, {}).update(cs)
    counters = sorted({c for cs in merged.values() for c in cs})
    lines = ["| kernel | dispatches | " + " | ".join(counters) + " | derived |", "|---" * (len(counters) + 3) + "|"]
    for k in sorted(merged, key=lambda k: -max(v[0] for v in merged[k].values())):
        if "ttgpu" not in k:
            continue
        cs = merged[k]
        v = {c: cs[c][0] for c in cs}
        n = max(x[1] for x in cs.values())
        der = []
        if "SQ_THREAD_CYCLES_VALU" in v and v.get("SQ_ACTIVE_INST_VALU"):
            der.append(f"VALU lanes active {100 * v['SQ_THREAD_CYCLES_VALU'] / v['SQ_ACTIVE_INST_VALU'] / 64:.1f} %")
        if "SQ_ACTIVE_INST_VALU" in v and v.get("GRBM_GUI_ACTIVE"):
            der.append(f"VALU busy {100 * v['SQ_ACTIVE_INST_VALU'] * 4 / (SIMDS * v['GRBM_GUI_ACTIVE'] / XCDS):.1f} %")
        hit, miss = v.get("TCC_HIT_sum"), v.get("TCC_MISS_sum")
        if hit is not None and miss is not None and hit + miss > 0:
            der.append(f"L2 hit {100 * hit / (hit + miss):.1f} %")
        if "SQ_VALU_MFMA_BUSY_CYCLES" in v and v.get("GRBM_GUI_ACTIVE"):
            der.append(f"MFMA busy {100 * v['SQ_VALU_MFMA_BUSY_CYCLES'] / (SIMDS * v['GRBM_GUI_ACTIVE'] / XCDS):.2f} %")
        if "SQ_INSTS_VALU_MFMA_MOPS_BF16" in v:
            der.append(f"bf16 MFMA {v['SQ_INSTS_VALU_MFMA_MOPS_BF16'] * 512 / 1e9:.3f} GFLOP/dispatch")
        row = " | ".join(f"{v[c]:.4g}" if c in v else "" for c in counters)
        lines.append(f"| {k} | {n} | {row} | {'; '.join(der)} |")
    return "\n".join(lines)


def summarize_pmc(d, prog="bench"):
    """Per-dispatch HBM traffic of each kernel from FETCH_SIZE / WRITE_SIZE runs of the program
    `prog` (output name of the rocprofv3 runs), each counter scaled by its reading for a plain
    device-to-device copy of COPY_MIB MiB (bytes moved / counter KiB)."""
    lines = []
    scale = {}
    for ctr in ("FETCH_SIZE", "WRITE_SIZE"):
        copy = _pmc_means(os.path.join(d, f"copy_{ctr}", f"copy_counter_collection.csv"))
        kib, _ = copy["__amd_rocclr_copyBuffer"]
        scale[ctr] = (COPY_MIB << 20) / kib
    bench = {ctr: _pmc_means(os.path.join(d, f"{prog}_{ctr}", f"{prog}_counter_collection.csv")) for ctr in ("FETCH_SIZE", "WRITE_SIZE")}
    lines.append("| kernel | dispatches | FETCH_SIZE KiB/dispatch | WRITE_SIZE KiB/dispatch | HBM read MB | HBM write MB | HBM total MB |")
    lines.append("|---|---|---|---|---|---|---|")
    machine = []
    for k in sorted(bench["FETCH_SIZE"], key=lambda k: -bench["FETCH_SIZE"][k][0]):
        if not k.startswith("ttgpu::"):
            continue
        f, n = bench["FETCH_SIZE"][k]
        w, _ = bench["WRITE_SIZE"].get(k, (0.0, 0))
        rb, wb = f * scale["FETCH_SIZE"], w * scale["WRITE_SIZE"]
        lines.append(f"| {k} | {n} | {f:.1f} | {w:.1f} | {rb / 1e6:.2f} | {wb / 1e6:.2f} | {(rb + wb) / 1e6:.2f} |")
        machine.append(f"traffic_bytes_per_dispatch {k.split('::')[-1]} {rb + wb:.0f}")
    head = [f"Calibration: a {COPY_MIB} MiB device-to-device copy reads {(COPY_MIB << 20) / scale['FETCH_SIZE']:.1f} KiB of "
            f"FETCH_SIZE and writes {(COPY_MIB << 20) / scale['WRITE_SIZE']:.1f} KiB of WRITE_SIZE, so bytes = "
            f"FETCH_SIZE KiB x {scale['FETCH_SIZE']:.1f} and WRITE_SIZE KiB x {scale['WRITE_SIZE']:.1f}.", ""]
    return "\n".join(head + lines + [""] + machine)


def load_traffic(kernel):
    """Calibrated HBM bytes per dispatch of `kernel` from the committed PMC summary, or None."""
    try:
        for line in open(TRAFFIC_SUMMARY):
            parts = line.split()
            if len(parts) == 3 and parts[0] == "traffic_bytes_per_dispatch" and parts[1] == kernel:
                return float(parts[2])
    except OSError:
        pass
    return None


COUNTER_SUMMARY = os.path.join(ROOT, "profiles", "counters_terrain_1080p.md")


def load_counter_bound(kernel):
    """What the committed hardware-counter summary says bounds `kernel`: the share of SIMD cycles
    issuing VALU work, the share of lanes active in them and the L2 hit rate, or None."""
    import re
    try:
        for line in open(COUNTER_SUMMARY):
            if line.startswith(f"| ttgpu::{kernel} |"):
                out = {}
                for key, pat in (("valu_busy", r"VALU busy ([0-9.]+) %"), ("valu_lanes_active", r"VALU lanes active ([0-9.]+) %"),
                                 ("l2_hit", r"L2 hit ([0-9.]+) %")):
                    m = re.search(pat, line)
                    if m:
                        out[key] = round(float(m.group(1)) / 100, 3)
                out["source"] = os.path.relpath(COUNTER_SUMMARY, ROOT)
                return out
    except OSError:
        pass
    return None


def copy_calibration(mib, repeats=4):
    """Plain device-to-device copies of a known size through the HIP runtime (one copy kernel each), so the
    FETCH_SIZE / WRITE_SIZE counters of a profiled run can be scaled to bytes."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    n = mib << 20
    a, b = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(a), C.c_size_t(n)) == 0 and hip.hipMalloc(C.byref(b), C.c_size_t(n)) == 0
    assert hip.hipMemset(a, 1, C.c_size_t(n)) == 0
    for _ in range(repeats):
        assert hip.hipMemcpy(b, a, C.c_size_t(n), 3) == 0  # hipMemcpyDeviceToDevice
    assert hip.hipDeviceSynchronize() == 0
    hip.hipFree(a)
    hip.hipFree(b)
    print(json.dumps({"copy_calibration_bytes": n, "copies": repeats}), flush=True)


def relmse(img, ref, eps=1e-2, ref_se=None):
    """mean over pixels and RGB channels of (I - I_ref)^2 / (I_ref^2 + eps), linear RGB.  With the
    reference's standard error, its own variance is taken out of the squared difference (it adds
    the same amount to every method)."""
    d2 = (img - ref) ** 2
    if ref_se is not None:
        d2 = d2 - ref_se ** 2
    return float(np.mean(d2 / (ref ** 2 + eps)))


GOLDEN = os.path.join(ROOT, "tests", "golden")
SCENES = {
    # the guided workloads: the Cornell box with its light behind a baffle, and the glass sphere
    # filled with a chromatic medium (the participating-media scene)
    "cornell_hidden_light": ("cornell_hidden_light", 8),
    "medium_sphere": ("medium_sphere", 16),
}


def relmse_equal_time(budget_s, size, guide_max_spp, repeats=3, scene_name="cornell_hidden_light"):
    """relMSE of plain pt2, vMF-tree, quadtree and learned guiding after the same wall time each
    (guide training included; scene upload and BVH build excluded), against the oracle's converged
    FP64 render of the same scene (tests/golden/<scene><size>_ref.npz, written by
    tests/golden/make_relmse_refs.py; its own noise is taken out).  Each method runs `repeats`
    times with different seeds; the median relMSE is reported (a single 1 s run varies by tens of
    percent)."""
    import threading
    from naivetrace_amd import abi, configs
    from naivetrace_amd.renderer import GpuRenderer
    builder, depth = SCENES[scene_name]
    scene = getattr(configs, builder)(size, size)
    f = np.load(os.path.join(GOLDEN, f"{scene_name}{size}_ref.npz"))
    assert int(f["width"]) == size and int(f["max_depth"]) == depth and int(f["mis_mode"]) == abi.MIS_CONSISTENT
    ref, ref_se = f["mean"].astype(np.float64), f["stderr"].astype(np.float64)
    n_sweeps = int(np.log2(guide_max_spp)) if guide_max_spp >= 2 else 0

    def timed(params, guided):
        with GpuRenderer(scene, params) as r:
            stamps = []
            r.set_pass_callback(lambda complete: stamps.append(time.perf_counter()))
            timer = threading.Timer(budget_s, r.request_stop)
            t0 = time.perf_counter()
            timer.start()
            r.run()
            timer.cancel()
            dt = time.perf_counter() - t0
            _, _, n = r.framebuffer()
            img = r.mean_image()
            res = {"relmse": relmse(img, ref, ref_se=ref_se), "relmse_uncorrected": round(relmse(img, ref), 7),
                   "spp": float(n.mean()), "wall_s": round(dt, 3)}
            if guided and len(stamps) > n_sweeps:
                res["training_s"] = round(stamps[n_sweeps] - t0, 3)
            return res

    out = {"scene": f"{scene_name} {size}x{size}, depth {depth}", "budget_s": budget_s,
           "reference": f"oracle FP64 CPU render, {int(f['spp'])} spp (tests/golden/{scene_name}{size}_ref.npz)",
           "reference_relmse_floor": round(float(np.mean(ref_se ** 2 / (ref ** 2 + 1e-2))), 8), "guide_max_spp": guide_max_spp}
    def median_of(make, guided):
        runs = [timed(make(rep), guided) for rep in range(repeats)]
        runs.sort(key=lambda r: r["relmse"])
        res = dict(runs[len(runs) // 2])
        res["relmse_runs"] = [round(r["relmse"], 7) for r in runs]
        return res

    def plain(rep):
        p = abi.default_params(size, size, max_depth=depth, seed=5 + 100 * rep)
        p.mis_mode = abi.MIS_CONSISTENT
        return p

    out["repeats"] = repeats
    out["plain"] = median_of(plain, False)
    for name, kind in (("vmf_tree", abi.GUIDE_VMF_TREE), ("quadtree", abi.GUIDE_QUADTREE), ("learned", abi.GUIDE_LEARNED)):
        def guided(rep, kind=kind):
            g = abi.default_params(size, size, max_depth=depth, seed=6 + 100 * rep, algo=abi.ALGO_PTG)
            g.guide_kind = kind
            g.guide_max_spp = guide_max_spp
            return g
        out[name] = median_of(guided, True)
    for name in ("vmf_tree", "quadtree", "learned"):
        out[f"gain_{name}"] = round(out["plain"]["relmse"] / max(out[name]["relmse"], 1e-30), 3)
    # The tree guides once more with their per-pass fit on the host threads (TTGPU_GUIDE_HOST_FIT=1,
    # one run each): what moving the fit to the device buys at equal time.
    for name, kind in (("vmf_tree", abi.GUIDE_VMF_TREE), ("quadtree", abi.GUIDE_QUADTREE)):
        g = abi.default_params(size, size, max_depth=depth, seed=6, algo=abi.ALGO_PTG)
        g.guide_kind = kind
        g.guide_max_spp = guide_max_spp
        os.environ["TTGPU_GUIDE_HOST_FIT"] = "1"
        try:
            res = timed(g, True)
        finally:
            os.environ.pop("TTGPU_GUIDE_HOST_FIT", None)
        res["gain"] = round(out["plain"]["relmse"] / max(res["relmse"], 1e-30), 3)
        out[f"{name}_host_fit"] = res
    return out


NN_FWD_FLOP_PER_RECORD = 2 * (38 * 64 + 64 * 64 + 64 * 64 + 64 * 80)  # 31,488: dense layers, true widths
BF16_DENSE_PEAK_TFLOPS = 2500.0


def nn_inference_roofline(size, guide_max_spp, spp=8):
    """Batched inference of the learned guide inside the wavefront (k_guide_infer): algorithmic
    dense-layer FLOPs (NN_FWD_FLOP_PER_RECORD per queued path) over its HIP-event time.  The frame
    (size x size, 2048 x 2048 = the 4,194,304-path wavefront by default) is one full wavefront per
    pass, so the first bounce of every pass queries the network for every path at once."""
    from naivetrace_amd import abi, configs
    from naivetrace_amd.renderer import GpuRenderer
    scene = configs.cornell_hidden_light(size, size)
    g = abi.default_params(size, size, spp=spp, max_depth=8, seed=6, algo=abi.ALGO_PTG)
    g.guide_kind = abi.GUIDE_LEARNED
    g.guide_max_spp = guide_max_spp
    with GpuRenderer(scene, g) as r:
        r.enable_kernel_timing(True)
        r.run()
        st = r.stats()
        infer_ms, infer_n = r.kernel_time("guide")
        train_ms, train_n = r.kernel_time("train")
        trace_ms, _ = r.kernel_time("trace")
        shade_ms, _ = r.kernel_time("shade")
    # Every queued path of every bounce is one query; rays_closest and the "guide" timer both
    # accumulate over all passes of the handle (training and rendering).
    records = st["rays_closest"]
    achieved = records * NN_FWD_FLOP_PER_RECORD / max(infer_ms * 1e-3, 1e-12) / 1e12
    return {"kernel": "k_guide_infer", "bound": "mfma", "unit": "TFLOP/s", "achieved": round(achieved, 2),
            "peak": BF16_DENSE_PEAK_TFLOPS, "frac": round(achieved / BF16_DENSE_PEAK_TFLOPS, 5),
            "flop_per_record": NN_FWD_FLOP_PER_RECORD, "queries": records, "launches": infer_n,
            "queries_per_launch": round(records / max(infer_n, 1)), "wavefront_paths": st["wavefront_paths"],
            "frame": [size, size], "spp": spp, "guide_max_spp": guide_max_spp,
            "avg_launch_ms": round(infer_ms / max(infer_n, 1), 4), "trace_ms_total": round(trace_ms, 2),
            "shade_ms_total": round(shade_ms, 2),
            "train_ms_total": round(train_ms, 2), "train_passes": train_n}


def media_throughput(width=1024, height=512, spp=8, passes=4, cpu_spp=8):
    """Plain pt2 through participating media at the media workload's resolution: the glass sphere
    filled with a chromatic Henyey-Greenstein medium (pinhole, depth 16), and the Earth atmosphere
    (exponential Rayleigh and Mie profiles, FP64 shell distances and altitudes) seen through an
    upward fisheye with the sun at 5 degrees (depth 8).  Mpaths/s over `passes` passes of `spp`
    after one warm-up pass, and the media kernels' share of the time; the oracle's Mpaths/s on the
    same frame at `cpu_spp`."""
    from naivetrace_amd import abi, configs
    from naivetrace_amd.renderer import GpuRenderer
    out = {}
    for name, scene, depth in (("medium_sphere", configs.medium_sphere(width, height), 16),
                               ("atmosphere", configs.atmosphere(width, height), 8)):
        p = abi.default_params(width, height, max_depth=depth, seed=3)
        with GpuRenderer(scene, p) as r:
            r.render_spp(spp)
            r.enable_kernel_timing(False)
            t0 = time.perf_counter()
            for _ in range(passes):
                r.render_spp(spp)
            dt = time.perf_counter() - t0
            r.enable_kernel_timing(True)
            c0 = r.stats()
            r.render_spp(spp)
            c1 = r.stats()
            kt = {k: r.kernel_time(k) for k in ("raygen", "trace", "shade", "shadow")}
        paths = width * height * spp * passes
        rays = c1["rays_closest"] - c0["rays_closest"]
        out[name] = {"mpaths_per_s": round(paths / dt / 1e6, 2), "width": width, "height": height, "max_depth": depth,
                     "spp": spp * passes, "rays_closest_per_path": round(rays / (width * height * spp), 3),
                     "kernel_ms_per_pass": {k: {"ms": round(v[0], 3), "launches": v[1]} for k, v in kt.items()}}
        if cpu_spp:
            try:
                out[name]["cpu_oracle"] = oracle_mpaths(scene, width, height, depth, cpu_spp)
            except Exception as e:  # reported, not fatal for the GPU number
                out[name]["cpu_oracle"] = {"error": str(e)}
    return out


def oracle_mpaths(scene, width, height, depth, spp, mis_mode=None):
    """The oracle's Mpaths/s (all host threads, render only) on the given frame and spp."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib
    from naivetrace_amd import abi
    oracle_lib.build()
    p = abi.default_params(width, height, max_depth=depth, seed=5)
    if mis_mode is not None:
        p.mis_mode = mis_mode
    oracle_lib.render(scene, p, spp, threads=os.cpu_count() or 1, with_sq=False)
    dt = oracle_lib.last_render_seconds()
    return {"mpaths_per_s": round(width * height * spp / dt / 1e6, 3), "cores": os.cpu_count() or 1,
            "sample": f"{width}x{height} x {spp} spp ({dt:.2f} s)"}


def cornell_throughput(size=256, depth=8, spp=64, passes=4, cpu_spp=32):
    """Plain pt2 on the Cornell box (36 triangles), 256x256, depth 8: GPU Mpaths/s over `passes`
    passes of `spp` samples per pixel (4.2 M paths each, the wavefront's capacity) after a
    warm-up pass; also over 8-spp passes (0.5 M paths, a quarter-full wavefront); and the
    oracle on `cpu_spp`."""
    from naivetrace_amd import abi, configs
    from naivetrace_amd.renderer import GpuRenderer
    scene = configs.cornell_box(size, size)
    p = abi.default_params(size, size, max_depth=depth, seed=3)
    with GpuRenderer(scene, p) as r:
        r.render_spp(spp)
        t0 = time.perf_counter()
        for _ in range(passes):
            r.render_spp(spp)
        dt = time.perf_counter() - t0
        t1 = time.perf_counter()
        for _ in range(spp // 8):
            r.render_spp(8)
        dt8 = time.perf_counter() - t1
    out = {"mpaths_per_s": round(size * size * spp * passes / dt / 1e6, 2), "width": size, "height": size, "max_depth": depth,
           "spp_per_pass": spp, "passes": passes, "mpaths_per_s_8spp_passes": round(size * size * spp / dt8 / 1e6, 2)}
    try:
        out["cpu_oracle"] = oracle_mpaths(scene, size, size, depth, cpu_spp)
    except Exception as e:  # reported, not fatal for the GPU number
        out["cpu_oracle"] = {"error": str(e)}
    return out


def cpu_baseline(scene, width, height, depth, rows, spp=2):
    """Oracle (FP64 C++ restatement of pt2, all host threads) on a bounded sample: `rows` rows x full
    width x `spp` spp (the full 1920x1080 frame at 2 spp takes about 10 s on 16 cores)."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib
    from naivetrace_amd import abi
    oracle_lib.build()
    threads = os.cpu_count() or 1
    # A width x rows image with the same horizontal field of view is exactly the central band of
    # rows of the full frame (pixel footprint 2 tan(fov/2)/width in both directions).
    p = abi.default_params(width, rows, max_depth=depth, seed=5)
    crop = scene
    oracle_lib.render(crop, p, spp, threads=threads, with_sq=False)
    dt = oracle_lib.last_render_seconds()
    paths = width * rows * spp
    return {"value": paths / dt / 1e6, "unit": "Mpaths/s", "cores": threads, "kind": "port",
            "sample": f"{rows} rows x {width} px x {spp} spp of the same scene ({paths} paths, {dt:.1f} s, oracle BVH build excluded)"}


def main():
    args = parse()
    if args.copy_calibration_mib:
        copy_calibration(args.copy_calibration_mib)
        return
    if args.summarize_pmc:
        print(summarize_pmc(args.summarize_pmc, args.pmc_program))
        return
    if args.summarize_counters:
        print(summarize_counters(args.summarize_counters))
        return
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; --gpus must be 1 (multi-GPU sharding is designed, not built)"}))
        sys.exit(2)
    from naivetrace_amd import abi, configs
    from naivetrace_amd.renderer import GpuRenderer

    if args.leg != "all":
        leg = {"nn": lambda: nn_inference_roofline(args.nn_size, args.nn_guide_max_spp),
               "media": media_throughput,
               "guided": lambda: relmse_equal_time(args.relmse_budget, args.relmse_size, args.guide_max_spp),
               "cornell": cornell_throughput}[args.leg]
        print(json.dumps({"leg": args.leg, "result": leg()}), flush=True)
        return

    t0 = time.time()
    scene = configs.terrain_instances(args.width, args.height)
    gen_s = time.time() - t0
    p = abi.default_params(args.width, args.height, max_depth=args.depth, seed=1)
    p.wavefront_paths = args.wavefront
    r = GpuRenderer(scene, p)
    st0 = r.stats()
    spp = args.spp_per_step
    for _ in range(args.warmup):
        r.render_spp(spp)
    r.reset()
    r.enable_kernel_timing(False)
    t1 = time.perf_counter()
    for _ in range(args.steps):
        r.render_spp(spp)
    t2 = time.perf_counter()
    st = r.stats()
    dt = t2 - t1
    paths = args.width * args.height * args.steps * spp
    value = paths / dt / 1e6

    # Kernel timing (HIP events on the library's own stream) over a separate timed pass.
    r.enable_kernel_timing(True)
    c0 = r.stats()
    nt = 1
    for _ in range(nt):
        r.render_spp(spp)
    c1 = r.stats()
    times = {k: r.kernel_time(k) for k in ("raygen", "trace", "shade", "shadow")}
    rays_closest = c1["rays_closest"] - c0["rays_closest"]
    rays_shadow = c1["rays_shadow"] - c0["rays_shadow"]
    paths_t = args.width * args.height * nt * spp
    # The roofline kernel: the longest of the per-ray / per-bounce kernels (the "raygen" timer also
    # holds the queue selections).
    dom = max(("trace", "shade", "shadow"), key=lambda k: times[k][0])
    ms_tot, launches = times[dom]
    avg_ms = ms_tot / max(launches, 1)
    # The closest-hit launches also trace the shadow rays (no shadow launches of their own): their
    # bytes count toward the traversal kernel.
    shadow_in_trace = times["shadow"][1] == 0
    if dom == "trace":
        alg_bytes = (TRACE_BYTES_PER_RAY * rays_closest + (SHADOW_BYTES_PER_RAY * rays_shadow if shadow_in_trace else 0)) / max(launches, 1)
    elif dom == "shadow":
        alg_bytes = SHADOW_BYTES_PER_RAY * rays_shadow / max(launches, 1)
    else:
        alg_bytes = SHADE_BYTES_PER_PATH * rays_closest / max(launches, 1)
    achieved = alg_bytes / (avg_ms * 1e-3) / 1e9
    # The trace kernels are templates on how they take shadow rays: <1> also traces them.
    kname = (f"k_trace<{1 if shadow_in_trace else 0}>" if dom == "trace"
             else "k_shade<false>" if dom == "shade" else f"k_{dom}")
    roofline = {"bound": "hbm", "achieved": round(achieved, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 5), "traffic": load_traffic(kname), "kernel": kname,
                "avg_launch_ms": round(avg_ms, 4), "counters": load_counter_bound(kname),
                "bytes_per_unit": {"trace": TRACE_BYTES_PER_RAY, "shade": SHADE_BYTES_PER_PATH, "shadow": SHADOW_BYTES_PER_RAY}[dom],
                "shadow_rays_in_trace": shadow_in_trace}
    if dom == "trace" and shadow_in_trace:
        roofline["bytes_per_unit"] = {"closest_hit_ray": TRACE_BYTES_PER_RAY, "shadow_ray": SHADOW_BYTES_PER_RAY}
    ktimes = {k: {"ms": round(v[0], 3), "launches": v[1]} for k, v in times.items()}
    r.close()

    guided = None
    nn_roof = None
    guided_media = None
    media = None
    if args.relmse_budget > 0:
        guided = relmse_equal_time(args.relmse_budget, args.relmse_size, args.guide_max_spp)
        nn_roof = nn_inference_roofline(args.nn_size, args.nn_guide_max_spp)
        if args.media:
            guided_media = relmse_equal_time(args.relmse_budget, args.relmse_size, args.guide_max_spp, scene_name="medium_sphere")
    if args.media:
        media = media_throughput()
    cornell = cornell_throughput() if args.media else None

    cpu = None
    if args.cpu_baseline:
        rows = args.cpu_sample_rows or args.height
        try:
            cpu = cpu_baseline(scene, args.width, args.height, args.depth, rows)
        except Exception as e:  # reported, not fatal for the GPU number
            cpu = {"error": str(e)}

    out = {
        "metric": METRIC, "value": round(value, 3), "unit": "Mpaths/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(dt / args.steps * 1e3, 3), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "fp32", "data": "synthetic",
        "config": {"workload": "terrain_instances: 1,008,288 tris (512x512 heightfield + 200 icospheres f=11), GGX/glass/mirror/"
                               "Lambert, 1024x512 HDR sky + sun disc, pinhole, 4 wavelengths/path",
                   "width": args.width, "height": args.height, "spp_per_step": spp, "spp_total": spp * args.steps, "max_depth": args.depth,
                   "triangles": scene.num_triangles, "wavefront_paths": st["wavefront_paths"]},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "relmse_equal_time": guided,
        "relmse_equal_time_media": guided_media,
        "media_throughput": media,
        "cornell_throughput": cornell,
        "roofline_nn": nn_roof,
        "detail": {"rays_closest_per_path": round(rays_closest / paths_t, 3), "rays_shadow_per_path": round(rays_shadow / paths_t, 3),
                   "mrays_per_s": round((rays_closest + rays_shadow) / (sum(v[0] for v in times.values()) * 1e-3) / 1e6, 1),
                   "kernel_ms": ktimes, "bvh_build_ms": round(st0["bvh_build_ms"], 1), "scene_gen_s": round(gen_s, 2),
                   "upload_ms": round(st0["upload_ms"], 1)},
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
