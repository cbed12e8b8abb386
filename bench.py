#!/usr/bin/env python3
"""Benchmark of the FDMAP time-stepping path on one MI355X.

Workload: the planar rate-and-state rupture, two blocks of 1601 x 801
points (h = 0.025 km) coupled by a frictional fault (slip law with strong
velocity weakening), LSRK(5,4) at CFL 0.5, built from its .in file by the
Fortran host.  A step is one full LSRK(5,4) step of the whole grid.

Prints one JSON line: FP64 updates/s (value), the roofline of the bulk
kernel measured with HIP events after the timed region, the FP32-bulk
throughput and its error against FP64 after the configuration's 4000 steps
(whatever --steps), and the CPU oracle timed on the host cores as the CPU
baseline.  Two more legs state the metric's other parts at their
configurations' own lengths: the rough fault with plasticity (2 x 4001 x
2001, 3000 steps, FP32-bulk against FP64: speed ratio and error) and the
adjoint gradient (2 x 801 x 401, 2000 steps: gradient time over forward
time with square-root checkpointing and with the fault trace kept, and the
finite-difference check).  --no-legs leaves them out.
"""
import argparse
import json
import os
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = ("updates/s & %HBM peak, FP32-bulk vs FP64 at stated L2 err; adjoint/fwd time")
HBM_PEAK_GBS = 8000.0
# algorithmic bytes per grid point per bulk launch: read F(6) + DF(6), write
# DF(6) + F(6), read 5 metric arrays; the first stage does not read DF
# (A1 = 0).  FP64: 232 B (184 B at stage 1); FP32-bulk: half.
BYTES_STAGE = {"fp64": (184.0, 232.0), "fp32": (92.0, 116.0)}
# what the interior tiles themselves must move, per point and stage: DF6 is
# neither read nor stored (no stage needs it); Ji is not read where the
# kernel forms it from the metrics (ji); the metrics take 4 FP32 deltas
# instead of 4 FP64 values where that encoding is exact (mc); the last
# stage of a step that another step of the same call follows does not store
# DF1..5


def kernel_min_bytes(prec, ns, ji=False, mc=False):
    """average bytes per point of the interior tiles over a step's stages"""
    e = 8.0 if prec == "fp64" else 4.0
    read = 6 * e + (16.0 if mc else 4 * e) + (0.0 if ji else e)
    tot = 0.0
    for s in range(1, ns + 1):
        tot += read + (5 * e if s > 1 else 0.0) + 6 * e + (5 * e if s < ns else 0.0)
    return tot / ns


def rel_l2(a, b):
    d = np.linalg.norm(np.asarray(b))
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / (d if d > 0 else 1.0))


def run_device(inpath, precision, steps, warmup, prof_steps, horizon=None):
    """Time `steps` steps after `warmup` untimed ones (the headline number),
    then `prof_steps` more with HIP events around every launch (kernel
    durations for the roofline).  horizon: keep stepping until that many
    steps in all, and return the fields and fault arrays there too (errors
    at the configuration's own length, whatever the timed steps)."""
    from fdmap_github_amd import host
    from fdmap_github_amd.device import Context

    from fdmap_github_amd import capi
    from fdmap_github_amd.device import FdmError

    hp = host.HostProblem(inpath, precision=precision)
    ctx = Context(hp.ptr)
    npts = hp.nx * hp.ny
    # the interior kernel's variant: Ji formed in the kernel (FP64, where the
    # given Ji is 1/(xq yr - xr yq) to the bit) and FP32-delta metrics (on
    # wherever fdm_create found them exact; setting the knob to 1 fails
    # where it did not)
    P = hp.ptr.contents
    ji = mc = False
    if precision == "fp64":
        m = {k: np.ctypeslib.as_array(getattr(P, k), shape=(hp.ny, hp.nx))
             for k in ("xq", "xr", "yq", "yr", "Ji")}
        ji = bool(np.array_equal(1.0 / (m["xq"] * m["yr"] - m["xr"] * m["yq"]), m["Ji"]))
        try:
            ctx._check(ctx.lib.fdm_tune(ctx.h, capi.FDM_TUNE_METRIC_F32, 1))
            mc = True
        except FdmError:
            mc = False
    ctx.set_fields(hp.fields())
    ctx.init_edges(hp.t)
    ctx.step(hp.t, hp.dt, 1, warmup)
    ctx.sync()
    t0 = time.perf_counter()
    ctx.step(hp.t, hp.dt, warmup + 1, steps)
    ctx.sync()
    el = time.perf_counter() - t0
    F, _ = ctx.get_fields()
    fault = {f: ctx.get_iface(0, f) for f in ("D", "V", "S")}
    ctx.profile_enable(True)
    ctx.sync()
    t0 = time.perf_counter()
    ctx.step(hp.t, hp.dt, warmup + steps + 1, prof_steps)
    ctx.sync()
    el_prof = time.perf_counter() - t0
    prof = ctx.profile_read()
    ctx.profile_enable(False)
    nstage = hp.ptr.contents.nstage
    done = warmup + steps + prof_steps
    Fh, fault_h = F, fault
    if horizon is not None and horizon > done:
        ctx.step(hp.t, hp.dt, done + 1, horizon - done)
        done = horizon
    if horizon is not None:
        Fh, _ = ctx.get_fields()
        fault_h = {f: ctx.get_iface(0, f) for f in ("D", "V", "S")}
    ctx.close()
    return dict(hp=hp, npts=npts, el=el, el_prof=el_prof, prof=prof, F=F, fault=fault,
                nstage=nstage, F_h=Fh, fault_h=fault_h, horizon=done, ji=ji, mc=mc)


def cpu_baseline(inpath, sample_steps):
    """Oracle (C restatement of the reference, OpenMP) on the same problem."""
    from fdmap_github_amd import host
    from oracle.binding import OracleContext

    threads = min(os.cpu_count() or 1, 16)
    hp = host.HostProblem(inpath, precision="fp64")
    o = OracleContext(hp.ptr, threads=threads)
    o.set_fields(hp.fields())
    o.init_edges(hp.t)
    o.step(hp.t, hp.dt, 1, 1)
    t0 = time.perf_counter()
    o.step(hp.t, hp.dt, 2, sample_steps)
    el = time.perf_counter() - t0
    return dict(value=hp.nx * hp.ny * sample_steps / el, unit="updates/s", cores=threads,
                kind="port",
                sample=f"{sample_steps} LSRK(5,4) steps of the same 2x(1601x801) problem "
                       f"({el:.1f} s wall on {threads} threads)")


def measured_traffic(name="bulk_interior_c2_fp64"):
    """HBM bytes per launch of the dominant kernel from the committed counter
    summary profiles/<name>_traffic.md (two rocprofv3 --pmc runs, FETCH_SIZE
    and WRITE_SIZE, each scaled by what the counter reads for a plain copy of
    known size)."""
    path = os.path.join(ROOT, "profiles", name + "_traffic.md")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        for line in f:
            if line.startswith("hbm_bytes_per_launch:"):
                return float(line.split(":", 1)[1])
    return None


def c3_measure(tmp, nx=4001, ny=2001, steps=3000, warmup=0, prof_steps=0):
    """Rough fault: a seeded band-limited self-similar profile (rms amplitude
    1e-2 of the fault length, wavelengths from 20 h to the fault length) as
    the shared edge of two curvilinear nx x ny blocks, C2's friction and
    prestress, Drucker-Prager plasticity (cohesion 0, friction 0.6); FP64 and
    FP32-bulk over the same steps, the FP32 error stated against FP64 after
    warmup + steps steps."""
    from fdmap_github_amd import inputs

    os.makedirs(tmp, exist_ok=True)
    h = 0.025
    x, y, n1, n2 = inputs.fractal_profile(nx, h, alpha=1e-2, seed=3)
    curve = os.path.join(tmp, "fault.bin")
    inputs.write_curve(curve, x, y, n1, n2)
    inpath = inputs.write(os.path.join(tmp, "c3.in"),
                          inputs.c2_planar_rs(name=os.path.join(tmp, "c3"), nx=nx, ny=ny, h=h,
                                              nsteps=steps + warmup + prof_steps,
                                              outputs=False, plastic=True, curve=curve))
    r64 = run_device(inpath, "fp64", steps, warmup, prof_steps)
    r32 = run_device(inpath, "fp32", steps, warmup, prof_steps)
    npts = r64["npts"]
    ups64 = npts * steps / r64["el"]
    ups32 = npts * steps / r32["el"]
    return dict(r64=r64, r32=r32, npts=npts, ups64=ups64, ups32=ups32, steps=steps, nx=nx, ny=ny,
                fp32={"updates_per_s": ups32, "speedup_vs_fp64": ups32 / ups64,
                      "ms_per_step": 1e3 * r32["el"] / steps,
                      "rel_l2_fields_vs_fp64": rel_l2(r32["F"], r64["F"]),
                      "rel_l2_slip_vs_fp64": rel_l2(r32["fault"]["D"], r64["fault"]["D"]),
                      "rel_l2_slip_velocity_vs_fp64": rel_l2(r32["fault"]["V"], r64["fault"]["V"]),
                      "after_steps": steps + warmup})


def run_c3(args, tmp):
    nx = 4001 if args.nx == 1601 else args.nx
    ny = 2001 if args.ny == 801 else args.ny
    steps = 3000 if args.steps == 4000 else args.steps
    m = c3_measure(tmp, nx, ny, steps, args.warmup, args.prof_steps)
    r64, r32 = m["r64"], m["r32"]
    out = {
        "metric": METRIC, "value": m["ups64"], "unit": "updates/s", "n_gpus": 1, "steps": steps,
        "warmup": args.warmup, "ms_per_step": 1e3 * r64["el"] / steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (rough-fault problem generated as an FDMAP .in file and curve file)",
        "config": {"workload": f"rough curvilinear fault with plasticity, 2 blocks x ({nx}x{ny}), "
                               "self-similar profile alpha 1e-2 seed 3, RFL slip law, "
                               "Drucker-Prager mu 0.6 b 0, LSRK(5,4) CFL 0.5",
                   "grid_points": m["npts"], "fault_nodes": nx},
        "fp32_bulk": m["fp32"],
        "avg_launch_ms": {prec: {k: r["prof"][k + "_ms"] / max(1, r["prof"][k + "_launches"])
                                 for k in ("bulk", "band", "edge")}
                          for prec, r in (("fp64", r64), ("fp32", r32))},
    }
    print(json.dumps(out), flush=True)


def run_c2_variant(args, tmp, het, cdiss):
    """C2 in a heterogeneous medium and/or with artificial dissipation: the
    same two blocks and fault.  het: rho, cs and cp vary smoothly by 10 %
    over the grid (seeded, read from a medium file); the interior kernel
    reads five more planes per point (rho, G, M, gamma, nu), 40 B more per
    point in FP64.  cdiss: Cdiss of both blocks (scaled by CFL/dt); the
    interior kernel reads the Jacobian, 8 B more per point.  FP32 halves
    both."""
    from fdmap_github_amd import inputs

    nx, ny = args.nx, args.ny
    med = None
    if het:
        rho, cs, cp = inputs.smooth_medium(nx, 2 * ny, 0.025, amp=0.1, seed=5)
        med = inputs.write_medium(os.path.join(tmp, "medium.bin"), rho, cs, cp)
    name = args.config
    inpath = inputs.write(os.path.join(tmp, name + ".in"),
                          inputs.c2_planar_rs(name=os.path.join(tmp, name), nx=nx, ny=ny,
                                              nsteps=args.steps + args.warmup + args.prof_steps,
                                              outputs=False, medium=med, Cdiss=cdiss))
    res = {}
    for prec in ("fp64",) if args.no_fp32 else ("fp64", "fp32"):
        r = run_device(inpath, prec, args.steps, args.warmup, args.prof_steps)
        ns, prof = r["nstage"], r["prof"]
        extra = (40.0 if het else 0.0) + (8.0 if cdiss else 0.0)
        if prec == "fp32":
            extra *= 0.5
        b1, b2 = (b + extra for b in BYTES_STAGE[prec])
        kpts = prof["bulk_points"]
        bytes_launch = kpts * (b1 + (ns - 1) * b2) / ns
        avg_ms = prof["bulk_ms"] / max(1, prof["bulk_launches"])
        achieved = bytes_launch / (avg_ms * 1e-3) / 1e9
        res[prec] = dict(r=r, ups=r["npts"] * args.steps / r["el"], avg_ms=avg_ms,
                         achieved=achieved, bytes_launch=bytes_launch, kpts=kpts)
    r64 = res["fp64"]
    out = {
        "metric": METRIC, "value": r64["ups"], "unit": "updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1e3 * r64["r"]["el"] / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (planar fault problem" + (" and seeded medium file)" if het else ")"),
        "config": {"workload": "planar rate-and-state rupture"
                               + (" in a heterogeneous medium (rho/cs/cp varying by 10 %, seed 5)"
                                  if het else "")
                               + (f" with artificial dissipation Cdiss {cdiss}" if cdiss else "")
                               + f", 2 blocks x ({nx}x{ny}), RFL slip law, LSRK(5,4) CFL 0.5",
                   "grid_points": r64["r"]["npts"], "fault_nodes": nx,
                   "dt": r64["r"]["hp"].dt},
        "roofline": {
            "bound": "hbm",
            "kernel": f"bulk_interior<double,64,4,0,true,{str(bool(het)).lower()},"
                      f"{str(bool(cdiss)).lower()},4,{str(r64['r']['ji']).lower()},"
                      f"{str(r64['r']['mc']).lower()},false>",
            "kernel_points": r64["kpts"], "achieved": r64["achieved"], "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": r64["achieved"] / HBM_PEAK_GBS,
            "traffic": measured_traffic(f"bulk_interior_{name}_fp64"),
            "alg_bytes_per_launch": r64["bytes_launch"], "avg_launch_ms": r64["avg_ms"],
        },
    }
    if "fp32" in res:
        r32 = res["fp32"]
        out["fp32_bulk"] = {
            "updates_per_s": r32["ups"], "speedup_vs_fp64": r32["ups"] / r64["ups"],
            "ms_per_step": 1e3 * r32["r"]["el"] / args.steps,
            "bulk_avg_launch_ms": r32["avg_ms"], "bulk_achieved_GBs": r32["achieved"],
            "rel_l2_fields_vs_fp64": rel_l2(r32["r"]["F"], r64["r"]["F"]),
            "rel_l2_slip_vs_fp64": rel_l2(r32["r"]["fault"]["D"], r64["r"]["fault"]["D"]),
            "rel_l2_slip_velocity_vs_fp64": rel_l2(r32["r"]["fault"]["V"],
                                                   r64["r"]["fault"]["V"]),
            "after_steps": args.steps + args.warmup,
        }
    print(json.dumps(out), flush=True)


def run_c2_sbp6(args, tmp):
    """C2 with the reference's default operator, SBP6 (domain.f90:94): the
    same grid, fault and byte count per point (the interior stencil reads a
    halo of 3 instead of 2 from LDS; the closures reach 6 points in
    instead of 4, so the interior tiles start 6 points from the block
    edges and the band is wider)."""
    from fdmap_github_amd import inputs

    nx, ny = args.nx, args.ny
    inpath = inputs.write(os.path.join(tmp, "c2sbp6.in"),
                          inputs.c2_planar_rs(name=os.path.join(tmp, "c2sbp6"), nx=nx, ny=ny,
                                              nsteps=args.steps + args.warmup + args.prof_steps,
                                              outputs=False, fdmethod="SBP6"))
    res = {}
    for prec in ("fp64",) if args.no_fp32 else ("fp64", "fp32"):
        r = run_device(inpath, prec, args.steps, args.warmup, args.prof_steps)
        ns, prof = r["nstage"], r["prof"]
        b1, b2 = BYTES_STAGE[prec]
        kpts = prof["bulk_points"]
        bytes_launch = kpts * (b1 + (ns - 1) * b2) / ns
        avg_ms = prof["bulk_ms"] / max(1, prof["bulk_launches"])
        res[prec] = dict(r=r, ups=r["npts"] * args.steps / r["el"], avg_ms=avg_ms, kpts=kpts,
                         achieved=bytes_launch / (avg_ms * 1e-3) / 1e9, bytes_launch=bytes_launch)
    r64 = res["fp64"]
    out = {
        "metric": METRIC, "value": r64["ups"], "unit": "updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1e3 * r64["r"]["el"] / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic (planar fault problem)",
        "config": {"workload": f"planar rate-and-state rupture on the SBP6 operator, 2 blocks x "
                               f"({nx}x{ny}), RFL slip law, LSRK(5,4) CFL 0.5",
                   "grid_points": r64["r"]["npts"], "fault_nodes": nx, "dt": r64["r"]["hp"].dt},
        "roofline": {
            "bound": "hbm",
            "kernel": f"bulk_interior<double,64,4,0,true,false,false,6,{str(r64['r']['ji']).lower()},"
                      f"{str(r64['r']['mc']).lower()},false>",
            "kernel_points": r64["kpts"], "achieved": r64["achieved"], "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": r64["achieved"] / HBM_PEAK_GBS,
            "traffic": measured_traffic("bulk_interior_c2sbp6_fp64"),
            "alg_bytes_per_launch": r64["bytes_launch"], "avg_launch_ms": r64["avg_ms"],
            "edge_kernel_avg_ms": prof["edge_ms"] / max(1, prof["edge_launches"]),
            "band_kernel_avg_ms": prof["band_ms"] / max(1, prof["band_launches"]),
        },
    }
    if "fp32" in res:
        r32 = res["fp32"]
        out["fp32_bulk"] = {
            "updates_per_s": r32["ups"], "speedup_vs_fp64": r32["ups"] / r64["ups"],
            "ms_per_step": 1e3 * r32["r"]["el"] / args.steps,
            "bulk_avg_launch_ms": r32["avg_ms"], "bulk_achieved_GBs": r32["achieved"],
            "rel_l2_fields_vs_fp64": rel_l2(r32["r"]["F"], r64["r"]["F"]),
            "rel_l2_slip_vs_fp64": rel_l2(r32["r"]["fault"]["D"], r64["r"]["fault"]["D"]),
            "rel_l2_slip_velocity_vs_fp64": rel_l2(r32["r"]["fault"]["V"],
                                                   r64["r"]["fault"]["V"]),
            "after_steps": args.steps + args.warmup,
        }
    print(json.dumps(out), flush=True)


def run_c2_pml(args, tmp):
    """C2 with a graded perfectly matched layer in both blocks (pmlx and
    pmly, n = 2, from 80 % of the half-widths outwards).  Per point per stage
    the layer kernel reads F (48 B), the coordinates (16 B) and, after stage 1,
    DF (40 B), and writes F and DF (96 B): 160 B at stage 1 and 200 B after, in
    FP64 (the field planes halve in FP32, the coordinates stay FP64).  A point
    that a direction damps also reads that direction's auxiliary fields (48
    B) and, after stage 1, their rates (48 B), and writes both (96 B): 144
    and 192 B more.  Elsewhere they are zero and stay zero.  The launch
    (bulk_layer) covers the whole stage."""
    from fdmap_github_amd import inputs

    nx, ny = args.nx, args.ny
    h = 0.025
    Lx, Ly = 0.5 * (nx - 1) * h, (ny - 1) * h
    layer = dict(pmlx=True, pmly=True, n=2.0, sigma=50.0 / (0.2 * Ly) ** 2, mx=-0.8 * Lx, px=0.8 * Lx,
                 my=-0.8 * Ly, py=0.8 * Ly)
    inpath = inputs.write(os.path.join(tmp, "c2pml.in"),
                          inputs.c2_planar_rs(name=os.path.join(tmp, "c2pml"), nx=nx, ny=ny,
                                              nsteps=args.steps + args.warmup + args.prof_steps,
                                              outputs=False, pml=layer))
    res = {}
    for prec in ("fp64",) if args.no_fp32 else ("fp64", "fp32"):
        r = run_device(inpath, prec, args.steps, args.warmup, args.prof_steps)
        ns, prof = r["nstage"], r["prof"]
        xg, yg = (np.ctypeslib.as_array(getattr(r["hp"].ptr.contents, k),
                                        shape=(r["hp"].ny, r["hp"].nx)) for k in ("x", "y"))
        damped = (float(np.mean((xg < layer["mx"]) | (xg > layer["px"])))
                  + float(np.mean((yg < layer["my"]) | (yg > layer["py"]))))
        b1, b2 = (160.0, 200.0) if prec == "fp64" else (88.0, 108.0)
        e = 1.0 if prec == "fp64" else 0.5
        b1, b2 = b1 + 144.0 * e * damped, b2 + 192.0 * e * damped
        kpts = prof["bulk_points"]
        bytes_launch = kpts * (b1 + (ns - 1) * b2) / ns
        avg_ms = prof["bulk_ms"] / max(1, prof["bulk_launches"])
        res[prec] = dict(r=r, ups=r["npts"] * args.steps / r["el"], avg_ms=avg_ms, kpts=kpts,
                         achieved=bytes_launch / (avg_ms * 1e-3) / 1e9, bytes_launch=bytes_launch)
    r64 = res["fp64"]
    out = {
        "metric": METRIC, "value": r64["ups"], "unit": "updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1e3 * r64["r"]["el"] / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic (planar fault problem)",
        "config": {"workload": f"planar rate-and-state rupture with a graded perfectly matched layer "
                               f"(n 2) in both blocks, 2 blocks x ({nx}x{ny}), RFL slip law, LSRK(5,4) CFL 0.5",
                   "grid_points": r64["r"]["npts"], "fault_nodes": nx, "dt": r64["r"]["hp"].dt},
        "roofline": {
            "bound": "hbm", "kernel": "bulk_layer<double,0,true,false> (a whole stage of a problem with a layer)",
            "kernel_points": r64["kpts"], "achieved": r64["achieved"], "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": r64["achieved"] / HBM_PEAK_GBS,
            "traffic": measured_traffic("bulk_pml_c2pml_fp64"),
            "alg_bytes_per_launch": r64["bytes_launch"], "avg_launch_ms": r64["avg_ms"],
        },
    }
    if "fp32" in res:
        r32 = res["fp32"]
        out["fp32_bulk"] = {
            "updates_per_s": r32["ups"], "speedup_vs_fp64": r32["ups"] / r64["ups"],
            "layer_avg_launch_ms": r32["avg_ms"], "layer_achieved_GBs": r32["achieved"],
            "rel_l2_fields_vs_fp64": rel_l2(r32["r"]["F"], r64["r"]["F"]),
            "rel_l2_slip_vs_fp64": rel_l2(r32["r"]["fault"]["D"], r64["r"]["fault"]["D"]),
            "after_steps": args.steps + args.warmup,
        }
    print(json.dumps(out), flush=True)


def run_m3(args, tmp):
    """Antiplane shear (mode 3): two blocks of 1601 x 801 points (h = 0.025
    km) side by side with a vertical aging-law fault between them, a free
    surface on top, built from its .in file.  Per point per stage the
    interior kernel reads vz, sxz, syz, their rates and the 5 metric planes
    and writes fields and rates: 136 B in FP64 (112 B at stage 1, where the
    rates are not read), half in FP32."""
    from fdmap_github_amd import inputs

    # each block is --ny wide and --nx high: C2's point count, turned upright
    inpath = inputs.write(os.path.join(tmp, "m3.in"),
                          inputs.antiplane_rs(name=os.path.join(tmp, "m3"), nx=args.ny, ny=args.nx,
                                              h=0.025,
                                              nsteps=args.steps + args.warmup + args.prof_steps,
                                              outputs=False, ld_width=4.0, ninfo=100000))
    res = {}
    for prec in ("fp64",) if args.no_fp32 else ("fp64", "fp32"):
        r = run_device(inpath, prec, args.steps, args.warmup, args.prof_steps)
        ns, prof = r["nstage"], r["prof"]
        b1, b2 = (112.0, 136.0) if prec == "fp64" else (56.0, 68.0)
        kpts = prof["bulk_points"]
        bytes_launch = kpts * (b1 + (ns - 1) * b2) / ns
        avg_ms = prof["bulk_ms"] / max(1, prof["bulk_launches"])
        res[prec] = dict(r=r, ups=r["npts"] * args.steps / r["el"], avg_ms=avg_ms,
                         achieved=bytes_launch / (avg_ms * 1e-3) / 1e9, bytes_launch=bytes_launch,
                         kpts=kpts)
    r64 = res["fp64"]
    out = {
        "metric": METRIC, "value": r64["ups"], "unit": "updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1e3 * r64["r"]["el"] / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (antiplane fault problem generated as an FDMAP .in file)",
        "config": {"workload": "antiplane shear (mode 3) rate-and-state rupture, 2 blocks "
                               f"x ({r64['r']['hp'].nx // 2}x{r64['r']['hp'].ny}) side by side, "
                               "vertical RAL fault, free surface, LSRK(5,4) CFL 0.5",
                   "grid_points": r64["r"]["npts"], "fault_nodes": r64["r"]["hp"].ny},
        "roofline": {
            "bound": "hbm", "kernel": "bulk_interior3<double,64,4,NT,4>",
            "kernel_points": r64["kpts"], "achieved": r64["achieved"], "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": r64["achieved"] / HBM_PEAK_GBS,
            "traffic": measured_traffic("bulk_interior3_m3_fp64"),
            "alg_bytes_per_launch": r64["bytes_launch"], "avg_launch_ms": r64["avg_ms"],
        },
    }
    if "fp32" in res:
        r32 = res["fp32"]
        out["fp32_bulk"] = {
            "updates_per_s": r32["ups"], "speedup_vs_fp64": r32["ups"] / r64["ups"],
            "ms_per_step": 1e3 * r32["r"]["el"] / args.steps,
            "bulk_avg_launch_ms": r32["avg_ms"], "bulk_achieved_GBs": r32["achieved"],
            "rel_l2_fields_vs_fp64": rel_l2(r32["r"]["F"], r64["r"]["F"]),
            "rel_l2_slip_vs_fp64": rel_l2(r32["r"]["fault"]["D"], r64["r"]["fault"]["D"]),
            "rel_l2_slip_velocity_vs_fp64": rel_l2(r32["r"]["fault"]["V"],
                                                   r64["r"]["fault"]["V"]),
            "after_steps": args.steps + args.warmup,
        }
    print(json.dumps(out), flush=True)


def run_c4(args, tmp):
    """Ensemble: scenarios with block sizes uniform in 401..2001 x 201..1001,
    lognormal fault shear prestress (mean 70 MPa, log sd 0.1, correlation
    length 1 km), uniform a in [0.008, 0.012]; FP32 fields, FP64 friction;
    tile shapes from the autotuner; every RK stage of all scenarios is a
    batched launch per kernel kind, and a step is one hipGraph launch."""
    import collections

    from fdmap_github_amd import capi, ensemble, host
    from fdmap_github_amd.device import Context

    steps = 2000 if args.steps == 4000 else args.steps
    scen = ensemble.c4_scenarios(count=args.scenarios, seed=0)
    cache = ensemble.load_cache(args.tune_cache)
    members, t, dt, npts, chosen = [], [], [], 0, collections.Counter()
    t_setup = time.perf_counter()
    for sc in scen:
        path = ensemble.write_scenario(tmp, sc, steps + args.warmup + 200)
        hp = host.HostProblem(path, precision="fp32")

        def make(hp=hp):
            c = Context(hp.ptr)
            c.set_fields(hp.fields())
            c.init_edges(hp.t)
            return c

        key = "fp32:%d:%d" % ensemble.size_class(hp.nx, hp.ny // 2)
        tile = ensemble.tune(make, key, cache)
        c = make()
        ensemble.apply_tile(c, tile)
        chosen[capi.TILE_SHAPES[tile]] += 1
        members.append(c)
        t.append(hp.t)
        dt.append(hp.dt)
        npts += hp.nx * hp.ny
        print(f"scenario {sc['index']}: {hp.nx} x {hp.ny // 2} x 2, tile {capi.TILE_SHAPES[tile]}",
              file=sys.stderr, flush=True)
    ensemble.save_cache(args.tune_cache, cache)
    t_setup = time.perf_counter() - t_setup
    ens = ensemble.Ensemble(members)
    ens.step(t, dt, 1, args.warmup)
    ens.sync()
    t0 = time.perf_counter()
    ens.step(t, dt, args.warmup + 1, steps)
    ens.sync()
    el = time.perf_counter() - t0
    ens.close()
    # the same batched launches made directly, without the graph
    eager_steps = min(100, steps)
    n0 = args.warmup + steps + 1
    os.environ["FDM_ENSEMBLE_GRAPH"] = "0"
    direct = ensemble.Ensemble(members)
    del os.environ["FDM_ENSEMBLE_GRAPH"]
    direct.step(t, dt, n0, 2)
    direct.sync()
    t0 = time.perf_counter()
    direct.step(t, dt, n0 + 2, eager_steps)
    direct.sync()
    el_direct = time.perf_counter() - t0
    direct.close()
    n0 += eager_steps + 2
    # the same members stepped one call per member and step
    t0 = time.perf_counter()
    for k in range(eager_steps):
        for m, c in enumerate(members):
            c.step(t[m], dt[m], n0 + k, 1)
    for c in members:
        c.sync()
    el_eager = time.perf_counter() - t0
    vmax = max(float(np.abs(c.get_iface(0, "V")).max()) for c in members)
    out = {
        "metric": METRIC, "value": npts * steps / el, "unit": "updates/s", "n_gpus": 1,
        "steps": steps, "warmup": args.warmup, "ms_per_step": 1e3 * el / steps,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32 fields, f64 friction",
        "data": "synthetic (seeded scenarios generated as FDMAP .in, stress and state files)",
        "config": {"workload": f"ensemble of {len(members)} two-block rate-and-state ruptures, "
                               "blocks uniform in 401..2001 x 201..1001, lognormal prestress, "
                               "uniform a, FP32-bulk, batched launches, one hipGraph launch per RK step",
                   "grid_points": npts, "scenarios": len(members)},
        "tile_choices": dict(chosen),
        "batched_direct_updates_per_s": npts * eager_steps / el_direct,
        "per_member_updates_per_s": npts * eager_steps / el_eager,
        "speedup_vs_per_member": (npts * steps / el) / (npts * eager_steps / el_eager),
        "max_slip_velocity": vmax,
        "setup_s": t_setup,
    }
    print(json.dumps(out), flush=True)


def c5_measure(tmp, steps=2000):
    """Adjoint gradient: the planar rate-and-state rupture (C2 parameters)
    on two blocks of 801 x 401 points with a free surface on top, 2000
    steps; misfit 0.5 dt sum (v - v_target)^2 of vx, vy at 32 free-surface
    receivers against the traces of a run whose fault shear prestress
    carries a seeded Gaussian random perturbation (1 MPa rms, correlation
    length 1 km).  Gradient with respect to the 801 fault shear-prestress
    values, a and b (and the initial state), by the hand-written adjoint
    (the fault trace kept in HBM, and with square-root checkpointing and
    recomputation); its time against one forward run, and
    central differences (eps = 1e-6) along one seeded direction per
    parameter."""
    from fdmap_github_amd import ensemble, host
    from fdmap_github_amd.adjoint import FaultInversion
    from fdmap_github_amd.device import Context

    nx, ny, h = 801, 401, 0.025
    rng = np.random.default_rng(5)
    sc = dict(index=0, nx=nx, ny=ny, a=0.010, S0=np.full(nx, 70.0), h=h)
    path = ensemble.write_scenario(tmp, sc, steps + 10, bcT="free")
    hp = host.HostProblem(path, precision="fp64")
    ctx = Context(hp.ptr)
    ctx.set_fields(hp.fields())
    ctx.init_edges(hp.t)
    ri = np.linspace(0.05 * (nx - 1), 0.95 * (nx - 1), 32).round().astype(np.int32)
    rj = np.full(32, hp.ny - 1, dtype=np.int32)
    n = nx
    p0 = {"S0": np.full(n, 70.0), "a": np.full(n, 0.010), "b": np.full(n, 0.014)}
    pert = ensemble.correlated_lognormal(n, h, 1.0, 1.0, 1.0, rng)
    pert = (np.log(pert) + 0.5) / np.std(np.log(pert))  # unit-variance Gaussian field
    inv = FaultInversion(ctx, hp.t, hp.dt, ri, rj, steps, interval=0)  # automatic policy
    target = inv.run(S0=p0["S0"] + pert, a=p0["a"], b=p0["b"])
    dt = hp.dt

    def misfit(rec):
        return 0.5 * dt * float(np.sum((rec - target) ** 2))

    # one plain forward run (fdm_step), after a short warm-up
    inv.reset()
    ctx.step(hp.t, dt, 1, 20)
    ctx.sync()
    inv.adj.set_param("S0", p0["S0"])
    inv.reset()
    t0 = time.perf_counter()
    ctx.step(hp.t, dt, 1, steps)
    ctx.sync()
    t_fwd = time.perf_counter() - t0
    vmax = ctx.max_slip_velocity()
    out_modes = {}
    grads = None
    for label, itv in (("auto", 0), ("sqrtN", -1)):
        fi = inv if itv == 0 else FaultInversion(ctx, hp.t, dt, ri, rj, steps, interval=itv)
        if fi is not inv:
            fi.F0, fi.DF0, fi.iface0 = inv.F0, inv.DF0, inv.iface0
        fi.run(**p0)  # warm-up of this workspace
        fi.adj.backward(dt * np.zeros((steps, 32, 2)))
        t0 = time.perf_counter()
        rec = fi.run(**p0)
        t1 = time.perf_counter()
        g = fi.adj.backward(dt * (rec - target))
        t2 = time.perf_counter()
        tm = fi.adj.timing()
        out_modes[label] = {"interval": fi.adj.interval, "forward_pass_s": t1 - t0,
                            "backward_pass_s": t2 - t1, "gradient_s": t2 - t0,
                            "ratio_to_forward": (t2 - t0) / t_fwd,
                            "device_ms": {k: round(v, 3) for k, v in tm.items()}}
        if grads is None:
            grads, J0 = g, misfit(rec)
        else:
            out_modes[label]["same_gradient_as_auto"] = all(
                np.array_equal(g[k], grads[k]) for k in ("S0", "a", "b", "Psi0"))
            fi.adj.close()
    # central differences at eps = 1e-6 along seeded directions (N(0, 1)
    # entries times 10 MPa for S0, a for a, 10 for b, 1 for the initial state)
    eps = 1e-6
    fd = {}
    for name, scale in (("S0", 10.0), ("a", p0["a"]), ("b", 10.0), ("Psi0", 1.0)):
        d = rng.standard_normal(n) * scale
        vals = []
        for sgn in (1.0, -1.0):
            if name == "Psi0":
                psi0 = inv.iface0[0]["Psi"].copy()
                inv.iface0[0]["Psi"] = psi0 + sgn * eps * d
                vals.append(misfit(inv.run(**p0)))
                inv.iface0[0]["Psi"] = psi0
            else:
                p = dict(p0)
                p[name] = p0[name] + sgn * eps * d
                vals.append(misfit(inv.run(**p)))
        fdv = (vals[0] - vals[1]) / (2 * eps)
        ad = float(grads[name] @ d)
        fd[name] = {"fd": fdv, "adjoint": ad,
                    "rel_err": abs(fdv - ad) / abs(ad) if ad != 0.0 else float(fdv != 0.0)}
        print(f"fd {name}: {fd[name]}", file=sys.stderr, flush=True)
    ratio = out_modes["auto"]["ratio_to_forward"]
    out = {
        "metric": METRIC, "value": ratio, "unit": "adjoint gradient time / forward time",
        "n_gpus": 1, "steps": steps, "warmup": 20, "ms_per_step": 1e3 * t_fwd / steps,
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (seeded .in, stress and state files; targets from a seeded "
                "prestress perturbation)",
        "config": {"workload": "adjoint gradient of a receiver misfit, 2 x (801 x 401) planar "
                               "rate-and-state rupture (RFL), free surface, 32 receivers, "
                               f"{steps} steps; fault trace kept in HBM (automatic policy; "
                               "square-root checkpointing with recomputation in modes.sqrtN)",
                   "grid_points": hp.nx * hp.ny, "fault_nodes": n, "receivers": 32},
        "forward_s": t_fwd, "forward_updates_per_s": hp.nx * hp.ny * steps / t_fwd,
        "modes": out_modes, "misfit": J0, "max_slip_velocity": vmax,
        "fd_check": {"eps": eps, **fd},
        "fd_max_rel_err": max(v["rel_err"] for v in fd.values()),
    }
    return out


def run_c5(args, tmp):
    print(json.dumps(c5_measure(tmp, 2000 if args.steps == 4000 else args.steps)), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=4000)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--nx", type=int, default=1601)
    ap.add_argument("--ny", type=int, default=801)
    ap.add_argument("--cpu-steps", type=int, default=40)
    ap.add_argument("--prof-steps", type=int, default=200,
                    help="steps timed after the headline ones with HIP events per launch")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fp32", action="store_true")
    ap.add_argument("--no-legs", action="store_true",
                    help="leave out the C3 (FP32-bulk against FP64 on the rough fault, 3000 "
                         "steps) and C5 (adjoint gradient time) legs of the default line")
    ap.add_argument("--horizon", type=int, default=4000,
                    help="steps after which the FP32-bulk error against FP64 is stated (C2's "
                         "own length), whatever --steps")
    ap.add_argument("--config", choices=("c2", "c2het", "c2diss", "c2pml", "c2sbp6", "m3", "c3", "c4",
                                         "c5"),
                    default="c2",
                    help="c2: planar rupture (the headline); c2het: the same in a "
                         "heterogeneous medium; c2diss: the same with artificial dissipation "
                         "(Cdiss 0.1); c2pml: the same inside a graded perfectly matched layer; "
                         "c2sbp6: the same on the SBP6 operator; m3: antiplane shear rupture, "
                         "2 x (801x1601); "
                         "c3: rough curvilinear fault with "
                         "off-fault plasticity, 2 x (4001x2001), FP64 and FP32-bulk; c4: 64 "
                         "uneven rupture scenarios advanced as one graph launch per step; c5: "
                         "adjoint gradient of a receiver misfit, 2 x (801x401), 2000 steps")
    ap.add_argument("--scenarios", type=int, default=64)
    ap.add_argument("--tune-cache", default="fdmap_tuning.json")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only; --gpus {args.gpus} is not supported "
              "(blocks would shard across GPUs as described in DESIGN.md)", file=sys.stderr)
        sys.exit(2)

    from fdmap_github_amd import inputs

    tmp = tempfile.mkdtemp(prefix="fdmap_bench_")
    if args.config == "m3":
        run_m3(args, tmp)
        return
    if args.config in ("c2het", "c2diss"):
        run_c2_variant(args, tmp, het=args.config == "c2het",
                       cdiss=0.1 if args.config == "c2diss" else 0.0)
        return
    if args.config == "c2pml":
        run_c2_pml(args, tmp)
        return
    if args.config == "c2sbp6":
        run_c2_sbp6(args, tmp)
        return
    if args.config == "c3":
        run_c3(args, tmp)
        return
    if args.config == "c4":
        run_c4(args, tmp)
        return
    if args.config == "c5":
        run_c5(args, tmp)
        return
    inpath = inputs.write(os.path.join(tmp, "c2.in"),
                          inputs.c2_planar_rs(name=os.path.join(tmp, "c2"), nx=args.nx,
                                              ny=args.ny,
                                              nsteps=max(args.horizon,
                                                         args.steps + args.warmup + args.prof_steps),
                                              outputs=False))
    horizon = None if args.no_fp32 else args.horizon
    r64 = run_device(inpath, "fp64", args.steps, args.warmup, args.prof_steps, horizon)
    npts = r64["npts"]
    prof = r64["prof"]
    ns = r64["nstage"]
    b1, b2 = BYTES_STAGE["fp64"]
    # one launch a stage: edge nodes, inner band and interior tiles; it
    # covers prof["bulk_points"] points
    kpts = prof["bulk_points"]
    bytes_launch = kpts * (b1 + (ns - 1) * b2) / ns
    avg_ms = prof["bulk_ms"] / max(1, prof["bulk_launches"])
    achieved = bytes_launch / (avg_ms * 1e-3) / 1e9
    ups = npts * args.steps / r64["el"]
    out = {
        "metric": METRIC,
        "value": ups,
        "unit": "updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * r64["el"] / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (planar fault problem generated as an FDMAP .in file)",
        "config": {
            "workload": "planar rate-and-state rupture, 2 blocks x (1601x801), h=0.025 km, "
                        "RFL slip law, LSRK(5,4) CFL 0.5, FP64",
            "grid_points": npts,
            "fault_nodes": args.nx,
        },
        "roofline": {
            "bound": "hbm",
            "kernel": f"bulk_interior<double,64,4,0,true,false,false,4,"
                      f"{str(r64['ji']).lower()},{str(r64['mc']).lower()},false> (SBP4 interior rates + "
                      "RK update, a whole stage: edge nodes and the points near edges ahead of "
                      "64x4 LDS tiles over the block interiors; non-temporal stores since "
                      "the 23 field, rate and metric planes exceed 256 MB; JI: Ji formed "
                      "from the metrics, MC: metrics read as FP32 deltas)",
            "kernel_points": kpts,
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": None,
            "alg_bytes_per_launch": bytes_launch,
            "kernel_min_bytes_per_launch": kpts * kernel_min_bytes("fp64", ns, r64["ji"], r64["mc"]),
            "avg_launch_ms": avg_ms,
            "launches": prof["bulk_launches"],
            "ms_per_step_with_events": 1e3 * r64["el_prof"] / args.prof_steps,
            "edge_kernel_avg_ms": prof["edge_ms"] / max(1, prof["edge_launches"]),
            "band_kernel_avg_ms": prof["band_ms"] / max(1, prof["band_launches"]),
            "hbm_frac_end_to_end": npts * (b1 + (ns - 1) * b2) * args.steps / r64["el"] / 1e9
                                   / HBM_PEAK_GBS,
        },
    }
    out["roofline"]["traffic"] = measured_traffic()
    if not args.no_fp32:
        r32 = run_device(inpath, "fp32", args.steps, args.warmup, args.prof_steps, horizon)
        ups32 = npts * args.steps / r32["el"]
        p32 = r32["prof"]
        c1, c2 = BYTES_STAGE["fp32"]
        avg32 = p32["bulk_ms"] / max(1, p32["bulk_launches"])
        k32 = p32["bulk_points"]
        # the stored planes of the FP32-bulk context: fields (two buffers),
        # rates and metrics, 23 planes of 4 bytes
        hp = r64["hp"]
        ws = 23 * 4 * hp.ny * (-(-hp.nx // 64) * 64 + 64)
        out["fp32_bulk"] = {
            "updates_per_s": ups32,
            "speedup_vs_fp64": ups32 / ups,
            "ms_per_step": 1e3 * r32["el"] / args.steps,
            "bulk_avg_launch_ms": avg32,
            "bulk_achieved_GBs": k32 * (c1 + (ns - 1) * c2) / ns / (avg32 * 1e-3) / 1e9,
            "working_set_MB": ws / 2 ** 20,
            "cache_resident": ws < 256 * 2 ** 20,
            "note": "the FP32 planes fit MI355X's 256 MB Infinity Cache: bulk_achieved_GBs is "
                    "cache-assisted, not an HBM figure" if ws < 256 * 2 ** 20 else "",
            "rel_l2_fields_vs_fp64": rel_l2(r32["F_h"], r64["F_h"]),
            "rel_l2_slip_vs_fp64": rel_l2(r32["fault_h"]["D"], r64["fault_h"]["D"]),
            "rel_l2_slip_velocity_vs_fp64": rel_l2(r32["fault_h"]["V"], r64["fault_h"]["V"]),
            "after_steps": r64["horizon"],
        }
    if not args.no_legs:
        t0 = time.perf_counter()
        m = c3_measure(os.path.join(tmp, "c3"))
        out["c3_rough_fault"] = {
            "workload": f"rough curvilinear fault with plasticity, 2 blocks x ({m['nx']}x{m['ny']}), "
                        "FP64 and FP32-bulk over the same 3000 steps",
            "steps": m["steps"], "fp64_updates_per_s": m["ups64"], **m["fp32"],
            "leg_s": time.perf_counter() - t0}
        t0 = time.perf_counter()
        r5 = c5_measure(os.path.join(tmp, "c5"))
        out["c5_adjoint"] = {
            "workload": r5["config"]["workload"],
            "gradient_over_forward_sqrtN_checkpoints": r5["modes"]["sqrtN"]["ratio_to_forward"],
            "gradient_over_forward_trace_kept": r5["modes"]["auto"]["ratio_to_forward"],
            "interval_sqrtN": r5["modes"]["sqrtN"]["interval"],
            "forward_s": r5["forward_s"], "modes": r5["modes"],
            "fd_eps": r5["fd_check"]["eps"], "fd_max_rel_err": r5["fd_max_rel_err"],
            "leg_s": time.perf_counter() - t0}
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(inpath, args.cpu_steps)
        out["cpu_baseline"]["gpu_over_cpu"] = ups / out["cpu_baseline"]["value"]
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
