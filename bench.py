"""Benchmark: FLIP substeps/s of the MI355X engine at 256^3, mixed-precision
refined PCG vs FP64 PCG at relative residual 1e-8.

Workload (per step): one FluidSimulation.update() of 1/240 s -- one CFL
substep of the whole per-substep path (cell sort, liquid SDF, P2G,
extrapolation, body force, pressure assembly + MIC(0)-PCG + projection,
constraints, G2P + RK3 + collision, removal) -- on the dam break at n^3 with
the static sphere obstacle: fluid block [0, 0.375) x [0, 0.625) x [0, 1),
8 particles per cell (seeded jitter, zero initial velocity), sphere r = 0.15 at
(0.6, 0.2, 0.5).  Inputs are resident in HBM before the timed region.

Prints one JSON line.  `value` is the substeps/s of the fastest
mixed-precision mode (FP32 PCG restarted inside FP64 iterative refinement,
FP32 PCG with FP64 reliable updates, or FP64 PCG with the MIC(0) application
in FP32; `mode` names it); the FP64 run, the ratio, per-kernel GPU times (HIP
events on the engine's stream) and the roofline of the dominant kernel are
reported beside it.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "blender-flip-fluids_amd"))
sys.path.insert(0, os.path.join(ROOT, "tests"))

HBM_PEAK_GBS = 8000.0
KERNELS = ["cell_sort", "liquid_sdf", "p2g", "extrapolate", "pressure_assembly", "mic0_factor", "spmv",
           "mic0_apply", "unused", "g2p_advect", "removal", "apply_pressure", "viscosity"]


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def make_sim(n, pos, solid, mode, tol, apic=False, warm=False, schedule=None):
    """solid: a nodal SDF array, a (vertices, triangles) mesh obstacle, or None.
    schedule: the MIC(0) application's schedule (None: the engine's default)."""
    from ffengine import FluidSimulation, MeshObject, TriangleMesh
    sim = FluidSimulation(n, n, n, 1.0 / n)
    if schedule is not None:
        sim.set_pressure_solver_preconditioner_schedule(schedule)
    if apic:
        sim.set_velocity_transfer_method_APIC()
    if warm:
        sim.set_pressure_solver_warm_start(True)
    sim.add_body_force(0.0, -9.81, 0.0)
    sim.PICFLIP_ratio = 0.05
    sim.CFL_condition_number = 5
    sim.enable_surface_reconstruction = False
    sim.pressure_solver_tolerance = tol
    sim.set_pressure_solver_precision(mode)
    if isinstance(solid, tuple):
        mo = MeshObject(n, n, n, 1.0 / n)
        mo.update_mesh_static(TriangleMesh(*solid))
        sim.add_mesh_obstacle(mo)
        sim._bench_obstacle = mo  # the simulation holds the object by pointer
    elif solid is not None:
        sim.set_solid_phi(solid)
    sim.load_marker_particle_data(len(pos), pos.tobytes(), np.zeros_like(pos).tobytes())
    sim.initialize()
    return sim


def mesh_obstacle_sdf(n, mesh, cpu, threads, reps=3):
    """Build time of the static solid SDF (domain box + the mesh obstacle) at
    n^3: this engine's C ABI call (host preparation, uploads, kernels and the
    read-back of the nodal grid), and the reference engine's
    _addStaticObjectsToSDF on `threads` host cores when its build is present."""
    import oracle_lib
    from ffengine import kernels
    dx = 1.0 / n
    kernels.solid_phi_meshes((n, n, n), dx, [mesh])  # warm-up: first allocation and module load
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        phi, draws = kernels.solid_phi_meshes((n, n, n), dx, [mesh])
        times.append(time.perf_counter() - t0)
    out = {"triangles": int(len(mesh[1])), "gpu_ms": round(1e3 * min(times), 3), "rand_draws": int(draws),
           "cpu_reference_ms": None, "cpu_threads": None, "identical_to_reference": None}
    if cpu and oracle_lib.reference_available():
        oracle_lib.probe().refprobe_set_threads(threads)
        oracle_lib.libc_srand(7)
        ref, seconds = oracle_lib.ref_solid_phi_meshes((n, n, n), dx, [mesh], 7, timed=True)
        oracle_lib.probe().refprobe_set_threads(1)
        oracle_lib.libc_srand(7)
        mine, _ = kernels.solid_phi_meshes((n, n, n), dx, [mesh])
        out.update(cpu_reference_ms=round(1e3 * seconds, 3), cpu_threads=threads,
                   identical_to_reference=bool(np.array_equal(mine.view(np.uint32), ref.view(np.uint32))))
    return out


def kernel_times(sim):
    from ctypes import byref, c_double, c_int, c_longlong, c_void_p
    from ffengine import pybindings as pb
    from ffengine.ffengine import ffengine as lib
    f = lib.FluidSimulation_get_kernel_timing
    pb.init_lib_func(f, [c_void_p, c_int, c_void_p, c_void_p, c_void_p], None)
    out = {}
    for i, name in enumerate(KERNELS):
        if name == "unused":
            continue
        ms, n, ok = c_double(), c_longlong(), c_int()
        f(sim(), i, byref(ms), byref(n), byref(ok))
        out[name] = {"ms": ms.value, "launches": n.value}
    return out


def enable_timing(sim, on):
    from ctypes import c_int, c_void_p
    from ffengine import pybindings as pb
    from ffengine.ffengine import ffengine as lib
    f = lib.FluidSimulation_enable_kernel_timing
    pb.init_lib_func(f, [c_void_p, c_int, c_void_p], None)
    pb.execute_lib_func(f, [sim(), 1 if on else 0])


def run_mode(n, pos, solid, mode, tol, steps, warmup, frame_dt, apic=False, warm=False, schedule=None,
             keep_state=False):
    """keep_state: also return the particles (positions, velocities) and the
    nodal solid SDF after the timed steps, for the CPU baseline."""
    import torch
    sim = make_sim(n, pos, solid, mode, tol, apic, warm, schedule)
    for s in range(warmup):
        sim.update(frame_dt)
        log("  warmup %s %d/%d" % (mode, s + 1, warmup))
    enable_timing(sim, True)
    torch.cuda.synchronize()
    substeps, iters, unknowns = 0, [], []
    t0 = time.perf_counter()
    for s in range(steps):
        sim.update(frame_dt)
        st = sim.get_frame_stats_data()
        ps = sim.get_last_pressure_solve_stats()
        substeps += st.substeps
        iters.append(st.pressure_solver_iterations)
        unknowns.append(ps["unknowns"])
        log("  %s step %d/%d: substeps=%d iters=%d unknowns=%d" % (mode, s + 1, steps, st.substeps,
                                                                   st.pressure_solver_iterations, ps["unknowns"]))
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    free, total = torch.cuda.mem_get_info()
    kt = kernel_times(sim)
    nparticles = sim.get_num_marker_particles()
    state = None
    if keep_state:
        p = np.frombuffer(sim.get_marker_particle_position_data_range(0, nparticles), np.float32).reshape(-1, 3)
        v = np.frombuffer(sim.get_marker_particle_velocity_data_range(0, nparticles), np.float32).reshape(-1, 3)
        state = (p.copy(), v.copy(), sim.get_solid_sdf().copy())
    del sim
    return {"elapsed_s": elapsed, "substeps": substeps, "iterations": iters, "unknowns": unknowns,
            "kernels": kt, "particles": nparticles, "device_bytes_used": total - free, "state": state}


def algorithmic_bytes(name, n, P, M_total, launches_per_sub, substeps, iters_total, mode):
    """Compulsory bytes per timed region for one kernel group (units below)."""
    N = n ** 3
    F = 3 * n * n * (n + 1)
    Nn = (n + 1) ** 3
    if name == "p2g":
        return substeps * (28 * P + 4 * N + 5 * F)          # 28 B/particle, 4 B/cell, 5 B/face
    if name == "spmv":
        # 4 coefficients, z and s read, the direction and its product written per row (z in FP32 beside FP64 vectors)
        per = 32 if mode in ("mixed", "mixed-reliable") else 64 if mode == "fp64" else 60
        return per * M_total
    if name == "mic0_apply":
        per = 96 if mode == "fp64" else 48                    # both sweeps: r, invdiag, 3 L, z per row
        return per * M_total
    if name == "g2p_advect":
        return substeps * (48 * P + 8 * F + 4 * Nn)
    if name == "extrapolate":
        return substeps * 2 * 9 * F
    if name == "liquid_sdf":
        return substeps * (12 * P + 8 * N)
    if name == "cell_sort":
        return substeps * (20 * P + 4 * N)
    return None


def sweep_kernel_name(fp64, schedule):
    """The MIC(0) sweep kernel the library runs for one precision and schedule, with the shape it was built for
    (columns: forward and backward launches; lines along j and k of a column, columns of a workgroup)."""
    from ctypes import byref, c_int, c_void_p
    from ffengine import pybindings as pb
    from ffengine.ffengine import ffengine as lib
    word = "double" if fp64 else "float"
    a, b, c = c_int(), c_int(), c_int()
    if schedule == 2:
        f = lib.FFAMD_mic0_column_shape
        pb.init_lib_func(f, [c_void_p] * 4, None)
        pb.execute_lib_func(f, [byref(a), byref(b), byref(c)])
        return "columnSweepKernel<%s> %dx%dx%d" % (word, a.value, b.value, c.value)
    if schedule == 5:
        f = lib.FFAMD_mic0_band_shape
        pb.init_lib_func(f, [c_int, c_void_p, c_void_p, c_void_p], None)
        pb.execute_lib_func(f, [1 if fp64 else 0, byref(a), byref(b)])
        return "micBandKernel<%s, %d, %d>" % (word, a.value, b.value)
    return "pencilSweepKernel<%s>" % word


def measured_traffic(kernel):
    """HBM bytes per dispatch of `kernel` from the committed PMC summaries
    (lines 'traffic <kernel> <bytes>' in profiles/*.md), or None when no
    summary covers this kernel build."""
    import glob
    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*.md"))):
        with open(path) as fh:
            for line in fh:
                parts = line.strip().strip("`").split()
                if len(parts) >= 2 and parts[0] == "traffic" and " ".join(parts[1:-1]) == kernel:
                    return int(parts[-1])
    return None


CALIBRATION = os.path.join(ROOT, "profiles", "cpu_baseline_dam_break_256.md")


def calibration_ratio():
    """The reference engine's substeps/s over the oracle's, both measured on
    the same host and thread count on the 256^3 scene (the line
    'calibration reference_over_port <ratio>' of the committed summary), or
    None."""
    if not os.path.isfile(CALIBRATION):
        return None
    with open(CALIBRATION) as fh:
        for line in fh:
            parts = line.strip().strip("`").split()
            if len(parts) == 3 and parts[:2] == ["calibration", "reference_over_port"]:
                return float(parts[2])
    return None


def cpu_baseline(state, n, tol, threads):
    """The oracle (this build's CPU restatement, tests/oracle_lib) timed on the
    host cores for one substep of the same scene: the GPU run's particles and
    solid SDF after its timed steps.  Its liquid SDF, P2G, SpMV, vector updates,
    G2P and advection run on `threads` threads (the same bits as serial); the
    MIC(0) factor and sweeps and the dot products are serial, as in the
    reference engine's PCG."""
    import oracle_lib
    pos, vel, solid = state
    oracle_lib.set_threads(threads)
    try:
        orc = oracle_lib.OracleSim((n, n, n), 1.0 / n, tol=tol)
        orc.set_solid_phi(solid)
        orc.load(pos, vel)
        orc.initialize()
        t0 = time.perf_counter()
        orc.step(1.0 / 240.0)
        el = time.perf_counter() - t0
    finally:
        oracle_lib.set_threads(1)
    ratio = calibration_ratio()
    out = {"value": round(1.0 / el, 5), "unit": "substeps/s", "cores": threads, "kind": "port",
           "sample": "the oracle (CPU restatement of the path) for one substep of 1/240 s of the same %d^3 scene "
                     "(%d particles: the GPU run's state after its timed steps, PCG rel res %g), %.1f s; liquid "
                     "SDF, P2G, SpMV, vector updates, G2P and advection on %d threads, MIC(0) and dots serial"
                     % (n, len(pos), tol, el, threads)}
    if ratio is not None:
        out["calibration"] = {"reference_over_port": ratio,
                              "reference_equivalent_substeps_per_s": round(ratio / el, 5),
                              "source": os.path.relpath(CALIBRATION, ROOT)}
    return out


def cpu_calibration(n, substeps, threads):
    """No GPU: the reference engine (oracle/_ref, built from its sources) and
    the oracle on the same host, the same thread count and the same scene (the
    n^3 dam break with the sphere obstacle, from rest, PCG to the reference's
    fixed 1e-9): one warm-up substep (builds the solid), then `substeps` timed
    substeps of 1/240 s each.  Prints one JSON line."""
    import oracle_lib
    from ffengine import scenes
    if not oracle_lib.reference_available():
        sys.exit("the reference build (oracle/_ref) is missing: run `make -C oracle ref`")
    dx = 1.0 / n
    pos = scenes.dam_break_particles(n, seed=0)
    verts, tris = scenes.sphere_mesh(subdivisions=5)
    out = {}
    log("reference engine n=%d threads=%d" % (n, threads))
    ref = oracle_lib.ReferenceSim((n,) * 3, dx, threads=threads)
    ref.load(pos)
    ref.add_mesh_obstacle((n,) * 3, dx, verts, tris)
    ref.initialize()
    ref.update(1.0 / 240.0)
    times = []
    for s in range(substeps):
        t0 = time.perf_counter()
        ref.update(1.0 / 240.0)
        times.append(time.perf_counter() - t0)
        log("  reference substep %d: %.2f s" % (s + 1, times[-1]))
    out["reference"] = {"substeps_per_s": len(times) / sum(times), "seconds": [round(t, 3) for t in times]}
    del ref
    log("oracle n=%d threads=%d" % (n, threads))
    oracle_lib.set_threads(threads)
    orc = oracle_lib.OracleSim((n,) * 3, dx, tol=1e-9)
    orc.set_solid_phi(oracle_lib.solid_phi_meshes((n,) * 3, dx, [(verts, tris)], 7)[0])
    orc.load(pos)
    orc.initialize()
    orc.step(1.0 / 240.0)
    times = []
    for s in range(substeps):
        t0 = time.perf_counter()
        orc.step(1.0 / 240.0)
        times.append(time.perf_counter() - t0)
        log("  oracle substep %d: %.2f s" % (s + 1, times[-1]))
    oracle_lib.set_threads(1)
    out["port"] = {"substeps_per_s": len(times) / sum(times), "seconds": [round(t, 3) for t in times]}
    ratio = out["reference"]["substeps_per_s"] / out["port"]["substeps_per_s"]
    line = {"metric": "CPU substeps/s at %d^3: reference engine vs the oracle, same host and threads" % n,
            "n": n, "threads": threads, "host_cpus": os.cpu_count(), "substeps": substeps,
            "reference": out["reference"], "port": out["port"], "reference_over_port": round(ratio, 4)}
    print(json.dumps(line), flush=True)


def precision_config(n, tol):
    """The precision configuration: one pressure solve + projection of a liquid
    slab over 40% of the height carrying smoothed Gaussian-noise velocities
    (0.5 m/s, 8-cell correlation), in every PCG mode.  Reports each mode's
    pressure error (relative L2) against the FP64 GPU solve, its iterations and
    the largest divergence left after the projection (max |rhs| of the
    projected field).  The FP64 GPU solve itself is checked against the FP64
    CPU oracle at 40^3 by the test suite."""
    import numpy as np
    from ffengine import kernels, scenes
    n3, dx, dt = (n, n, n), 1.0 / n, 1.0 / 240.0
    log("precision slab n=%d" % n)
    phi, uvw = scenes.precision_slab(n, seed=0)
    weights = kernels.face_weights(n3, kernels.solid_box_phi(n3, dx))
    div0 = float(np.abs(kernels.pressure_system(n3, dx, dt, uvw, weights, phi)["rhs"]).max())
    res, ref = {}, None
    for mode, name in ((0, "fp64"), (1, "mixed"), (2, "mixed-reliable"), (3, "fp32-preconditioner")):
        t0 = time.perf_counter()
        p, uvw2, _, it, err, ok = kernels.pressure_solve(n3, dx, dt, uvw, weights, phi, tol=tol, max_iter=20000,
                                                         mode=mode)
        wall = time.perf_counter() - t0
        div = float(np.abs(kernels.pressure_system(n3, dx, dt, uvw2, weights, phi)["rhs"]).max())
        if ref is None:
            ref = p.astype(np.float64)
        l2 = float(np.linalg.norm(p.astype(np.float64) - ref) / max(np.linalg.norm(ref), 1e-300))
        res[name] = {"iterations": int(it), "residual_inf": float(err), "success": bool(ok),
                     "pressure_rel_l2_vs_fp64": l2, "divergence_max_after": div,
                     "wall_s_with_host_copies": round(wall, 3)}
        log("  %s: iters %d residual %.3g rel L2 %.3g div %.3g (%.1fs)" % (name, it, err, l2, div, wall))
    line = {"metric": "pressure rel L2 vs FP64 PCG and max post-projection divergence, precision slab %d^3" % n,
            "value": res["mixed"]["pressure_rel_l2_vs_fp64"], "unit": "relative L2", "n_gpus": 1,
            "higher_is_better": False, "data": "synthetic",
            "config": {"workload": "liquid slab over 40%% of %d^3, smoothed Gaussian-noise MAC velocity "
                                   "(0.5 m/s, 8-cell correlation, seed 0), dt 1/240 s, PCG rel res %g" % (n, tol),
                       "grid": n},
            "divergence_max_before": div0, "modes": res}
    print(json.dumps(line), flush=True)


def splash_config(n, steps, warmup, tol, mode):
    """The large single-GPU configuration: a sphere of liquid (r = 0.2) falling
    into a pool over 30% of the height, 8 particles per liquid cell."""
    import torch
    _, total = torch.cuda.mem_get_info()
    log("splash n=%d: seeding particles" % n)
    from ffengine import scenes
    pos = scenes.splash_particles(n)
    log("  %d particles" % len(pos))
    res = run_mode(n, pos, None, mode, tol, steps, warmup, 1.0 / 240.0)
    rate = res["substeps"] / res["elapsed_s"]
    P = res["particles"]
    kt = res["kernels"]
    M_total = sum(u * it for u, it in zip(res["unknowns"], res["iterations"]))
    peak_used = res.get("device_bytes_used", 0)
    gbs = {}
    for k, v in kt.items():
        b = algorithmic_bytes(k, n, P, M_total, 1, res["substeps"], sum(res["iterations"]), mode)
        if b is not None and v["ms"] > 0:
            gbs[k] = round(b / (v["ms"] * 1e-3) / 1e9, 1)
    line = {"metric": "FLIP substeps/s, splash %d^3" % n, "value": round(rate, 4), "unit": "substeps/s",
            "n_gpus": 1, "steps": steps, "warmup": warmup, "higher_is_better": True, "data": "synthetic",
            "dtype": "f32+f64" if mode != "fp64" else "f64", "mode": mode,
            "config": {"workload": "sphere of liquid r=0.2 at (0.5, 0.65, 0.5) falling into a pool over 30%% of "
                                   "%d^3, %d particles, frame 1/240 s, PCG rel res %g" % (n, len(pos), tol),
                       "grid": n, "particles": len(pos)},
            "particle_updates_per_s": round(rate * P, 1),
            "pressure_iterations": res["iterations"], "unknowns": res["unknowns"],
            "kernel_ms": {k: round(v["ms"], 3) for k, v in kt.items()}, "kernel_gb_per_s": gbs,
            "device_memory_gb": round(peak_used / 1e9, 2), "device_memory_total_gb": round(total / 1e9, 1)}
    print(json.dumps(line), flush=True)


def moving_config(n, steps, warmup, tol, mode, speed):
    """The 256^3 dam break with its sphere obstacle (the 20480-triangle
    icosphere MeshObject) animated: it moves along +z at `speed` m/s, each
    frame's MeshObject_update_mesh_animated giving the previous, current and
    next frame's meshes, so the solid (with its face velocities, the cells'
    solid weights and the pocket conditioning) is rebuilt every substep.  The
    same run with the sphere static is timed beside it."""
    import torch
    from ffengine import FluidSimulation, MeshObject, TriangleMesh, scenes
    frame_dt = 1.0 / 240.0
    pos = scenes.dam_break_particles(n, seed=0)
    v, t = scenes.sphere_mesh(subdivisions=5)
    d = np.array([0.0, 0.0, speed * frame_dt], np.float32)
    out = {}
    for moving in (False, True):
        sim = FluidSimulation(n, n, n, 1.0 / n)
        sim.add_body_force(0.0, -9.81, 0.0)
        sim.PICFLIP_ratio = 0.05
        sim.CFL_condition_number = 5
        sim.enable_surface_reconstruction = False
        sim.pressure_solver_tolerance = tol
        sim.set_pressure_solver_precision(mode)
        mo = MeshObject(n, n, n, 1.0 / n)
        if moving:
            mo.update_mesh_animated(TriangleMesh(v - d, t), TriangleMesh(v, t), TriangleMesh(v + d, t))
        else:
            mo.update_mesh_static(TriangleMesh(v, t))
        sim.add_mesh_obstacle(mo)
        sim.load_marker_particle_data(len(pos), pos.tobytes(), np.zeros_like(pos).tobytes())
        sim.initialize()
        iters, substeps, elapsed = [], 0, 0.0
        for f in range(warmup + steps):
            if moving and f > 0:
                c = v + f * d
                mo.update_mesh_animated(TriangleMesh(c - d, t), TriangleMesh(c, t), TriangleMesh(c + d, t))
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            sim.update(frame_dt)
            torch.cuda.synchronize()
            if f >= warmup:
                elapsed += time.perf_counter() - t0
                st = sim.get_frame_stats_data()
                substeps += st.substeps
                iters.append(st.pressure_solver_iterations)
            log("  %s frame %d/%d" % ("moving" if moving else "static", f + 1, warmup + steps))
        vel = sim.get_solid_velocity_field()
        out["moving" if moving else "static"] = {
            "substeps_per_s": round(substeps / elapsed, 4), "ms_per_substep": round(1e3 * elapsed / substeps, 2),
            "pressure_iterations": iters, "particles": sim.get_num_marker_particles(),
            "max_solid_speed": round(max(float(np.abs(a).max()) for a in vel), 4)}
        del sim, mo
    rate = out["moving"]["substeps_per_s"]
    line = {"metric": "FLIP substeps/s, dam break %d^3 with an animated sphere obstacle" % n, "value": rate,
            "unit": "substeps/s", "n_gpus": 1, "steps": steps, "warmup": warmup, "higher_is_better": True,
            "data": "synthetic", "dtype": "f32+f64" if mode != "fp64" else "f64", "mode": mode,
            "config": {"workload": "dam break %d^3, %d particles, the 20480-triangle sphere MeshObject (r 0.15 at "
                                   "(0.6, 0.2, 0.5)) animated at %g m/s along +z, frame 1/240 s, PCG rel res %g"
                                   % (n, len(pos), speed, tol), "grid": n, "particles": len(pos)},
            "moving": out["moving"], "static": out["static"],
            "rebuild_ms_per_substep": round(out["moving"]["ms_per_substep"] - out["static"]["ms_per_substep"], 2)}
    print(json.dumps(line), flush=True)


def properties_config(n, steps, warmup, tol, mode, visc, tension):
    """The 256^3 dam break with its sphere obstacle (the 20480-triangle
    icosphere MeshObject) run three ways: plain, with a constant viscosity
    (every substep runs the viscosity solve after the body forces: the
    reference's ViscositySolver system, solved on the GPU by
    Jacobi-preconditioned CG to the reference's tolerance 1e-4), and with
    surface tension (every substep computes the curvature grid and the
    cluster status, and the pressure solve takes the tension terms).
    Reports each run's substep rate and the stages' shares; the line's
    value is the viscous run's rate."""
    import torch
    from ffengine import FluidSimulation, MeshObject, TriangleMesh, scenes
    frame_dt = 1.0 / 240.0
    pos = scenes.dam_break_particles(n, seed=0)
    v, t = scenes.sphere_mesh(subdivisions=5)
    out = {}
    for kind in ("plain", "viscous", "tension"):
        sim = FluidSimulation(n, n, n, 1.0 / n)
        sim.add_body_force(0.0, -9.81, 0.0)
        sim.PICFLIP_ratio = 0.05
        sim.CFL_condition_number = 5
        sim.enable_surface_reconstruction = False
        sim.pressure_solver_tolerance = tol
        sim.set_pressure_solver_precision(mode)
        if kind == "viscous":
            sim.viscosity = visc
        if kind == "tension":
            sim.surface_tension = tension
        mo = MeshObject(n, n, n, 1.0 / n)
        mo.update_mesh_static(TriangleMesh(v, t))
        sim.add_mesh_obstacle(mo)
        sim.load_marker_particle_data(len(pos), pos.tobytes(), np.zeros_like(pos).tobytes())
        sim.initialize()
        iters, viters, vms, vrows, substeps, elapsed = [], [], [], [], 0, 0.0
        for f in range(warmup + steps):
            if f == warmup:
                enable_timing(sim, True)  # counts the timed frames only
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            sim.update(frame_dt)
            torch.cuda.synchronize()
            if f >= warmup:
                elapsed += time.perf_counter() - t0
                st = sim.get_frame_stats_data()
                substeps += st.substeps
                iters.append(st.pressure_solver_iterations)
                if kind == "viscous":
                    vs = sim.get_last_viscosity_solve_stats()
                    viters.append(vs["iterations"])
                    vrows.append(vs["unknowns"])
                    vms.append(round(sim.get_last_substep_phase_ms(8), 2))
            log("  %s frame %d/%d" % (kind, f + 1, warmup + steps))
        rec = {"substeps_per_s": round(substeps / elapsed, 4), "ms_per_substep": round(1e3 * elapsed / substeps, 2),
               "pressure_iterations": iters, "particles": sim.get_num_marker_particles()}
        if kind == "viscous":
            rec.update({"viscosity_iterations": viters, "viscosity_rows": vrows, "viscosity_ms_last_substep": vms,
                        "viscosity_ms_per_substep": round(kernel_times(sim)["viscosity"]["ms"] / substeps, 2)})
        out[kind] = rec
        del sim, mo
    line = {"metric": "FLIP substeps/s, dam break %d^3 with viscosity %g" % (n, visc),
            "value": out["viscous"]["substeps_per_s"], "unit": "substeps/s", "n_gpus": 1, "steps": steps,
            "warmup": warmup, "higher_is_better": True, "data": "synthetic",
            "dtype": "f32+f64" if mode != "fp64" else "f64", "mode": mode,
            "config": {"workload": "dam break %d^3, %d particles, the 20480-triangle sphere MeshObject (r 0.15 at "
                                   "(0.6, 0.2, 0.5)), frame 1/240 s, PCG rel res %g; viscous: constant viscosity %g "
                                   "(solver tolerance 1e-4); tension: surface tension %g"
                                   % (n, len(pos), tol, visc, tension), "grid": n, "particles": len(pos)},
            "plain": out["plain"], "viscous": out["viscous"], "tension": out["tension"]}
    print(json.dumps(line), flush=True)


def adjoint_config(n, substeps, checkpoint_every, fd_faces, eps, tol, dt):
    """The differentiation configuration: a dam break (block [0, 0.375) x
    [0, 0.625) x [0, 1), 8 particles per cell outside the walls) whose initial
    particle velocities are G2P of an initial MAC field (zero: the dam at
    rest), run for `substeps` substeps of dt.  Loss = squared L2 distance of
    the particle density after the last substep to a target density from
    the same run started from a seeded perturbation (smoothed noise,
    0.2 m/s) of the initial field.  Times the forward (with checkpoints every
    `checkpoint_every` substeps) and the backward (recomputation + adjoint),
    then checks the gradient by central differences on `fd_faces` seeded
    faces (forwards with the recorded masks) and along one smooth direction
    at three step sizes.  The map has jumps the adjoint does not see (the
    collision response's 0.1 dx path search; a face losing its last particle
    in P2G), crossed more often the larger the step; below the jumps the
    float32 state's rounding sets a noise floor."""
    import numpy as np
    from ffengine import kernels, scenes
    from ffengine.rollout import Rollout
    n3, dx = (n, n, n), 1.0 / n
    log("adjoint configuration n=%d, %d substeps, checkpoints every %d" % (n, substeps, checkpoint_every))
    pos = scenes.dam_break_particles(n, seed=0)
    solid = kernels.solid_box_phi(n3, dx)
    c = np.floor(pos / dx).astype(int)
    free = np.ones(len(pos), bool)
    for o in range(8):
        a, b, e = o & 1, (o >> 1) & 1, o >> 2
        free &= solid[c[:, 2] + e, c[:, 1] + b, c[:, 0] + a] > 0
    pos = np.ascontiguousarray(pos[free])
    shapes = [(n, n, n + 1), (n, n + 1, n), (n + 1, n, n)]
    init = [np.zeros(s, np.float32) for s in shapes]
    target_init = scenes.noise_mac_field(n, seed=1, amplitude=0.2, correlation=8.0)
    ro = Rollout(n3, dx, pos, dt=dt, substeps=substeps, checkpoint_every=checkpoint_every, tol=tol, max_iter=5000)
    target = ro.forward(*target_init).astype(np.float64)

    def loss(rho):
        return float(((rho.astype(np.float64) - target) ** 2).sum())

    t0 = time.perf_counter()
    rho = ro.forward(*init)
    t_fwd = time.perf_counter() - t0
    moved, fwd_iters, _ = ro.stats()
    L0 = loss(rho)
    t0 = time.perf_counter()
    g = ro.backward((2.0 * (rho.astype(np.float64) - target)).astype(np.float32))
    t_bwd = time.perf_counter() - t0
    _, _, bwd_iters = ro.stats()
    log("  %d particles, loss %.6g, forward %.2fs (%d PCG iterations, %d collision moves), backward %.2fs "
        "(%d adjoint PCG iterations)" % (len(pos), L0, t_fwd, fwd_iters, moved, t_bwd, bwd_iters))
    scale = max(float(np.abs(a).max()) for a in g)
    rng = np.random.default_rng(2)
    cand = [(d, i) for d in range(3) for i in np.flatnonzero(np.abs(g[d]).ravel() > 0.01 * scale)]
    picks = [cand[int(q)] for q in rng.choice(len(cand), size=min(fd_faces, len(cand)), replace=False)]
    steps = [eps]
    pairs = {e: [] for e in steps}
    t0 = time.perf_counter()
    for q, (d, i) in enumerate(picks):
        for e in steps:
            plus = [a.copy() for a in init]
            minus = [a.copy() for a in init]
            plus[d].ravel()[i] += e
            minus[d].ravel()[i] -= e
            h = float(plus[d].ravel()[i]) - float(minus[d].ravel()[i])
            fd = (loss(ro.forward(*plus, freeze=True)) - loss(ro.forward(*minus, freeze=True))) / h
            pairs[e].append((fd, float(g[d].ravel()[i])))
        if q % 8 == 7:
            log("  central differences: %d of %d faces (%.0fs)" % (q + 1, len(picks), time.perf_counter() - t0))
    t_fd = time.perf_counter() - t0

    def fd_stats(e):
        v = np.array(pairs[e])
        err = np.abs(v[:, 0] - v[:, 1]) / scale
        rel = np.abs(v[:, 0] - v[:, 1]) / np.maximum(np.abs(v[:, 1]), 1e-300)
        return {"eps": e, "max_err_over_max_grad": float(err.max()), "median_err_over_max_grad": float(np.median(err)),
                "median_rel_err": float(np.median(rel)), "sign_agreement": int((np.sign(v[:, 0]) == np.sign(v[:, 1])).sum()),
                "correlation": float(np.corrcoef(v[:, 0], v[:, 1])[0, 1]) if len(v) > 2 else None}
    direction = scenes.noise_mac_field(n, seed=3, amplitude=1.0, correlation=8.0)
    dad = sum(float(np.dot(a.astype(np.float64).ravel(), b.astype(np.float64).ravel())) for a, b in zip(g, direction))
    dirs = []
    for tdir in (1e-6, 1e-5, 1e-4):
        lp = loss(ro.forward(*[a + tdir * b for a, b in zip(init, direction)], freeze=True))
        mp = ro.stats()[0]
        lm = loss(ro.forward(*[a - tdir * b for a, b in zip(init, direction)], freeze=True))
        mm = ro.stats()[0]
        dfd = (lp - lm) / (2 * tdir)
        dirs.append({"step": tdir, "fd": dfd, "fd_over_adjoint": dfd / dad, "collision_moves": [mp, mm]})
    stats = [fd_stats(e) for e in steps]
    for s in stats:
        log("  central differences on %d faces, eps %g: error max %.3g, median %.3g of max |grad|, median relative "
            "%.3g; sign agreement %d/%d; correlation %.4f" % (len(picks), s["eps"], s["max_err_over_max_grad"],
                                                             s["median_err_over_max_grad"], s["median_rel_err"],
                                                             s["sign_agreement"], len(picks), s["correlation"]))
    for r in dirs:
        log("  direction, step %g: fd %.6g adjoint %.6g ratio %.4f (collision moves %s)"
            % (r["step"], r["fd"], dad, r["fd_over_adjoint"], r["collision_moves"]))
    line = {"metric": "differentiable rollout %d^3, %d substeps: seconds for the gradient of the density loss "
                      "wrt the initial MAC velocity" % (n, substeps),
            "value": round(t_fwd + t_bwd, 3), "unit": "s", "n_gpus": 1, "higher_is_better": False,
            "data": "synthetic", "dtype": "f32+f64",
            "config": {"workload": "dam break %d^3 (%d particles outside the walls), %d substeps of %.6g s, "
                                   "checkpoints every %d, PCG rel res %g (forward and adjoint)"
                                   % (n, len(pos), substeps, dt, checkpoint_every, tol),
                       "grid": n, "particles": len(pos)},
            "forward_s": round(t_fwd, 3), "backward_s": round(t_bwd, 3),
            "substeps_per_s_forward": round(substeps / t_fwd, 2),
            "pcg_iterations": {"forward": fwd_iters, "adjoint": bwd_iters}, "collision_moves": moved,
            "loss": L0, "grad_max_abs": scale,
            "central_differences": {"faces": len(picks), "face_pool": "faces with |grad| > 1% of max",
                                    "steps": stats,
                                    "direction": {"adjoint": dad, "unit_amplitude_noise_field": True, "steps": dirs}}}
    ro.close()
    print(json.dumps(line), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--config", default="dam-break",
                    choices=["dam-break", "precision", "splash", "adjoint", "moving", "properties",
                             "cpu-calibration"],
                    help="dam-break: the 256^3 headline benchmark (default); precision: the 384^3 slab "
                         "pressure-accuracy comparison; splash: the 512^3 splash; adjoint: the 128^3 "
                         "differentiable rollout with its finite-difference check; moving: the 256^3 dam break "
                         "with its sphere obstacle animated, beside the static run; properties: the 256^3 dam "
                         "break plain, with a constant viscosity and with surface tension; cpu-calibration (no GPU, "
                         "needs the reference build): the reference engine against the oracle on the host")
    ap.add_argument("--speed", type=float, default=0.3, help="moving: the sphere's speed along +z (m/s)")
    ap.add_argument("--viscosity", type=float, default=0.5, help="properties: the constant viscosity")
    ap.add_argument("--surface-tension", type=float, default=0.2, help="properties: the surface tension constant")
    ap.add_argument("--substeps", type=int, default=32, help="adjoint: substeps of the rollout")
    ap.add_argument("--checkpoint-every", type=int, default=8, help="adjoint: checkpoint spacing")
    ap.add_argument("--fd-faces", type=int, default=64, help="adjoint: faces checked by central differences")
    ap.add_argument("--fd-eps", type=float, default=1e-3, help="adjoint: central-difference step (m/s)")
    ap.add_argument("--dt", type=float, default=1.0 / 240.0, help="adjoint: substep length (s)")
    ap.add_argument("--obstacle", default="mesh", choices=["mesh", "phi"],
                    help="dam-break: the sphere as a static MeshObject (the reference's obstacle path) or as a "
                         "nodal SDF set directly")
    ap.add_argument("--transfer", default="flip", choices=["flip", "apic"],
                    help="dam-break: velocity transfer method (the headline uses FLIP)")
    ap.add_argument("--no-warm-extra", action="store_true",
                    help="dam-break: skip the warm-started runs reported beside the headline")
    ap.add_argument("--warm-start", action="store_true",
                    help="dam-break: FP64 PCG modes start from the previous substep's pressure (the headline "
                         "starts from 0, as the reference does)")
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=4)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--n", type=int, default=None, help="grid edge (default 256, 384 or 512 by --config)")
    ap.add_argument("--tol", type=float, default=1e-8)
    ap.add_argument("--cpu-threads", type=int, default=None,
                    help="host threads of the CPU baseline (default: min(16, cpu count))")
    ap.add_argument("--cpu-substeps", type=int, default=3, help="cpu-calibration: timed substeps per engine")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--schedule", type=int, default=None, choices=[2, 4, 5],
                    help="MIC(0) application: 2 = columns of lines, 4 = line pipeline, 5 = bands of hyperplanes from a "
                         "replayed graph (default: the engine's)")
    ap.add_argument("--modes", default="fp64,mixed,mixed-reliable,fp32-preconditioner",
                    help="comma list of PCG modes: fp64, mixed (FP32 PCG restarted in FP64 refinement), "
                         "mixed-reliable (FP32 PCG with FP64 reliable updates), fp32-preconditioner (FP64 "
                         "PCG with the MIC(0) application in FP32)")
    args = ap.parse_args()
    cpu_threads = args.cpu_threads or min(16, os.cpu_count() or 1)
    if args.config == "cpu-calibration":
        cpu_calibration(args.n or 256, args.cpu_substeps, cpu_threads)
        return
    if args.gpus != 1:
        print("bench.py runs on one GPU: the engine keeps a whole simulation on one device "
              "(multi-GPU slab decomposition is design-only); got --gpus %d" % args.gpus, file=sys.stderr)
        sys.exit(2)
    import torch
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)
    torch.cuda.set_device(0)
    from ffengine import kernels, scenes

    if args.config == "precision":
        precision_config(args.n or 384, args.tol)
        return
    if args.config == "adjoint":
        adjoint_config(args.n or 128, args.substeps, args.checkpoint_every, args.fd_faces, args.fd_eps, args.tol,
                       args.dt)
        return
    if args.config == "moving":
        modes = [m for m in args.modes.split(",") if m]
        moving_config(args.n or 256, args.steps, args.warmup, args.tol,
                      modes[0] if len(modes) == 1 else "fp32-preconditioner", args.speed)
        return
    if args.config == "properties":
        modes = [m for m in args.modes.split(",") if m]
        properties_config(args.n or 256, args.steps, args.warmup, args.tol,
                          modes[0] if len(modes) == 1 else "fp32-preconditioner", args.viscosity,
                          args.surface_tension)
        return
    if args.config == "splash":
        modes = [m for m in args.modes.split(",") if m]
        splash_config(args.n or 512, args.steps, args.warmup, args.tol, modes[0] if len(modes) == 1 else "mixed")
        return
    n = args.n or 256
    dx = 1.0 / n
    frame_dt = 1.0 / 240.0
    # one plain device-to-device copy of exactly 512 MiB before the timed
    # region: its counters in a profile calibrate the HBM byte counts
    cal_src = torch.empty(64 << 20, dtype=torch.float64, device="cuda")
    cal_dst = torch.empty_like(cal_src)
    cal_dst.copy_(cal_src)
    torch.cuda.synchronize()
    del cal_src, cal_dst
    log("scene n=%d" % n)
    pos = scenes.dam_break_particles(n, seed=0)
    if args.obstacle == "mesh":
        # the sphere as the reference takes it: a static MeshObject obstacle
        solid = scenes.sphere_mesh(subdivisions=5)
    else:
        solid = scenes.union_phi(kernels.solid_box_phi((n, n, n), dx), scenes.sphere_phi_nodes(n))
    modes = [m for m in args.modes.split(",") if m]
    if not set(modes) <= {"fp64", "mixed", "mixed-reliable", "fp32-preconditioner"} or not modes:
        sys.exit("--modes takes fp64, mixed, mixed-reliable and/or fp32-preconditioner")
    results = {}
    for q, mode in enumerate(modes):
        log("mode %s" % mode)
        results[mode] = run_mode(n, pos, solid, mode, args.tol, args.steps, args.warmup, frame_dt,
                                 args.transfer == "apic", args.warm_start, args.schedule,
                                 keep_state=(q == 0 and not args.no_cpu))
    state = results[modes[0]].pop("state")
    for r in results.values():
        r.pop("state", None)
    # headline: the faster mixed-precision mode, else FP64
    mixed_modes = [m for m in ("mixed-reliable", "mixed", "fp32-preconditioner") if m in results]
    rate = lambda m: results[m]["substeps"] / results[m]["elapsed_s"]  # noqa: E731
    main_mode = max(mixed_modes, key=rate) if mixed_modes else "fp64"
    mixed, fp64 = results.get(main_mode) if mixed_modes else None, results.get("fp64")
    head = results[main_mode]
    value = head["substeps"] / head["elapsed_s"]
    fp64_rate = fp64["substeps"] / fp64["elapsed_s"] if fp64 else None

    # dominant kernel of the headline run by measured time
    P = head["particles"]
    kt = head["kernels"]
    dom = max((k for k in kt if algorithmic_bytes(k, n, P, 1, 1, 1, 1, "mixed") is not None),
              key=lambda k: kt[k]["ms"])
    M_total = 0
    iters = head["iterations"]
    for u, it in zip(head["unknowns"], iters):
        M_total += u * it
    bytes_ = algorithmic_bytes(dom, n, P, M_total, 1, head["substeps"], sum(iters), main_mode)
    achieved = bytes_ / (kt[dom]["ms"] * 1e-3) / 1e9 if kt[dom]["ms"] > 0 else 0.0
    launches = max(kt[dom]["launches"], 1)
    traffic, kname = None, dom
    if dom == "mic0_apply":
        kname = sweep_kernel_name(main_mode == "fp64", args.schedule or 2)
        traffic = measured_traffic(kname)
    # algorithmic HBM bytes / time of every kernel group that has a byte model
    # (SpMV, the transfers, the preconditioner, ...), as a fraction of 8 TB/s
    hbm_fraction = {}
    for k, v in kt.items():
        b = algorithmic_bytes(k, n, P, M_total, 1, head["substeps"], sum(iters), main_mode)
        if b is not None and v["ms"] > 0:
            hbm_fraction[k] = round(b / (v["ms"] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)
    roofline = {"bound": "hbm", "achieved": round(achieved, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": traffic, "kernel": kname,
                "avg_launch_us": round(kt[dom]["ms"] * 1e3 / launches, 3),
                "algorithmic_bytes_per_launch": int(bytes_ / launches)}

    mesh_sdf = None
    if args.obstacle == "mesh":
        log("mesh obstacle SDF build")
        mesh_sdf = mesh_obstacle_sdf(n, solid, not args.no_cpu, cpu_threads)

    cpu = None
    if not args.no_cpu and state is not None:
        log("cpu baseline: the oracle, one substep at n=%d on %d threads" % (n, cpu_threads))
        cpu = cpu_baseline(state, n, args.tol, cpu_threads)
    del state

    # the same two solvers started from the previous substep's pressure (an
    # option of this engine; the reference's PCG starts from 0): reported
    # beside the headline, never as it
    warm = {}
    if not args.warm_start and not args.no_warm_extra and args.transfer == "flip":
        for mode in dict.fromkeys(["fp64", main_mode]):
            log("warm-started %s" % mode)
            r = run_mode(n, pos, solid, mode, args.tol, args.steps, args.warmup, frame_dt, False, True)
            warm[mode] = {"substeps_per_s": round(r["substeps"] / r["elapsed_s"], 4), "pressure_iterations": r["iterations"]}
    line = {
        "metric": "FLIP substeps/s at 256^3, mixed vs FP64 PCG at rel res 1e-8; % HBM peak",
        "value": round(value, 4), "unit": "substeps/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(1e3 * head["elapsed_s"] / args.steps, 3),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32+f64" if main_mode != "fp64" else "f64",
        "data": "synthetic",
        "config": {"workload": "dam break %d^3 + static sphere obstacle (%s), %d particles, frame 1/240 s, "
                               "PCG rel res %g%s" % (n, "icosphere MeshObject, %d triangles" % len(solid[1])
                                                     if args.obstacle == "mesh" else "nodal SDF", len(pos), args.tol,
                                                     ", APIC transfer" if args.transfer == "apic" else ""),
                   "grid": n, "particles": len(pos)},
        "mode": main_mode,
        "transfer": args.transfer,
        "warm_start": bool(args.warm_start),
        "warm_started_pcg": warm or None,
        "substeps_per_s": {m: round(rate(m), 4) for m in results},
        "fp64_substeps_per_s": round(fp64_rate, 4) if fp64_rate else None,
        "mixed_over_fp64": round(value / fp64_rate, 4) if (fp64_rate and mixed) else None,
        "pressure_iterations": {m: results[m]["iterations"] for m in results},
        "kernel_ms": {m: {k: round(v["ms"], 3) for k, v in results[m]["kernels"].items()} for m in results},
        "roofline": roofline,
        "hbm_fraction_by_group": hbm_fraction,
        "mesh_obstacle_sdf": mesh_sdf,
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
