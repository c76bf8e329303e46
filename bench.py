#!/usr/bin/env python3
"""Benchmark of the explicit hex8 neo-Hookean path on one MI355X.

Workload (default): 100^3 hex8 unit cube (1.0M elements, 1.03M nodes, 2x2x2 Gauss), interior nodes
perturbed by U(-0.1h, 0.1h) (SplitMix64 seed 0x4D50530001), compressible neo-Hookean E=1e6 Pa,
nu=0.3, rho=1000; bottom face clamped, top face prescribed z-velocity ramped to 0.1 m/s over the
first 100 steps; lumped mass, central difference, dt = 0.5 x stable dt recomputed every step.

A step = one explicit step of the whole mesh (element forces, CSR gather, central-difference update,
stable-dt reduction).  `value` = element-Gauss-point updates per second of the FP64 form over the timed
steps (inputs resident in HBM; wall clock between two device synchronisations).  The FP32-element /
FP64-accumulate form is reported beside it with its displacement error against the FP64 form.

A GPU reaches its steady rate on this workload only after some 30-60 ms of it: started cold, the first ~200
steps run up to 10% slower (0.157 falling to 0.141 ms per step over the first ten 20-step chunks), whether the
solve starts from rest or from a moving state, and an HBM-bound warm-up (the copy probe) does not shorten it,
while a solve that has run 400 steps is at 0.141 ms from its first chunk.  So before each leg's warm-up steps
a separate solver of the same workload runs PREWARM_STEPS steps and is closed; the measured solver's graphs
are captured before that, so that no host work idles the GPU between the pre-warm and the timed steps.  The
measured solver still runs exactly `--warmup` untimed steps, then the timed ones.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "v.1.1_amd"))
sys.path.insert(0, os.path.join(ROOT, "tests"))

import numpy as np  # noqa: E402

import mps_gpu as G  # noqa: E402
from mps_gpu import configs  # noqa: E402

HBM_PEAK_GBS = 8000.0
FP64_PEAK_TFLOPS = 78.6
VALU_ISSUE_PEAK = 256 * 2.4e9  # MI355X: 256 CUs x 2.4 GHz, one wave64 VALU instruction per CU per cycle
TRAFFIC_TABLE = os.path.join(ROOT, "profiles", "hex8_cube100_hbm_traffic.md")
# the dominant kernel: k_elem<T, nodes, law, viscosity, energies, 32-bit node offsets>
ELEM_KERNEL = "k_elem<double,8,0,false,false,true>"


def measured_traffic(kernel):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 FETCH_SIZE/WRITE_SIZE summary
    (copy-kernel-calibrated, one row per kernel: | `name` | fetch KiB | write KiB | fetched MB | written MB |
    total MB | ...).  None when the summary or the row is absent."""
    try:
        with open(TRAFFIC_TABLE) as f:
            for line in f:
                cells = [c.strip() for c in line.strip().strip("|").split("|")]
                if len(cells) >= 6 and cells[0] == f"`{kernel}`":
                    return float(cells[5].replace(",", "")) * 1e6
    except OSError:
        pass
    return None


def measured_valu_per_wave(kernel):
    """VALU instructions per wave of `kernel` from the committed rocprofv3 SQ_INSTS_VALU/SQ_WAVES table
    (| `name` | VALU instructions / wave | VALU busy | resident cycles | waiting |), or None."""
    try:
        with open(TRAFFIC_TABLE) as f:
            for line in f:
                cells = [c.strip() for c in line.strip().strip("|").split("|")]
                if len(cells) == 5 and cells[0] == f"`{kernel}`":
                    return float(cells[1].replace(",", ""))
    except OSError:
        pass
    return None


def note(msg):
    """Progress line on stderr (the JSON result is the only stdout line)."""
    print(f"bench: {msg}", file=sys.stderr, flush=True)


PATCH = 256  # elements per patch of the element kernel (MPS_PATCH)
PREWARM_STEPS = 400  # steps of a separate solver of the same workload before each leg's warm-up (about 60 ms)


def elem_kernel_bytes(ne, nn, nen, n_part, per_elem_mat):
    """Algorithmic HBM bytes of one element-kernel launch: per element its node references + l0 8 (+
    material 24 when per element) + patch contribution list 2 nen; per partial its offset 2 + FP64 force
    write 24; per node X and u, 24 B each (read once).  Node references: hex8 conn 4 nen; tet4 (node
    staging) the local indices 2 nen per element and the patch node id 4 per partial."""
    n_patch = -(-ne // PATCH)
    refs = ne * 4 * nen if nen == 8 else ne * 2 * nen + n_part * 4
    return refs + ne * (8 + (24 if per_elem_mat else 0) + 2 * nen) + n_part * (2 + 24) + 4 * (n_patch + 1) \
        + nn * (24 + 24)


def node_kernel_bytes(nn, n_part):
    """Algorithmic HBM bytes of one node-kernel launch between two steps of a launch: per node CSR offset 4, BC
    info 4, u and the half-step velocity w read 48 and written 48, mass 8; per partial its index 4 and FP64 force
    read 24."""
    return nn * (4 + 4 + 48 + 48 + 8) + n_part * (4 + 24)


def step_bytes(ne, nn, nen, n_part, per_elem_mat):
    """Algorithmic HBM bytes of one whole step (element + node kernels)."""
    return elem_kernel_bytes(ne, nn, nen, n_part, per_elem_mat) + node_kernel_bytes(nn, n_part)


def run_gpu(cfg, precision, warmup, steps, prof_steps=None, energy_every=0):
    """Warm-up, then `steps` timed steps (graph replay, no per-kernel events), then `prof_steps` (default
    `steps`) more steps launched one by one with HIP events around every kernel on the solver's stream:
    the per-kernel averages and the event-timed step rate come from that second region.  The
    displacement returned is the one after warm-up + timed steps."""
    prof_steps = steps if prof_steps is None else prof_steps
    m = cfg["mesh"]
    total = warmup + steps + prof_steps

    def solver(n_steps, ee):
        return G.Solver(m, law=cfg["law"], E=cfg["E"], nu=cfg["nu"], rho=cfg["rho"], dir_dof=cfg["dir_dof"],
                        dir_val=cfg["dir_val"], bc_mode=G.BC_VELOCITY, vel_ramp_steps=100, scale=cfg["scale"],
                        n_steps=n_steps, precision=precision, energy_every=ee, history_cap=n_steps if ee else 0)

    s = solver(total, energy_every)
    # graph capture and instantiation of the warm-up and timed chunks stay outside the clock, and before the
    # pre-warm, so that the GPU does not idle between it and the timed steps
    s.prepare_run(warmup)
    s.prepare_run(steps)
    if PREWARM_STEPS > 0:  # a separate solver brings the GPU to its steady rate (module docstring)
        w = solver(PREWARM_STEPS, energy_every)
        rc, rep = w.run(PREWARM_STEPS)
        assert rc == 0, rep
        w.close()
    rc, rep = s.run(warmup)
    assert rc == 0, rep
    s.prepare_run(steps)  # finds the graphs captured above (their key is the chunk length and energy phase)
    t0 = time.perf_counter()
    rc, rep = s.run(steps)
    t1 = time.perf_counter()
    assert rc == 0 and rep["steps"] == warmup + steps, (rc, rep)
    u, v, a = s.get_state()
    hist = None
    if energy_every:
        hist = s.history(0, warmup + steps)
        hist.update(s.energy_balance(0, warmup + steps))
    s.profile(True)
    t2 = time.perf_counter()
    rc, rep2 = s.run(prof_steps)
    t3 = time.perf_counter()
    assert rc == 0, rep2
    kt = s.kernel_times()
    n_part = s.layout()["n_part"]  # partial forces: distinct nodes per patch, in the library's element order
    s.close()
    return dict(wall_s=t1 - t0, device_ms=rep["device_ms"], kt=kt, u=u, rep=rep, hist=hist,
                events_ms_per_step=(t3 - t2) * 1e3 / prof_steps, n_part=n_part)


def energy_leg(cfg, warmup, steps, plain_ms):
    """The FP64 leg with DEFO_ENERGY, KIN_ENERGY, VOLUME, EXTERNAL_ENERGY and the work sums every step: cost
    against the plain step, and the energy balance (lumped kinetic + deformation energy - work of the loads and
    supports, from the end of step 1) at the last step."""
    r = run_gpu(cfg, G.PREC_FP64, warmup, steps, energy_every=1)
    h = r["hist"]
    E = h["e_def"] + h["e_kin_lumped"]
    W = h["w_ext"] + h["w_react"]
    B = (E - E[0]) - W
    scale = max(abs(W[-1]), abs(h["e_def"][-1] - h["e_def"][0]) + h["e_kin_lumped"][-1])
    ms = r["wall_s"] * 1e3 / steps
    ke = r["kt"]["element"]
    return {"ms_per_step": ms, "overhead_vs_plain": ms / plain_ms - 1.0,
            "element_avg_ms": ke[0] / max(ke[1], 1),
            "energy_pass_avg_ms": r["kt"]["energy"][0] / max(r["kt"]["energy"][1], 1),
            "balance_residual_rel": float(abs(B[-1]) / scale), "work_J": float(W[-1]),
            "e_def_J": float(h["e_def"][-1]), "e_kin_J": float(h["e_kin"][-1])}


def tet_leg(warmup, steps):
    """80^3 hex grid split into 6 tets each (3.07M tet4, 1 GP), 15% node perturbation, per-element E and nu:
    FP64 and FP32-element throughput over `steps` steps and their displacement difference."""
    cfg = configs.config(2)
    m = cfg["mesh"]
    r64 = run_gpu(cfg, G.PREC_FP64, warmup, steps)
    r32 = run_gpu(cfg, G.PREC_FP32_ELEM, warmup, steps)
    ne = m["n_elem"]
    n_part = r64["n_part"]
    e64 = r64["kt"]["element"][0] / max(r64["kt"]["element"][1], 1)
    n64 = r64["kt"]["node"][0] / max(r64["kt"]["node"][1], 1)
    return {"workload": f"{ne} tet4 (80^3 x 6), 15% perturbation, per-element E log-U[1e5,1e7], nu U[0.2,0.45], "
                        f"{warmup} + {steps} steps",
            "fp64_gp_per_s": ne * steps / r64["wall_s"], "fp64_ms_per_step": r64["wall_s"] * 1e3 / steps,
            "fp32_gp_per_s": ne * steps / r32["wall_s"], "fp32_ms_per_step": r32["wall_s"] * 1e3 / steps,
            "fp32_speedup": r64["wall_s"] / r32["wall_s"],
            "max_rel_disp_err_fp32_vs_fp64": float(np.abs(r32["u"] - r64["u"]).max() / np.abs(r64["u"]).max()),
            "fp64_element_avg_ms": e64, "fp64_node_avg_ms": n64,
            "fp32_element_avg_ms": r32["kt"]["element"][0] / max(r32["kt"]["element"][1], 1),
            "fp32_node_avg_ms": r32["kt"]["node"][0] / max(r32["kt"]["node"][1], 1), "partials": n_part,
            "step_algorithmic_bytes": step_bytes(ne, m["n_nodes"], 4, n_part, True)}


def cpu_baseline(cfg, budget_s=12.0):
    """Oracle (the CPU restatement of the reference loop) on the same mesh, all host threads (max 16)."""
    import oracle_ctypes as O
    m = cfg["mesh"]
    nt = max(1, min(16, os.cpu_count() or 1))

    def timed(nsteps, threads):
        p = O.OracleProblem(m, law=cfg["law"], E=cfg["E"], nu=cfg["nu"], rho=cfg["rho"], dir_dof=cfg["dir_dof"],
                            dir_val=cfg["dir_val"], bc_mode=O.BC_VELOCITY, vel_ramp_steps=100, scale=cfg["scale"],
                            n_steps=nsteps, sum_order=O.SUM_ELEMENT, n_threads=threads)
        t = time.perf_counter()
        r = p.run()
        assert r["rc"] == 0
        return time.perf_counter() - t

    out = {}
    for threads in (nt, 1):
        t_a = timed(1, threads)
        t_b = timed(3, threads)
        per = max((t_b - t_a) / 2, 1e-6)
        n = int(max(2, min(400, (budget_s if threads > 1 else budget_s / 2) / per)))
        t_c = timed(1 + n, threads)
        per = (t_c - t_a) / n
        gp = m["n_elem"] * (8 if m["nen"] == 8 else 1)
        out[threads] = dict(value=gp / per, steps=n, per_step_s=per)
    return nt, out


def plain_solve(c, precision):
    """One solve alone through the single-solve path with plain kernel launches (no graph replay)."""
    with G.Solver(c["mesh"], E=c["E"], nu=c["nu"], dir_dof=c["dir_dof"], dir_val=c["dir_val"],
                  n_steps=c["n_steps"], precision=precision) as s:
        s.set_graphs(False)
        t = time.perf_counter()
        rc, rep = s.run(c["n_steps"])
        dt = time.perf_counter() - t
        assert rc == 0 and rep["status"] == G.MPS_DONE, rep
        return dt, s.get_state()[0]


def batch_leg(precision, n_inst=512, steps=1000, plain_sample=48):
    """512 independent cubes n^3, n ~ U{6..40}, 1000 steps each, in one arena; hipGraph replay on the grid that the autotuner fixes,
    against the same solves launched one at a time with plain launches (random sample)."""
    sols = configs.batch_meshes(n_inst, steps=steps)
    gp = sum(c["mesh"]["n_elem"] * 8 for c in sols) * steps
    with G.Batch(arena_bytes=16 << 30, max_instances=n_inst, precision=precision, steps_per_launch=32) as b:
        t = time.perf_counter()
        slots = [b.add(c["mesh"], E=c["E"], nu=c["nu"], dir_dof=c["dir_dof"], dir_val=c["dir_val"],
                       n_steps=steps) for c in sols]
        b.sync()
        t_admit = time.perf_counter() - t
        bs, gm = b.autotune()
        t0 = time.perf_counter()
        b.step(steps)
        wall = time.perf_counter() - t0
        assert all(b.query(s_)["status"] == G.MPS_DONE for s_ in slots)
        rng = np.random.default_rng(3)
        pick = sorted(rng.choice(n_inst, plain_sample, replace=False))
        plain_t, err = 0.0, 0.0
        for i in pick:
            dt, u = plain_solve(sols[i], precision)
            plain_t += dt
            ub = b.get_state(slots[i])[0]
            assert np.array_equal(ub, u)  # same solve alone and in the batch: identical
            if precision == G.PREC_FP32_ELEM and i == pick[0]:
                _, u64 = plain_solve(sols[i], G.PREC_FP64)
                err = float(np.abs(u - u64).max() / np.abs(u64).max())
    return {"workload": f"{n_inst} clamped cubes n^3, n~U{{6..40}}, E log-U[1e5,1e7], nu U[0.2,0.45], "
                        f"{steps} steps each, hipGraph replay of {32}-step launches",
            "precision": "fp32-element" if precision == G.PREC_FP32_ELEM else "fp64",
            "elements": sum(c["mesh"]["n_elem"] for c in sols), "wall_s": wall, "solves_per_s": n_inst / wall,
            "elem_gp_updates_per_s": gp / wall, "autotuned": {"elem_block": bs, "grid_mult": gm},
            "admission_s": t_admit,
            "plain_one_at_a_time_solves_per_s": plain_sample / plain_t, "plain_sample": plain_sample,
            "speedup_vs_plain": (n_inst / wall) / (plain_sample / plain_t),
            "batch_equals_alone": True,
            **({"max_rel_disp_err_vs_fp64": err} if precision == G.PREC_FP32_ELEM else {})}


def serving_leg(lambdas, n_req=200, precision=G.PREC_FP32_ELEM, plain_sample=32, oracle_sample=4):
    """Poisson arrivals at rate lam of hex8 boxes (N_e log-U[1e3,2e5], aspect U[1,4], steps U{500..5000});
    requests are admitted by device footprint into the running batch (continuous batching).  Each rate serves
    n_req requests (its own draws); the `oracle_sample` cheapest requests of the last rate are checked against the
    FP64 oracle on the host."""
    import threading
    import oracle_ctypes as O
    points = []
    last = None
    with G.Server(arena_bytes=16 << 30, max_instances=1024, precision=precision, steps_per_launch=32) as srv:
        for li, lam in enumerate(lambdas):
            reqs = configs.serving_requests(n_req, seed=configs.SEED_CFG4 + li)
            srv.reset_stats()
            rng = np.random.default_rng(int(lam))
            ids = []

            def producer():
                for c in reqs:
                    ids.append(srv.submit(c["mesh"], E=c["E"], nu=c["nu"], dir_dof=c["dir_dof"],
                                          dir_val=c["dir_val"], n_steps=c["n_steps"]))
                    time.sleep(rng.exponential(1.0 / lam))
            th = threading.Thread(target=producer)
            th.start()
            th.join()
            assert srv.drain(600.0) == 0
            st = srv.stats()
            us = []
            for rid in ids:
                rc, u, _, _ = srv.result(rid)
                assert rc == 0
                us.append(u)
            points.append({"lambda_per_s": lam, "requests": n_req, "solves_per_s": st["solves_per_s"],
                           "p50_ms": st["p50_ms"], "p99_ms": st["p99_ms"], "max_ms": st["max_ms"],
                           "queue_p50_ms": st["queue_p50_ms"], "completed": st["completed"],
                           "elem_block": st["elem_block"], "grid_mult": st["grid_mult"],
                           "mixes": st["tunings"]})
            note(f"serving lambda={lam:g}/s: {st['solves_per_s']:.1f} solves/s, p50 {st['p50_ms']:.0f} ms, "
                 f"p99 {st['p99_ms']:.0f} ms, launch shape bs {st['elem_block']}, grid x{st['grid_mult']}")
            last = (reqs, us)
    # one-at-a-time plain launches of a sample of the same request distribution
    reqs, us = last
    rng = np.random.default_rng(5)
    pick = sorted(rng.choice(n_req, plain_sample, replace=False))
    plain_t = sum(plain_solve(reqs[i], precision)[0] for i in pick)
    plain_rate = plain_sample / plain_t
    for p_ in points:
        p_["speedup_vs_plain"] = p_["solves_per_s"] / plain_rate
    # served results against the FP64 oracle (the cheapest requests, so the host check stays short)
    cost = [r["mesh"]["n_elem"] * r["n_steps"] for r in reqs]
    worst = 0.0
    for i in np.argsort(cost)[:oracle_sample]:
        r = reqs[int(i)]
        o = O.OracleProblem(r["mesh"], E=r["E"], nu=r["nu"], dir_dof=r["dir_dof"], dir_val=r["dir_val"],
                            n_steps=r["n_steps"], sum_order=O.SUM_ELEMENT,
                            n_threads=max(1, min(16, os.cpu_count() or 1))).run()
        worst = max(worst, float(np.abs(us[int(i)] - o["u"]).max() / np.abs(o["u"]).max()))
    assert worst <= (1e-6 if precision == G.PREC_FP32_ELEM else 1e-12), worst
    return {"workload": f"{n_req} requests per rate: hex8 boxes N_e log-U[1e3,2e5], aspect U[1,4], "
                        "steps U{500..5000}, Poisson arrivals",
            "precision": "fp32-element" if precision == G.PREC_FP32_ELEM else "fp64",
            "points": points, "plain_one_at_a_time_solves_per_s": plain_rate, "plain_sample": plain_sample,
            "max_rel_disp_err_vs_fp64_oracle": worst, "oracle_checked_requests": oracle_sample}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-fp32", action="store_true")
    ap.add_argument("--no-energy", action="store_true", help="skip the energies-every-step leg")
    ap.add_argument("--no-batch", action="store_true", help="skip the batched (512 solves) leg")
    ap.add_argument("--no-serve", action="store_true", help="skip the serving (Poisson arrivals) leg")
    ap.add_argument("--no-tet", action="store_true", help="skip the 3.07M-tet4 leg")
    ap.add_argument("--lambdas", default="50,100,200,500,1000,2000")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only; --gpus {args.gpus} is not supported "
              "(independent solves shard trivially, a single mesh would need an interface-force exchange)",
              file=sys.stderr)
        sys.exit(2)

    cfg = configs.config(1)
    m = cfg["mesh"]
    ne, nn = m["n_elem"], m["n_nodes"]
    gp_per_step = ne * 8

    note(f"workload {ne} hex8 elements, {nn} nodes; copy probe")
    copy_gbs = G.bandwidth_probe(1 << 30, 20)
    note(f"copy ceiling {copy_gbs:.0f} GB/s; FP64 leg")
    r64 = run_gpu(cfg, G.PREC_FP64, args.warmup, args.steps)
    note(f"FP64 leg {r64['wall_s'] * 1e3 / args.steps:.4f} ms/step")
    value = gp_per_step * args.steps / r64["wall_s"]
    ems, en = r64["kt"]["element"]
    nms, nn_l = r64["kt"]["node"]
    elem_avg_ms = ems / max(en, 1)
    node_avg_ms = nms / max(nn_l, 1)
    n_part = r64["n_part"]
    eb = elem_kernel_bytes(ne, nn, 8, n_part, False)
    sb = step_bytes(ne, nn, 8, n_part, False)
    achieved = eb / (elem_avg_ms * 1e-3) / 1e9
    valu_wave = measured_valu_per_wave(ELEM_KERNEL)
    n_waves = -(-ne // PATCH) * (PATCH // 64)
    valu_peak = VALU_ISSUE_PEAK  # wave64 VALU instructions per second (one per CU per cycle)
    valu = None if valu_wave is None else {
        "achieved": valu_wave * n_waves / (elem_avg_ms * 1e-3), "peak": valu_peak, "unit": "wave-instr/s",
        "frac": valu_wave * n_waves / (elem_avg_ms * 1e-3) / valu_peak, "instr_per_wave": valu_wave}
    # the per-element-slot byte model of a two-kernel design that writes one force per (element, slot):
    # conn 4 nen + force write 3 nen 8 per element, X and u 48 per node
    slot_model_bytes = ne * (4 * 8 + 3 * 8 * 8) + nn * (3 * 8 + 24)
    out = {
        "metric": "elem-GP updates/s (1M hex8 NH explicit) + batched solves/s, p99 latency",
        "value": value,
        "unit": "elem-GP updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": r64["wall_s"] * 1e3 / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "100^3 hex8 cube, 10% seeded node perturbation, compressible neo-Hookean "
                               "E=1e6 nu=0.3 rho=1000, bottom clamped, top z-velocity ramp 0.1 m/s, "
                               "dt=0.5 x stable dt, FP64",
                   "n_elem": ne, "n_nodes": nn, "gauss_points": 8, "form": "fp64"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": measured_traffic(ELEM_KERNEL),
                     "traffic_source": os.path.relpath(TRAFFIC_TABLE, ROOT),
                     "kernel": f"{ELEM_KERNEL} (hex8 element forces + stable dt)",
                     "kernel_avg_ms": elem_avg_ms, "algorithmic_bytes_per_launch": eb,
                     "measured_copy_ceiling_gbs": copy_gbs,
                     "binding_resource": "valu" if valu is not None and valu["frac"] > achieved / HBM_PEAK_GBS
                     else "hbm",
                     "valu_check": valu,
                     "slot_model_bytes_per_launch": slot_model_bytes,
                     "slot_model_frac": slot_model_bytes / (elem_avg_ms * 1e-3) / 1e9 / HBM_PEAK_GBS},
        "kernels": {"element_avg_ms": elem_avg_ms, "node_avg_ms": node_avg_ms, "partials": n_part,
                    "timing": "kernel averages from HIP events around every launch over a second region of "
                              f"{args.steps} steps launched one by one ({r64['events_ms_per_step']:.4f} ms/step); "
                              "value and ms_per_step from the graph-replayed timed region",
                    "node_algorithmic_bytes": node_kernel_bytes(nn, n_part),
                    "node_achieved_gbs": node_kernel_bytes(nn, n_part) / (node_avg_ms * 1e-3) / 1e9,
                    "step_algorithmic_bytes": sb,
                    "step_hbm_frac": sb / (r64["wall_s"] / args.steps) / 1e9 / HBM_PEAK_GBS},
    }
    if not args.no_fp32:
        note("FP32-element leg")
        r32 = run_gpu(cfg, G.PREC_FP32_ELEM, args.warmup, args.steps)
        v32 = gp_per_step * args.steps / r32["wall_s"]
        err = float(np.abs(r32["u"] - r64["u"]).max() / np.abs(r64["u"]).max())
        e32, n32 = r32["kt"]["element"]
        out["fp32_elem"] = {"value": v32, "ms_per_step": r32["wall_s"] * 1e3 / args.steps,
                            "speedup_vs_fp64": v32 / value, "max_rel_disp_err_vs_fp64": err,
                            "element_avg_ms": e32 / max(n32, 1),
                            "node_avg_ms": r32["kt"]["node"][0] / max(r32["kt"]["node"][1], 1)}
    if not args.no_energy:
        note("FP64 leg with energies every step")
        out["energies_every_step"] = energy_leg(cfg, args.warmup, args.steps, r64["wall_s"] * 1e3 / args.steps)
        note(f"energies every step {out['energies_every_step']['ms_per_step']:.4f} ms/step "
             f"(+{100 * out['energies_every_step']['overhead_vs_plain']:.1f}%)")
    if not args.no_tet:
        note("tet4 leg (80^3 x 6 tets, per-element materials)")
        out["tet4"] = tet_leg(args.warmup, 500)
        note(f"tet4 FP64 {out['tet4']['fp64_ms_per_step']:.4f} ms/step, FP32 {out['tet4']['fp32_ms_per_step']:.4f}")
    if not args.no_batch:
        note("batched leg (512 solves)")
        out["batched"] = batch_leg(G.PREC_FP32_ELEM)
        note(f"batched {out['batched'].get('solves_per_s', 0):.1f} solves/s")
    if not args.no_serve:
        note("serving leg")
        out["serving"] = serving_leg([float(x) for x in args.lambdas.split(",")])
    if not args.no_cpu:
        note("CPU baseline (oracle, bounded sample)")
        nt, cb = cpu_baseline(cfg)
        out["cpu_baseline"] = {"value": cb[nt]["value"], "unit": "elem-GP updates/s", "cores": nt, "kind": "port",
                               "sample": f"same 1M-hex8 workload, {cb[nt]['steps']} steps after a 1-step set-up "
                                         f"run (set-up excluded), oracle element-order, {nt} threads"}
        out["cpu_baseline_seq"] = {"value": cb[1]["value"], "cores": 1, "steps": cb[1]["steps"]}
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
