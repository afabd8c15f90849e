"""Benchmark: converged SCFT solves per second on one MI355X.

Workload (one "step" = one converged solve): AB diblock double gyroid
(Ia-3d), N=100, blocks 36/64, chi N=20, b=1, ds=0.5 (200 contour steps),
cubic cell starting at a=16, 64^3 grid, seeded initial field (first 20 stars
~ N(0, 0.1) per monomer, seed 20261201), Anderson mixing (N_hist=20) with
unit-cell relaxation through scf_stress to residual 1e-9 -- the reference's
ITERATE/iterate_AM path on the GPU hot path.

Prints one JSON line with the headline value, the roofline of the fused
contour step (HIP-event timing of its kernels inside the timed region) and
the reference Fortran+MKL-FFTW program timed on the host (cpu_baseline).

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]
"""
import argparse
import json
import os
import re
import shutil
import subprocess
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
# HBM bytes per launch of each step kernel at the gyroid 64^3 workload (both
# sweeps), measured with rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE on
# `bench.py --traffic-probe`, each scaled by the same counter on a 256 MiB
# device copy (reads 2.0 x FETCH_SIZE, writes 1.0 x WRITE_SIZE):
# profiles/k_step_gyroid64_hbm_traffic.md
TRAFFIC = {"step_a": 28.93e6, "step_z0": 21.74e6, "step_c": 21.03e6, "step_z1": 10.93e6}
TRAFFIC_SOURCE = ("constant: rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE of `bench.py --traffic-probe`, "
                  "scaled by a 256 MiB copy (profiles/k_step_gyroid64_hbm_traffic.md); not "
                  "measured in this run")
WORKLOAD = "gyroid_Ia-3d_64^3_N100_f0.36_chiN20_ds0.5_a16_AM_domain"
# the gyroid at its equilibrium period: the same chemistry, started from the
# principal (211) star at a = 36, cell relaxed (the reference program
# converges this start to a = 38.89; tests/golden/conv_gyr64.npz)
PERIOD_WORKLOAD = "gyroid_Ia-3d_64^3_N100_f0.36_chiN20_ds0.5_a36_principal211_AM_domain"


def load_workload():
    d = np.load(os.path.join(ROOT, "tests", "golden", "gyr64.npz"))
    return {k: d[k] for k in d.files}


def gyroid_system():
    from pscf_amd.system import diblock
    return diblock(0.36, 100.0, 20.0, dim=3, crystal_system="cubic", cell_param=[16.0],
                   ngrid=[64, 64, 64], chain_step=0.5, group_name="I a -3 d")


def kernel_bytes(Ms, Mk):
    """Algorithmic HBM bytes per launch of each contour-step kernel for ONE
    sweep (every array the kernel must read or write, once), with Ms stored
    points of a real field (all N1 N2 N3, or those of the symmetric planes) and
    Mk half-grid points: FP64 real fields 8 B/point, packed spectra 8 B per
    stored point, factors e1, e2 (Ms) and k1, k2 (Mk):
      step_a : spectrum C in, q1, e2, e1 in, q out, A, B out
      step_z0: A, B in and out, k1, k2 in
      step_c : A, B in, e1 in, q1 out, C out
      step_z1: C in and out, k2 in"""
    return {"step_a": 56.0 * Ms, "step_z0": 32.0 * Ms + 16.0 * Mk,
            "step_c": 40.0 * Ms, "step_z1": 16.0 * Ms + 8.0 * Mk}


def cpu_baseline(g, n_gpu_iter, workdir):
    """The reference program (oracle/_ref/pscf, flang -O2 + MKL's FFTW3 API,
    one core) on the same workload, bounded to its first Anderson iterations.
    Reports its per-iteration cost scaled by the GPU solve's iteration count."""
    ref = os.path.join(ROOT, "oracle", "_ref", "pscf")
    if not os.path.exists(ref):
        return None
    from pscf_amd import fieldio, scf
    sysm = gyroid_system()
    B = scf.Basis.from_tables(g)
    fieldio.write_field(os.path.join(workdir, "in.omega"), g["omega"], sysm, B, g["star_count"])
    max_itr = 1
    param = sysm.to_param() + (
        "ITERATE\ninput_filename\n'in.omega'\noutput_prefix\n'out/'\nmax_itr\n%d\n"
        "error_max\n1.0E-09\ndomain\nT\nitr_algo\n'AM'\nN_hist\n20\n\nFINISH\n" % max_itr)
    with open(os.path.join(workdir, "param"), "w") as f:
        f.write(param)
    os.makedirs(os.path.join(workdir, "out"), exist_ok=True)
    env = dict(os.environ, MKL_NUM_THREADS="1", OMP_NUM_THREADS="1")
    t0 = time.perf_counter()
    with open(os.path.join(workdir, "param")) as fin:
        r = subprocess.run(["bash", "-c", "ulimit -s unlimited; %s" % ref], stdin=fin,
                           cwd=workdir, env=env, capture_output=True, text=True, timeout=600)
    wall = time.perf_counter() - t0
    if r.returncode != 0:
        return {"error": "reference run failed: " + r.stderr[-300:]}
    out = open(os.path.join(workdir, "out", "out")).read()
    scf_time = float(re.search(r"^scf_time\s*\n\s*(\S+)", out, re.M).group(1))
    itr = int(re.search(r"^iterations\s*\n\s*(\S+)", out, re.M).group(1))
    # scf_time covers the initial density() plus `itr` iterations of
    # density() + scf_stress(): per-iteration cost ~ scf_time / (itr + 1)
    t_iter = scf_time / (itr + 1)
    return {"value": 1.0 / (t_iter * n_gpu_iter), "unit": "solves/s", "cores": 1,
            "kind": "reference", **host_cpu(),
            "sample": "reference pscf (flang -O2, MKL FFTW3 API, MKL_NUM_THREADS=1), same "
                      "workload, ITERATE AM max_itr=%d: scf_time %.2f s for %d iterations -> "
                      "%.3f s/iteration x %d GPU iterations per solve (wall %.1f s incl. "
                      "make_basis)" % (max_itr, scf_time, itr, t_iter, n_gpu_iter, wall)}


def host_cpu():
    """Model name of the host CPU and the cores this process may use."""
    model = None
    try:
        for ln in open("/proc/cpuinfo"):
            if ln.startswith("model name"):
                model = ln.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return {"cpu_model": model, "nproc": len(os.sched_getaffinity(0))}


def gyroid_at_period_leg(L, g, B, steps, error_max=1e-9):
    """Converged solves/s of the double gyroid that the workload's chemistry
    forms at its equilibrium period: start from the principal star at a = 36,
    Anderson mixing with cell relaxation to residual 1e-9 (1 warm-up solve,
    then `steps` timed).  Checks that the state is ordered (f below the
    Flory-Huggins value) and reports it against the reference program's
    converged state of the same start (tests/golden/conv_gyr64.npz)."""
    import torch
    from pscf_amd import iterate, scf
    from pscf_amd.system import diblock
    sysm = diblock(0.36, 100.0, 20.0, dim=3, crystal_system="cubic", cell_param=[36.0],
                   ngrid=[64, 64, 64], chain_step=0.5, group_name="I a -3 d")
    _, G0, _ = iterate.unit_cell(L, 3, "cubic", [36.0])
    S = scf.SCFSystem(sysm, B, G0, lib=L)
    am = iterate.AndersonMixing(S, n_hist=20, domain=True)
    om0 = np.zeros_like(g["omega"])
    om0[:, 0] = g["omega"][:, 0]
    om0[0, 1], om0[1, 1] = 0.05, -0.05

    def solve():
        S.set_cell(G0)
        return am.run(om0, error_max=error_max, max_itr=2000)

    solve()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    res = [solve() for _ in range(steps)]
    torch.cuda.synchronize()
    el = time.perf_counter() - t0
    r = res[-1]
    f_fh = S.free_energy_FH()
    line = {"metric": "converged SCFT solves/s, gyroid 64^3 at its equilibrium period",
            "value": steps / el, "unit": "solves/s", "workload": PERIOD_WORKLOAD,
            "iterations_per_solve": [x.itr for x in res], "converged": [x.converge for x in res],
            "final_cell_a": float(r.cell_param[0]), "f_helmholtz": r.f_helmholtz,
            "f_flory_huggins": f_fh, "ordered": bool(r.f_helmholtz < f_fh - 1e-3),
            "ms_per_iteration": el / sum(x.itr for x in res) * 1e3}
    ref = os.path.join(ROOT, "tests", "golden", "conv_gyr64.npz")
    if os.path.exists(ref):
        d = np.load(ref)
        line["reference_f_helmholtz"] = float(d["f_helmholtz"])
        line["reference_cell_a"] = float(d["cell_param"][0])
        line["rel_diff_f_vs_reference"] = abs(r.f_helmholtz / float(d["f_helmholtz"]) - 1.0)
    return {"line": line, "omega": r.omega, "cell_a": float(r.cell_param[0]),
            "seconds_per_solve": el / steps}


def batch_cpu_baseline(batch_res, max_cores=16):
    """All-cores estimate for the batched leg: one reference process
    (oracle/_ref/pscf, one thread each) per phase, run concurrently, each
    timing its first Anderson iteration (scf_time of ITERATE with max_itr 1:
    the initial density() and one iteration); the batch's instances then cost
    their phase's time per iteration times the iterations the GPU solve took,
    spread over the host's cores (at most 16, the share of one GPU)."""
    ref = os.path.join(ROOT, "oracle", "_ref", "pscf")
    if not os.path.exists(ref):
        return None
    from pscf_amd import fieldio, scf
    insts = batch_instances(batch_res["instances"])
    first = {}
    for i, (ph, sysm, g, om) in enumerate(insts):
        first.setdefault(ph, i)
    procs = {}
    tmp = tempfile.mkdtemp(prefix="pscf_cpu_batch_")
    env = dict(os.environ, MKL_NUM_THREADS="1", OMP_NUM_THREADS="1")
    t0 = time.perf_counter()
    try:
        for ph, i in first.items():
            _, sysm, g, om = insts[i]
            wd = os.path.join(tmp, ph)
            os.makedirs(os.path.join(wd, "out"))
            fieldio.write_field(os.path.join(wd, "in.omega"), om, sysm, scf.Basis.from_tables(g),
                                g["star_count"])
            with open(os.path.join(wd, "param"), "w") as f:
                f.write(sysm.to_param() + "ITERATE\ninput_filename\n'in.omega'\noutput_prefix\n"
                        "'out/'\nmax_itr\n1\nerror_max\n1.0E-08\ndomain\nF\nitr_algo\n'AM'\n"
                        "N_hist\n20\n\nFINISH\n")
            fin = open(os.path.join(wd, "param"))
            procs[ph] = (subprocess.Popen(["bash", "-c", "ulimit -s unlimited; %s" % ref], stdin=fin,
                                          cwd=wd, env=env, stdout=subprocess.DEVNULL,
                                          stderr=subprocess.DEVNULL), fin, wd)
        t_iter = {}
        for ph, (p, fin, wd) in procs.items():
            p.wait(timeout=600)
            fin.close()
            out = open(os.path.join(wd, "out", "out")).read()
            scf_time = float(re.search(r"^scf_time\s*\n\s*(\S+)", out, re.M).group(1))
            itr = int(re.search(r"^iterations\s*\n\s*(\S+)", out, re.M).group(1))
            t_iter[ph] = scf_time / (itr + 1)
        wall = time.perf_counter() - t0
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    hc = host_cpu()
    cores = max(1, min(max_cores, hc["nproc"]))
    work = sum(t_iter[ph] * it for (ph, *_), it in zip(insts, batch_res["iterations"]))
    conv = batch_res["converged"]
    return {"value": conv / (work / cores), "unit": "solves/s", "cores": cores, "kind": "reference",
            "seconds_per_iteration": t_iter, "cpu_model": hc["cpu_model"], "nproc": hc["nproc"],
            "sample": "estimate: reference pscf (flang -O2, MKL FFTW3 API, 1 thread per process), "
                      "one process per phase run concurrently for one Anderson iteration (wall "
                      "%.1f s incl. make_basis); each of the %d instances costs its phase's "
                      "s/iteration x the iterations of its GPU solve, %d converged instances over "
                      "%d cores" % (wall, len(insts), conv, cores)}


# ---------------------------------------------------------------- batched leg
# 64 AB diblock melts (N=100, ds=1) with chi N ~ U[12, 30], f_A ~ U[0.2, 0.5]
# and a phase drawn per instance: lamellae in a tetragonal cell on 32^3,
# hexagonal cylinders (3D cell) on 48^3, BCC or gyroid on 64^3.  Each runs
# its own Anderson history (fixed cell) to residual 1e-8.  Starting field:
# the phase's principal star (lamellae: (001), cylinders: (100), BCC: (110),
# gyroid: (211)) at amplitude +-chi/4 in omega_A/omega_B, and the other
# stars 2..10 seeded N(0, chi/20).
BATCH_PHASES = {   # tables, crystal system, cell, grid, group, principal star
    "lam": ("lam_tet32", "tetragonal", [16.0, 16.0], [32, 32, 32], "P 4/m m m", 2),
    "hex": ("hex48", "hexagonal", [19.0, 19.0], [48, 48, 48], "P 6/m m m", 2),
    "bcc": ("bcc64", "cubic", [18.0], [64, 64, 64], "I m -3 m", 1),
    "gyr": ("gyr64", "cubic", [36.0], [64, 64, 64], "I a -3 d", 1),
}
BATCH_SEED = 20261203


def batch_instances(n=64, seed=BATCH_SEED):
    from pscf_amd.system import diblock
    rng = np.random.default_rng(seed)
    tables = {}
    out = []
    for _ in range(n):
        ph = ["lam", "hex", "bcc", "gyr"][int(rng.integers(4))]
        chiN = float(rng.uniform(12.0, 30.0))
        fA = float(rng.uniform(0.2, 0.5))
        tname, cs, cell, grid, group, principal = BATCH_PHASES[ph]
        if tname not in tables:
            d = np.load(os.path.join(ROOT, "tests", "golden", tname + ".npz"))
            tables[tname] = {k: d[k] for k in d.files}
        g = tables[tname]
        sysm = diblock(fA, 100.0, chiN, dim=3, crystal_system=cs, cell_param=cell, ngrid=grid,
                       chain_step=1.0, group_name=group)
        nstar = len(g["star_count"])
        chi = chiN / 100.0
        om = np.zeros((2, nstar))
        om[:, 1:10] = rng.normal(0.0, 0.05 * chi, size=(2, 9))
        om[0, principal] = 0.25 * chi
        om[1, principal] = -0.25 * chi
        out.append((ph, sysm, g, om))
    return out


def batch_leg(L, n_inst=64, n_loop=16, error_max=1e-8, max_itr=300):
    """Converged solves/s of the batched solver over all instances, and of a
    per-instance loop (the plain single-system path) over every (n_inst /
    n_loop)-th instance."""
    import torch
    from pscf_amd import batch, iterate
    insts = batch_instances(n_inst)
    B = batch.BatchSolver(n_hist=20, domain=False, error_max=error_max, max_itr=max_itr, lib=L)
    for ph, sysm, g, om in insts:
        B.add(batch.make_system(sysm, g, lib=L), om)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    B.solve()
    torch.cuda.synchronize()
    t_batch = time.perf_counter() - t0
    res = [B.result(i) for i in range(n_inst)]
    del B
    conv_b = sum(r.converge for r in res)
    stride = max(1, n_inst // n_loop)
    sub = list(range(0, n_inst, stride))[:n_loop]
    t_loop = 0.0
    conv_l = 0
    same = 0
    for i in sub:
        ph, sysm, g, om = insts[i]
        S = batch.make_system(sysm, g, lib=L)
        am = iterate.AndersonMixing(S, n_hist=20, domain=False)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        r = am.run(om, error_max=error_max, max_itr=max_itr)
        torch.cuda.synchronize()
        t_loop += time.perf_counter() - t0
        conv_l += r.converge
        same += (r.itr == res[i].itr and r.converge == res[i].converge)
        del am, S
    phases = {}
    for ph, *_ in insts:
        phases[ph] = phases.get(ph, 0) + 1
    v_b = conv_b / t_batch
    v_l = conv_l / t_loop if t_loop > 0 else None
    return {"metric": "batched converged SCFT solves/s", "value": v_b, "unit": "solves/s",
            "instances": n_inst, "converged": conv_b, "phases": phases,
            "seconds": t_batch, "iterations": [r.itr for r in res],
            "loop_value": v_l, "loop_instances": len(sub), "loop_converged": conv_l,
            "loop_seconds": t_loop, "speedup_vs_loop": (v_b / v_l) if v_l else None,
            "loop_matches_batch": same,
            "workload": "64 AB diblocks N=100 ds=1, chiN~U[12,30], fA~U[0.2,0.5], "
                        "phases lam(32^3)/hex(48^3)/bcc,gyr(64^3) from their principal star, "
                        "AM n_hist=20, fixed cell, residual 1e-8, max_itr 300, seed %d" % BATCH_SEED}


# --------------------------------------------------------------- adjoint leg
def adjoint_leg(L, g, omega, cell_a, t_solve, reps=3):
    """Cost of the reverse-mode gradient of L = sum_r (phi_A(r) - phi_t(r))^2
    (phi_t: first 20 gyroid stars, amplitude 0.1 around 0.36, seed 2026) with
    respect to omega(r), the cell a and f_A at the converged gyroid."""
    import torch
    from pscf_amd import adjoint, batch
    sysm = gyroid_system()
    sysm.cell_param = [float(cell_a)]
    S = batch.make_system(sysm, g, lib=L)
    dev = "cuda"
    rng = np.random.default_rng(2026)
    tst = np.zeros((1, S.N_star))
    tst[0, 0] = 0.36
    tst[0, 1:20] = rng.normal(size=19)
    tst[0, 1:20] *= 0.1 / np.abs(tst[0, 1:20]).max()
    phi_t = adjoint.stars_to_grid(S, torch.tensor(tst, device=dev))[0].detach()
    omg = adjoint.stars_to_grid(S, torch.tensor(omega, device=dev)).detach()
    fwd, bwd = [], []
    for _ in range(reps + 1):
        om = omg.clone().requires_grad_(True)
        cp = torch.tensor([float(cell_a)], dtype=torch.float64, requires_grad=True)
        fA = torch.tensor(0.36, dtype=torch.float64, requires_grad=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        rho, Q = adjoint.density(S, om, cp, torch.stack([fA * 100.0, (1.0 - fA) * 100.0]))
        loss = ((rho[0] - phi_t) ** 2).sum()
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        loss.backward()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        fwd.append(t1 - t0)
        bwd.append(t2 - t1)
    f_ms = float(np.median(fwd[1:])) * 1e3
    b_ms = float(np.median(bwd[1:])) * 1e3
    return {"metric": "adjoint gradient cost", "forward_density_ms": f_ms, "backward_ms": b_ms,
            "gradient_over_density": (f_ms + b_ms) / f_ms,
            "gradient_over_solve": (f_ms + b_ms) * 1e-3 / t_solve,
            "wrt": ["omega(r)", "cell a", "f_A"],
            "loss": "sum_r (phi_A - phi_t)^2, gyroid 64^3 at the converged state"}


def jacobian_leg(L, cuts=(17, 33), reps=3):
    """Newton-Raphson Jacobian of the BCC 32^3 melt (N=100, f=0.25, chi N=20,
    a=18): the N_cut * N_monomer perturbed density() calls of
    response_pd_omega (src/response_pd_mod.f90:114-124, increment 1e-8), one
    by one as the reference makes them and grouped through density_many
    (one launch set), each at the seeded star field; the results must agree
    bit for bit."""
    from pscf_amd import scf
    from pscf_amd.system import diblock
    from pscf_amd import iterate
    d = np.load(os.path.join(ROOT, "tests", "golden", "bcc32.npz"))
    g = {k: d[k] for k in d.files}
    sysm = diblock(0.25, 100.0, 20.0, dim=3, crystal_system="cubic", cell_param=[18.0],
                   ngrid=[32, 32, 32], chain_step=1.0, group_name="I m -3 m")
    _, G, _ = iterate.unit_cell(L, 3, "cubic", [18.0])
    S = scf.SCFSystem(sysm, scf.Basis.from_tables(g), G, lib=L)
    om = np.asarray(g["omega"], dtype=np.float64)
    out = []
    for cut in cuts:
        fields = []
        for j in range(1, cut):
            for beta in range(2):
                w = om.copy()
                w[beta, j] += 1.0e-8
                fields.append(w)
        fields = np.array(fields)
        t_one, t_many = [], []
        for r in range(reps + 1):
            t0 = time.perf_counter()
            one = [S.density(w, with_q=False)[0] for w in fields]
            t1 = time.perf_counter()
            many = S.density_many(fields, with_q=False)[0]
            t2 = time.perf_counter()
            t_one.append(t1 - t0)
            t_many.append(t2 - t1)
        same = all(np.array_equal(a, b) for a, b in zip(one, many))
        a_ms = float(np.median(t_one[1:])) * 1e3
        b_ms = float(np.median(t_many[1:])) * 1e3
        out.append({"n_cut": cut, "density_calls": len(fields), "serial_ms": a_ms,
                    "grouped_ms": b_ms, "speedup": a_ms / b_ms, "bitwise_equal": bool(same)})
    return {"metric": "Newton-Raphson Jacobian (perturbed density() calls)",
            "workload": "BCC 32^3 AB diblock, N=100, f=0.25, chi N=20, ds=1", "cases": out}


def design_leg(L, n_inst=32, seed=20261204):
    """Batching plus differentiation: ABA triblock (N=100, blocks 20/60/20)
    + A homopolymer (length 50, phi_h ~ U[0.05, 0.2]), chi N ~ U[15, 25],
    ds = 0.5, contour slabs checkpointed every 14 steps.
    (1) Gradient cost on 96^3 grids: the gradient of sum_r (phi_A - t)^2 in
        omega(r), f_A and phi_h for n_inst instances on seeded fields, one
        backward pass per instance against one grouped backward
        (adjoint.Group).
    (2) The descent of pscf_amd.design toward seeded target periods
        d_t ~ U[12.5, 15.5] for the same instances as lamellae (1D cells, 96
        points): |sigma(d_t)| per iteration."""
    import torch
    from pscf_amd import adjoint, design, scf
    from pscf_amd.system import System
    rng = np.random.default_rng(seed)
    blends = [design.Blend(f_A=0.4, phi_h=float(rng.uniform(0.05, 0.2)),
                           chi_N=float(rng.uniform(15.0, 25.0))) for _ in range(n_inst)]
    n = 96
    basis = scf.Basis(np.zeros((1, 3)), np.ones(1), np.ones(1), np.zeros(1), np.zeros((1, 3)))
    G0 = np.eye(3) * (2.0 * np.pi / 24.0)
    systems = []
    for b in blends:
        s = b.system(24.0, n, 0.5)
        s = System(kuhn=s.kuhn, chains=s.chains, phi_chain=s.phi_chain, chi=s.chi, dim=3,
                   crystal_system="cubic", cell_param=[24.0], ngrid=[n, n, n], chain_step=0.5,
                   group_name="P 1")
        S = scf.SCFSystem(s, basis, G0, lib=L)
        S.set_checkpoint(14)
        systems.append(S)
    oms = [torch.tensor(0.1 * rng.standard_normal((2, n, n, n)), device="cuda") for _ in blends]
    tgt = torch.tensor(0.5 + 0.1 * rng.standard_normal((n, n, n)), device="cuda")

    def leaves(b):
        fA = torch.tensor(b.f_A, dtype=torch.float64, requires_grad=True)
        ph = torch.tensor(b.phi_h, dtype=torch.float64, requires_grad=True)
        Lb = torch.stack([50.0 * fA, 100.0 * (1.0 - fA), 50.0 * fA,
                          torch.tensor(50.0, dtype=torch.float64)])
        return fA, ph, Lb, torch.stack([1.0 - ph, ph])

    cp = torch.tensor([24.0], dtype=torch.float64)
    torch.cuda.synchronize()
    t_fwd = t_bwd = 0.0
    loop_grads = []
    for i, (b, S) in enumerate(zip(blends, systems)):
        fA, ph, Lb, phis = leaves(b)
        om = oms[i].clone().requires_grad_(True)
        t0 = time.perf_counter()
        rho, Q = adjoint.density(S, om, cp, Lb, phis)
        loss = ((rho[0] - tgt) ** 2).sum()
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        loss.backward()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        t_fwd += t1 - t0
        t_bwd += t2 - t1
        loop_grads.append((fA.grad.item(), ph.grad.item()))
    G = adjoint.Group(systems)
    res = {}
    for rep in range(2):       # the first grouped pass builds and captures the launch set
        lv = [leaves(b) for b in blends]
        om = [o.clone().requires_grad_(True) for o in oms]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        outs = G.density(om, [cp] * n_inst, [x[2] for x in lv], [x[3] for x in lv])
        loss = sum(((rho[0] - tgt) ** 2).sum() for rho, _ in outs)
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        loss.backward()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        res = {"forward_s": t1 - t0, "backward_s": t2 - t1}
        same = all(lv[i][0].grad.item() == loop_grads[i][0] and lv[i][1].grad.item() == loop_grads[i][1]
                   for i in range(n_inst))
    del G, outs, loss, om
    systems.clear()
    torch.cuda.empty_cache()
    grad_cost = {"instances": n_inst, "grid": [n, n, n], "checkpoint_stride": 14,
                 "forward_s_total": t_fwd, "backward_s_loop": t_bwd,
                 "backward_s_grouped": res["backward_s"],
                 "grouped_speedup": t_bwd / res["backward_s"],
                 "backward_over_forward_grouped": res["backward_s"] / t_fwd,
                 "grouped_equals_loop": bool(same)}
    # (2) descent toward target periods, lamellae on 96 points
    tables = design.lamellar_tables(n)
    target = [float(x) for x in rng.uniform(12.5, 15.5, n_inst)]
    om0 = np.zeros((2, n // 2 + 1))
    t0 = time.perf_counter()
    starts = []
    for b in blends:
        o = om0.copy()
        o[0, 1] = 0.25 * b.chi_N / 100.0 * 4.0
        o[1, 1] = -o[0, 1]
        starts.append((o, o))
    _, hist = design.fit_spacing(blends, target, starts, tables, n, 0.5, iters=4, lib=L)
    t_design = time.perf_counter() - t0
    sig = [float(np.abs(h["sigma"]).max()) for h in hist]
    return {"metric": "batched adjoint gradients with checkpointing (ABA + A blends)",
            "gradient_cost_96cubed": grad_cost,
            "descent": {"instances": n_inst, "grid": [n], "iterations": len(hist) - 1,
                        "max_abs_sigma_per_iteration": sig, "wall_s": t_design,
                        "final_f_A_range": [float(hist[-1]["f_A"].min()), float(hist[-1]["f_A"].max())],
                        "final_phi_h_range": [float(hist[-1]["phi_h"].min()),
                                              float(hist[-1]["phi_h"].max())]}}


def traffic_probe():
    import torch
    from pscf_amd import iterate, scf
    from pscf_amd._lib import lib
    L = lib()
    g = load_workload()
    sysm = gyroid_system()
    _, G0, _ = iterate.unit_cell(L, 3, "cubic", [16.0])
    S = scf.SCFSystem(sysm, scf.Basis.from_tables(g), G0, lib=L)
    S.use_graph(False)
    for _ in range(2):
        S.density(g["omega"])
    x = torch.ones(32 * 1024 * 1024, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    for _ in range(3):
        y.copy_(x)
    torch.cuda.synchronize()
    print("traffic probe done", flush=True)


def task_scaling(L, counts=(1, 2, 4, 8, 16)):
    """Contour-step cost versus sweeps per launch: one BCC 64^3 system whose
    chemistry holds n identical AB diblock species (N=100, f=0.25, ds=1), so
    every launch carries 2n sweeps.  Prints per-chain step and kernel times."""
    import torch
    from pscf_amd import iterate, scf
    from pscf_amd.system import System
    d = np.load(os.path.join(ROOT, "tests", "golden", "bcc64.npz"))
    g = {k: d[k] for k in d.files}
    B = scf.Basis.from_tables(g)
    _, G, _ = iterate.unit_cell(L, 3, "cubic", [18.0])
    out = []
    for n in counts:
        chi = 0.2
        s = System(kuhn=[1.0, 1.0], chains=[[(1, 25.0), (2, 75.0)]] * n, phi_chain=[1.0 / n] * n,
                   chi=np.array([[0, chi], [chi, 0]]), dim=3, crystal_system="cubic",
                   cell_param=[18.0], ngrid=[64, 64, 64], chain_step=1.0, group_name="I m -3 m")
        S = scf.SCFSystem(s, B, G, lib=L)
        S.density(g["omega"])
        S.profile_sweeps(1)
        for _ in range(3):
            S.density(g["omega"])
        ms, cnt = S.profile_sweeps(0)
        step = float(ms[4]) / max(int(cnt[4]), 1) * 1e3
        ks = []
        for kind in range(4):
            S.density(g["omega"])
            ks.append(S.profile_step_kernel(kind, 50, reps=50))
        torch.cuda.synchronize()
        row = {"chains": n, "sweeps_per_launch": 2 * n, "step_us": step, "step_us_per_chain": step / n,
               "kernel_us_per_chain": dict(zip(["step_a", "step_z0", "step_c", "step_z1"],
                                               [k / n for k in ks]))}
        print(json.dumps(row), flush=True)
        out.append(row)
        del S
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-batch", action="store_true", help="skip the batched-solves leg")
    ap.add_argument("--no-adjoint", action="store_true", help="skip the gradient-cost leg")
    ap.add_argument("--no-jacobian", action="store_true", help="skip the Newton Jacobian leg")
    ap.add_argument("--no-design", action="store_true",
                    help="skip the batched-gradient / inverse-design leg")
    ap.add_argument("--task-scaling", action="store_true",
                    help="only print contour-step cost versus sweeps per launch (BCC 64^3)")
    ap.add_argument("--traffic-probe", action="store_true",
                    help="only run two eagerly launched density() calls of the workload and a "
                         "256 MiB device copy (the HBM counter runs under rocprofv3 --pmc)")
    args = ap.parse_args()
    if args.traffic_probe:
        traffic_probe()
        return
    if args.task_scaling:
        from pscf_amd._lib import lib as _lib
        task_scaling(_lib())
        return
    if args.gpus != 1:
        print("bench.py measures one GPU: the library has no multi-GPU path "
              "(independent solves would shard across GPUs without communication)")
        sys.exit(2)

    import torch
    from pscf_amd import iterate, scf
    from pscf_amd._lib import lib

    assert torch.cuda.is_available(), "bench.py needs a HIP device"
    L = lib()
    g = load_workload()
    sysm = gyroid_system()
    B = scf.Basis.from_tables(g)
    _, G0, _ = iterate.unit_cell(L, 3, "cubic", [16.0])
    S = scf.SCFSystem(sysm, B, G0, lib=L)
    am = iterate.AndersonMixing(S, n_hist=20, domain=True)

    def solve():
        S.set_cell(G0)
        return am.run(g["omega"], error_max=1e-9, max_itr=2000)

    for _ in range(args.warmup):
        r = solve()
    torch.cuda.synchronize()
    S.profile_sweeps(1)            # HIP events around every captured sweep
    t0 = time.perf_counter()
    results = [solve() for _ in range(args.steps)]
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms, n = S.profile_sweeps(0)
    r = results[-1]
    iters = [x.itr for x in results]
    f_fh = S.free_energy_FH()

    M = 64 * 64 * 17               # stored points: Ia-3d's sweeps keep 17 of 64 planes
    Mk = 33 * 64 * 64
    # whole captured sweeps (slot 4): milliseconds and contour steps advanced
    steps_timed = int(n[4])
    t_step_ms = float(ms[4]) / max(steps_timed, 1)
    # per-kernel durations in place: density() at the converged field with
    # every kernel launched once per contour step (the sweep's own order, on
    # the stream the sweeps use), its start and end recorded as HIP events by
    # its own dispatch (execution time, no launch gaps)
    names = ["step_a", "step_z0", "step_c", "step_z1"]
    S.profile_sweeps(2)
    for _ in range(5):
        S.density(r.omega)
    torch.cuda.synchronize()
    kms, kn = S.profile_sweeps(0)
    kavg_us = {nm: float(kms[i]) / max(int(kn[i]), 1) * 1e3 for i, nm in enumerate(names)}
    kb = {nm: 2 * v for nm, v in kernel_bytes(M, Mk).items()}   # qf and qr sweeps per launch
    dom = max(names, key=kavg_us.get)           # each kernel runs once per contour step
    achieved = kb[dom] / (kavg_us[dom] * 1e-6) / 1e9
    bytes_step = sum(kb.values())

    gyr = gyroid_at_period_leg(L, g, B, steps=args.steps)

    extra = {"gyroid_at_period": gyr["line"]}
    if not args.no_adjoint:
        extra["adjoint"] = adjoint_leg(L, g, gyr["omega"], gyr["cell_a"], gyr["seconds_per_solve"])
    if not args.no_jacobian:
        extra["jacobian"] = jacobian_leg(L)
    if not args.no_design:
        extra["design"] = design_leg(L)
    if not args.no_batch:
        extra["batch"] = batch_leg(L)
        if not args.no_cpu_baseline:
            extra["batch"]["cpu_baseline_all_cores"] = batch_cpu_baseline(extra["batch"])

    cpu = None
    if not args.no_cpu_baseline:
        wd = tempfile.mkdtemp(prefix="pscf_cpu_")
        try:
            cpu = cpu_baseline(g, int(np.mean(iters)), wd)
        finally:
            shutil.rmtree(wd, ignore_errors=True)

    line = {
        "metric": "converged SCFT solves/s at 64^3 FP64",
        "value": args.steps / elapsed,
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": elapsed / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": WORKLOAD, "grid": [64, 64, 64], "contour_steps": 200,
                   "iterations_per_solve": iters, "converged": [x.converge for x in results],
                   "final_cell_a": float(r.cell_param[0]), "f_helmholtz": r.f_helmholtz,
                   "f_flory_huggins": f_fh,
                   "final_state": ("disordered melt (f = Flory-Huggins f; a = 16 is far from the "
                                   "gyroid period -- see gyroid_at_period)"
                                   if abs(r.f_helmholtz - f_fh) < 1e-8 else "ordered"),
                   "ms_per_iteration": elapsed / sum(iters) * 1e3},
        "roofline": {"bound": "hbm", "kernel": "k_step_" + dom[5:] + "<64,64> (both sweeps)",
                     "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": TRAFFIC.get(dom),
                     "traffic_source": TRAFFIC_SOURCE,
                     "bytes_per_launch": kb[dom], "kernel_avg_us": kavg_us,
                     "kernel_timing": "in place: 5 density() calls at the converged field, each "
                                      "kernel once per contour step, start/end HIP events recorded "
                                      "by each dispatch (hipExtLaunchKernelGGL; %d launches of "
                                      "the dominant kernel)"
                                      % int(kn[names.index(dom)]),
                     "kernel_achieved_gbs": {nm: kb[nm] / (kavg_us[nm] * 1e-6) / 1e9
                                             for nm in names},
                     "step_us_graph": t_step_ms * 1e3, "steps_timed": steps_timed,
                     "step_bytes": bytes_step,
                     "step_achieved_gbs": bytes_step / (t_step_ms * 1e-3) / 1e9,
                     "step_frac": bytes_step / (t_step_ms * 1e-3) / 1e9 / HBM_PEAK_GBS},
        "cpu_baseline": cpu,
    }
    line.update(extra)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
