"""What is measured of this framework: calls of its public entry points that
circuit simulation consists of, over the range of sizes it is used at.

kinds
  tran     CircuitEngine.run_transient on a prepared engine: the whole path
           (eval, stamping, LU, Newton, step control, waveforms to the host)
  newton   the device Newton solve behind DC and single-step use, on a packed
           Monte Carlo batch
  lu       SparseLU.refactor + solve of a new matrix on an analysed pattern,
           in FP64, or FP32 with FP64 refinement
  lut      SparseLU.solve_transpose (adjoint / sensitivity direction)
  host     vajax_amd.sparse.solve on host buffers, as the reference's solver
           call is used
  build    DeviceCircuit.build_system: device eval and stamping alone

Circuits are the framework's own synthetic ones (RC ladder, ring oscillator,
CMOS gate DAGs, packed Monte Carlo batches, array multipliers); the seed draws
topology, device sizes, states and matrix values.
"""

import math
from types import SimpleNamespace

import numpy as np
import torch

from vajax_amd import _lib as L
from vajax_amd import generators as G
from vajax_amd import sparse, vacask
from vajax_amd.engine import AdaptiveConfig, CircuitEngine, DeviceCircuit
from vajax_amd.models import VT, mosfet_cache
from vajax_amd.topology import build_topology


def listed():
    return [
        # one linear solve of a ring's matrix through the host call: the
        # smallest use, all latency
        {"name": "host_ring101", "kind": "host", "circuit": "ring", "size": 101},
        # a linear RC network on a fixed grid (interconnect, filters)
        {"name": "tran_rc200", "kind": "tran", "circuit": "rc", "size": 200, "steps": 200,
         "precision": "f64"},
        # an oscillator: the usual small nonlinear bench circuit
        {"name": "tran_ring101", "kind": "tran", "circuit": "ring", "size": 101, "steps": 60,
         "precision": "f64"},
        # a logic block: the ordinary circuit size
        {"name": "tran_dag2000", "kind": "tran", "circuit": "dag", "size": 2000, "steps": 20,
         "precision": "f64"},
        # the same with the full EKV 2.6 transistor and FP32 factors
        {"name": "tran_ekv5001_f32", "kind": "tran", "circuit": "dag_ekv26", "size": 5001,
         "steps": 10, "precision": "f32"},
        # a large circuit's power-up
        {"name": "tran_dag65000", "kind": "tran", "circuit": "dag", "size": 65000, "steps": 8,
         "precision": "f64"},
        # Monte Carlo: many instances of one block advanced together
        {"name": "newton_batch64x1000", "kind": "newton", "circuit": "batch", "size": 1000,
         "instances": 64},
        # the linear solver alone at three sizes, both precisions
        {"name": "lu_dag777", "kind": "lu", "circuit": "dag", "size": 777, "precision": "f64"},
        {"name": "lu_dag20000_f32", "kind": "lu", "circuit": "dag", "size": 20000,
         "precision": "f32"},
        {"name": "lu_dag65000", "kind": "lu", "circuit": "dag", "size": 65000,
         "precision": "f64"},
        # sensitivities of a medium block
        {"name": "lut_dag5000", "kind": "lut", "circuit": "dag", "size": 5000,
         "precision": "f64"},
        # device eval and stamping of the large circuit
        {"name": "build_dag65000", "kind": "build", "circuit": "dag", "size": 65000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tran", "tran", "newton", "lu", "lu", "lut", "host", "build"])
    if kind == "tran":
        circuit = rng.choice(["rc", "ring", "dag", "dag", "dag_ekv26", "mult"])
        c = {"kind": kind, "circuit": circuit, "precision": rng.choice(["f64", "f64", "f32"])}
        if circuit == "rc":
            c.update(size=_log_int(rng, 20, 1000), steps=rng.randint(40, 200))
        elif circuit == "ring":
            c.update(size=2 * _log_int(rng, 5, 150) + 1, steps=rng.randint(20, 60))
        elif circuit == "mult":
            c.update(size=rng.randint(4, 20), steps=rng.randint(3, 5))
        else:
            n = _log_int(rng, 60, 40000 if circuit == "dag" else 12000)
            most = 30 if circuit == "dag" else 12
            c.update(size=n, steps=max(4, min(most, 200000 // n)))
        return c
    if kind == "newton":
        n = _log_int(rng, 60, 2000)
        return {"kind": kind, "circuit": "batch", "size": n,
                "instances": rng.randint(3, max(4, min(64, 64000 // n)))}
    if kind == "build":
        return {"kind": kind, "circuit": "dag", "size": _log_int(rng, 60, 60000)}
    circuit = rng.choice(["rc", "dag", "dag", "dag", "mult"])
    size = {"rc": _log_int(rng, 20, 3000), "mult": rng.randint(3, 24),
            "dag": _log_int(rng, 60, {"lu": 60000, "lut": 20000, "host": 3000}[kind])}[circuit]
    c = {"kind": kind, "circuit": circuit, "size": size}
    if kind != "host":
        c["precision"] = rng.choice(["f64", "f64", "f32"])
    return c


# ---- circuits -------------------------------------------------------------


def _netlist(case, seed):
    n, circuit = case["size"], case["circuit"]
    if case["kind"] == "build":
        # the pattern is fixed by the size; the seed varies the devices
        return G.monte_carlo(G.gate_dag(n, seed=n), seed)
    if circuit == "rc":
        return G.rc_ladder(n, seed=seed)
    if circuit == "ring":
        return G.ring_oscillator(n, seed=seed)
    if circuit == "dag":
        return G.gate_dag(n, seed=seed)
    if circuit == "dag_ekv26":
        return G.gate_dag(n, seed=seed, model="ekv26")
    if circuit == "mult":
        # the topology is fixed by the size; the seed varies the devices and
        # the operands
        rng = np.random.default_rng(seed)
        text = G.array_multiplier_testbench(n, a_bits=rng.integers(0, 2, n).tolist(),
                                            b_bits=rng.integers(0, 2, n).tolist())
        return G.monte_carlo(vacask.load("", text=text), seed)
    if circuit == "batch":
        return G.batch_mc(case["instances"], n, ragged=(), seed=seed)
    raise ValueError(circuit)


def _cuda(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device="cuda")


def _matrix(topo, net, rng, dt=1e-12):
    """Values of a transient Newton matrix on the circuit's CSR pattern: per
    device conductances and charge derivatives over dt in the shapes and
    magnitudes that circuits have, sources, and gmin on the diagonal."""
    v = np.zeros(topo.nse)
    for name, ms in topo.models.items():
        n = ms.count
        if name in ("resistor", "capacitor"):
            p = net.groups[name].params["r" if name == "resistor" else "c"]
            g = 1.0 / p if name == "resistor" else np.asarray(p) / dt
            g = g * rng.uniform(0.9, 1.1, n)
            j = np.stack([g, -g, -g, g], axis=1)
        else:  # drain, gate, source, bulk
            on = np.minimum(np.exp(rng.normal(-12.0, 2.5, n)), 2e-3)  # cut off to fully on
            gd, gg = on * rng.uniform(0.02, 1.0, n), on * rng.uniform(0.1, 1.0, n)
            gs = -(gd + gg) * rng.uniform(1.0, 1.3, n)
            gb = -(gd + gg + gs)
            w, ln = net.groups[name].params["w"], net.groups[name].params["l"]
            cg = (0.01 * w * ln + 2e-10 * w) / dt
            cj = 5e-10 * w / dt
            j = np.zeros((n, 4, 4))
            for col, x in enumerate((gd, gg, gs, gb)):
                j[:, 0, col] += x
                j[:, 2, col] -= x
            for a, b, c in ((1, 2, cg), (1, 0, cg), (0, 3, cj), (2, 3, cj)):
                j[:, a, a] += c
                j[:, b, b] += c
                j[:, a, b] -= c
                j[:, b, a] -= c
            j = j.reshape(n, 16)
        pos = ms.csr_pos
        ok = pos >= 0
        v += np.bincount(pos[ok], weights=j[ok], minlength=topo.nse)
    v[topo.diag_pos] += 1e-12
    for key, s in (("b_p", 1.0), ("b_n", -1.0), ("bt_p", 1.0), ("bt_n", -1.0)):
        p = topo.vs_pos.get(key, np.zeros(0, np.int64))
        v[p[p >= 0]] += s
    return v


def _product(topo, v, x, transpose=False):
    """A x (A^T x) in extended precision, rounded to 64 bits."""
    rows = np.repeat(np.arange(topo.n_augmented), np.diff(topo.indptr))
    cols = topo.indices
    out, src = (cols, rows) if transpose else (rows, cols)
    t = v.astype(np.longdouble) * x.astype(np.longdouble)[src]
    order = np.argsort(out, kind="stable")
    at = np.concatenate([[0], np.cumsum(np.bincount(out, minlength=topo.n_augmented))])
    return np.add.reduceat(t[order], at[:-1]).astype(np.float64)


def _system(case, seed):
    """(topology, first matrix, new matrix, right-hand side, its solution):
    the new matrix of the pass is another Newton iterate's, and the solution is
    an update of some millivolts."""
    net = _netlist(case, seed)
    topo = build_topology(net)
    rng = np.random.default_rng([seed, 1])
    first = _matrix(topo, net, rng)
    new = _matrix(topo, net, rng)
    x = rng.normal(0.0, 1e-2, topo.n_augmented)
    x[topo.n_unknowns:] *= 1e-2  # branch currents
    b = _product(topo, new, x, case["kind"] == "lut")
    return topo, first, new, b, x


def _state_vector(topo, rng):
    """Node voltages inside the rails as a transient meets them (ground first,
    then branch currents)."""
    x = np.zeros(topo.n_total + topo.n_vsources)
    x[1:topo.n_total] = rng.uniform(0.0, 1.0, topo.n_total - 1)
    x[topo.n_total:] = rng.normal(0.0, 1e-4, topo.n_vsources)
    return x


# ---- what a program holds before the call ---------------------------------


def prepare(case, seed):
    kind = case["kind"]
    s = SimpleNamespace(kind=kind, precision=case.get("precision", "f64"))
    if kind == "tran":
        net = _netlist(case, seed)
        eng = CircuitEngine(net)
        eng.parse()
        eng.options.fixed_step_transient = case["circuit"] == "rc"
        cfg = AdaptiveConfig(integration_method="gear2")
        dt = 2e-12 if case["circuit"] == "mult" else 1e-12
        if case["circuit"] == "rc":
            cfg.tran_fs = 1.0

        def plan(steps):
            eng.prepare(t_stop=10e-9, dt=dt, adaptive_config=cfg, precision=case["precision"],
                        use_graph=True, max_steps=steps + 1)

        plan(2)  # the symbolic analysis, which an engine keeps
        eng.run_transient()
        plan(case["steps"])
        s.engine = eng
    elif kind == "newton":
        net = _netlist(case, seed)
        topo = build_topology(net)
        dc = DeviceCircuit(topo, net)
        rng = np.random.default_rng([seed, 2])
        # the first steps of a power-up from rest: the supplies a few
        # millivolts up, the history empty
        x = 1e-3 * _state_vector(topo, rng)
        s.vs = _cuda(rng.uniform(0.0, 2e-2, topo.n_vsources))
        s.isv = _cuda(np.zeros(net.isources.count))
        s.x, s.q = _cuda(x), _cuda(np.zeros(topo.n_unknowns))
        s.c0 = 1.0 / 1e-12
        s.circuit = dc
        s.solve = dc.make_nr_solve(use_graph=True)
        s.solve(s.x, s.vs, s.isv, s.q, s.c0)  # the symbolic analysis
    elif kind == "build":
        net = _netlist(case, seed)
        topo = build_topology(net)
        rng = np.random.default_rng([seed, 3])
        s.circuit = DeviceCircuit(topo, net)
        s.x, s.vs = _cuda(_state_vector(topo, rng)), _cuda(rng.uniform(0, 1, topo.n_vsources))
        s.isv = _cuda(np.zeros(net.isources.count))
        s.q = [_cuda(rng.normal(0.0, 1e-15, topo.n_unknowns)) for _ in range(2)]
        s.c = (1.5e12, -2e12, 0.5e12)
    else:
        topo, first, new, b, _ = _system(case, seed)
        s.topo = topo
        if kind == "host":
            s.a, s.b = new, b
            sparse.solve(topo.indptr, topo.indices, first, b)
            return s
        s.lu = sparse.SparseLU(topo.indptr, topo.indices)
        s.prec = L.VJX_PREC_F32 if case["precision"] == "f32" else L.VJX_PREC_F64
        s.refine = 1 if case["precision"] == "f32" else 0
        s.a, s.b = _cuda(new), _cuda(b)
        s.out = torch.empty_like(s.b)
        torch.cuda.synchronize()
        if kind == "lut":
            s.lu.solve_transpose(_cuda(first), s.b, s.out, s.prec, s.refine)
        else:
            s.lu.analyze(first)
            s.lu.refactor(_cuda(first), s.prec)
    return s


def run(s):
    if s.kind == "tran":
        r = s.engine.run_transient()
        return {"times": r.times, "V": r.stats["V_out"], "I": r.stats["I_out"]}
    if s.kind == "newton":
        r = s.solve(s.x, s.vs, s.isv, s.q, s.c0)
        return {"X": r[0], "iterations": r[1], "Q": r[4], "dQdt": r[5], "I": r[6]}
    if s.kind == "build":
        r = s.circuit.build_system(s.x, s.vs, s.isv, Q_prev=s.q[0], Q_prev2=s.q[1], c0=s.c[0],
                                   c1=s.c[1], c2=s.c[2])
        return {k: r[k] for k in ("csr_data", "f", "Q", "max_res_contrib", "I_vsource")}
    if s.kind == "host":
        return sparse.solve(s.topo.indptr, s.topo.indices, s.a, s.b)
    if s.kind == "lut":
        s.lu.solve_transpose(s.a, s.b, s.out, s.prec, s.refine)
    else:
        s.lu.refactor(s.a, s.prec)
        s.lu.solve(s.a, s.b, s.out, s.refine)
    return s.out


# ---- the least work of a pass ---------------------------------------------


def _sizes(case):
    """(unknowns, matrix entries, devices, doubles per device, LU entries)."""
    n = case["size"]
    if case["circuit"] == "rc":
        return n + 2, 3 * n + 3, 2 * n, 1, 3 * n
    if case["circuit"] == "ring":
        return n + 2, 5 * n + 3, 3 * n, 8, 7 * n
    if case["circuit"] == "mult":
        return 32 * n * n, 255 * n * n, 65 * n * n, 11, 600 * n * n
    k = case.get("instances", 1)
    per = 52 if case["circuit"] == "dag_ekv26" else 11
    return k * (2 * n + 130), k * 15 * n, k * 4 * n, per, k * 40 * n


def work(case):
    n, nnz, dev, per, lu = _sizes(case)
    # factorisation: each multiplier updates about ten entries of its row
    fact = 20.0 * lu
    solve = 4.0 * lu
    ev = (250.0 if per < 52 else 6000.0) * dev
    build = 8.0 * (per * dev + nnz + 4 * n)
    kind = case["kind"]
    if kind == "tran":
        it = 2 * case["steps"]
        return {"bytes": it * build + 8.0 * case["steps"] * n, "flops": it * (fact + solve + ev)}
    if kind == "newton":
        return {"bytes": 3 * build, "flops": 3 * (fact + solve + ev)}
    if kind == "build":
        return {"bytes": build, "flops": ev}
    return {"bytes": 8.0 * (nnz + 2 * n), "flops": fact + solve}


def tolerance(case):
    # measured between two elimination orders of the same systems (largest
    # relative differences seen: solves 2e-16 in FP64 and 1.3e-14 with FP32
    # factors, Newton 6e-17, waveforms 1.7e-14 and 3.5e-12), with room for
    # larger sizes.  EKV 2.6 waveforms follow their step sizes, which the
    # error estimate sets from a difference of nearly equal voltages: 1.4e-7
    # after 27 steps.
    kind, f32 = case["kind"], case.get("precision") == "f32"
    if kind == "tran":
        if case["circuit"] == "dag_ekv26":
            return {"rel": 1e-6, "max": 1e-5}
        return {"rel": 2e-11, "max": 1e-9} if f32 else {"rel": 1e-12, "max": 1e-10}
    if kind in ("lu", "lut") and f32:
        return {"rel": 2e-13, "max": 2e-11}
    if kind == "build":  # exponentials of another library: 2.5e-14
        return {"rel": 1e-13, "max": 1e-11}
    return {"rel": 1e-14, "max": 1e-12}


# ---- 64-bit values without the framework's numerics -----------------------


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lu", "lut", "host"):
        return _system(case, seed)[4]
    if kind == "build":
        return _exact_build(case, seed)
    if kind == "tran" and case["circuit"] == "rc" and case["precision"] == "f64":
        return _exact_rc(case, seed)
    return None  # thousands of nonlinear unknowns: no plain solver in reach


def _exact_build(case, seed):
    net = _netlist(case, seed)
    topo = build_topology(net)
    rng = np.random.default_rng([seed, 3])
    X = _state_vector(topo, rng)
    vs = rng.uniform(0, 1, topo.n_vsources)
    qp = [rng.normal(0.0, 1e-15, topo.n_unknowns) for _ in range(2)]
    c0, c1, c2 = 1.5e12, -2e12, 0.5e12
    gmin = 1e-12
    ms = topo.models["mosfet"]
    sgn, vgoff, phi, gam, beta0, theta, cgs, cgd, cgb, cdb, csb = mosfet_cache(
        net.groups["mosfet"].params)
    d, g, s, b = (X[ms.node_terms[:, k]] for k in range(4))
    vgp = sgn * (g - b) + vgoff
    g2 = 0.5 * gam
    t = vgp + g2 * g2
    lo = t <= 1e-12
    sq = np.sqrt(np.where(lo, 1.0, t))
    vp = np.where(lo, vgp - phi - gam * gam / 2, vgp - phi - gam * (sq - g2))
    dvp = np.where(lo, 1.0, 1.0 - gam / (2 * sq))
    arg = phi + vp + 4 * VT
    low = arg <= 1e-24
    sa = np.sqrt(np.where(low, 1.0, arg))
    n = np.where(low, 1.0 + gam / 2 * 1e48, 1.0 + gam / (2 * sa))
    dn = np.where(low, 0.0, -gam / (4 * np.where(low, 1.0, arg) * sa))
    den = 1 + theta * vp
    beta, dbeta = beta0 / den, -beta0 * theta / (den * den)

    def interp(u):
        e = np.exp(-np.abs(u))
        sp = np.maximum(u, 0) + np.log1p(e)
        return sp, sp * np.where(u >= 0, 1 / (1 + e), e / (1 + e))

    lf, ff = interp(0.5 * (vp - sgn * (s - b)) / VT)
    lr, fr = interp(0.5 * (vp - sgn * (d - b)) / VT)
    isp = 2 * n * beta * VT * VT
    idf = lf * lf - lr * lr
    cur = sgn * isp * idf
    gg = (2 * VT * VT * (dn * beta + n * dbeta) * idf + isp * (ff - fr) / VT) * dvp
    gs, gd = -isp * ff / VT, isp * fr / VT
    gb = -(gg + gs + gd)
    j = np.zeros((ms.count, 4, 4))
    for k, x in enumerate((gd, gg, gs, gb)):
        j[:, 0, k] += x
        j[:, 2, k] -= x
    for a, k, c in ((1, 2, cgs), (1, 0, cgd), (1, 3, cgb), (0, 3, cdb), (2, 3, csb)):
        j[:, a, a] += c0 * c
        j[:, k, k] += c0 * c
        j[:, a, k] -= c0 * c
        j[:, k, a] -= c0 * c
    zero = np.zeros(ms.count)
    fr_ = np.stack([cur, zero, -cur, zero], axis=1)
    q = np.stack([cgd * (d - g) + cdb * (d - b),
                  cgs * (g - s) + cgd * (g - d) + cgb * (g - b),
                  cgs * (s - g) + csb * (s - b),
                  -(cgb * (g - b) + cdb * (d - b) + csb * (s - b))], axis=1)
    nse, nu = topo.nse, topo.n_unknowns
    pos = ms.csr_pos
    ok = pos >= 0
    csr = np.bincount(pos[ok], weights=j.reshape(-1, 16)[ok], minlength=nse)
    csr[topo.diag_pos] += gmin
    for key, v in (("b_p", 1.0), ("b_n", -1.0), ("bt_p", 1.0), ("bt_n", -1.0)):
        p = topo.vs_pos[key]
        csr[p[p >= 0]] += v
    r = ms.res_idx
    ok = r >= 0
    f = np.bincount(r[ok], weights=fr_[ok], minlength=nu)
    Q = np.bincount(r[ok], weights=q[ok], minlength=nu)
    p_, n_ = topo.vs_node_p, topo.vs_node_n
    i_vs = np.where(p_ > 0, -f[np.maximum(p_ - 1, 0)], 0.0)
    np.add.at(f, p_[p_ > 0] - 1, X[topo.n_total:][p_ > 0])
    np.add.at(f, n_[n_ > 0] - 1, -X[topo.n_total:][n_ > 0])
    f = f + c0 * Q + c1 * qp[0] + c2 * qp[1] + gmin * X[1:topo.n_total]
    res = np.concatenate([f, X[p_] - X[n_] - vs])
    return {"csr_data": csr, "f": res, "Q": Q, "max_res_contrib": None, "I_vsource": i_vs}


def _exact_rc(case, seed):
    """BDF2 on a fixed grid for the linear ladder, by dense 64-bit solves."""
    net = _netlist(case, seed)
    topo = build_topology(net)
    nt = topo.n_total
    r, c = topo.models["resistor"], topo.models["capacitor"]
    Gm, Cm = np.zeros((nt, nt)), np.zeros((nt, nt))
    for ms, val, M in ((r, 1.0 / np.asarray(net.groups["resistor"].params["r"]), Gm),
                       (c, np.asarray(net.groups["capacitor"].params["c"]), Cm)):
        a, b = ms.node_terms[:, 0], ms.node_terms[:, 1]
        for i, j, sg in ((a, a, 1.0), (b, b, 1.0), (a, b, -1.0), (b, a, -1.0)):
            np.add.at(M, (i, j), sg * val)
    src = int(topo.vs_node_p[0])
    free = np.array([k for k in range(1, nt) if k != src])
    dt = 1e-12
    A = Gm + 1.5 / dt * Cm + 1e-12 * np.eye(nt)
    inv = np.linalg.inv(A[np.ix_(free, free)])
    S = case["steps"]
    V = np.zeros((S + 1, nt))
    I = np.zeros((S + 1, 1))
    times = np.arange(S + 1) * dt
    q1, q2 = np.zeros(nt), np.zeros(nt)  # the DC point of the undriven ladder is zero
    for k in range(1, S + 1):
        t = k * dt
        vin = min(t / 10e-12, 1.0)
        rhs = -(-2.0 / dt * q1 + 0.5 / dt * q2)[free] - A[np.ix_(free, [src])][:, 0] * vin
        V[k, src] = vin
        V[k, free] = inv @ rhs
        res = A[np.ix_(free, free)] @ V[k, free] - rhs
        V[k, free] -= inv @ res
        q2, q1 = q1, Cm @ V[k]
        I[k, 0] = -(Gm @ V[k])[src]
    return {"times": times, "V": V, "I": I}
