"""The work that users of this framework have it do, as timed cases.

Seven kinds of case, each through the public entry points of the package:

* ``solve``    -- a whole run: ``solve(problem)`` from the start address, its report and its
  final vector (set-up, stepping and read-out together, as a script does it).
* ``advance``  -- an equilibrated run goes on for some steps and its vector is read out for a
  checkpoint: the steady state of a long calculation.
* ``sweep``    -- a batch of independent runs over u from their specifications to their
  histories (``BatchedRuns``).
* ``overlap``  -- ``dot(v, w)`` and ``dot(v, op, w)`` of two replicas' vectors.
* ``gradient`` -- dE/du and dE/dt of the K-step deterministic projector energy.
* ``product``  -- ``mul!(w, H, v)`` and its pullback for a caller that differentiates through it.
* ``ground``   -- ground-state energies by Lanczos (the exact answers runs are held against).
"""
import ctypes
import math

import numpy as np
import torch

from __graft_entry__ import load_package

rimu = load_package()


# ---- cases ------------------------------------------------------------------------------
def listed():
    return [
        # the smallest run anyone does: a chain whose exact energy is known, 1000 integer
        # walkers (tens of microseconds of work a step: launches and latency)
        dict(name="solve_real10_1e3", kind="solve", model="real", M=10, N=10, u=6.0, style="integer",
             walkers=1000.0, dtau=1e-3, steps=1000, initiator=False, project=True),
        # the reference's benchmark "(10, 20) Mom space with projected energy and initiator"
        dict(name="solve_mom20_initiator", kind="solve", model="mom", M=20, N=10, u=1.0, style="dynamic",
             walkers=4e4, dtau=1e-4, steps=1500, initiator=True, project=True),
        # the reference's benchmark "(50, 50) Real space": 99-bit addresses
        dict(name="solve_real50_5e4", kind="solve", model="real", M=50, N=50, u=6.0, style="dynamic",
             walkers=5e4, dtau=1e-4, steps=1000, initiator=False, project=False),
        # the reference's "2D Hubbard" system, two fermion components on 4 x 4 sites, exact
        # vector-matrix products on the sparse vector
        dict(name="solve_fermi4x4_exact", kind="solve", model="fermi", M=16, N=2, u=1.0, style="exact",
             walkers=1e6, dtau=0.02, steps=400, initiator=False, project=False),
        # the largest: 1e8 walkers of 20 bosons on 20 sites, semistochastic FP64 amplitudes
        dict(name="advance_real20_1e8", kind="advance", model="real", M=20, N=20, u=6.0, style="dynamic",
             walkers=1e8, dtau=1e-3, steps=50, initiator=False, project=False),
        # momentum space, integer walkers: thousands of excitations per address
        dict(name="advance_mom16_2e7", kind="advance", model="mom", M=16, N=16, u=4.0, style="integer",
             walkers=2e7, dtau=5e-4, steps=50, initiator=False, project=True),
        # two-word addresses at a production walker number
        dict(name="advance_real50_5e6", kind="advance", model="real", M=50, N=50, u=6.0, style="dynamic",
             walkers=5e6, dtau=1e-3, steps=100, initiator=False, project=False),
        # 64 runs of uneven M, N, u and walker number advanced together, from their specs on
        dict(name="sweep_64_runs", kind="sweep", runs=64, walkers=1e5, steps=1000),
        # the estimators of a replica pair at a reporting step: norm, correlator and energy
        dict(name="overlap_real20_pair", kind="overlap", M=20, N=20, u=6.0, entries=400_000),
        # gradients of the projector energy at four u, dimension 1,352,078
        dict(name="gradient_real12", kind="gradient", M=12, N=12, rhs=4, steps=300, dtau=1e-3),
        # one product and its pullback inside somebody else's optimisation, dimension 92,378
        dict(name="product_real10", kind="product", M=10, N=10, rhs=1),
        # exact energies of four u on 11 sites, dimension 352,716
        dict(name="ground_real11", kind="ground", M=11, N=11, rhs=4),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["solve", "solve", "advance", "advance", "sweep", "overlap", "gradient", "product", "ground"])
    u = round(rng.uniform(1.0, 8.0), 3)
    if kind == "solve":
        model = rng.choice(["real", "real", "mom", "wide", "bose2d", "fermi"])
        if model == "real":
            M = rng.randint(8, 24)
            return dict(kind="solve", model="real", M=M, N=M - rng.randint(0, 3), u=u,
                        style=rng.choice(["integer", "dynamic"]), walkers=round(_log(rng, 500, 2e5)), dtau=1e-3,
                        steps=rng.randint(400, 1000), initiator=rng.random() < 0.3, project=rng.random() < 0.5)
        if model == "mom":
            N = rng.randint(6, 14)
            return dict(kind="solve", model="mom", M=rng.randint(N, 20), N=N, u=round(rng.uniform(0.5, 4.0), 3),
                        style=rng.choice(["integer", "dynamic"]), walkers=round(_log(rng, 1e3, 1e5)), dtau=1e-4,
                        steps=rng.randint(400, 1000), initiator=rng.random() < 0.5, project=True)
        if model == "wide":
            M = rng.randint(34, 60)
            return dict(kind="solve", model="real", M=M, N=M - rng.randint(0, 3), u=u, style="dynamic",
                        walkers=round(_log(rng, 5e3, 2e5)), dtau=1e-4, steps=rng.randint(400, 1000),
                        initiator=rng.random() < 0.3, project=False)
        if model == "bose2d":
            side = rng.randint(3, 8)
            return dict(kind="solve", model="bose2d", M=side * side, N=side * side, u=u, style="dynamic",
                        walkers=round(_log(rng, 5e3, 2e5)), dtau=1e-4, steps=rng.randint(400, 800),
                        initiator=False, project=False)
        return dict(kind="solve", model="fermi", M=16, N=2, u=round(rng.uniform(0.5, 4.0), 3), style="exact",
                    walkers=1e6, dtau=0.02, steps=rng.randint(200, 500), initiator=False, project=False)
    if kind == "advance":
        model = rng.choice(["real", "mom", "wide"])
        if model == "real":
            M = rng.randint(14, 26)
            return dict(kind="advance", model="real", M=M, N=M - rng.randint(0, 3), u=u,
                        style=rng.choice(["integer", "dynamic", "dynamic"]), walkers=round(_log(rng, 2e5, 4e7)),
                        dtau=1e-3, steps=rng.randint(20, 50), initiator=rng.random() < 0.25, project=False)
        if model == "mom":
            N = rng.randint(10, 16)
            return dict(kind="advance", model="mom", M=rng.randint(N, 18), N=N, u=round(rng.uniform(1.0, 4.0), 3),
                        style=rng.choice(["integer", "integer", "dynamic"]), walkers=round(_log(rng, 2e5, 5e6)),
                        dtau=5e-4, steps=rng.randint(20, 50), initiator=rng.random() < 0.25, project=True)
        M = rng.randint(34, 60)
        return dict(kind="advance", model="real", M=M, N=M - rng.randint(0, 3), u=u, style="dynamic",
                    walkers=round(_log(rng, 1e5, 5e6)), dtau=1e-3, steps=rng.randint(20, 100), initiator=False,
                    project=False)
    if kind == "sweep":
        return dict(kind="sweep", runs=rng.randint(16, 256), walkers=round(_log(rng, 1e4, 1e5)),
                    steps=rng.randint(300, 1000))
    if kind == "overlap":
        M = rng.randint(14, 26)
        return dict(kind="overlap", M=M, N=M, u=u, entries=round(_log(rng, 2e4, 4e5)))
    M = rng.randint(8, 12) if kind != "ground" else rng.randint(7, 11)
    N = max(4, M - rng.randint(0, 3))
    if kind == "gradient":
        return dict(kind="gradient", M=M, N=N, rhs=rng.randint(1, 4), steps=rng.randint(60, 300), dtau=1e-3)
    return dict(kind=kind, M=M, N=N, rhs=rng.randint(1, 4))


# ---- set-up -------------------------------------------------------------------------------
def _hamiltonian(case):
    M, N, u = case["M"], case["N"], case["u"]
    if case["model"] == "real":
        return rimu.HubbardReal1D(rimu.near_uniform(N, M), u=u, t=1.0)
    if case["model"] == "mom":
        onr = [0] * M
        onr[M // 2 - 1] = N                      # the zero-momentum condensate
        return rimu.HubbardMom1D(rimu.BoseFS(*onr), u=u)
    side = math.isqrt(M)
    grid = rimu.PeriodicBoundaries(side, side)
    if case["model"] == "bose2d":
        return rimu.HubbardRealSpace(rimu.near_uniform(N, M), geometry=grid, u=[[u]])
    address = rimu.FermiFS2C(M, (1, 1), (2, 1), (1, -1), (2, -1))
    return rimu.HubbardRealSpace(address, geometry=grid, u=[[0.0, u], [u, 0.0]])


_STYLES = {"integer": rimu.IsStochasticInteger, "dynamic": rimu.IsDynamicSemistochastic,
           "exact": rimu.IsDeterministic}


def _problem(case, seed, last_step):
    h = _hamiltonian(case)
    address = h.starting_address()
    population = 10 + seed % 7                   # the start vector, also where nothing is drawn
    style = _STYLES[case["style"]]()
    start = rimu.PDVec((address, population), style=style, initiator=case["initiator"])
    post = (rimu.ProjectedEnergy(h, address),) if case["project"] else ()
    return rimu.ProjectorMonteCarloProblem(
        h, start_at=start, style=style, time_step=case["dtau"], last_step=last_step,
        target_walkers=case["walkers"], post_step_strategy=post, random_seed=seed)


def _us(seed, rhs):
    rng = np.random.default_rng(seed)
    return [float(x) for x in rng.uniform(1.0, 8.0, rhs)]


def _chains(case, seed):
    return [rimu.HubbardReal1D(rimu.near_uniform(case["N"], case["M"]), u=u, t=1.0)
            for u in _us(seed, case["rhs"])]


def _hopped(M, N, n, rng):
    """About n distinct addresses of a Mott-like chain: the uniform filling after a few random
    hops, as bit strings, ascending, with their occupation numbers."""
    occ = np.zeros((int(1.6 * n), M), dtype=np.int16)
    occ[:, :N] = 1
    rows = np.arange(len(occ))
    for k in range(10):
        site = rng.integers(0, M, len(occ))
        to = (site + rng.choice([-1, 1], len(occ))) % M
        go = (occ[rows, site] > 0) & (rng.random(len(occ)) < 0.8)
        occ[rows[go], site[go]] -= 1
        occ[rows[go], to[go]] += 1
    keys, first = np.unique(_bits(occ), return_index=True)
    keep = np.sort(rng.permutation(len(keys))[:n])
    return keys[keep], occ[first[keep]]


def _bits(occ):
    keys = np.zeros(len(occ), dtype=np.uint64)
    shift = np.zeros(len(occ), dtype=np.uint64)
    one = np.uint64(1)
    for m in range(occ.shape[1]):
        n = occ[:, m].astype(np.uint64)
        keys |= ((one << n) - one) << shift
        shift += n + one
    return keys


def _pair(case, seed):
    """Two replicas' vectors on mostly the same addresses."""
    rng = np.random.default_rng(seed)
    keys, occ = _hopped(case["M"], case["N"], case["entries"], rng)
    out = []
    for _ in range(2):
        sel = rng.random(len(keys)) < 0.9
        out.append((keys[sel], occ[sel], rng.standard_exponential(int(sel.sum())) + 1.0))
    return out


def _states(case):
    """Number of addresses of the case's space."""
    if case["model"] == "fermi":
        return math.comb(case["M"], case["N"]) ** 2
    return math.comb(case["M"] + case["N"] - 1, case["N"])


def _buffers(case):
    """Host arrays a run's vector is read into: a stored entry holds one walker or more, so
    half as many again as the target walkers is room enough."""
    n = int(min(_states(case), 1.5 * case["walkers"] + 2000))
    kw = 2 if _hamiltonian(case).key_words == 2 else 1
    return {"keys": np.zeros(n * kw, dtype=np.int64), "vals": np.zeros(
        n, dtype=np.int64 if case["style"] == "integer" else np.float64), "used": 0, "kw": kw}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        return {"kind": kind, "problem": _problem(case, seed, case["steps"]), "out": _buffers(case)}
    if kind == "advance":
        # grown to the target walker number and settled there; chains take a longer time step
        # until then, so that the steps to be timed find the steady distribution over addresses
        longer = 5 if case["model"] == "real" else 1
        sim = rimu.init(_problem(dict(case, dtau=longer * case["dtau"]), seed, 0))
        while sim.step < 2000 and not sim.aborted:
            sim.solve_(last_step=sim.step + 100)
            if sim.columns["norm"][-1] > 0.95 * case["walkers"]:
                break
        sim.solve_(last_step=sim.step + 200)
        sim.shift_parameters.time_step = case["dtau"]
        sim.solve_(last_step=sim.step + 50)
        return {"kind": kind, "sim": sim, "steps": case["steps"], "out": _buffers(case)}
    if kind == "sweep":
        specs = rimu.u_sweep_specs(case["runs"], rng_seed=seed)
        for i, s in enumerate(specs):
            s.seed = seed + i
            s.target_walkers = min(s.target_walkers, case["walkers"])
        room = int(case["runs"] * (1.5 * case["walkers"] + 2000))
        return {"kind": kind, "specs": specs, "steps": case["steps"], "room": room}
    if kind == "overlap":
        h = rimu.HubbardReal1D(rimu.near_uniform(case["N"], case["M"]), u=case["u"], t=1.0)
        style = rimu.IsDeterministic()
        vecs = []
        for keys, _, vals in _pair(case, seed):
            eng = rimu._native.Engine(h.descriptor(), style.descriptor(), seed, len(keys) + 1, len(keys) + 4096)
            eng.upload(keys, vals)
            vecs.append(rimu.DeviceDVec(eng, h, style))
        return {"kind": kind, "vecs": vecs, "ops": (h, rimu.G2RealCorrelator(1), rimu.DensityMatrixDiagonal(1))}
    chains = _chains(case, seed)
    d = rimu.DenseHamiltonians(chains)
    st = {"kind": kind, "d": d, "case": case}
    rng = np.random.default_rng(seed + 1)
    if kind == "product":
        st["v"] = rng.standard_normal((d.dim, d.R))
        st["ybar"] = rng.standard_normal((d.dim, d.R))
    else:
        st["v0"] = d.unit_vector(chains[0].starting_address())
        st["shift"] = np.zeros(d.R)
    return st


def _report(columns, n):
    return {name: np.asarray(col[-n:], dtype=np.float64) for name, col in columns.items()}


def _read(engine, out):
    """The engine's vector into the host arrays (ascending addresses), as a checkpoint reads it."""
    n = ctypes.c_int64(0)
    native = rimu._native
    native.check(native.lib().rimu_vector_download(engine._h, out["keys"].ctypes.data, out["vals"].ctypes.data,
                                                   len(out["vals"]), ctypes.byref(n)))
    for a, kw in ((out["keys"], out["kw"]), (out["vals"], 1)):
        a[n.value * kw:out["used"] * kw] = 0       # what a longer vector left there
    out["used"] = n.value
    return {"keys": out["keys"], "vals": out["vals"], "length": n.value}


def run(state):
    kind = state["kind"]
    if kind == "solve":
        sim = rimu.solve(state["problem"])
        df = sim.DataFrame()
        vector = _read(sim.engine, state["out"])
        sim.close()
        return {"report": {c: df[c].to_numpy(np.float64) for c in df.columns}, **vector}
    if kind == "advance":
        sim, n = state["sim"], state["steps"]
        sim.solve_(last_step=sim.step + n)
        return {"report": _report(sim.columns, n), **_read(sim.engine, state["out"])}
    if kind == "sweep":
        b = rimu.BatchedRuns(state["specs"], history_steps=state["steps"])
        b.step(state["steps"])
        hist = b.history()
        status, length = b.status()
        keys, vals = (np.zeros(state["room"], dtype=np.int64) for _ in range(2))
        at = 0
        for r in range(b.n):
            k, v = b.vector(r)
            keys[at:at + len(k)], vals[at:at + len(k)] = k, v
            at += len(k)
        b.close()
        return {"history": hist, "status": status, "length": length, "keys": keys, "vals": vals}
    if kind == "overlap":
        left, right = state["vecs"]
        return {"dot": rimu.dot(left, right), "ops": list(rimu.dot(left, state["ops"], right))}
    d = state["d"]
    if kind == "gradient":
        c = state["case"]
        res = d.projector_energy(c["steps"], c["dtau"], state["shift"], state["v0"])
        return {k: res[k] for k in ("energy", "grad_u", "grad_t", "hf_u", "hf_t", "v")}
    if kind == "product":
        y, pullback = d.rrule_mul(state["v"])
        vbar, ubar, tbar = pullback(state["ybar"])
        return {"y": y, "vbar": vbar, "ubar": ubar, "tbar": tbar}
    return {"energy": d.ground_state(state["v0"])[0]}


# ---- what a pass cannot do without -----------------------------------------------------------
def _dim(case):
    return math.comb(case["M"] + case["N"] - 1, case["N"])


def work(case):
    kind = case["kind"]
    if kind in ("solve", "advance"):
        # per step the vector is read and written once, and every walker makes an attempt (a
        # random number of ten rounds, a hop and its matrix element: about 200 operations)
        walkers = float(case["walkers"])
        key = 16 if case["M"] + case["N"] > 65 else 8
        entries = {"exact": 14_400.0, "integer": 0.6 * walkers, "dynamic": 0.6 * walkers}[case["style"]]
        if case["model"] == "real":
            entries = min(entries, float(_dim(case)))
        attempts = 20 * entries if case["style"] == "exact" else walkers
        share = 0.5 if kind == "solve" else 1.0     # a whole run grows from one address
        return {"bytes": share * case["steps"] * 2 * entries * (key + 8) + entries * (key + 8),
                "flops": share * case["steps"] * (200 * attempts + 50 * entries)}
    if kind == "sweep":
        walkers = case["runs"] * case["walkers"] / 4
        return {"bytes": case["steps"] * (walkers * 16.0 + case["runs"] * 48.0),
                "flops": case["steps"] * 200.0 * walkers}
    if kind == "overlap":
        n = case["entries"] * 0.9
        return {"bytes": 2 * n * 16.0, "flops": n * 2 * 0.65 * case["M"] * 100.0}
    D, R = float(_dim(case)), case["rhs"]
    product = {"bytes": D * (8 + 16 * R), "flops": D * 1.1 * case["M"] * (2 * R + 20)}
    times = {"gradient": 3 * case.get("steps", 0), "product": 2.5, "ground": 100}[kind]
    return {k: times * x for k, x in product.items()}


# ---- the same in 64 bits without the framework -------------------------------------------------
def _basis(M, N):
    """Occupation numbers (dim, M) of every N-boson address of M modes."""
    table = [np.full((1, 1), n, dtype=np.int64) for n in range(N + 1)]   # one mode, n bosons
    for _ in range(M - 1):
        table = [np.concatenate([np.pad(table[n - k], ((0, 0), (0, 1)), constant_values=k) for k in range(n + 1)])
                 for n in range(N + 1)]
    return table[N]


def _table(M, N, device):
    """Interaction sum n(n-1)/2 of every address, and per hop (neighbour row, -sqrt factor)."""
    occ = _basis(M, N)
    keys = _bits(occ)
    order = np.argsort(keys)
    occ, keys = occ[order], keys[order]
    diag = torch.from_numpy((occ * (occ - 1) / 2).sum(1)).to(device)
    hops = []
    for m in range(M):
        for to in ((m + 1) % M, (m - 1) % M):
            go = occ[:, m] > 0
            new = occ.copy()
            new[:, m] -= go
            new[:, to] += go
            row = np.searchsorted(keys, _bits(new))
            amp = -np.sqrt(np.where(go, occ[:, m] * (occ[:, to] + 1.0), 0.0))
            hops.append((torch.from_numpy(row).to(device), torch.from_numpy(amp).to(device)[:, None]))
    return keys, diag[:, None], hops


def _kinetic(hops, v):
    out = torch.zeros_like(v)
    for row, amp in hops:
        out += amp * v[row]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "overlap":
        (tk, _, tv), (uk, occ, uv) = _pair(case, seed)

        def amplitude(keys):
            at = np.minimum(np.searchsorted(tk, keys), len(tk) - 1)
            return np.where(tk[at] == keys, tv[at], 0.0)

        own = amplitude(uk) * uv
        M = case["M"]
        n = occ.astype(np.float64)
        energy = math.fsum(own * case["u"] * (n * (n - 1)).sum(1) / 2)
        for m in range(M):
            for to in ((m + 1) % M, (m - 1) % M):
                go = occ[:, m] > 0
                new = occ[go].copy()
                new[:, m] -= 1
                new[:, to] += 1
                energy -= math.fsum(np.sqrt(n[go, m] * (n[go, to] + 1)) * amplitude(_bits(new)) * uv[go])
        g2 = math.fsum(own * (n * np.roll(n, -1, axis=1)).sum(1)) / M
        return {"dot": math.fsum(own), "ops": [energy, g2, math.fsum(own * n[:, 0])]}
    if kind not in ("gradient", "product", "ground"):
        return None                               # random walks have no such value
    device = "cuda" if torch.cuda.is_available() else "cpu"
    M, N, R = case["M"], case["N"], case["rhs"]
    us = torch.tensor(_us(seed, R), dtype=torch.float64, device=device)
    keys, diag, hops = _table(M, N, device)
    H = lambda v: diag * (us * v) + _kinetic(hops, v)  # noqa: E731
    rng = np.random.default_rng(seed + 1)
    if kind == "product":
        v = torch.from_numpy(rng.standard_normal((len(keys), R))).to(device)
        ybar = torch.from_numpy(rng.standard_normal((len(keys), R))).to(device)
        ky = _kinetic(hops, ybar)
        return {"y": H(v).cpu().numpy(), "vbar": (diag * (us * ybar) + ky).cpu().numpy(),
                "ubar": (ybar * diag * v).sum(0).cpu().numpy(), "tbar": (v * ky).sum(0).cpu().numpy()}
    start = np.zeros((1, M), dtype=np.int64)
    start[0] = rimu.near_uniform(N, M).onr
    v = torch.zeros((len(keys), R), dtype=torch.float64, device=device)
    v[int(np.searchsorted(keys, _bits(start))[0])] = 1.0
    if kind == "ground":
        # Lanczos with 64-bit sums to well past convergence of the lowest value
        a, b, prev, beta = [], [], torch.zeros_like(v), torch.zeros(R, dtype=torch.float64, device=device)
        for _ in range(min(160, len(keys))):
            w = H(v) - beta * prev
            alpha = (v * w).sum(0)
            w -= alpha * v
            a.append(alpha.cpu().numpy())
            prev, beta = v, w.square().sum(0).sqrt()
            b.append(beta.cpu().numpy())
            v = w / beta
        a, b = np.array(a), np.array(b)
        low = [np.linalg.eigvalsh(np.diag(a[:, i]) + np.diag(b[:-1, i], 1) + np.diag(b[:-1, i], -1))[0]
               for i in range(R)]
        return {"energy": np.array(low)}
    dtau, path = case["dtau"], [v]
    for _ in range(case["steps"]):
        path.append(path[-1] - dtau * H(path[-1]))
    v = path[-1]
    vv = (v * v).sum(0)
    kv = _kinetic(hops, v)
    hf_u, hf_t = (v * diag * v).sum(0) / vv, (v * kv).sum(0) / vv
    energy = us * hf_u + hf_t
    lam = 2 * (H(v) - energy * v) / vv
    grad_u, grad_t = hf_u.clone(), hf_t.clone()
    for x in reversed(path[:-1]):
        kl = _kinetic(hops, lam)
        grad_u -= dtau * (lam * diag * x).sum(0)
        grad_t -= dtau * (x * kl).sum(0)
        lam = lam - dtau * (diag * (us * lam) + kl)
    out = {"energy": energy, "grad_u": grad_u, "grad_t": grad_t, "hf_u": hf_u, "hf_t": hf_t, "v": v}
    return {k: x.cpu().numpy() for k, x in out.items()}
