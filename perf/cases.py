"""Performance cases: what a user of the framework has it do, through its public
entry points, over the range of sizes, directions, precisions and kernel
families.  A case is a dict of plain values; ``prepare`` makes the solver with
its systems loaded, ``run`` is one call of the solver as a program makes it,
``work`` the bytes and operations that call cannot do without and ``exact`` the
same result in 64-bit torch, written from the equations alone.

Kinds of case (``case["kind"]``):

* ``duffing``: forced Duffing oscillators, zero-order hold, final states and
  the largest amplitude over a window of last steps (a frequency response);
* ``two_dof``: many two-DOF systems forward, each with its own excitation (a
  parameter sweep; the library's headline workload);
* ``sweep``: copies of one small system against every signal of an excitation
  set (the Cartesian product), final states or the recorded trajectory;
* ``batch``: chains of uneven size and step count forward in one call;
* ``gradient``: the energy gradient (forward and adjoint) of chains;
* ``differentiate``: the autograd function, forward and backward, with
  coefficients as the parameters;
* ``serve``: requests of registered systems through the pool.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from pasif_amd import adjoint as ADJ
from pasif_amd import autograd as AG
from pasif_amd import serving as SRV
from pasif_amd import workloads as W

SIZES = (1, 2, 4, 8, 16, 32, 64)


def listed():
    return [
        # one oscillator, a short run: what a single call costs
        {"name": "duffing_1", "kind": "duffing", "n": 1, "steps": 1000, "window": 200},
        # a frequency response: 64 oscillators, one frequency each
        {"name": "duffing_64", "kind": "duffing", "n": 64, "steps": 10000, "window": 2000},
        # a parameter sweep of two-DOF systems (the library's headline workload)
        {"name": "two_dof_4096", "kind": "two_dof", "n": 4096, "steps": 20000},
        # copies of a small system against a set of 50 excitations, final states
        {"name": "sweep_16x50", "kind": "sweep", "n": 16, "dof": 4, "signals": 50,
         "steps": 16000, "save": 0},
        # the same with the trajectory recorded (an odd count of copies)
        {"name": "trajectory_33x50", "kind": "sweep", "n": 33, "dof": 4, "signals": 50,
         "steps": 8000, "save": 16},
        # a batch of uneven sizes and step counts, single precision
        {"name": "batch_f32", "kind": "batch", "n": 6000, "tmin": 1000, "tmax": 10000,
         "bits": 32},
        # the energy gradient of many 16-DOF chains (the differentiation workload)
        {"name": "gradient_16dof", "kind": "gradient", "n": 8192, "dof": 16, "tmin": 10000,
         "tmax": 10000, "bits": 64},
        # the energy gradient of a batch of uneven sizes and step counts
        {"name": "gradient_batch", "kind": "gradient", "n": 4096, "dof": 0, "tmin": 1000,
         "tmax": 10000, "bits": 64},
        # an optimisation step: autograd forward and backward
        {"name": "differentiate", "kind": "differentiate", "n": 777, "dof": 16, "steps": 3000},
        # chains longer than the lanes of a wave
        {"name": "gradient_150dof", "kind": "gradient", "n": 48, "dof": 150, "tmin": 1000,
         "tmax": 1000, "bits": 64},
        # single large systems
        {"name": "gradient_2001dof", "kind": "gradient", "n": 2, "dof": 2001, "tmin": 300,
         "tmax": 300, "bits": 64},
        # requests of registered systems admitted, advanced and collected
        {"name": "serve_60", "kind": "serve", "n": 60, "systems": 32, "tmin": 1000,
         "tmax": 10000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["duffing", "two_dof", "sweep", "trajectory", "batch", "gradient",
                       "gradient_batch", "gradient_long", "gradient_large", "differentiate",
                       "serve"])
    if kind == "duffing":
        steps = _log_int(rng, 1000, 10000)
        return {"kind": kind, "n": _log_int(rng, 1, 2048), "steps": steps,
                "window": rng.randint(1, steps // 2)}
    if kind == "two_dof":
        return {"kind": kind, "n": _log_int(rng, 100, 4096), "steps": _log_int(rng, 2000, 20000)}
    if kind in ("sweep", "trajectory"):
        return {"kind": "sweep", "n": _log_int(rng, 1, 33), "dof": rng.choice([1, 2, 3, 4, 5, 6]),
                "signals": rng.randint(1, 50), "steps": _log_int(rng, 1000, 8000),
                "save": rng.randint(8, 64) if kind == "trajectory" else 0}
    if kind == "batch":
        tmax = _log_int(rng, 2000, 10000)
        return {"kind": kind, "n": _log_int(rng, 300, 6000), "tmin": rng.randint(500, 1500),
                "tmax": tmax, "bits": rng.choice([32, 64])}
    if kind == "gradient":
        t = _log_int(rng, 1000, 8000)
        return {"kind": kind, "n": _log_int(rng, 300, 6000), "dof": rng.randint(6, 16),
                "tmin": t, "tmax": t, "bits": rng.choice([64, 64, 32])}
    if kind == "gradient_batch":
        return {"kind": "gradient", "n": _log_int(rng, 300, 4096), "dof": 0,
                "tmin": rng.randint(500, 1500), "tmax": _log_int(rng, 2000, 10000), "bits": 64}
    if kind == "gradient_long":
        t = _log_int(rng, 200, 1000)
        return {"kind": "gradient", "n": _log_int(rng, 4, 48), "dof": _log_int(rng, 70, 200),
                "tmin": t, "tmax": t, "bits": rng.choice([64, 64, 32])}
    if kind == "gradient_large":
        t = _log_int(rng, 100, 300)
        return {"kind": "gradient", "n": rng.randint(1, 3), "dof": _log_int(rng, 700, 2001),
                "tmin": t, "tmax": t, "bits": 64}
    if kind == "differentiate":
        return {"kind": kind, "n": _log_int(rng, 50, 777), "dof": rng.randint(4, 16),
                "steps": _log_int(rng, 500, 3000)}
    return {"kind": kind, "n": rng.randint(5, 60), "systems": rng.randint(4, 32),
            "tmin": rng.randint(500, 1500), "tmax": _log_int(rng, 2000, 10000)}


# ------------------------------------------------------------------ inputs
def _workload(case, seed):
    """The systems, excitations and step counts of a case."""
    kind = case["kind"]
    if kind == "duffing":
        w = W.duffing(n_systems=case["n"], steps=case["steps"], seed=seed)
        return w
    if kind == "two_dof":
        return W.two_dof(n_systems=case["n"], steps=case["steps"], seed=seed)
    if kind == "sweep":
        t = case["steps"]
        w = W.heterogeneous(case["n"], tmin=t, tmax=t, seed=seed, n_signals=case["signals"],
                            dof_choices=[case["dof"]], dof_probs=[1.0])
        w.exc_of_system, w.steps_of_system, w.numsteps = None, None, t
        return w
    if kind == "differentiate":
        t = case["steps"]
        w = W.heterogeneous(case["n"], tmin=t, tmax=t, seed=seed, dof_choices=[case["dof"]],
                            dof_probs=[1.0])
        w.steps_of_system, w.numsteps = None, t
        return w
    return _batch(case, seed)


def _batch(case, seed):
    """Chains of one size (``dof``) or of the batch's sizes in its proportions
    (``dof`` 0), every size's count and the step counts being the case's and
    the coefficients and signals the seed's."""
    n, t0, t1 = case["n"], case["tmin"], case["tmax"]
    one = case.get("dof", 0)
    fixed = np.random.default_rng([n, one, t0, t1])
    dofs = np.full(n, one) if one else np.sort(fixed.choice(SIZES, size=n, p=W.DOF_PROBS))
    parts = [W.heterogeneous(int((dofs == d).sum()), tmin=t0, tmax=t0, n_signals=1,
                             seed=[seed, int(d)], dof_choices=[int(d)], dof_probs=[1.0])
             for d in np.unique(dofs)]
    order = fixed.permutation(n)
    steps = np.exp(fixed.uniform(np.log(t0), np.log(t1), n)).astype(np.int64)
    rng = np.random.default_rng([seed, 1])
    vecs = []
    for name in ("vecM", "vecB", "vecK", "vecGamma", "vecLambda", "vecForce", "vecQ0"):
        every = [x for p in parts for x in getattr(p, name)]
        vecs.append([every[i] for i in order])
    bank = SRV.signal_bank(rng, 64, t1)
    return W.Workload("chains", *vecs, bank, 1000, t1 if t0 == t1 else int(steps.max()),
                      exc_of_system=rng.integers(0, 64, n),
                      steps_of_system=None if t0 == t1 else steps,
                      interp=W.linear_interp_matrix(10))


def _stiffness_params(w):
    """Parameters of an optimisation: every system's K diagonal and Lambda."""
    out = []
    for s in range(w.n_systems):
        d = (w.vecM[s].shape[0] - 1) // 2
        out.append([("K", d + i, i) for i in range(d)] + [("Lambda", i) for i in range(d)])
    return out


def _requests(case, seed):
    """The served library and its signals (the seed's) and the requests
    (library positions, signals and steps: the case's)."""
    lib = SRV.SystemLibrary(seed=seed)
    bank = SRV.signal_bank(np.random.default_rng([seed, 7]), 16, case["tmax"])
    stream = SRV.RequestStream(lib, case["n"], case["n"], 16, tmin=case["tmin"],
                               tmax=case["tmax"], max_systems=case["systems"])
    return lib, bank, [stream[k] for k in range(case["n"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        lib, bank, reqs = _requests(case, seed)
        pool = SRV.Pool(checkpoint_every=256, steps_per_tick=5000, hbm_budget=20e9)
        pool.set_bank(bank, 1000, W.linear_interp_matrix(10))
        pool.register_library(lib)
        return {"case": case, "pool": pool, "requests": reqs}
    w = _workload(case, seed)
    if kind == "differentiate":
        prob = AG.DifferentiableProblem(w, _stiffness_params(w))
        q0 = torch.tensor(prob.q00(), requires_grad=True)
        theta = torch.tensor(prob.theta0(), requires_grad=True)
        return {"case": case, "problem": prob, "q0": q0, "theta": theta}
    p = W.make_solver(w)
    if kind == "gradient":
        p.setJacobianBlocks(ADJ.energy_gradient_blocks(w))
    if case.get("bits", 64) == 32:
        p.setPrecision(32)
    return {"case": case, "solver": p}


# --------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "duffing":
        return state["solver"].getMaxAmplitudes(case["window"])
    if kind == "sweep" and case["save"]:
        return state["solver"].getTrajectory(case["save"])
    if kind in ("two_dof", "sweep", "batch"):
        return state["solver"].getAmplitudes()
    if kind == "gradient":
        return state["solver"].getGradient()
    if kind == "differentiate":
        q0, theta = state["q0"], state["theta"]
        q0.grad = theta.grad = None
        q = AG.rk4_solve(state["problem"], q0, theta)
        (0.5 * (q * q).sum()).backward()
        return q.detach(), q0.grad, theta.grad
    pool = state["pool"]
    groups = [g for g in ([r for r in state["requests"] if r.adjoint],
                          [r for r in state["requests"] if not r.adjoint]) if g]
    jobs = [pool.submit_group(g) for g in groups]
    while not all(pool.finished(j) for j in jobs):
        pool.tick(wait=True)
    pool.collect_groups(jobs, groups)
    reqs = [r for g in groups for r in g]
    return (np.concatenate([r.result for r in reqs]),
            np.concatenate([r.grad for r in reqs if r.adjoint] or [np.zeros(0)]))


# ------------------------------------------------ equations, term by term
class _Terms:
    """Every term of a batch's right-hand side, flat over all systems:
    ``kinds[k] = (out row, factor rows [k + 1], coefficient)`` for products
    of k + 1 states, the forced rows, and per row its system's step count."""

    def __init__(self, systems, steps, exc):
        rows = [[], [], []]
        self.par = []                    # (system, forward row, factor rows, scale) per parameter
        force, q0, row_steps, row_exc = [], [], [], []
        off = 0
        self.offsets = [0]
        for s, (m, A, G, L, f, q, params) in enumerate(systems):
            n = len(m)
            D = -1.0 / m
            for kind, (ix, v) in enumerate((A, G, L)):
                rows[kind].append((ix + off, D[ix[:, 0]] * v))
            for p in params:
                self.par.append((s, off + p[0], [off + c for c in p[1]], D[p[0]]))
            force.append(-D * f)
            q0.append(q)
            row_steps.append(np.full(n, steps[s]))
            row_exc.append(np.full(n, exc[s]))
            off += n
            self.offsets.append(off)
        self.n = off
        self.kinds = [(np.concatenate([r[0] for r in rk]), np.concatenate([r[1] for r in rk]))
                      for rk in rows]
        self.force, self.q0 = np.concatenate(force), np.concatenate(q0)
        self.row_steps, self.row_exc = np.concatenate(row_steps), np.concatenate(row_exc)
        self.steps = int(self.row_steps.max())

    def counts(self):
        """Terms of each system by number of factors, its rows and forced rows."""
        sysof = np.repeat(np.arange(len(self.offsets) - 1), np.diff(self.offsets))
        S = len(self.offsets) - 1
        per = [np.bincount(sysof[ix[:, 0]], minlength=S) for ix, _ in self.kinds]
        forced = np.bincount(sysof[np.flatnonzero(self.force)], minlength=S)
        npar = np.zeros((S, 2), dtype=np.int64)
        for s, _, fs, _ in self.par:
            npar[s, 0 if len(fs) == 1 else 1] += 1
        return per, forced, np.diff(self.offsets), npar


def _mat(*ms):
    ms = [m.tocoo() for m in ms]
    ix = np.stack([np.concatenate([m.row for m in ms]), np.concatenate([m.col for m in ms])], 1)
    return ix.astype(np.int64), np.concatenate([m.data for m in ms])


def _tens(t, order):
    return (np.asarray(t.indices, dtype=np.int64).reshape(-1, order),
            np.asarray(t.val, dtype=np.float64).reshape(-1))


def _energy_params(K, L, n):
    """Rows and factors of the K-diagonal and Lambda parameters of a chain."""
    d = (n - 1) // 2
    return [(d + i, [i]) for i in range(d)] + [(int(r[0]), [int(x) for x in r[1:]]) for r in L[0]]


def _terms_of(case, seed):
    """(_Terms, excitations, interpolation rows or None, sample rate) of a case."""
    if case["kind"] == "serve":
        lib, bank, reqs = _requests(case, seed)
        reqs = [r for r in reqs if r.adjoint] + [r for r in reqs if not r.adjoint]
        systems, steps, exc = [], [], []
        for r in reqs:
            for k, t, e in zip(r.keys, r.steps, r.exc_ids):
                y = lib.flat[int(k)]
                A = _mat(_Csr(y.csr, y.n))
                G, L = (np.asarray(y.gamma[0], dtype=np.int64).reshape(-1, 3), y.gamma[1]), \
                    (np.asarray(y.lam[0], dtype=np.int64).reshape(-1, 4), y.lam[1])
                # the library's arrays are scaled by -1/m already
                par = _energy_params(None, L, y.n) if r.adjoint else []
                systems.append((-np.ones(y.n), A, G, L, -np.asarray(y.force), np.asarray(y.q0),
                                par))
                steps.append(int(t))
                exc.append(int(e))
        T = _Terms(systems, steps, exc)
        T.adjoint_systems = np.concatenate([np.full(len(r.keys), r.adjoint) for r in reqs])
        # forces of scaled arrays pass unscaled
        T.force = np.concatenate([np.asarray(lib.flat[int(k)].force) for r in reqs
                                  for k in r.keys])
        return T, bank, W.linear_interp_matrix(10), 1000
    w = _workload(case, seed)
    systems = []
    want = case["kind"] in ("gradient", "differentiate")
    for s in range(w.n_systems):
        m = np.asarray(w.vecM[s].diagonal(), dtype=np.float64)
        L = _tens(w.vecLambda[s], 4)
        systems.append((m, _mat(w.vecB[s], w.vecK[s]), _tens(w.vecGamma[s], 3), L,
                        np.asarray(w.vecForce[s]), np.asarray(w.vecQ0[s]),
                        _energy_params(None, L, len(m)) if want else []))
    S = w.n_systems
    steps = w.steps_of_system if w.steps_of_system is not None else np.full(S, w.numsteps)
    if w.exc_of_system is None:          # every system against every signal
        E = len(w.excitations)
        systems, steps = systems * E, np.tile(steps, E)
        exc = np.repeat(np.arange(E), S)
    else:
        exc = w.exc_of_system
    return _Terms(systems, steps, exc), w.excitations, w.interp, w.sample_rate


class _Csr:
    """Row, column and value arrays of a CSR triple (data, indices, indptr)."""

    def __init__(self, parts, n):
        self.data, self.col, ptr = (np.asarray(x) for x in parts)
        self.row = np.repeat(np.arange(n), np.diff(ptr))

    def tocoo(self):
        return self


# -------------------------------------------------------------------- work
def work(case):
    T, exc, interp, _ = _terms_of(case, 1)
    (a, g, l_), forced, rows, npar = T.counts()
    steps = T.row_steps[np.asarray(T.offsets[:-1])].astype(np.float64)
    fwd = 4 * (2 * a + 3 * g + 4 * l_ + 2 * forced) + 12 * rows
    adj = 4 * (2 * a + 6 * g + 12 * l_ + 3 * npar[:, 0] + 5 * npar[:, 1]) \
        + 12 * (rows + npar.sum(1)) + 2 * rows
    both = np.zeros(len(rows), dtype=bool)
    if case["kind"] in ("gradient", "differentiate"):
        both[:] = True
    elif case["kind"] == "serve":
        both = T.adjoint_systems.astype(bool)
    # the autograd function calls the forward solve and then the adjoint
    again = 2.0 if case["kind"] == "differentiate" else 1.0
    flops = float((steps * (fwd * again + np.where(both, adj, 0))).sum())
    el = 4 if case.get("bits", 64) == 32 else 8
    used = np.unique(T.row_exc)
    data = el * sum(len(v) for _, v in T.kinds) + el * 2 * T.n
    data += el * len(used) * min(exc.shape[1], T.steps + 1)
    data += 8 * (T.n + int(npar.sum()))
    if case.get("save"):
        data += 8 * T.n * (T.steps // case["save"])
    return {"bytes": float(data), "flops": flops}


# ------------------------------------------------------------------- exact
class _Flat:
    """The right-hand side of ``_Terms`` (and its adjoint) on one device."""

    def __init__(self, T, exc, interp, rate):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.T, self.h = T, 1.0 / rate
        ten = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=self.dev)  # noqa: E731
        self.kinds = [([ten(ix[:, c]) for c in range(ix.shape[1])], ten(v)) for ix, v in T.kinds
                      if len(v)]
        self.frow = ten(np.flatnonzero(T.force))
        fr = np.flatnonzero(T.force)
        self.fval, self.fexc = ten(T.force[fr]), ten(T.row_exc[fr].astype(np.int64))
        self.q0, self.rsteps = ten(T.q0), ten(T.row_steps.astype(np.int64))
        self.even = bool((T.row_steps == T.steps).all())
        e = ten(np.asarray(exc, dtype=np.float64))
        L = e.shape[1]
        n = torch.arange(T.steps, device=self.dev)
        zero = torch.zeros(e.shape[0], 2, dtype=e.dtype, device=self.dev)

        def at(i):                       # sample i, 0 from the signal's end on
            return torch.cat([e, zero], 1)[:, torch.clamp(i, max=L)]

        if interp is None:               # e[n] in the first three stages, e[n + 1] in the last
            self.u = [torch.where((k > 0) & (k < L), at(k), torch.zeros((), dtype=e.dtype,
                                                                       device=self.dev))
                      for k in (n, n, n + 1)]
        else:
            m = ten(np.asarray(interp, dtype=np.float64))
            Wd = m.shape[1]
            self.u = []
            for hs in (2 * n, 2 * n + 1, 2 * n + 2):
                i, j = hs // Wd, hs % Wd
                v = m[1][j] * at(i) + m[0][j] * at(i + 1)
                self.u.append(torch.where((i > 0) & (i < L), v, torch.zeros_like(v)))
        self.u = [x.t().contiguous() for x in self.u]

    def rhs(self, y, u):
        k = torch.zeros_like(y)
        for ix, v in self.kinds:
            p = v * y[ix[1]]
            for f in ix[2:]:
                p = p * y[f]
            k.index_add_(0, ix[0], p)
        k.index_add_(0, self.frow, self.fval * u[self.fexc])
        return k

    def stages(self, q, n):
        h = self.h
        u0, u1, u3 = (x[n] for x in self.u)
        k1 = self.rhs(q, u0)
        y2 = q + 0.5 * h * k1
        k2 = self.rhs(y2, u1)
        y3 = q + 0.5 * h * k2
        k3 = self.rhs(y3, u1)
        y4 = q + h * k3
        k4 = self.rhs(y4, u3)
        return y2, y3, y4, k1 + 2 * k2 + 2 * k3 + k4

    def step(self, q, n):
        qn = q + (self.h / 6) * self.stages(q, n)[3]
        return qn if self.even else torch.where(self.rsteps > n, qn, q)

    def forward(self, each=None):
        q = self.q0.clone()
        for n in range(self.T.steps):
            q = self.step(q, n)
            if each is not None:
                each(n, q)
        return q

    def adjoint(self, lam, path, discrete):
        """lambda and the parameters' accumulators at step 0 from ``lam`` at
        the last step; ``path[n]`` is the state after n steps."""
        T = self.T
        terms = []                       # (out, own, set points, coefficient)
        for ix, v in self.kinds:
            for c in range(1, len(ix)):
                terms.append((ix[c], ix[0], [ix[b] for b in range(1, len(ix)) if b != c], v))
        acc = {}
        for j, (_, r, fs, s) in enumerate(T.par):
            acc.setdefault(len(fs), []).append((T.n + j, r, fs, s))
        ten = lambda x: torch.as_tensor(np.asarray(x), device=self.dev)  # noqa: E731
        for nf, rows in acc.items():
            terms.append((ten([r[0] for r in rows]), ten([r[1] for r in rows]),
                          [ten([r[2][b] for r in rows]) for b in range(nf)],
                          ten([r[3] for r in rows])))
        na = T.n + len(T.par)
        sysof = np.repeat(np.arange(len(T.offsets) - 1), np.diff(T.offsets))
        st = T.row_steps[np.asarray(T.offsets[:-1])]
        asteps = ten(np.concatenate([st[sysof], st[np.asarray([p[0] for p in T.par],
                                                              dtype=np.int64)]]).astype(np.int64))
        z = torch.zeros(na, dtype=lam.dtype, device=self.dev)
        z[:T.n] = lam
        h = self.h

        def g(y, x):
            k = torch.zeros_like(y)
            for out, own, fs, v in terms:
                p = v * y[own]
                for f in fs:
                    p = p * x[f]
                k.index_add_(0, out, p)
            return k

        for n in range(T.steps, 0, -1):
            if discrete:
                x1 = path[n - 1]
                x2, x3, x4, _ = self.stages(x1, n - 1)
                m4 = g((h / 6) * z, x4)
                m3 = g((h / 3) * z + h * m4, x3)
                m2 = g((h / 3) * z + 0.5 * h * m3, x2)
                zn = z + (m4 + m3 + m2 + g((h / 6) * z + 0.5 * h * m2, x1))
            else:
                xc, xp = path[n], path[n - 1]
                xm = 0.5 * (xc + xp)
                k1 = g(z, xc)
                k2 = g(z + 0.5 * h * k1, xm)
                k3 = g(z + 0.5 * h * k2, xm)
                zn = z + (h / 6) * (k1 + 2 * k2 + 2 * k3 + g(z + h * k3, xp))
            z = zn if self.even else torch.where(asteps >= n, zn, z)
        return z

    def by_system(self, z):
        """[lambda ; accumulators] of each system in turn."""
        T = self.T
        npar = np.bincount([p[0] for p in T.par], minlength=len(T.offsets) - 1).astype(np.int64)
        po = np.concatenate([[0], np.cumsum(npar)]) + T.n
        idx = np.concatenate([np.concatenate([np.arange(T.offsets[s], T.offsets[s + 1]),
                                              np.arange(po[s], po[s + 1])])
                              for s in range(len(npar))])
        return z.cpu().numpy()[idx]


def exact(case, seed):
    """What ``run`` returns, in 64-bit torch from the equations; None where
    that takes long."""
    kind = case["kind"]
    T, exc, interp, rate = _terms_of(case, seed)
    both = kind in ("gradient", "differentiate")
    # seconds: launches, and the terms' memory traffic
    terms = sum(len(v) * ix.shape[1] for ix, v in T.kinds)
    est = T.steps * 4 * (3 if both else 1) * (1.6e-4 + terms * 3e-10)
    if kind == "serve" or est > 27 or (both and T.steps * T.n > 6e9):
        return None
    F = _Flat(T, exc, interp, rate)
    if kind == "duffing":
        top = torch.zeros_like(F.q0)
        first = T.steps - case["window"]

        def each(n, q):
            if n >= first:
                torch.maximum(top, q.abs(), out=top)

        q = F.forward(each)
        return q.cpu().numpy(), top.cpu().numpy()
    if kind == "sweep" and case["save"]:
        slots = T.steps // case["save"]
        rec = torch.zeros(slots, T.n, dtype=torch.float64, device=F.dev)

        def each(n, q):
            if n % case["save"] == 0 and n // case["save"] < slots:
                rec[n // case["save"]] = q

        F.forward(each)
        out = np.zeros((T.n + 1, slots))
        out[0] = np.arange(slots) * case["save"] / rate
        out[1:] = rec.t().cpu().numpy()
        return out
    if not both:
        return F.forward().cpu().numpy()
    path = torch.empty(T.steps + 1, T.n, dtype=torch.float64, device=F.dev)
    path[0] = F.q0

    def keep(n, q):
        path[n + 1] = q

    q = F.forward(keep)
    if kind == "gradient":
        lam = torch.zeros_like(q)
        lam[torch.as_tensor(np.asarray(T.offsets[1:]) - 1, device=F.dev)] = 1.0
        return F.by_system(F.adjoint(lam, path, False))
    z = F.adjoint(q, path, True).cpu().numpy()
    return q.cpu().numpy(), z[:T.n], z[T.n:]
