"""The row kernel (one workgroup per system, units of rows over its threads)
against the oracle at the edges of its layout: rows of more terms than a
thread takes, rows nothing reads, one to eight units per thread, chains just
above the automatic choice's line, per-step outputs, both precisions, both
adjoints; its stored path against recomputed segments bitwise, and the solvers
against each other.  FP64 within 1e-10 per output (``oracle.parity``), FP32
within the tolerances of ``test_gpu_forward`` (1e-4 of the FP32 oracle)."""
import numpy as np
import pytest

from oracle import parity as PAR
from pasif_amd import adjoint as ADJ
from pasif_amd import workloads as W
from pasif_amd.PASIf import coo_tensor
from tests.helpers import dense_chain, random_system, side_by_side
from tests.test_gpu_adjoint import oracle_gradient
from tests.test_gpu_exact_adjoint import oracle_exact
from tests.test_gpu_forward import oracle_run, rel_err

pytestmark = pytest.mark.gpu


def _sizes(w):
    return [m.shape[0] for m in w.vecM]


def _check(g, ref, sizes, what):
    r = PAR.report(g, np.asarray(ref).reshape(-1), sizes)
    assert r.max_rel < PAR.TOL64, (what, r.as_dict())


def _coo(t):
    c = coo_tensor(list(t.dimensions))
    c.val, c.indices = np.asarray(t.val, dtype=np.float64), np.asarray(t.indices)
    return c


def _dense(n, seed):
    """Random coupled systems with rows of many terms (more than a thread
    takes), rows nothing reads and forces on several rows."""
    rng = np.random.default_rng(seed)
    cols = [[] for _ in range(7)]
    for k in range(2):
        M, B, K, G, L, _, f, q0 = random_system(rng, n + 3 * k, nnzA=14 * n, nG=9 * n, nL=3 * n,
                                                scale=0.02)
        for c, x in zip(cols, (M, B, K, _coo(G), _coo(L), f, q0)):
            c.append(x)
    exc = rng.normal(size=(2, 40))
    return W.Workload("dense", *cols, exc, 200, 150, exc_of_system=np.array([1, 0]),
                      steps_of_system=np.array([150, 97]), interp=W.linear_interp_matrix(5))


@pytest.mark.parametrize("n,kernel", [(2, "big"), (65, "big"), (150, "auto")])
def test_rows_dense_couplings(n, kernel):
    print(f"[gpu case] rows: dense couplings, {n} rows", flush=True)
    w = _dense(n, n)
    J = ADJ.energy_gradient_inputs(w, [[("K", 0, int(k.col[0]))] if int(k.row[0]) == 0 else
                                       [("Lambda", 0), ("Gamma", 1)] for k in w.vecK])
    p = W.make_solver(w)
    p.setKernel(kernel)
    p.setJacobian(*J.as_args())
    assert p.kernelInfo()["kernel"] == "big"
    q = p.getAmplitudes()
    _check(q, oracle_run(w).q, _sizes(w), "forward")
    g = p.getGradient()                       # automatic interval: stored path
    _check(g, oracle_gradient(w, J, 64), J.sizes, "reference adjoint")
    for k in (1, 7, 150):
        p.setTuning(checkpoint_every=k)
        np.testing.assert_array_equal(p.getGradient(), g)
    p.setAdjointMode("exact")
    x = p.getGradient()
    _check(x, oracle_exact(w, J), J.sizes, "exact adjoint")
    p.setTuning(checkpoint_every=0)
    np.testing.assert_array_equal(p.getGradient(), x)
    p.setSolver("plain")
    np.testing.assert_array_equal(p.getGradient(), x)
    np.testing.assert_array_equal(p.getAmplitudes(), q)
    p.setSolver("graph", steps_per_launch=13, launches_per_graph=3)
    p.setAdjointMode("reference")
    np.testing.assert_array_equal(p.getGradient(), g)


@pytest.mark.parametrize("d,steps", [(65, 130), (255, 70), (256, 20), (520, 12), (1030, 8)])
def test_rows_chains_by_units_per_thread(d, steps):
    print(f"[gpu case] rows: chains of {d} DOF", flush=True)
    w = W.chains(n_systems=3, d=d, steps=steps, steps_per_sample=10)
    w.steps_of_system = np.array([steps, 1, steps - 3])
    w.vecQ0 = [np.random.default_rng(s).normal(0, 0.3, 2 * d + 1) for s in range(3)]
    J = ADJ.energy_gradient_inputs(w)
    p = W.make_solver(w)
    p.setKernel("big")            # a lane group of 64 still holds the 65-DOF chain forward
    p.setJacobian(*J.as_args())
    assert p.kernelInfo()["kernel"] == "big"
    _check(p.getAmplitudes(), oracle_run(w).q, _sizes(w), "forward")
    _check(p.getGradient(), oracle_gradient(w, J, 16), J.sizes, "reference adjoint")
    p.setAdjointMode("exact")
    _check(p.getGradient(), oracle_exact(w, J, 16), J.sizes, "exact adjoint")


def test_rows_trajectory_window_and_fp32():
    print("[gpu case] rows: 70-DOF chains, trajectory, window, FP32, cartesian", flush=True)
    w = W.chains(n_systems=2, d=70, steps=90, steps_per_sample=10)
    w.steps_of_system = np.array([90, 41])
    p = W.make_solver(w)
    tr = p.getTrajectory(saveSteps=7)
    ref = oracle_run(w, save_steps=7, window=20)
    assert rel_err(tr[1:].T, ref.traj.reshape(ref.traj.shape[0], -1)) < 1e-10
    q, mx = p.getMaxAmplitudes(window=20)
    _check(q, ref.q, _sizes(w), "states beside the window")
    _check(mx, ref.maxabs, _sizes(w), "window")
    p.setSolver("plain")
    q2, mx2 = p.getMaxAmplitudes(window=20)
    np.testing.assert_array_equal(q2, q)
    np.testing.assert_array_equal(mx2, mx)
    p.setSolver("persistent")
    p.setPrecision(32)
    assert rel_err(p.getAmplitudes(), oracle_run(w, dtype=np.float32).q, 1e-4) < 1e-4
    w.exc_of_system = w.steps_of_system = None
    p = W.make_solver(w)
    _check(p.getAmplitudes(), oracle_run(w).q, _sizes(w) * 2, "cartesian")


def test_rows_trajectory_and_window_of_a_system_no_lane_layout_holds():
    print("[gpu case] rows: dense couplings, trajectory, window", flush=True)
    w = _dense(150, 150)
    p = W.make_solver(w)
    assert p.kernelInfo()["kernel"] == "big"
    tr = p.getTrajectory(saveSteps=7)
    ref = oracle_run(w, save_steps=7, window=20)
    assert rel_err(tr[1:].T, ref.traj.reshape(ref.traj.shape[0], -1)) < 1e-10
    q, mx = p.getMaxAmplitudes(window=20)
    _check(q, ref.q, _sizes(w), "states beside the window")
    _check(mx, ref.maxabs, _sizes(w), "window")


@pytest.mark.parametrize("kernel", ["auto", "big"])
def test_rows_a_long_chain_beside_a_dense_system(kernel):
    """Instances of one launch that divide LDS differently: a chain of 2,001 DOF
    and a dense system of 150, which do not fit LDS together."""
    print(f"[gpu case] rows: 2001-DOF chain beside a dense 150-DOF system, {kernel}", flush=True)
    w = side_by_side([W.chains(1, 2001, 20, steps_per_sample=10), dense_chain(150, 20)], [12, 20])
    J = ADJ.energy_gradient_inputs(w)
    p = W.make_solver(w)
    p.setKernel(kernel)
    _check(p.getAmplitudes(), oracle_run(w).q, _sizes(w), "forward")
    p.setJacobian(*J.as_args())
    assert p._rowInfo(True)["rows"] == 2
    g = p.getGradient()
    _check(g, oracle_gradient(w, J, 16), J.sizes, "reference adjoint")
    p.setTuning(checkpoint_every=5)
    np.testing.assert_array_equal(p.getGradient(), g)
    p.setAdjointMode("exact")
    _check(p.getGradient(), oracle_exact(w, J, 16), J.sizes, "exact adjoint")
