"""The stored path of an adjoint solve is extra: it takes what the solve's own
buffers leave, so a solve whose buffers fit runs however little is left
beside them -- with a path for some waves or for none.  One whose buffers do
not fit runs its lane groups in pieces."""
import numpy as np
import pytest
import torch

from pasif_amd import adjoint as ADJ
from pasif_amd import workloads as W

pytestmark = pytest.mark.gpu


def _leave(nbytes):
    """Tensors that leave about ``nbytes`` of the device's memory free (a large
    one takes a little less off the free memory than its size)."""
    held = []
    while (over := torch.cuda.mem_get_info()[0] - int(nbytes)) > 4 << 20:
        held.append(torch.empty(over, dtype=torch.uint8, device="cuda"))
    return held


def _problem(steps):
    w = W.chains(n_systems=4096, d=16, steps=steps, steps_per_sample=10)
    w.excitations = np.asarray(w.excitations)[:3]
    w.exc_of_system = np.arange(4096) % 3
    return w, W.make_solver(w), ADJ.energy_gradient_inputs(w)


def test_path_takes_what_the_run_buffers_leave():
    steps = 100_000
    print(f"[gpu case] path memory: 4096 16-DOF chains x {steps} steps, little memory free",
          flush=True)
    w, p, J = _problem(steps)
    p.setJacobian(*J.as_args())
    p.setTuning(checkpoint_every=256)     # checkpoints, no path
    ref = p.getGradient()
    del p
    p = W.make_solver(w)
    p.setJacobian(*J.as_args())
    fp = p._runFootprint(True)            # packed and uploaded, nothing run
    # the solve's own buffers take 79 % of what is left free (it may take 80)
    hold = _leave(fp["run"] / 0.79)
    try:
        g = p.getGradient()
        again = p.getGradient()
    finally:
        del hold
        torch.cuda.empty_cache()
    np.testing.assert_array_equal(g, ref)
    np.testing.assert_array_equal(again, ref)


def test_idle_path_memory_makes_way():
    print("[gpu case] path memory: a pool's bank and a trajectory beside idle path memory",
          flush=True)
    from pasif_amd import serving
    w, p, J = _problem(2_000)
    p.setJacobian(*J.as_args())
    g = p.getGradient()
    free = torch.cuda.mem_get_info()[0]
    kept = p._trimMemory()
    assert kept > 1 << 30
    assert torch.cuda.mem_get_info()[0] > free
    assert p._trimMemory() == 0
    np.testing.assert_array_equal(p.getGradient(), g)   # takes it anew
    hold = _leave(256 << 20)
    try:
        pool = serving.Pool()
        pool.set_bank(np.zeros((64, 1 << 20)), 1000, None)    # 512 MiB of 256 free
        pool.close()
        assert p._trimMemory() == 0
        # a path from what is left now
        np.testing.assert_array_equal(p.getGradient(), g)
    finally:
        del hold
        torch.cuda.empty_cache()


def test_trajectory_rows_with_little_memory_left():
    print("[gpu case] trajectory rows, 40 MiB beside a trajectory of 130", flush=True)
    w = W.two_dof(n_systems=4096, steps=2000)
    p = W.make_solver(w)
    ref = p.getTrajectory(saveSteps=2)                  # 131 MB, kept by the handle
    del p
    p = W.make_solver(w)
    p.getAmplitudes()
    hold = _leave(180 << 20)
    try:
        tr = p.getTrajectory(saveSteps=2)
    finally:
        del hold
        torch.cuda.empty_cache()
    np.testing.assert_array_equal(tr, ref)


def test_solve_in_pieces_when_memory_is_short():
    print("[gpu case] 4096 16-DOF chains x 30000 steps in pieces", flush=True)
    w, p, J = _problem(30_000)
    w.steps_of_system = np.random.default_rng(0).integers(1, 30_001, 4096)
    w.steps_of_system[::2] = 30_000
    p = W.make_solver(w)
    p.setJacobian(*J.as_args())
    ref = p.getGradient()
    del p
    p = W.make_solver(w)
    p.setJacobian(*J.as_args())
    fp = p._runFootprint(True)
    hold = _leave(fp["run"] * 0.9)
    try:
        g = p.getGradient()
        again = p.getGradient()
        p.setSolver("graph", steps_per_launch=9_000, launches_per_graph=4)
        graph = p.getGradient()
    finally:
        del hold
        torch.cuda.empty_cache()
    np.testing.assert_array_equal(g, ref)
    np.testing.assert_array_equal(again, ref)
    np.testing.assert_array_equal(graph, ref)


def test_handles_of_several_threads_share_the_path_memory():
    print("[gpu case] path memory: three threads, four gradients each, trims between", flush=True)
    import threading
    cases = []
    for n, d, steps in ((512, 16, 900), (64, 4, 2500), (3, 300, 60)):
        w = W.chains(n_systems=n, d=d, steps=steps, steps_per_sample=10, seed=n)
        J = ADJ.energy_gradient_inputs(w)
        p = W.make_solver(w)
        p.setJacobian(*J.as_args())
        cases.append((p, p.getGradient()))
    bad = []

    def run(k):
        p, ref = cases[k]
        for i in range(4):
            if not np.array_equal(p.getGradient(), ref):
                bad.append((k, i))
            if k == i % 3:
                p._trimMemory()

    threads = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
