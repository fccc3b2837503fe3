"""The trajectory by rows (transposed on the device) against the solver's own
slot order, exactly: tiles of 32 x 32 values whole, one over and one short,
one slot, one row, both precisions."""
import ctypes as C

import numpy as np
import pytest

from pasif_amd import adjoint as ADJ
from pasif_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,steps,save,bits", [(1, 70, 70, 64), (8, 64, 2, 64), (11, 66, 2, 64),
                                               (13, 31, 1, 32), (43, 99, 3, 32), (200, 40, 7, 64)])
def test_trajectory_rows_are_the_slots_transposed(n, steps, save, bits):
    print(f"[gpu case] trajectory rows: {n} systems, {steps} / {save}, FP{bits}", flush=True)
    w = W.two_dof(n_systems=n, steps=steps)
    p = W.make_solver(w)
    p.setPrecision(bits)
    rows = p.getTrajectory(save)
    slots = p._getTrajectory(save).reshape(steps // save, 4 * n)
    np.testing.assert_array_equal(rows[1:], slots.T)
    np.testing.assert_array_equal(rows[0], np.arange(steps // save) * save / w.sample_rate)


@pytest.mark.parametrize("window,save", [(1, 0), (16, 17), (29, 3), (33, 16), (1000, 1)])
@pytest.mark.parametrize("even", [True, False])
def test_window_and_saved_steps_are_the_states_of_every_step(even, window, save):
    """Steps of the window, saved steps and the others run in loops of their
    own: the amplitudes and the saved states are those of the states after
    every step, for windows that begin inside a chunk of samples, before the
    first step and at a different step in each lane of a wave."""
    print(f"[gpu case] window {window}, save {save}, even {even}", flush=True)
    n = 70
    w = W.duffing(n_systems=n, steps=50)
    steps = np.full(n, 50)
    if not even:
        steps = np.arange(n) % 50 + 1
        w.steps_of_system = steps
    p = W.make_solver(w)
    per = w.vecM[0].shape[0]
    every = p._getTrajectory(1).reshape(-1, per * n)
    q, mx = p.getMaxAmplitudes(window=window)
    rows = np.repeat(np.arange(n), per)
    for r in range(per * n):
        s = steps[rows[r]]
        assert q[r] == every[s - 1, r], r
        assert mx[r] == np.abs(every[max(0, s - window):s, r]).max(), r
    if save:
        saved = p._getTrajectory(save).reshape(-1, per * n)
        np.testing.assert_array_equal(saved, every[::save][:saved.shape[0]])


def test_a_buffer_too_small_says_what_is_needed():
    """A solve into a buffer too small is refused with the length it needs, and
    its amplitude window is there all the same."""
    print("[gpu case] output buffers too small", flush=True)
    w = W.chains(3, 2, 40, steps_per_sample=10)
    p = W.make_solver(w)
    p.setJacobian(*ADJ.energy_gradient_inputs(w).as_args())
    q, mx = p.getMaxAmplitudes(window=9)
    small = np.full(4, 7.0)
    buf = small.ctypes.data_as(C.POINTER(C.c_double))
    p._setAmplitudeWindow(5)
    n = C.c_size_t(0)
    lib, h = p._pl, p._h
    assert lib.pasif_get_amplitudes(h, buf, 4, C.byref(n)) == 1 and n.value == q.size
    five = np.empty(q.size)
    assert lib.pasif_get_max_amplitudes(h, five.ctypes.data_as(C.POINTER(C.c_double)), q.size,
                                        None) == 0
    p._setAmplitudeWindow(0)
    np.testing.assert_array_equal(five, p.getMaxAmplitudes(window=5)[1])
    for f in (lib.pasif_get_trajectory, lib.pasif_get_trajectory_rows):
        n.value = 0
        assert f(h, 8, buf, 4, C.byref(n)) == 1 and n.value == 5 * q.size
    n.value = 0
    g = p.getGradient()
    assert lib.pasif_get_gradient(h, 0, buf, 4, C.byref(n)) == 1 and n.value == g.size
    np.testing.assert_array_equal(small, 7.0)
