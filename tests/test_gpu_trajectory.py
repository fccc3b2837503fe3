"""The trajectory by rows (transposed on the device) against the solver's own
slot order, exactly: tiles of 32 x 32 values whole, one over and one short,
one slot, one row, both precisions."""
import numpy as np
import pytest

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
