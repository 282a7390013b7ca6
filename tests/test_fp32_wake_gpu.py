"""Free-wake steps in the FP32 mode, whose self-induction splits a chunk of pieces over a workgroup's
waves, against the oracle: fewer pieces than waves, points that do not fill a block of 128, several
blocks and chunks.

Tolerance: a pair's angle is a few 2^-24 off, and a sum of terms of either sign some ten times that:
1e-5 of the largest velocity, so dt times that for the positions, which are what the self-induction moves."""

import numpy as np
import pytest

from oracle import oracle as O
from oracle import wake_oracle as WO
from pyvl_amd import _lib
from pyvl_amd import geometry as G
from pyvl_amd.solver import FlowConditionsUniform, HeaveFrame, make_wing_wake_solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_span,rows", [(1, 2), (1, 40), (5, 17), (16, 15), (31, 64), (40, 70)])
def test_fp32_free_wake_step(n_span, rows):
    dt, vinf = 0.25, np.array([1.0, 0.0, 0.0])
    frame = HeaveFrame(0.1, 0.6)
    sol = make_wing_wake_solver(n_span, 3, 8.0, 1.0, frame, FlowConditionsUniform(*vinf), rows, dt, mode="free",
                                induction_precision=_lib.PVL_FP32)
    w, rng = sol.wake, np.random.default_rng(n_span + rows)
    te = np.asarray(w.bordering_nodes, np.int64).reshape(-1, 2)
    r = np.arange(rows + 1)
    pos = np.empty((te.shape[0], 2, rows + 1, 3))
    pos[...] = sol.p0[te][:, :, None, :]
    pos[..., 0] += r * dt
    pos[..., 2] += 0.2 * np.sin(0.7 * pos[..., 1] + 0.3 * r) * (r > 0)
    circ = rng.normal(size=(te.shape[0], rows))
    d = w.save()
    d.update(wake_positions=pos, circulation=circ, step_count=rows + 2, current_time=(rows + 1) * dt)
    w.set_state(d)
    sol.iteration = rows + 2
    pos0, elements, _ = G.flat_wing(n_span, 3, 8.0, 1.0)
    ow = WO.OracleWake(w.bordering_nodes, w.shedding_lines, w.adjacent_surfaces, 1e-6, 0.0, rows)
    ow.wake_positions[...], ow.circulation[...] = pos, circ
    ow.step_count, ow.current_time = rows + 2, (rows + 1) * dt
    WO.step(rows + 2, dt, O.mesh_from_elements(pos0.shape[0], elements), pos0, frame, vinf, 1e-6, ow, free=True)
    sol.step()
    wp, _ = w.state()
    v = np.max(np.abs((ow.wake_positions[:, :, 1:] - pos[:, :, :-1]) / dt))
    assert np.max(np.abs(wp - ow.wake_positions)) <= dt * 1e-5 * v
