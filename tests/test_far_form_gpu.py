"""The far form of the induction kernels (angle / h as a polynomial of h^2 / B^2 for points at
least four segment lengths away, decided by the boxes of a wave's points and of a group of lines)
against the oracle, at the sizes where its rule can go wrong: groups and waves that are partly
near, wakes shorter than a piece of sixteen segments, odd strip counts, a single strip, points on
the extension of the segments (cut off), segments shorter than the cut-off.

Tolerance: the oracle's own rounding of h^2 and of a difference of two atan2 values is what
separates the two (1e-12 of the largest velocity, the bound of the other parity tests)."""

import numpy as np
import pytest

from oracle import wake_oracle as WO
from oracle import oracle as O
from pyvl_amd import geometry as G
from pyvl_amd.cvl import Mesh
from pyvl_amd.solver import FlowConditionsUniform, HeaveFrame, make_wing_wake_solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_span,rows,flat", [(1, 3, False), (5, 17, False), (16, 15, True), (17, 33, False),
                                              (40, 64, True)])
def test_free_wake_step_near_and_far_pieces(n_span, rows, flat):
    """One free-wake step from a wake that is mostly far from itself: straight (every node on the
    extension of its column's streamwise segments) or deformed."""
    dt, vinf = 0.25, np.array([1.0, 0.0, 0.0])
    frame = HeaveFrame(0.1, 0.6)
    sol = make_wing_wake_solver(n_span, 3, 8.0, 1.0, frame, FlowConditionsUniform(*vinf), rows, dt, mode="free")
    w, rng = sol.wake, np.random.default_rng(n_span + rows)
    te = np.asarray(w.bordering_nodes, np.int64).reshape(-1, 2)
    pos = np.empty((te.shape[0], 2, rows + 1, 3))
    r = np.arange(rows + 1)
    pos[...] = sol.p0[te][:, :, None, :]
    pos[..., 0] += r * dt
    if not flat:
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
    g_o, _, _ = WO.step(rows + 2, dt, O.mesh_from_elements(pos0.shape[0], elements), pos0, frame, vinf, 1e-6, ow,
                        free=True)
    g = sol.step().numpy()
    wp, wc = w.state()
    assert np.linalg.norm(g - g_o) <= 1e-12 * np.linalg.norm(g_o)
    # positions move by dt times the velocity: the velocity's bound, scaled
    v = np.max(np.abs((ow.wake_positions[:, :, 1:] - pos[:, :, :-1]) / dt))
    assert np.max(np.abs(wp - ow.wake_positions)) <= dt * 1e-12 * v + 1e-14
    assert np.linalg.norm(wc - ow.circulation) <= 1e-12 * np.linalg.norm(ow.circulation)
