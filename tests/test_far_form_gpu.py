"""The far form of the induction kernels (angle / h as a polynomial of h^2 / B^2 for points at
least four segment lengths away, decided by the boxes of a wave's points and of a group of lines)
against the oracle, at the sizes where its rule can go wrong: groups and waves that are partly
near, wakes shorter than a piece of sixteen segments, odd strip counts, a single strip, points on
the extension of the segments (cut off), segments shorter than the cut-off.

Tolerance: the oracle's own rounding of h^2 and of a difference of two atan2 values is what
separates the two (1e-12 of the largest velocity, the bound of the other parity tests)."""

import ctypes as C

import numpy as np
import pytest

from oracle import wake_oracle as WO
from oracle import oracle as O
from pyvl_amd import _lib
from pyvl_amd import geometry as G
from pyvl_amd.cvl import Mesh
from pyvl_amd.device import DeviceArray
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


@pytest.mark.parametrize("n_pts", [1, 63, 64, 65, 127, 128, 129, 200])
@pytest.mark.parametrize("lo,hi", [(2.05, 40.0), (1.9, 2.1), (0.05, 3.0)])
def test_point_velocity_near_and_far_lines(n_pts, lo, hi):
    """Sums whose waves are all far from a line, all at the border of the rule (two lengths from the
    midpoint), or near: points around the lines of a small mesh with one zero-length line (a
    collapsed panel edge), some of them on a line's extension (cut off)."""
    rng = np.random.default_rng(n_pts)
    pos, el, _ = G.flat_wing(3, 2, 3.0, 2.0)
    pos[:, 2] += 0.05 * rng.normal(size=pos.shape[0])
    pos[el[1][1]] = pos[el[1][0]]
    m, t = Mesh(pos.shape[0], el), O.mesh_from_elements(pos.shape[0], el)
    e = rng.integers(0, len(el), n_pts)
    a, b = (pos[np.array([el[i][k] for i in e])] for k in (2, 3))
    d = rng.normal(size=(n_pts, 3))
    r = rng.uniform(lo, hi, (n_pts, 1)) * np.linalg.norm(b - a, axis=1, keepdims=True)
    pts = 0.5 * (a + b) + r * d / np.linalg.norm(d, axis=1, keepdims=True)
    pts[::7] = (b + lo * (b - a))[::7]
    pts = np.ascontiguousarray(pts)
    circ = rng.normal(size=m.n_surfaces)
    want = O.point_velocity(t, pos, circ, pts, 1e-6)
    got = m.point_velocity(1e-6, pos, circ, pts)
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))


def test_noalloc_holds_meshes_near_its_scratch_limit():
    """Line records alone near the fixed scratch: the smaller chunk count is taken, by both entry
    points, and the call is not refused."""
    _lib.call("pvl_init", 0)
    pos, el = G.uv_sphere(512, 300, sigma=1e-4, seed=1)
    m, rng = Mesh(pos.shape[0], el), np.random.default_rng(2)
    assert 88 * m.n_lines + 24 * 512 * 1000 > (32 << 20) > 88 * m.n_lines + 24 * 128 * 1000
    pts = DeviceArray.from_numpy(rng.normal(0.0, 1.5, (1000, 3)))
    dpos, circ = DeviceArray.from_numpy(pos), DeviceArray.from_numpy(rng.normal(size=m.n_surfaces))
    out = []
    for name in ("pvl_point_velocity", "pvl_point_velocity_noalloc"):
        v = DeviceArray((1000, 3))
        _lib.check(getattr(_lib.load(), name)(m._device(), C.c_double(1e-6), dpos.cptr, circ.cptr, C.c_uint(1000),
                                              pts.cptr, v.cptr, C.c_int(0), C.c_int(_lib.PVL_FP64)), name)
        out.append(v.numpy())
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n_span,n_chord", [(1, 1), (9, 7), (64, 31), (32, 64), (59, 50)])
def test_assembly_at_every_run_length(n_span, n_chord):
    """The normal-reduced matrix on both sides of the surface counts where the groups per wave change
    (2,048 and about 2,900), a single surface, and a last group that is not full."""
    rng = np.random.default_rng(n_span)
    pos, el, _ = G.flat_wing(n_span, n_chord, 8.0, 1.0)
    pos[:, 2] += 0.1 * np.sin(3.0 * pos[:, 0]) + 0.002 * rng.normal(size=pos.shape[0])
    m, t = Mesh(pos.shape[0], el), O.mesh_from_elements(pos.shape[0], el)
    nrm, cps = O.surface_normal(t, pos), O.surface_center(t, pos)
    rows = rng.permutation(m.n_surfaces)[:200]
    c, n = np.ascontiguousarray(cps[rows]), np.ascontiguousarray(nrm[rows])
    got, want = m.induction_matrix3(1e-6, pos, c, n), O.induction_matrix3(t, pos, c, n, 1e-6)
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("n_pts", [65, 3968, 3969, 4100])
def test_point_velocity_fp32_points_per_lane(n_pts):
    """FP32 on both sides of the point count where a lane takes two points (32 chunks of lines: 32
    blocks of 128), against FP64: a pair's angle is a few 2^-24 off, a sum of terms of either sign some
    ten times that, so 1e-5 of the largest velocity."""
    pos, el = G.uv_sphere(64, 64, sigma=1e-3, seed=3)
    m, rng = Mesh(pos.shape[0], el), np.random.default_rng(n_pts)
    assert (m.n_lines + 255) // 256 == 32
    pts, circ = rng.normal(0.0, 1.5, (n_pts, 3)), rng.normal(size=m.n_surfaces)
    want = m.point_velocity(1e-6, pos, circ, pts)
    got = m.point_velocity(1e-6, pos, circ, pts, precision=_lib.PVL_FP32)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))
