"""Large solids in the soft step: the extrapolation's fronts where the box of
target cells does not fit one workgroup's LDS.

* nz = 572, r_ball = 0.39: a solid of 223 cells' radius, below the 224 from
  which fronts are launches: the walk runs over the list of words in global
  memory;
* nz = 640, r_ball = 0.4, zone of 16 cells instead of 8: more fronts than the
  twelve launches, one workgroup takes the others in global memory;
* a batch of both sizes beside small cases, zones of 16 cells: the launches
  serve all of them (one workgroup in LDS takes the small cases' last
  fronts; nz = 64 lists more cells than it keeps factors of).

Bar: from the GPU's own velocity and dt the oracle's reference-map ENO3, pin,
reinit and extrapolation give the same eta and phi bit for bit.  And a step of
a large solid costs little more than one of a small solid on the same grid
(bars between the two figures measured, in parentheses)."""
import ctypes
import time

import numpy as np
import pytest

from oracle import kernels as K
from oracle.drivers import SoftSphereCase
from oracle.reinit import distance

pytestmark = pytest.mark.gpu


def check_map(case, dt, nz, r_ball, G=1.0, zone=None):
    cpu = SoftSphereCase(grid_size_z=nz, r_ball=r_ball, G=G, solver="exact")
    dx = cpu.dx
    zone = cpu.extrap_zone if zone is None else zone
    u_z, u_r = (np.asarray(u, dtype=np.float64) for u in case.velocity())
    K.advect_refmap_via_eno3(cpu.eta1, cpu.eta2, u_z, u_r, dt, dx)
    pinned = -np.sqrt((cpu.eta1 - cpu.Z_cm) ** 2 + (cpu.eta2 - cpu.R_cm) ** 2) + r_ball
    phi = np.where(cpu.ball_phi > -3 * dx, pinned, cpu.ball_phi)
    d, masked = distance(phi, dx, zone)
    phi = np.where(masked, phi, d)
    assert np.array_equal(case.phi(), phi)
    chi = 0 * phi
    K.smooth_Heaviside(chi, phi, cpu.moll_zone)
    K.extrapolate_eta_with_least_squares(chi > 0.5, phi, cpu.eta1, cpu.eta2, cpu.ball_phi_double,
                                         cpu.eta1_double, cpu.eta2_double, zone, cpu.nr, cpu.z)
    e1, e2 = case.eta()
    assert np.array_equal(e1, cpu.eta1) and np.array_equal(e2, cpu.eta2)


def test_walk_over_the_listed_words():
    from pyaxisymflow_amd.stepper import SoftSphereStepper

    print("nz 572", flush=True)
    st = SoftSphereStepper(grid_size_z=572, r_ball=0.39)
    st.step(1)
    check_map(st, st.dt(), 572, 0.39)


def test_more_fronts_than_launches():
    from pyaxisymflow_amd import _lib
    from pyaxisymflow_amd.stepper import SoftSphereStepper

    print("nz 640, zone of 16 cells", flush=True)
    st = SoftSphereStepper(grid_size_z=640, r_ball=0.4)
    st.cfg.extrap_zone = st.cfg.reinit_band = 16 * st.cfg.dx
    wide = ctypes.c_void_p()
    _lib.call("axs_soft_stepper_create", ctypes.byref(st.cfg), ctypes.byref(st._bufs),
              ctypes.byref(wide))
    _lib.load().axs_soft_stepper_destroy(st._h)
    st._h = wide
    st.step(1)
    assert st.lsq_sweeps_last() > 12
    check_map(st, st.dt(), 640, 0.4, zone=16 * st.cfg.dx)


@pytest.mark.parametrize("large", [(572, 0.39), (640, 0.4)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_batch_of_large_and_small(monkeypatch, precision, large):
    from pyaxisymflow_amd import stepper
    from pyaxisymflow_amd.stepper import SoftSphereBatch

    state = stepper._soft_case_state

    def wide_zone(obj, *args, **kw):
        state(obj, *args, **kw)
        obj.cfg.extrap_zone = obj.cfg.reinit_band = 16 * obj.cfg.dx

    monkeypatch.setattr(stepper, "_soft_case_state", wide_zone)
    print(f"batch {precision} {large}", flush=True)
    specs = [(64, 0.15, 2.0), (*large, 1.0), (128, 0.15, 1.0)]
    b = SoftSphereBatch(max_cases=3, precision=precision)
    cases = [b.add(grid_size_z=nz, r_ball=r, G=G) for nz, r, G in specs]
    b.step(1)
    for c, (nz, r, G) in zip(cases, specs):
        assert c.scalars()[7] > 12  # fronts
        check_map(c, c.scalars()[1], nz, r, G, zone=16 * c.cfg.dx)
    alone = SoftSphereBatch(max_cases=1, precision=precision)
    a = alone.add(grid_size_z=128, r_ball=0.15, G=1.0)
    alone.step(4)
    b.step(3)
    for x, y in zip([a.vorticity(), *a.eta(), a.phi()],
                    [cases[2].vorticity(), *cases[2].eta(), cases[2].phi()]):
        assert np.array_equal(x, y)


def step_us(nz, r_ball):
    from pyaxisymflow_amd.stepper import SoftSphereStepper

    st = SoftSphereStepper(grid_size_z=nz, r_ball=r_ball)
    st.step(8)
    best = float("inf")
    for _ in range(5):
        st.synchronize()
        t = time.perf_counter()
        st.step(16)
        st.synchronize()
        best = min(best, (time.perf_counter() - t) / 16 * 1e6)
    return best


# one workgroup that walked the whole box at every front: 2.83 at 1024, now 1.78; fits
# of a front by one workgroup per component: 1.96 at 2048, now 1.51; two
# atomics on one line by every segment of the target rows: 1.46 at 4096, now 1.19
@pytest.mark.parametrize("nz,bar", [(1024, 2.2), (2048, 1.72), (4096, 1.32)])
def test_a_large_solid_costs_little_more(nz, bar):
    large, small = step_us(nz, 0.4), step_us(nz, 0.05)
    print(f"nz {nz}: {large:.0f} and {small:.0f} us per step", flush=True)
    assert large / small < bar
