"""The soft step's extrapolation by fronts: where its shapes change.

The step splits the reference's sweeps (extrapolate_using_least_squares.hpp:142-446)
into fronts found from the flags alone: a cell's sweep is its 8-neighbour
distance from the known set within the target set.  The CPU test pins that
on the oracle's sweep loop; the GPU tests step grids that take each branch:

* nz = 64: the band is a larger share of the grid than the factors kept
  (a sixteenth of the doubled grid), so the solve pass factors the rest;
* nz = 194: rows that end inside a 32-cell flag word;
* nz = 640, r_ball = 0.4: the target box (536 rows of 18 words) does not fit
  the walk's LDS words (7168) and runs on global words;
* nz = 320, r_ball = 0.3: fronts of more cells than the solve workgroup's
  512 threads.
"""
import numpy as np
import pytest

from oracle import kernels as K
from oracle.drivers import SoftSphereCase
from oracle.lsq import extrapolate_using_least_squares_till_first_order
from oracle.reinit import distance


def fronts(known, target):
    """Front number of every target cell (0 known, -1 never reached)."""
    lev = np.where(known, 0, -1)
    level = 0
    while True:
        k = np.pad(lev >= 0, 1)
        n0, n1 = lev.shape
        near = np.zeros_like(known)
        for a in range(3):
            for b in range(3):
                near |= k[a:a + n0, b:b + n1]
        new = near & target & (lev < 0)
        if not new.any():
            return lev, level
        level += 1
        lev[new] = level


@pytest.mark.parametrize("seed", range(6))
def test_fronts_are_the_oracle_s_sweeps(seed):
    rng = np.random.default_rng(seed)
    n = 40
    z = (np.arange(n) + 0.5) / n
    # targets with holes and separate parts, known cells inside them
    field = sum(rng.standard_normal() * np.cos(rng.uniform(1, 9) * z[:, None] * np.pi
                                               + rng.uniform(0, 6))
                * np.cos(rng.uniform(1, 9) * z[None, :] * np.pi) for _ in range(4))
    target = field > np.quantile(field, 0.45)
    known = field > np.quantile(field, 0.8 if seed % 2 else 0.97)
    lev, levels = fronts(known, target)
    # the loop cut after s sweeps has filled exactly the first s fronts: run
    # it on the targets of those fronts alone
    for s in range(levels + 1):
        cur = known.astype(np.int16)
        tgt = (target & (lev >= 0) & (lev <= s)).astype(np.int16)
        e = np.ascontiguousarray(np.where(known, 1.0 + z[None, :], 0.0))
        got = extrapolate_using_least_squares_till_first_order(cur, tgt, e, e.copy(), z, z)
        assert got == s
        assert np.array_equal(cur != 0, (lev >= 0) & (lev <= s))
    cur = known.astype(np.int16)
    e = np.ascontiguousarray(np.where(known, 1.0 + z[None, :], 0.0))
    assert extrapolate_using_least_squares_till_first_order(
        cur, target.astype(np.int16), e, e.copy(), z, z) == levels
    assert np.array_equal(cur != 0, lev >= 0)


@pytest.mark.gpu
@pytest.mark.parametrize("nz,r_ball", [(64, 0.15), (194, 0.15), (320, 0.3), (640, 0.4)])
def test_one_step_s_map_is_the_oracle_s(nz, r_ball):
    """From the GPU's own velocity and dt the oracle's reference-map ENO3,
    pin, reinit and extrapolation give the GPU's eta and phi bit for bit."""
    from pyaxisymflow_amd.stepper import SoftSphereStepper

    cpu = SoftSphereCase(grid_size_z=nz, r_ball=r_ball, solver="exact")
    gpu = SoftSphereStepper(grid_size_z=nz, r_ball=r_ball)
    gpu.step(1)
    u_z, u_r = gpu.velocity()
    dx = cpu.dx
    K.advect_refmap_via_eno3(cpu.eta1, cpu.eta2, u_z, u_r, gpu.dt(), dx)
    pinned = -np.sqrt((cpu.eta1 - cpu.Z_cm) ** 2 + (cpu.eta2 - cpu.R_cm) ** 2) + r_ball
    phi = np.where(cpu.ball_phi > -3 * dx, pinned, cpu.ball_phi)
    d, masked = distance(phi, dx, cpu.reinit_band)
    phi = np.where(masked, phi, d)
    assert np.array_equal(gpu.phi(), phi)
    chi = 0 * phi
    K.smooth_Heaviside(chi, phi, cpu.moll_zone)
    K.extrapolate_eta_with_least_squares(chi > 0.5, phi, cpu.eta1, cpu.eta2, cpu.ball_phi_double,
                                         cpu.eta1_double, cpu.eta2_double, cpu.extrap_zone, cpu.nr,
                                         cpu.z)
    e1, e2 = gpu.eta()
    assert np.array_equal(e1, cpu.eta1) and np.array_equal(e2, cpu.eta2)
