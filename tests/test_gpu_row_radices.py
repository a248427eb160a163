"""Row transforms whose DFT has radices 7, 8, 11 and 13, and the launch shapes
of long rows: the lengths here give each of these radices, alone and mixed,
rows of one wavefront and of the most threads, each count of butterflies per
thread, and the chirp-z lengths that pass over a shorter one with a lone
radix 2.

Bars (FP64): relative L2 against the exact discrete solutions 1e-12, as for
the other lengths: a DFT of N <= 8192 points adds at most about
eps log2(N) = 3e-15 to each of the two row passes, the radial solves are the
same.  A batch that mixes lengths runs its rows with the threads of
the longest: the bits of a case stay those it has alone."""
import numpy as np
import pytest

from oracle import implicit_diffusion as O
from oracle.stokes import exact_stokes_solve

pytestmark = pytest.mark.gpu

PERIODIC = "homogenous_neumann_along_r_and_periodic_along_z"


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def solve(nr, nz, w, **kw):
    from pyaxisymflow_amd.kernels.FastDiagonalisationStokesSolver import (
        FastDiagonalisationStokesSolver,
    )

    psi = np.zeros_like(w)
    FastDiagonalisationStokesSolver(nr, nz, 1.0 / nz, **kw).solve(solution_field=psi, rhs_field=w)
    return psi


# even nz: DFTs of nz / 2 = 7, 11, 13, 56 = 8 x 7, 16 x 7,
# 32 x 11, 128 x 7, 7 x 11 x 13, 256 x 7, 2 x 7 x 11 x 13; odd nz: 7, 91, 4095
@pytest.mark.parametrize("nz", [14, 22, 26, 112, 224, 704, 1792, 2002, 3584, 4004, 7, 91, 4095])
def test_neumann_rows(nz):
    nr = 9
    w = np.random.default_rng(nz).standard_normal((nr, nz))
    print(f"rows of {nz}", flush=True)
    assert rel_l2(solve(nr, nz, w), exact_stokes_solve(w, 1.0 / nz)) < 1e-12


@pytest.mark.parametrize("nz", [7, 77, 154, 1456, 2002, 4004])
def test_periodic_rows(nz):
    nr = 6
    w = np.random.default_rng(nz).standard_normal((nr, nz))
    print(f"periodic rows of {nz}", flush=True)
    psi = solve(nr, nz, w, bc_type=PERIODIC)
    assert rel_l2(psi, exact_stokes_solve(w, 1.0 / nz, PERIODIC)) < 1e-12


# DFTs of nz + 1 points: 7, 13, 2 x 7 x 13, 4004; chirp-z of 2049 (4500
# points instead of 4320), 1363 and 1501 points
@pytest.mark.parametrize("nz", [6, 12, 181, 4003, 2048, 1362, 1500])
def test_sine_rows(nz):
    from pyaxisymflow_amd.kernels.implicit_diffusion_solver import ImplicitEulerDiffusionStepper

    nr, dx, nu = 7, 1.0 / nz, 1.5e-3
    dt = dx**2 / 4 / nu
    w = np.random.default_rng(nz).standard_normal((nr, nz))
    out = w.copy()
    print(f"sine rows of {nz}", flush=True)
    ImplicitEulerDiffusionStepper(time_step=dt, kinematic_viscosity=nu, grid_size_r=nr,
                                  grid_size_z=nz, dx=dx).step(vorticity_field=out, dt=dt)
    assert rel_l2(out, O.exact_implicit_diffusion(w, nu * dt, dx)) < 1e-12


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_batch_rows_keep_a_case_s_bits(precision):
    """Rows of 64 points alone, then beside rows of 182 and of 154 points
    (chirp-z in a batch); and the 154-point case alone."""
    from pyaxisymflow_amd.stepper import SoftSphereBatch

    def bits(c):
        return [c.vorticity(), c.psi(), *c.eta(), c.phi()]

    print(f"mixed rows, {precision}", flush=True)
    alone = {}
    for nz in (64, 154):
        b = SoftSphereBatch(max_cases=1, precision=precision)
        c = b.add(grid_size_z=nz, G=2.0)
        b.step(4)
        alone[nz] = bits(c)
    mix = SoftSphereBatch(max_cases=3, precision=precision)
    cases = {nz: mix.add(grid_size_z=nz, G=2.0) for nz in (64, 154, 182)}
    mix.step(4)
    for nz in (64, 154):
        for a, m in zip(alone[nz], bits(cases[nz])):
            assert np.array_equal(a, m), nz
