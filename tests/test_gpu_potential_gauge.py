"""Mode 0 of the potential inside the column pass: its last equation is
phi_hat_0[nr - 1] = 0, whichever row of its segment that is.  nr one past,
at and one short of multiples of the segment heights (4, 8, 16), the
smallest grid, a grid wide enough for the timed layouts, and one with fewer
modes than a workgroup takes; a compatible and an incompatible rhs.

Bars (FP64): 1e-12 against the exact route for nz <= 256, 1e-10 beyond (the
condition number grows as nz^2), and the gauge itself: the mean over z of
the last row is phi_hat_0[nr - 1] / nz = 0 up to the row transform's
round-off, 16 eps of the field's largest value."""
import numpy as np
import pytest

from oracle import potential as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,nr", [(4, 3), (5, 8), (64, 9), (64, 15), (64, 16), (64, 17), (97, 33),
                                   (256, 129), (1024, 257), (16, 1025)])
def test_gauge_row(nz, nr):
    from pyaxisymflow_amd.kernels.FastDiagonalisationPotentialSolver import (
        FastDiagonalisationPotentialSolver,
    )

    dx = 1.0 / nz
    raw = np.random.default_rng(nz + nr).standard_normal((nr, nz))
    st = FastDiagonalisationPotentialSolver(grid_size_r=nr, grid_size_z=nz, dx=dx)
    for rhs in (O.make_compatible(raw.copy(), dx), raw):
        print(f"potential {nz}x{nr}", flush=True)
        phi = np.zeros_like(rhs)
        st.solve(solution_field=phi, rhs_field=rhs)
        exact = O.exact_potential_solve(rhs, dx)
        err = np.linalg.norm(phi - exact) / np.linalg.norm(exact)
        assert err < (1e-12 if nz <= 256 else 1e-10)
        assert abs(phi[-1].mean()) <= 16 * np.finfo(float).eps * np.abs(phi).max()
