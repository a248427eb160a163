"""The reinit's launch shapes (axs_reinit.hip: by the number of 8 x 32
tiles, at most 1024 or more) against the CPU restatement, bit for bit: a grid
on each side of the line, ragged tiles, and sweep counts that leave a last
launch of 1, 2 or 3 sweeps."""
import numpy as np
import pytest

from oracle.reinit import distance as cpu_distance

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(120, 250), (256, 1024), (261, 1030)])
@pytest.mark.parametrize("iterations", [1, 6, 7, 13])
def test_reinit_shapes_match_oracle_bitwise(shape, iterations):
    from pyaxisymflow_amd.levelset import distance

    nr, nz = shape  # 128, 1024 and 1089 tiles
    dx = 1.0 / nz
    Z, R = np.meshgrid((np.arange(nz) + 0.5) * dx, (np.arange(nr) + 0.5) * dx)
    phi = np.maximum(0.08 - np.sqrt((Z - 0.4) ** 2 + R**2),
                     0.05 - np.sqrt((Z - 0.73) ** 2 + (R - 0.09) ** 2))
    phi = 0.3 * np.tanh(6.0 * phi)
    got = distance(phi, dx=dx, narrow=8 * dx, iterations=iterations)
    want, masked = cpu_distance(phi, dx, 8 * dx, iterations)
    assert np.array_equal(got.mask, masked)
    assert np.array_equal(np.asarray(got), want)
