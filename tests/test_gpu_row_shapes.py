"""Launch shapes of long rows (axs_anysize.hip): a row transform takes no
longer than its length explains.

The implicit step's two sine row passes are most of its time at these sizes.
Bars on the ratio of two steps of the same build on the same card, between
what shapes whose waves spread over the four SIMDs give and what 320-thread
rows gave (in parentheses): 1024 rows of 2250 against 2304 points 1.25
(1.62), 2560 against 2880 points 0.92 (1.30); 160 rows, each alone on its
compute unit, of 3375 against 3125 points 1.13 (1.41), of 4000 against 4096
points 0.97 (1.09)."""
import time

import pytest

pytestmark = pytest.mark.gpu


def step_us(points, nr):
    import torch

    from pyaxisymflow_amd.kernels.implicit_diffusion_solver import ImplicitEulerDiffusionStepper

    nz, nu = points - 1, 1.5e-3
    dx = 1.0 / nz
    dt = dx**2 / 4 / nu
    st = ImplicitEulerDiffusionStepper(dt, nu, nr, nz, dx)
    w = torch.randn((nr, nz), dtype=torch.float64, device="cuda")
    st.step(w, dt)
    best = float("inf")
    for _ in range(8):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(20):
            st.step(w, dt)
        torch.cuda.synchronize()
        best = min(best, (time.perf_counter() - t) / 20 * 1e6)
    return best


@pytest.mark.parametrize("nr,points,other,bar", [(1024, 2250, 2304, 1.42), (1024, 2560, 2880, 1.1),
                                                 (160, 3375, 3125, 1.26), (160, 4000, 4096, 1.04)])
def test_long_rows_take_what_their_length_explains(monkeypatch, nr, points, other, bar):
    monkeypatch.setenv("AXS_TRIDIAG_LK", "8,2")  # one column layout for both
    a, b = step_us(points, nr), step_us(other, nr)
    print(f"{nr} rows: {points} points {a:.1f} us, {other} points {b:.1f} us", flush=True)
    assert a / b < bar
