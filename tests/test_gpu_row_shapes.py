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

import numpy as np
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


@pytest.mark.parametrize("implicit", [False, True])
def test_a_case_keeps_its_bits_in_a_batch(implicit):
    """96 rows alone, 384 in a batch of four: rows of 2518 points (cosine, FFTs of
    2700) and of 1258 (sine, the same) have one shape for few rows and another
    for many, and a row's rounding depends on it."""
    from pyaxisymflow_amd import workloads
    from pyaxisymflow_amd.stepper import RigidBatchStepper, RigidBodyStepper

    nz, nr = (1258, 96) if implicit else (2518, 96)
    args = []
    for seed in (0, 1):
        sp = workloads.case_spec(seed)
        sp.update(nz=nz, nr=nr)
        a = workloads.rigid_case_args(sp, workloads.case_inputs(sp, nz, nr)[1])
        if implicit:
            a.update(nu=1e-3, implicit_diffusion=True)
        args.append(a)
    cases = [args[q % 2] for q in range(4)]
    print(f"{nz} x {nr}, implicit {implicit}", flush=True)
    many = RigidBatchStepper(nz, nr, 1.0, cases, r_len=nr / nz)
    many.step(4)
    for q in (0, 3):
        one = RigidBodyStepper(nz, nr, 1.0, r_len=nr / nz, **cases[q])
        one.step(4)
        assert np.isfinite(one.vorticity()).all()
        assert np.array_equal(many.vorticity(q), one.vorticity())
        assert np.array_equal(many.drag_history(q), one.drag_history())
