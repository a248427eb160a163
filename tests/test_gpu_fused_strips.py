"""The rigid step's fused kernel with strips for 256, 512 and 768 threads (by
the number of 54 x 16-cell tiles in a launch): a case alone and in batches
on the other sides of each change, with ragged tile edges.

Bar: the same bits (a cell's arithmetic and the order of the force sum do
not depend on the strips), fields and drag.  That the 256-thread strips
match the oracle at these precisions is test_gpu_batch.py's and
test_gpu_stepper.py's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# tiles alone -> in the batch: 12 -> 24, 252, 264, 516, 1020, 1032;
# 256 -> 512; 260 -> 520; 512 -> 1024; 520 -> 1040
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nz,nr,batch", [(128, 64, n) for n in (2, 21, 22, 43, 85, 86)]
                         + [(432, 512, 2), (540, 416, 2), (864, 512, 2), (1026, 410, 2)])
def test_case_alone_equals_in_a_batch(nz, nr, batch, precision):
    from pyaxisymflow_amd import workloads
    from pyaxisymflow_amd.stepper import RigidBatchStepper, RigidBodyStepper

    args = []
    for seed in (0, 1):
        sp = workloads.case_spec(seed)
        sp.update(nz=nz, nr=nr)
        args.append(workloads.rigid_case_args(sp, workloads.case_inputs(sp, nz, nr)[1]))
    cases = [args[q % 2] for q in range(batch)]
    print(f"strips {nz}x{nr} x {batch} {precision}", flush=True)
    many = RigidBatchStepper(nz, nr, 1.0, cases, r_len=nr / nz, precision=precision)
    many.step(6)
    for q in (0, 1, batch - 1):
        one = RigidBodyStepper(nz, nr, 1.0, r_len=nr / nz, precision=precision, **cases[q])
        one.step(6)
        assert np.isfinite(one.vorticity()).all()
        assert np.array_equal(many.vorticity(q), one.vorticity())
        assert np.array_equal(many.drag_history(q), one.drag_history())
