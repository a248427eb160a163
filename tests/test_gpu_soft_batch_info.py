"""axs_soft_batch_info: the most extrapolation sweeps of a step are those of
the finished runs, read without touching the device (also while another
stream is being captured)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
def test_most_sweeps_of_the_finished_runs(use_graph):
    import torch

    from pyaxisymflow_amd.stepper import SoftSphereBatch

    b = SoftSphereBatch(max_cases=2, use_graph=use_graph)
    cases = [b.add(grid_size_z=64, G=0.1), b.add(grid_size_z=128)]
    assert b.info()[:2] == (2, 0)
    most = 0
    for _ in range(6):
        b.step(1)
        most = max(most, *(int(c.scalars()[7]) for c in cases))  # waits for the step
        assert b.info()[1] == most > 0
    x = torch.zeros(8, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        x += 1
        info = b.info()
    assert info[:2] == (2, most)
    before = b.info()
    b.step(16)
    after = b.info()  # not waited for: of the runs that have finished
    b.synchronize()
    assert before[1] <= after[1] <= b.info()[1]
