"""Restart lengths past what the solution kernel's LDS holds (8000): the update reads the rows of the
steps that were taken and no others, whatever those hold."""
import numpy as np
import pytest
import torch

from test_gpu_gmres_cycle import _solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("restart", [8000, 8001])
def test_rows_past_the_last_step_are_not_read(restart):
    """As in test_solution_meets_its_tolerance, on a basis that starts as NaN."""
    print(f"case: restart {restart}", flush=True)
    s, A, b = _solver(600, restart, 11, 0.3)
    s.V.fill_(float("nan"))
    x, k = s.solve(b, 0.0, 1e-8, 3)
    assert 1 <= k < 600
    r = A.cpu() @ x.cpu() - b.cpu()
    assert float(torch.linalg.vector_norm(r)) < 1.01e-8 * float(torch.linalg.vector_norm(b))
    assert np.isfinite(x.cpu().numpy()).all()
