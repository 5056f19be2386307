"""The ion-fluid launch at the edges of its register layouts (4 x 4 tiles up to 88 points, 6 x 6 up to
128, 8 x 10 above; few points, where the row layout has more groups than it needs): the comparison
with the oracle, and its tolerances, of test_fluid_launch_against_oracle at other sizes."""
import pytest

from test_gpu_glow_coupled import test_fluid_launch_against_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Np", [6, 22, 23, 75, 88, 89, 128, 129])
def test_layout_edges(Np):
    check(Np)
