"""The blocked schedule and elimination of test_plan0d_tiles at the windows and slot counts that its
cases leave out: 20 columns (lmax = 5, five column groups), 17 (lmax = 3), more than eight tiles."""
import pytest

from test_plan0d_tiles import test_blocked_schedule_reproduces_lu as check


@pytest.mark.parametrize("Nr,lmax,nproc", [(20, 5, 3), (21, 5, 1), (18, 3, 2), (330, 1, 3)])
def test_schedule(Nr, lmax, nproc):
    check(Nr, lmax, nproc)
