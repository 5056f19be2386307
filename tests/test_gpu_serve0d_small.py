"""Small e-e batches in the serving loop: at most two at once, whatever the number of workers, with the
results of one at a time."""
import dataclasses

import numpy as np
import pytest

from conftest import XSEC_FILE

pytestmark = pytest.mark.gpu


def _run(workers):
    from boltzmann_amd.serve0d import Request, ServingEngine
    rng = np.random.default_rng(4)
    grids = [(16, 1, 1), (16, 1, 2), (16, 1, 3), (20, 1, 3), (16, 2, 3), (20, 2, 3)]
    reqs = [Request(i, *grids[i % 6], float(10.0 ** rng.uniform(0.0, 1.8)), 1e-4) for i in range(24)]
    eng = ServingEngine(XSEC_FILE, 8 << 30, max_iter=40, ee_workers=workers)
    eng.run([dataclasses.replace(r, arrival=0.0) for r in reqs[:6]], realtime=False)      # warm-up
    res, st = eng.run(reqs, realtime=True)
    return {r.rid: r for r in res}


def test_at_most_two_at_once():
    print("case: 24 e-e requests over six grids, four workers and one", flush=True)
    four, one = _run(4), _run(1)
    spans = sorted({(r.batch, r.admitted, r.done) for r in four.values()}, key=lambda s: s[1])
    assert len(spans) >= 6
    for _, t, _ in spans:
        assert sum(a <= t < d for _, a, d in spans) <= 2
    assert set(four) == set(one)
    for k in four:
        assert four[k].status == one[k].status             # (one without a fixed point among them)
        assert four[k].energy == one[k].energy and np.array_equal(four[k].rates, one[k].rates)
