"""An ensemble without its members' second accumulators (SOLAR_STEP_STORE_ALL,
or too little device memory) stores q after every stage: the same bits as the
stored-q schedule, in every stage tile shape, with one state less per member."""
import numpy as np
import pytest

from solar_amd import Ensemble
from tests.test_gpu_ensemble import _members, _run

pytestmark = pytest.mark.gpu


def test_store_all_equals_stored_q(monkeypatch):
    mems, q0s = _members()
    with Ensemble(mems) as ens:
        want, held = _run(ens, q0s, 3), ens.info()["device_bytes"]
    monkeypatch.setenv("SOLAR_STEP_STORE_ALL", "1")
    with Ensemble(mems) as ens:
        assert held - ens.info()["device_bytes"] == sum(q.nbytes for q in q0s)
        runs = [_run(ens, q0s, 3)]
        ens.autotune(reps=1)
        runs.append(_run(ens, q0s, 3))
        for k, m in enumerate(mems):  # each shape that divides n, the widest first
            n = m["n"]
            shapes = [s for s in ((64, 8), (32, 8), (16, 16)) if n % s[0] == 0 and n % s[1] == 0]
            ens.set_tiles(k, (*shapes[0], 9, 16, 16, 13))
        runs.append(_run(ens, q0s, 3))
    for got in runs:
        for k in range(len(mems)):
            assert np.array_equal(got[k], want[k]), k
