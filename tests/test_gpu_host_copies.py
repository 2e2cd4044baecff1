"""Host arrays to and from the device: below and above the size from which the
copies go through pinned staging in several threads, with pieces and parts
that end short, from and into the middle of a larger array, and two handles
from two threads."""
import threading

import numpy as np
import pytest

from solar_amd import Ensemble, Solver, background

pytestmark = pytest.mark.gpu


def _solver(n, nr):
    bg = background(1, nr)
    return Solver(n, nr, *bg, max(1, round(0.08 * nr)), 0.1)


def _state(n, nr, seed):
    return np.random.default_rng(seed).standard_normal((6, 5, nr, n, n))


# 31.5 MB; 33.7 MB (parts of 12 MiB and less); 63.9 MB; 129.6 MB
@pytest.mark.parametrize("n,nr", [(48, 57), (48, 61), (47, 120), (60, 150)])
def test_round_trip(n, nr):
    q = _state(n, nr, n)
    with _solver(n, nr) as s:
        s.set_state(q)
        assert np.array_equal(s.get_state(), q)
        s.set_state(q[::-1].copy())
        assert np.array_equal(s.get_state(), q[::-1])


def test_round_trip_ensemble():
    n, nr = 64, 70
    gr, c2, rho0, g0 = background(1, nr)
    member = dict(n=n, nr=nr, gr=gr, c2=c2, rho0=rho0, g0=g0, sponge_len=6, a_sponge=0.1, dt=1e-4)
    q = [_state(n, nr, m) for m in range(2)]
    with Ensemble([member] * 2) as e:
        for m in (1, 0):
            e.set_state(m, q[m])
        for m in (0, 1):
            assert np.array_equal(e.get_state(m), q[m])


def test_two_handles_from_two_threads():
    n, nr = 60, 100
    ok = [False, False]

    def work(t):
        q = _state(n, nr, 10 + t)
        with _solver(n, nr) as s:
            for _ in range(3):
                s.set_state(q)
                ok[t] = bool(np.array_equal(s.get_state(), q))
                if not ok[t]:
                    return

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert ok == [True, True]
