"""Stages that compute the ghost cells of their own tiles: chunks of one to six
planes, with an odd last plane pair, panels that are one tile wide, tiles that
reach a panel edge past a narrower last tile, single shells, and the first
sizes that keep separate gathers.  Held to the CPU restatement bit for bit.
"""
import numpy as np
import pytest

import oracle
from solar_amd import Solver, background, generate_ic
from tests.test_gpu_fp32 import _float_storage_steps

pytestmark = pytest.mark.gpu


def _inputs(n, nr):
    if nr == 1:  # a shell: r = 1, no radial derivative
        q = np.random.default_rng(n).standard_normal((6, 5, 1, n, n))
        return tuple(np.array([v]) for v in (0.85, 1.3, 0.9, 0.4)), q, 1, 0.5 * (np.pi / 2) / (n - 1) / np.sqrt(1.3)
    gr, c2, rho0, g0 = background(1, nr)
    q, _ = generate_ic(1, n, nr, gr, c2, n + nr, [1e-3, 1e-6, 6.0])
    q += 1e-4 * np.random.default_rng(n + nr).standard_normal(q.shape)
    dt = 0.5 * min(gr[1] - gr[0], gr[0] * (np.pi / 2) / (n - 1))
    return (gr, c2, rho0, g0), q, max(1, round(0.08 * nr)), dt


def _check(n, nr, bits, steps):
    print(f"[case] stage ghosts n={n} nr={nr} bits={bits}", flush=True)
    bg, q, length, dt = _inputs(n, nr)
    with Solver(n, nr, *bg, length, 0.1, state_bits=bits) as s:
        s.set_state(q)
        s.rk4(steps, dt)
        got = s.get_state()
    o = oracle.Oracle(n, nr, *bg, length, 0.1)
    want = _float_storage_steps(o, q, steps, dt) if bits == 32 else o.rk4(q, steps, dt)[0]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("n,nr", [(16, 13), (16, 64), (18, 21), (33, 12), (25, 26), (48, 31), (32, 75), (40, 30)])
def test_short_chunks(n, nr, bits):
    _check(n, nr, bits, 2)


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("n", [16, 17, 33, 64, 67, 128, 130])
def test_shells(n, bits):
    _check(n, 1, bits, 3)


@pytest.mark.parametrize("chunks", [1, 4, 8, 24])
def test_chunks_forced(chunks, monkeypatch):
    monkeypatch.setenv("SOLAR_STAGE_CHUNKS", str(chunks))
    _check(32, 24, 64, 2)
