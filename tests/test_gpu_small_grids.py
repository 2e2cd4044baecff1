"""Grids whose tiles do not fill the chip, which the launchers split into short
radial chunks: one-plane and two-plane chunks, chunks that end inside the
boundary closures or the filter's zeroed end planes, and a last chunk that is
shorter than the others.  The forward step is held to the CPU restatement bit
for bit; the adjoint step, whose planes do not depend on the split, to the
same step in one chunk.
"""
import numpy as np
import pytest

import oracle
from solar_amd import Solver, background, generate_ic
from tests.test_gpu_fp32 import _float_storage_steps

pytestmark = pytest.mark.gpu

SIZES = [(16, 12), (16, 29), (32, 13), (48, 25), (20, 17)]


def _inputs(n, nr):
    gr, c2, rho0, g0 = background(1, nr)
    q, _ = generate_ic(1, n, nr, gr, c2, n + nr, [1e-3, 1e-6, 6.0])
    q += 1e-4 * np.random.default_rng(nr).standard_normal(q.shape)
    dt = 0.5 * min(gr[1] - gr[0], gr[0] * (np.pi / 2) / (n - 1))
    return (gr, c2, rho0, g0), q, max(1, round(0.08 * nr)), dt


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("n,nr", SIZES)
def test_short_chunks_match_the_oracle(n, nr, bits):
    print(f"[case] small grid n={n} nr={nr} bits={bits}", flush=True)
    bg, q, length, dt = _inputs(n, nr)
    with Solver(n, nr, *bg, length, 0.1, state_bits=bits) as s:
        s.set_state(q)
        s.rk4(3, dt)
        got = s.get_state()
    o = oracle.Oracle(n, nr, *bg, length, 0.1)
    want = _float_storage_steps(o, q, 3, dt) if bits == 32 else o.rk4(q, 3, dt)[0]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n,nr", [s for s in SIZES if s[0] % 16 == 0])
def test_short_adjoint_chunks_match_one_chunk(n, nr, monkeypatch):
    print(f"[case] small grid adjoint n={n} nr={nr}", flush=True)
    bg, lam, length, dt = _inputs(n, nr)

    def step():
        with Solver(n, nr, *bg, length, 0.1) as s:
            return s.adj_step(lam, dt)

    got = step()
    monkeypatch.setenv("SOLAR_ADJ_STAGE_CHUNKS", "1")
    monkeypatch.setenv("SOLAR_ADJ_FILTER_CHUNKS", "1")
    assert np.array_equal(got, step())
