"""The stage kernel's tiles: every width of a panel the tiles do not divide
(one column or row left for the last tile, rows that begin inside a 64-byte
segment, one shell), against the CPU restatement bit for bit; and the 64-wide
tiles of panels from 128 with a c^2 field, kept divergences and a
tangent-linear run, against the oracle or the same run with 32-wide tiles.
"""
import numpy as np
import pytest

import oracle
from solar_amd import Solver, background, generate_ic
from tests.test_gpu_fp32 import _float_storage_steps

pytestmark = pytest.mark.gpu


def _inputs(n, nr, seed=5):
    gr, c2, rho0, g0 = background(1, nr) if nr > 1 else (np.full(1, 0.7), np.ones(1), np.ones(1), np.zeros(1))
    q = 1e-4 * np.random.default_rng(seed + n).standard_normal((6, 5, nr, n, n))
    if nr > 1:
        q += generate_ic(1, n, nr, gr, c2, seed, [1e-3, 1e-6, 6.0])[0]
    h = gr[0] * (np.pi / 2) / (n - 1)
    return (gr, c2, rho0, g0), q, max(1, round(0.08 * nr)), 0.5 * min(h, gr[1] - gr[0] if nr > 1 else h)


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("n,nr", [(17, 13), (33, 12), (50, 12), (65, 12), (72, 12), (129, 12), (33, 1), (137, 1)])
def test_partial_tiles_match_the_oracle(n, nr, bits):
    print(f"[case] stage tiles n={n} nr={nr} bits={bits}", flush=True)
    bg, q, length, dt = _inputs(n, nr)
    with Solver(n, nr, *bg, length, 0.1, state_bits=bits) as s:
        s.set_state(q)
        s.rk4(2, dt)
        got = s.get_state()
    o = oracle.Oracle(n, nr, *bg, length, 0.1)
    want = _float_storage_steps(o, q, 2, dt) if bits == 32 else o.rk4(q, 2, dt)[0]
    assert np.array_equal(got, want)


# 13 planes: the step's buffers stay in the last-level cache (plain stores);
# 24: they do not (non-temporal)
@pytest.mark.parametrize("nr", [13, 24])
def test_wide_tiles_with_a_c2_field_match_the_oracle(nr):
    n = 128
    bg, q, length, dt = _inputs(n, nr)
    c2 = bg[1][None, :, None, None] * (1 + 0.02 * np.random.default_rng(3).random((6, nr, n, n)))
    o = oracle.Oracle(n, nr, *bg, length, 0.1)
    o.set_c2_field(c2)
    with Solver(n, nr, *bg, length, 0.1) as s:
        s.set_c2_field(c2)
        s.set_state(q)
        s.rk4(1, dt)
        assert np.array_equal(s.get_state(), o.rk4(q, 1, dt)[0])


@pytest.mark.parametrize("nr", [14, 24])
def test_wide_tiles_gradient_and_tangent_linear(nr, monkeypatch):
    n, steps = 128, 3
    bg, q, length, dt = _inputs(n, nr)
    rng = np.random.default_rng(8)
    rec = np.array([[p, 6, 5 + p, 100] for p in range(6)])
    data, dc2 = 1e-4 * rng.standard_normal((steps, 6)), 1e-2 * rng.standard_normal((6, nr, n, n))

    def run():
        with Solver(n, nr, *bg, length, 0.1) as s:
            s.set_receivers(rec)
            J, grad, seis = s.misfit_gradient(q, steps, dt, data, 1)
            return J, grad, seis, s.tangent_linear(q, steps, dt, dc2)

    wide = run()
    monkeypatch.setenv("SOLAR_STAGE_TI", "32")
    monkeypatch.setenv("SOLAR_STAGE_TJ", "8")
    for a, b in zip(wide, run()):
        assert np.array_equal(a, b)
    assert np.abs(wide[1]).max() > 0 and np.abs(wide[3]).max() > 0
