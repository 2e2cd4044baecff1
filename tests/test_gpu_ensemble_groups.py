"""Ensemble gathers split a panel size's members by their number: a group of
many members runs long radial chunks, a group of few short ones, down to one
plane.  Every member equals its single-grid run bit for bit."""
import numpy as np
import pytest

from solar_amd import Ensemble, Solver, background, generate_ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[(16, 12)] * 6 + [(16, 45)] * 6, [(32, 13)], [(16, 14), (48, 33), (64, 12)]])
def test_groups_of_few_and_of_many_members(sizes):
    print(f"[case] ensemble groups {sizes}", flush=True)
    members, states = [], []
    for m, (n, nr) in enumerate(sizes):
        gr, c2, rho0, g0 = background(1, nr)
        members.append(dict(n=n, nr=nr, gr=gr, c2=c2, rho0=rho0, g0=g0, sponge_len=max(1, round(0.08 * nr)), a_sponge=0.1,
                            dt=0.4 * min(gr[1] - gr[0], gr[0] * (np.pi / 2) / (n - 1))))
        states.append(generate_ic(0, n, nr, gr, c2, 7 + m, [1e-3, 0.05, 0.0])[0]
                      + 1e-5 * np.random.default_rng(m).standard_normal((6, 5, nr, n, n)))
    with Ensemble(members) as e:
        for m, q in enumerate(states):
            e.set_state(m, q)
        e.rk4(3)
        got = [e.get_state(m) for m in range(len(sizes))]
    for m, d in enumerate(members):
        with Solver(d["n"], d["nr"], d["gr"], d["c2"], d["rho0"], d["g0"], d["sponge_len"], d["a_sponge"]) as s:
            s.set_state(states[m])
            s.rk4(3, d["dt"])
            assert np.array_equal(got[m], s.get_state()), m
