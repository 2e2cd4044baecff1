"""Forward runs with a 3-D c^2 field where the plain run takes a special route:
one shell, grids whose stages compute their own ghost cells, partial tiles, an
FP32 state.  With a field those stages go back to the gathered ghosts; held to
the CPU restatement bit for bit, and so are the steps after the field is taken
away again."""
import numpy as np
import pytest

import oracle
from solar_amd import Solver
from tests.test_gpu_fp32 import _float_storage_steps
from tests.test_gpu_stage_ghosts import _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("n,nr", [(32, 1), (33, 1), (16, 13), (25, 26), (48, 31), (32, 75)])
def test_c2_field(n, nr, bits):
    print(f"[case] c2 field n={n} nr={nr} bits={bits}", flush=True)
    bg, q, length, dt = _inputs(n, nr)
    c2 = bg[1][None, :, None, None] * (1 + 0.05 * np.random.default_rng(n).random((6, nr, n, n)))

    def steps(o, q):
        return _float_storage_steps(o, q, 2, dt) if bits == 32 else o.rk4(q, 2, dt)[0]

    with_field, plain = (oracle.Oracle(n, nr, *bg, length, 0.1) for _ in range(2))
    with_field.set_c2_field(c2)
    with Solver(n, nr, *bg, length, 0.1, state_bits=bits) as s:
        s.set_c2_field(c2)
        s.set_state(q)
        s.rk4(2, dt)
        mid = s.get_state()
        assert np.array_equal(mid, steps(with_field, q))
        s.set_c2_field(None)
        s.rk4(2, dt)
        assert np.array_equal(s.get_state(), steps(plain, mid))
