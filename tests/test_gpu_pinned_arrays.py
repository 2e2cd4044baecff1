"""Pinned host arrays above the size from which pageable ones are staged: whole
arrays, and the middle of a larger pinned allocation."""
import ctypes

import numpy as np
import pytest
import torch

from solar_amd import Solver, background

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("skip", [0, 4097])
def test_pinned_round_trip(skip):
    n, nr = 48, 70  # 38.7 MB
    print(f"[case] pinned arrays n={n} nr={nr} from element {skip}", flush=True)
    shape = (6, 5, nr, n, n)
    count = int(np.prod(shape))
    q, out = (torch.zeros(count + skip, dtype=torch.float64, pin_memory=True)[skip:] for _ in range(2))
    q.copy_(torch.from_numpy(np.random.default_rng(skip).standard_normal(count)))
    ptr = lambda t: ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))  # noqa: E731
    with Solver(n, nr, *background(1, nr), 6, 0.1) as s:
        for _ in range(2):
            assert s.lib.solar_set_state(s.h, ptr(q)) == 0
            assert s.lib.solar_get_state(s.h, ptr(out)) == 0
            assert torch.equal(q, out)
            out.zero_()
        assert np.array_equal(s.get_state().ravel(), q.numpy())
