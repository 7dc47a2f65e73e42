"""Seed lists around the length from which they are copied in place of riding in launches, and their owners' reuse of
the memory right after a call.  Labels equal the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2


@pytest.mark.parametrize("n", [511, 512, 513, 640, 4095, 4096, 4097])
def test_lists_around_the_copy(vf, n):
    dims = (18, 17, 40)
    rng = np.random.default_rng(n)
    grid = (rng.random(dims) < 0.8).astype(np.uint16)
    at = np.argwhere(grid)
    at = at[rng.choice(len(at), n, replace=False)]
    seeds = np.concatenate([at, np.arange(n)[:, None] + 2], 1).astype(np.uint32)
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        for shift in (0, 1):
            own = np.roll(seeds, shift, 0).copy()
            want = O.naive(grid, own, MAN)
            g.fracture_naive(own, MAN)
            own[:] = 0  # the caller's again
            np.testing.assert_array_equal(g.read(), want)
        if n <= 4096:
            own = seeds.copy()
            own[:, 3] = 2 + own[:, 3] % 254
            want = O.flood(grid, own, 26)
            g.fracture_flood(own, CHE)
            own[:] = 0
            np.testing.assert_array_equal(g.read(), want)
