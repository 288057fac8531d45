"""Every line length the solver takes, on each of the three FFT passes."""
import numpy as np
import pytest

import _oracle as O
from filsim_amd import abi, api, params
from helpers import random_segments, rel

pytestmark = pytest.mark.gpu

LENGTHS = sorted(n for n in
                 {2 ** a * 3 ** b * 5 ** c for a in range(1, 11)
                  for b in range(7) for c in range(5)}
                 if 16 <= n <= 1024)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("part", range(4))
def test_line_lengths(cuda, axis, part):
    """Even 2^a 3^b 5^c from 16 to 1024, a quarter of them per test: every
    radix (2-6, 8, 9, 10, 12, 16), first, inner and last in a plan. Bounds:
    1e-12 (FP64, the solver's parity bar) and 1e-5 (FP32) of the velocities'
    norm; angular velocities are differences of the velocity field over a
    radius (a = 1), so theirs is of the larger of |W| and |V| / a, which in
    the most elongated of these boxes is 70 |W|."""
    for k, n in enumerate(LENGTHS):
        if k % 4 != part:
            continue
        grid = [18, 20, 16]
        grid[axis] = n
        fp = params.fcm_params(tuple(grid))
        Y, F, T = random_segments(fp, 60, seed=n)
        Vo, Wo = O.mobility(fp, Y, F, T)
        for prec, bar in ((abi.FS_FP64, 1e-12), (abi.FS_FP32, 1e-5)):
            with api.Fcm(fp, 60, precision=prec) as fcm:
                V, W = fcm.mobility_host(Y, F, T)
            ew = np.linalg.norm(W - Wo)
            top = max(np.linalg.norm(Wo), np.linalg.norm(Vo) / fp.a)
            assert rel(V, Vo) <= bar and ew <= bar * top, (grid, prec)
