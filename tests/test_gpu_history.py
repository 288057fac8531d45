"""The Broyden history's coefficients on both sides of the line at which they
are added up where they are used."""
import numpy as np
import pytest

from helpers import rel, to_dev
from sysfix import config
from filsim_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfil", [1, 91, 92])  # 1, 8 and 9 partial sums
def test_solve_with_history(cuda, nfil):
    """Two columns against the same products in numpy, FP64: 1e-12 covers the
    order of sums of 16,000 terms and the solver's column normalisation."""
    torch = cuda
    nw = 30
    sp, nws, props, st = config(grid=160, nfil=nfil, nw=nw, seed=2, barrier=0)
    g = api.System(sp, nws, props)
    g.set_state(**st)
    g.initial_guess()
    g.forces(1)
    g.build_jacobian(1)
    rng = np.random.default_rng(nfil)
    n = 6 * nfil * nw

    def solve(b, it):
        x = torch.zeros(n, dtype=torch.float64, device="cuda")
        g.jsolve(to_dev(torch, b), x, it)
        return x.cpu().numpy()

    cols, bs = [], rng.standard_normal((4, n))

    def expect(b):
        return solve(b, 0) + sum(C * (D @ b) for C, D in cols)

    for it in range(2):
        E, En, upd = bs[it], bs[it + 1], rng.standard_normal(n)
        dE = En - E
        nrm = np.linalg.norm(dE)
        C, D = -(expect(dE) + upd) / nrm, dE / nrm
        g.broyden_update(to_dev(torch, E), to_dev(torch, En),
                         to_dev(torch, upd), it)
        cols.append((C, D))
        assert rel(solve(bs[3], it + 1), expect(bs[3])) <= 1e-12
