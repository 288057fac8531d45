"""The network's inference pass in one launch, at the edges of its tiles."""
import os
import sys

import numpy as np
import pytest

from filsim_amd import api

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n_in,width,n_out", [
    (1, 4, 16, 1),         # one row, one step of k, one output
    (16, 28, 20, 17),      # a part of the second tile of 16
    (17, 32, 260, 33),     # a second workgroup; a 17th tile of a layer
    (50, 36, 256, 180),
    (33, 1532, 256, 384),  # long rows
    (40, 30, 32, 12),      # an input row that is no whole load
    (9, 64, 1024, 48),     # too many weights: by layers
])
def test_forward_at_tile_edges(cuda, rows, n_in, width, n_out):
    """Against the FP64 oracle with the same BF16 rounding points; 2e-3 for the
    hidden values that FP32 sums round to the other BF16 neighbour. Then the
    outputs over the inputs' memory, and rows that hold a NaN or an infinity,
    which must not reach the other rows."""
    torch = cuda
    rng = np.random.default_rng(rows + n_in)
    mlp = api.Mlp(n_in, n_out, width=width, seed=3)
    mu = rng.standard_normal(n_in).astype(np.float32) * 0.1
    sig = (1 + rng.random(n_in)).astype(np.float32)
    tau = (0.5 + rng.random(n_out)).astype(np.float32)
    mlp.set_norm(mu, sig, tau)
    X = rng.standard_normal((rows, n_in)).astype(np.float32)
    for skip in (None, rng.standard_normal((n_out, n_in)) * 0.05):
        if skip is not None:
            mlp.set_skip(skip)
        yn, _, _, _ = M.forward(mlp.get_params(), mlp.dims, X, mu, sig, tau,
                                skip=skip)
        Yo = yn * tau
        dX = torch.tensor(X, device="cuda")
        Y = torch.full((rows, n_out), 7.0, dtype=torch.float32, device="cuda")
        mlp.forward(dX, Y)
        assert np.linalg.norm(Y.cpu().numpy() - Yo) < 2e-3 * np.linalg.norm(Yo)
        both = torch.zeros(rows * max(n_in, n_out), dtype=torch.float32,
                           device="cuda")
        Xs = both[:rows * n_in].view(rows, n_in)
        Ys = both[:rows * n_out].view(rows, n_out)
        Xs.copy_(dX)
        mlp.forward(Xs, Ys)
        assert np.linalg.norm(Ys.cpu().numpy() - Yo) < 2e-3 * np.linalg.norm(Yo)
        dX[rows // 2, 0] = float("nan")
        dX[rows - 1, n_in - 1] = float("inf")
        Z = torch.zeros_like(Y)
        mlp.forward(dX, Z)
        keep = [r for r in range(rows) if r not in (rows // 2, rows - 1)]
        assert torch.equal(Z[keep], Y[keep])


@pytest.mark.parametrize("skip,rows", [(False, 36864), (False, 36865),
                                       (True, 81920), (True, 81921)])
def test_many_rows_of_a_narrow_net(cuda, skip, rows):
    """The most rows in one launch and the fewest by layers, of the narrowest
    net. Bound as above."""
    torch = cuda
    rng = np.random.default_rng(rows)
    n_in, n_out = 28, 12
    mlp = api.Mlp(n_in, n_out, width=16, seed=3)
    S = rng.standard_normal((n_out, n_in)) * 0.05 if skip else None
    if skip:
        mlp.set_skip(S)
    one, zero = np.ones(n_in, np.float32), np.zeros(n_in, np.float32)
    X = rng.standard_normal((rows, n_in)).astype(np.float32)
    Yo, _, _, _ = M.forward(mlp.get_params(), mlp.dims, X, zero, one,
                            np.ones(n_out, np.float32), skip=S)
    Y = torch.full((rows, n_out), 7.0, dtype=torch.float32, device="cuda")
    mlp.forward(torch.tensor(X, device="cuda"), Y)
    Y = Y.cpu().numpy()
    assert np.linalg.norm(Y - Yo) < 2e-3 * np.linalg.norm(Yo)
    for r in (0, 15, 16, rows - 1):
        assert np.linalg.norm(Y[r] - Yo[r]) < 2e-2 * np.linalg.norm(Yo[r]), r
