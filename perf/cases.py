"""The performance cases of the framework.

What a user of the library has it do, through its public entry points: the
FCM mobility solve (`Fcm.mobility`, the hot call of every simulation) from
the smallest suspensions to the largest, in both precisions and at both
Gaussian supports in use; the collision barrier on its own; the warm start's
network; whole implicit timesteps of swimming filaments; and a batched
parameter sweep. Segments lie on filaments (chains of beads 2.2 radii apart),
as in every simulation.

Case kinds and their sizes
  fcm      nx, ny, nz, ngd (12: dx = a/1.86; 20: the reference's own
           dx = sigma_dip/1.5), prec (32 or 64), nfil filaments x nw segments
  barrier  nx, ny, nz, nfil, nw: link + apply
  mlp      rows, nw: the network's forward pass for `rows` filaments
  step     grid, nfil, nw, steps: restore a state, advance, read the state
  sweep    nsys, steps: the same for a batch of suspensions
"""
import math

import numpy as np
import torch

from filsim_amd import abi, api, params

F64 = torch.float64
DL = 2.2  # segment spacing in radii


def listed():
    return [
        # a 16 x 15 suspension on 64^3, the smallest simulated: the solve is
        # launches and latency
        dict(name="fcm_64_240_f64", kind="fcm", nx=64, ny=64, nz=64, ngd=12,
             prec=64, nfil=16, nw=15),
        # one point of a parameter sweep (grids 32..128, 15-40 segments):
        # mixed precision, a length that is no power of two
        dict(name="fcm_96_1350_f32", kind="fcm", nx=96, ny=96, nz=96, ngd=12,
             prec=32, nfil=50, nw=27),
        # an elongated channel (the reference runs 4:1:1 boxes) with ragged
        # lengths and an odd segment count
        dict(name="fcm_320x80x90_2997_f64", kind="fcm", nx=320, ny=80, nz=90,
             ngd=12, prec=64, nfil=111, nw=27),
        # the reference's own resolution: 20 support points per dimension
        dict(name="fcm_192_ngd20_2400_f64", kind="fcm", nx=192, ny=192,
             nz=192, ngd=20, prec=64, nfil=80, nw=30),
        # the benchmark suspension, 1,000 x 30 at 256^3: every Broyden
        # iteration of a mixed-precision step is one of these
        dict(name="fcm_256_30k_f32", kind="fcm", nx=256, ny=256, nz=256,
             ngd=12, prec=32, nfil=1000, nw=30),
        # the same in full precision
        dict(name="fcm_256_30k_f64", kind="fcm", nx=256, ny=256, nz=256,
             ngd=12, prec=64, nfil=1000, nw=30),
        # the largest suspension, 8,000 x 30 at 512^3
        dict(name="fcm_512_240k_f32", kind="fcm", nx=512, ny=512, nz=512,
             ngd=12, prec=32, nfil=8000, nw=30),
        # the barrier of the largest suspension: a new cell list, then the
        # pair forces
        dict(name="barrier_512_240k", kind="barrier", nx=512, ny=512, nz=512,
             nfil=8000, nw=30),
        # the warm start's guess for the benchmark suspension, one call a step
        dict(name="mlp_forward_1000", kind="mlp", rows=1000, nw=30),
        # a small simulation from rest, four steps between two outputs
        dict(name="step_64_16x15_f64", kind="step", grid=64, nfil=16, nw=15,
             steps=4),
        # the benchmark suspension's first step from rest (some sixty
        # iterations)
        dict(name="step_256_1000x30_f64", kind="step", grid=256, nfil=1000,
             nw=30, steps=1),
        # a sweep of eight small suspensions advanced together
        dict(name="sweep_8_f64", kind="sweep", nsys=8, steps=2),
    ]


# lengths 2^a 3^b 5^c the solver takes (even), for the drawn grids
LENGTHS = [n for n in range(32, 513, 2)
           if any(2 ** a * 3 ** b * 5 ** c == n for a in range(10)
                  for b in range(6) for c in range(4))]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: mostly mobility solves, grids of 32^3 to 512^3 points
    (cubic or not), dilute to as dense as the listed ones, both precisions;
    now and then a barrier, a network call, a small run or a sweep."""
    u = rng.random()
    if u < 0.7:
        # powers of two half of the time, as most runs choose them
        pool = rng.choice([LENGTHS, [32, 64, 128, 256, 512]])
        edge = math.exp(rng.uniform(math.log(32), math.log(512)))
        near = [n for n in pool if edge / 2 <= n <= edge * 1.5] or [64]
        n = [rng.choice(near) for _ in range(3)]
        if rng.random() < 0.4:
            n = [n[0]] * 3
        prec = rng.choice([32, 64])
        while n[0] * n[1] * n[2] * (prec // 32) > 512 ** 3:
            n[n.index(max(n))] = 128
        ngd = 20 if rng.random() < 0.2 else 12
        nw = rng.randint(5, 40)
        # segments per grid point: up to 2e-3 at a/1.86 and, by volume, a
        # fifth of it at the finer reference resolution
        dens = math.exp(rng.uniform(math.log(1e-4), math.log(2e-3)))
        if ngd == 20:
            dens /= 5
        nfil = max(1, int(n[0] * n[1] * n[2] * dens / nw))
        return dict(kind="fcm", nx=n[0], ny=n[1], nz=n[2], ngd=ngd, prec=prec,
                    nfil=nfil, nw=nw)
    if u < 0.8:
        n = [rng.choice([64, 96, 128, 160, 256, 384, 512]) for _ in range(3)]
        nw = rng.randint(5, 40)
        dens = math.exp(rng.uniform(math.log(2e-4), math.log(1.8e-3)))
        return dict(kind="barrier", nx=n[0], ny=n[1], nz=n[2],
                    nfil=max(1, int(n[0] * n[1] * n[2] * dens / nw)), nw=nw)
    if u < 0.88:
        return dict(kind="mlp", rows=_log_int(rng, 16, 8000),
                    nw=rng.randint(8, 40))
    if u < 0.95:
        g = rng.choice([64, 72, 96, 128])
        nw = rng.randint(8, 20)
        return dict(kind="step", grid=g, nw=nw, steps=rng.randint(1, 2),
                    nfil=max(2, int(g ** 3 * rng.uniform(4e-4, 1.2e-3) / nw)))
    return dict(kind="sweep", nsys=rng.randint(2, 8), steps=rng.randint(1, 2))


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------
def _fp(case):
    n = (case["nx"], case["ny"], case["nz"])
    return (params.reference_fcm_params(n) if case.get("ngd") == 20
            else params.fcm_params(n))


def _chains(box, nfil, nw, seed):
    """Unwrapped bead positions of nfil gently curved filaments anywhere in
    the box (np x 3, device)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    L = torch.tensor(box, dtype=F64, device="cuda")
    head = torch.rand((nfil, 1, 3), generator=g, dtype=F64, device="cuda") * L
    t = torch.randn((nfil, 1, 3), generator=g, dtype=F64, device="cuda")
    bend = torch.randn((nfil, nw, 3), generator=g, dtype=F64, device="cuda")
    t = t / t.norm(dim=-1, keepdim=True)
    t = t + 0.05 * bend.cumsum(1)
    t = t / t.norm(dim=-1, keepdim=True)
    X = head + DL * (t.cumsum(1) - t)
    return X.reshape(-1, 3).contiguous(), L, g


def _fcm_inputs(case, seed):
    X, L, g = _chains(params.box(_fp(case)), case["nfil"], case["nw"], seed)
    Y = torch.fmod(X, L)  # as the timestep passes it: may be negative
    F = torch.randn(Y.shape, generator=g, dtype=F64, device="cuda")
    T = torch.randn(Y.shape, generator=g, dtype=F64, device="cuda")
    return Y, F, T


def _barrier_inputs(case, seed):
    fp = params.fcm_params((case["nx"], case["ny"], case["nz"]))
    X, L, g = _chains(params.box(fp), case["nfil"], case["nw"], seed)
    F0 = torch.randn(X.shape, generator=g, dtype=F64, device="cuda")
    return fp, X, torch.fmod(X, L), F0


def _mlp_inputs(case, seed):
    nw = case["nw"]
    n_in, n_out = 24 * nw - 4, 6 * nw
    r = np.random.default_rng(seed)
    dims = [n_in, 256, 256, 256, n_out]
    p = np.concatenate([np.concatenate([
        r.standard_normal(a * b) * math.sqrt(2.0 / a),
        0.01 * r.standard_normal(b)])
        for a, b in zip(dims, dims[1:])]).astype(np.float32)
    mu = r.standard_normal(n_in).astype(np.float32)
    sigma = np.exp(0.5 * r.standard_normal(n_in)).astype(np.float32)
    tau = np.exp(r.standard_normal(n_out) - 3).astype(np.float32)
    S = (0.05 * r.standard_normal((n_out, n_in))).astype(np.float32)
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.randn((case["rows"], n_in), generator=g, device="cuda")
    X = X * torch.tensor(sigma, device="cuda") + torch.tensor(mu, device="cuda")
    return dims, p, mu, sigma, tau, S, X.contiguous()


def _swimmers(grid, nfil, nw, seed):
    """Parameters and initial state of nfil swimming filaments at rest."""
    fp = params.fcm_params(grid)
    sp = params.sim_params(fp, dt=0.005, tol=1e-6, maxiter=100,
                           precision=abi.FS_FP64, barrier_on=1)
    r = np.random.default_rng(seed)
    props = params.swimming_props(
        nfil, nw, kap=1000.0, phases=list(r.uniform(0, 2 * math.pi, nfil)))
    X, q = api.make_filaments(params.box(fp), [nw] * nfil, dL=DL, min_sep=DL,
                              seed=seed + 1, gpu=True)
    return sp, [nw] * nfil, props, dict(X=X, Xs=X, Xt=X, q=q, qs=q, qt=q)


def _with_copy(setup):
    """The system that steps and one that keeps the state it starts from."""
    sp, nws, props, state = setup
    pair = []
    for _ in range(2):
        s = api.System(sp, nws, props)
        s.set_state(U=np.zeros((s.np, 3)), Us=np.zeros((s.np, 3)),
                    Ut=np.zeros((s.np, 3)), lam=np.zeros((s.nlam, 3)),
                    lam1=np.zeros((s.nlam, 3)), lam2=np.zeros((s.nlam, 3)),
                    F=np.zeros((s.np, 3)), TAU=np.zeros((s.np, 3)), **state)
        pair.append(s)
    return pair


# the sweep's suspensions: grids of the sweep's range, a few filaments each
SWEEP = ((32, 6, 7), (48, 10, 10), (64, 16, 15), (96, 30, 20))


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "fcm":
        s["Y"], s["F"], s["T"] = _fcm_inputs(case, seed)
        s["V"], s["W"] = torch.empty_like(s["Y"]), torch.empty_like(s["Y"])
        s["fcm"] = api.Fcm(_fp(case), s["Y"].shape[0], precision=(
            abi.FS_FP64 if case["prec"] == 64 else abi.FS_FP32))
    elif kind == "barrier":
        fp, s["X"], s["Y"], s["F0"] = _barrier_inputs(case, seed)
        sf = np.repeat(np.arange(case["nfil"]), case["nw"])
        si = np.tile(np.arange(case["nw"]), case["nfil"])
        s["cb"] = api.Colbar(params.colbar_params(fp), sf, si)
    elif kind == "mlp":
        dims, p, mu, sigma, tau, S, s["X"] = _mlp_inputs(case, seed)
        m = api.Mlp(dims[0], dims[-1], width=256)
        m.set_params(p)
        m.set_norm(mu, sigma, tau)
        m.set_skip(S)
        s["mlp"] = m
        s["Y"] = torch.empty((case["rows"], dims[-1]), device="cuda")
    elif kind == "step":
        s["sys"], s["start"] = _with_copy(
            _swimmers(case["grid"], case["nfil"], case["nw"], seed))
    else:
        s["pairs"] = [_with_copy(_swimmers(*SWEEP[k % len(SWEEP)],
                                           seed + 100 * k))
                      for k in range(case["nsys"])]
        s["batch"] = api.Batch([p[0] for p in s["pairs"]])
    return s


# ---------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------
# what a run keeps of a state: everything a restart needs
FIELDS = ("X", "Xt", "U", "Ut", "q", "qt", "lam1", "lam2")


def run(s):
    kind = s["kind"]
    if kind == "fcm":
        s["fcm"].mobility(s["Y"], s["F"], s["T"], s["V"], s["W"],
                          stream=torch.cuda.current_stream())
        return s["V"], s["W"]
    if kind == "barrier":
        st = torch.cuda.current_stream()
        F = s["F0"].clone()
        s["cb"].link(s["X"], stream=st)
        return F, s["cb"].apply(s["Y"], 1, F, stream=st)
    if kind == "mlp":
        s["mlp"].forward(s["X"], s["Y"], stream=torch.cuda.current_stream())
        return s["Y"]
    if kind == "step":
        s["sys"].copy_filaments(s["start"])
        its = [s["sys"].timestep(nt + 1) for nt in range(s["case"]["steps"])]
        st = s["sys"].get_state()
        return its, {k: st[k] for k in FIELDS}
    for live, start in s["pairs"]:
        live.copy_filaments(start)
    its = [s["batch"].timestep(nt + 1) for nt in range(s["case"]["steps"])]
    out = [live.get_state() for live, _ in s["pairs"]]
    return sum(its, []), {k: np.concatenate([o[k] for o in out])
                          for k in FIELDS}


# ---------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------
def _solve_work(N, npt, ngd):
    """One mobility solve: positions, forces, torques in, velocities out;
    six real 3D transforms, the projection, and per segment and support
    point the force and torque terms both ways."""
    return (15.0 * 8 * npt,
            6 * 2.5 * N * math.log2(N) + 15.0 * N + 2 * 22.0 * npt * ngd ** 3)


def _step_work(grid, nfil, nw, steps):
    # about ten iterations a step, one solve each beside the guess's; state
    # in and out; the block-tridiagonal Jacobian (12 x 12 blocks)
    npt = nfil * nw
    b, f = _solve_work(grid ** 3, npt, 12)
    return (steps * (11 * b + 8.0 * 33 * npt * 2),
            steps * (11 * f + npt / 2 * 6 * 12.0 ** 3 +
                     10 * npt / 2 * 6 * 144.0))


def work(case):
    kind = case["kind"]
    if kind == "fcm":
        b, f = _solve_work(case["nx"] * case["ny"] * case["nz"],
                           case["nfil"] * case["nw"], case["ngd"])
    elif kind == "barrier":
        # positions twice (the list's and the current ones), forces in and
        # out; about 14 candidate pairs a segment
        npt = case["nfil"] * case["nw"]
        b, f = 8.0 * 3 * npt * 4 + 8.0 * npt, npt * 14 * 20.0
    elif kind == "mlp":
        nw, r = case["nw"], case["rows"]
        a, o = 24 * nw - 4, 6 * nw
        wts = a * 256 + 2 * 256 * 256 + 256 * o + a * o
        b, f = 4.0 * r * (a + o) + 2.0 * wts, 2.0 * r * wts
    elif kind == "step":
        b, f = _step_work(case["grid"], case["nfil"], case["nw"],
                          case["steps"])
    else:
        b = f = 0.0
        for k in range(case["nsys"]):
            x, y = _step_work(*SWEEP[k % len(SWEEP)], case["steps"])
            b, f = b + x, f + y
    return dict(bytes=b, flops=f)


# ---------------------------------------------------------------------
# the same in 64 bits, with torch alone
# ---------------------------------------------------------------------
def _fcm_exact(case, seed):
    Y, F, T = _fcm_inputs(case, seed)
    fp = _fp(case)
    n, ngd, dx = (case["nx"], case["ny"], case["nz"]), case["ngd"], fp.dx
    N = n[0] * n[1] * n[2]
    i = torch.arange(ngd, device="cuda")
    s2, d2 = fp.sigma ** 2, fp.sigma_dip ** 2
    G = 0.5 * T

    def chunks():
        step = max(1, 4_000_000 // ngd ** 3)
        for a in range(0, Y.shape[0], step):
            sl = slice(a, a + step)
            y = Y[sl]
            p = torch.trunc(y / dx).long()[:, :, None] - ngd // 2 + 1 + i
            xx = p.double() * dx - y[:, :, None]
            g = torch.exp(-xx * xx / (2 * s2)) / math.sqrt(2 * math.pi * s2)
            d = torch.exp(-xx * xx / (2 * d2)) / math.sqrt(2 * math.pi * d2)
            h = -xx / d2 * d
            q = [p[:, k] % n[k] for k in range(3)]
            at = ((q[0][:, :, None, None] * n[1] + q[1][:, None, :, None]) *
                  n[2] + q[2][:, None, None, :])

            def prod(a3, b3, c3):
                return (a3[:, 0, :, None, None] * b3[:, 1, None, :, None] *
                        c3[:, 2, None, None, :])
            yield (sl, at, prod(g, g, g), prod(h, d, d), prod(d, h, d),
                   prod(d, d, h))

    f = torch.zeros((3, N), dtype=F64, device="cuda")
    for sl, at, m, gx, gy, gz in chunks():
        b = [v[:, None, None, None] for v in G[sl].unbind(1)]
        t = (b[2] * gy - b[1] * gz, b[0] * gz - b[2] * gx,
             b[1] * gx - b[0] * gy)
        for c in range(3):
            f[c].index_add_(0, at.reshape(-1), (
                F[sl, c][:, None, None, None] * m + t[c]).reshape(-1))
    k = [torch.cat([torch.arange(m // 2 + 1), torch.arange(m // 2 + 1 - m, 0)])
         .to("cuda", F64) * (2 * math.pi / (m * dx)) for m in n]
    kx, ky = k[0][:, None, None], k[1][None, :, None]
    kz = k[2][None, None, :n[2] // 2 + 1]
    fh = [torch.fft.rfftn(f[c].reshape(n)) for c in range(3)]
    del f
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    kf = (kx * fh[0] + ky * fh[1] + kz * fh[2]) / k2
    u = torch.empty((3, N), dtype=F64, device="cuda")
    for c, kc in enumerate((kx, ky, kz)):
        w = (fh[c] - kc * kf) / (k2 * fp.mu)
        w[0, 0, 0] = 0
        fh[c] = None
        w = torch.fft.ifftn(w, dim=(0, 1))
        w[..., 0] = w[..., 0].real.to(w.dtype)  # a real line's end terms
        w[..., -1] = w[..., -1].real.to(w.dtype)
        u[c] = torch.fft.irfft(w, n=n[2], dim=2).reshape(-1)
    V, W = torch.empty_like(Y), torch.empty_like(Y)
    for sl, at, m, gx, gy, gz in chunks():
        a, b, c = (u[j][at] for j in range(3))

        def tot(v):
            return dx ** 3 * v.flatten(1).sum(1)
        V[sl] = torch.stack([tot(a * m), tot(b * m), tot(c * m)], 1)
        W[sl] = -0.5 * torch.stack([tot(c * gy - b * gz), tot(a * gz - c * gx),
                                    tot(b * gx - a * gy)], 1)
    return V, W


def _barrier_exact(case, seed):
    fp, X, Y, F = _barrier_inputs(case, seed)
    cp = params.colbar_params(fp)
    L = torch.tensor(list(cp.box), dtype=F64, device="cuda")
    npt, nw = X.shape[0], case["nw"]
    M = [int(v / (2.5 * cp.a)) for v in cp.box]
    m = torch.tensor(M, device="cuda")
    frac = Y / L - torch.floor(Y / L)
    c = torch.minimum((frac * m).long(), m - 1)
    cell = (c[:, 0] * M[1] + c[:, 1]) * M[2] + c[:, 2]
    ids = torch.argsort(cell)
    count = torch.bincount(cell, minlength=M[0] * M[1] * M[2])
    first = count.cumsum(0) - count
    me = torch.arange(npt, device="cuda")
    R2 = (2 * cp.a) ** 2
    cut = 1.21 * R2
    for o in range(27):
        d = torch.tensor([o // 9 - 1, o // 3 % 3 - 1, o % 3 - 1],
                         device="cuda")
        q = (c + d) % m
        nc = (q[:, 0] * M[1] + q[:, 1]) * M[2] + q[:, 2]
        for k in range(int(count.max())):
            j = ids[(first[nc] + k).clamp(max=npt - 1)]
            near = (k < count[nc]) & (j != me)
            near &= ~((me // nw == j // nw) & ((me - j).abs() == 1))
            r = Y - Y[j]
            r = r - L * torch.floor(r / L + 0.5)
            r2 = (r * r).sum(1)
            near &= r2 < cut
            r = torch.where((r2 < cp.cap ** 2)[:, None],
                            r / r2.sqrt()[:, None] * cp.cap, r)
            r2 = r2.clamp(min=cp.cap ** 2)
            pre = ((cut - r2) / (cut - R2)) ** 4 * cp.fs_over_2a
            F = F + torch.where(near[:, None], pre[:, None] * r, 0.0)
    return F, None  # the minimum is over the pairs the cells visit


def _mlp_exact(case, seed):
    dims, p, mu, sigma, tau, S, X = _mlp_inputs(case, seed)

    def dev(a):
        return torch.tensor(a, device="cuda").double()
    x = h = (X.double() - dev(mu)) / dev(sigma)
    at = 0
    for k, (a, b) in enumerate(zip(dims, dims[1:])):
        Wt = dev(p[at:at + a * b].reshape(b, a)).t().contiguous()
        h = h @ Wt + dev(p[at + a * b:at + a * b + b])
        at += a * b + b
        if k < 3:
            h = h.clamp(min=0)
    return dev(tau) * (h + x @ dev(S).t().contiguous())


def exact(case, seed):
    if case["kind"] == "fcm":
        return _fcm_exact(case, seed)
    if case["kind"] == "barrier":
        return _barrier_exact(case, seed)
    if case["kind"] == "mlp":
        return _mlp_exact(case, seed)
    return None  # a whole implicit step has no short restatement
