"""Performance cases of the framework: what its users run, from the smallest to
the largest calls, each through the public entry points.

A case is a dict of plain values with a ``kind``:

``solve3d``    HelmholtzSolver3D: the fused Chebyshev x Fourier^2 Helmholtz
               solve (a simulation's time step, a served 3D request);
``chain``      the drop-in sequence scalar_product -> banded solver ->
               backward of a 1D space or a TensorProductSpace (a shenfun
               program moved to the GPU as it stands): chebyshev.la.Helmholtz
               for Chebyshev spaces, la.SolverGeneric1ND for Legendre ones;
``transform``  TensorProductSpace.forward and backward (projection with the
               mass solve, and evaluation: what every pseudo-spectral step
               does);
``convolve``   TensorProductSpace.convolve on the 3/2-rule dealiased space
               (the nonlinear term of such a step);
``batch2d``    BatchedHelmholtz2D: many uneven 2D Legendre x Fourier problems
               in one call.

Inputs are smooth random fields (spectral coefficients N(0, 1) with an
algebraic decay), as the solvers meet them.  ``exact`` recomputes the outputs
in float64 with torch and numpy only.
"""
import math

import numpy as np
import torch

import shenfun_amd as sfa

DEV = "cuda"


def listed():
    return [
        # a small 3D solve: the low end of the served 3D shapes, where the
        # launches count
        dict(name="solve3d_32", kind="solve3d", Nx=32, Ny=32, Nz=32, bc="D", alpha=1.0,
             precision="fp64"),
        # the benchmark's shape in both forms
        dict(name="solve3d_256_fp64", kind="solve3d", Nx=256, Ny=256, Nz=256, bc="D", alpha=1.0,
             precision="fp64"),
        dict(name="solve3d_256_mixed", kind="solve3d", Nx=256, Ny=256, Nz=256, bc="D", alpha=1.0,
             precision="mixed"),
        # the largest benchmarked shape
        dict(name="solve3d_512_mixed", kind="solve3d", Nx=512, Ny=512, Nz=512, bc="D", alpha=1.0,
             precision="mixed"),
        # a grid that is no power of two, Neumann ends
        dict(name="solve3d_ragged", kind="solve3d", Nx=180, Ny=150, Nz=200, bc="N", alpha=7.5,
             precision="fp64"),
        # the drop-in chain in 3D
        dict(name="chain3d_cheb_128", kind="chain", family="chebyshev", dim=3, Nx=128, Ny=128,
             Nz=128, bc="D", alpha=1.0),
        # the 2D Poisson demo
        dict(name="chain2d_leg_64", kind="chain", family="legendre", dim=2, Nx=64, Ny=1, Nz=64,
             bc="D", alpha=0.0),
        # the largest 2D problem of the served mix, Neumann ends
        dict(name="chain2d_leg_512", kind="chain", family="legendre", dim=2, Nx=512, Ny=1, Nz=256,
             bc="N", alpha=25.0),
        # one 1D problem
        dict(name="chain1d_cheb_1024", kind="chain", family="chebyshev", dim=1, Nx=1024, Ny=1,
             Nz=1, bc="D", alpha=12.0),
        # the transforms of a channel-flow-like grid
        dict(name="transform3d_192", kind="transform", family="chebyshev", dim=3, Nx=192, Ny=96,
             Nz=160, bc="N"),
        # a dealiased product
        dict(name="convolve3d_64", kind="convolve", Nx=64, Ny=64, Nz=64, bc="D"),
        # a batch of uneven 2D problems
        dict(name="batch2d_1024", kind="batch2d", n=1024, hi_x=512, hi_y=256, bc="D", mode="wide",
             sizes_seed=0),
    ]


# ------------------------------------------------------------------ drawn cases
def _logint(rng, lo, hi, step=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return max(lo, min(hi, v))


def _shape3(rng, lo, hi, cap):
    """Three log-uniform lengths, the last even, at most cap points."""
    while True:
        s = (_logint(rng, lo, hi), _logint(rng, lo, hi), _logint(rng, lo, hi, 2))
        if s[0] * s[1] * s[2] <= cap:
            return s


def draw(rng):
    kind = rng.choice(["solve3d", "solve3d", "solve3d", "chain", "chain", "chain", "transform",
                       "transform", "convolve", "batch2d"])
    bc = rng.choice("DN")
    alpha = round(rng.uniform(0.5, 50.0), 3)
    if kind == "solve3d":
        form = rng.choice(["ragged", "pow2", "mixed"])
        if form == "ragged":
            Nx, Ny, Nz = _shape3(rng, 16, 320, 6_000_000)
        else:
            Nx = rng.choice([64, 128, 256])
            Ny, Nz = (rng.choice([32, 64, 128, 256]) for _ in range(2))
        return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, bc=bc, alpha=alpha,
                    precision="mixed" if form == "mixed" else "fp64")
    if kind == "chain":
        dim = rng.choice([1, 2, 3])
        family = rng.choice(["chebyshev", "legendre"])
        if dim == 1:
            Nx, Ny, Nz = _logint(rng, 64, 4096 if family == "chebyshev" else 1024), 1, 1
        elif dim == 2:
            Nx, Ny, Nz = _logint(rng, 32, 512), 1, _logint(rng, 32, 512, 2)
        else:
            Nx, Ny, Nz = _shape3(rng, 16, 256, 3_000_000)
        return dict(kind=kind, family=family, dim=dim, Nx=Nx, Ny=Ny, Nz=Nz, bc=bc, alpha=alpha)
    if kind == "transform":
        family = rng.choice(["chebyshev", "chebyshev", "legendre"])
        dim = rng.choice([2, 3])
        Nx, Ny, Nz = _shape3(rng, 16, 384, 4_000_000)
        return dict(kind=kind, family=family, dim=dim, Nx=Nx, Ny=Ny if dim == 3 else 1, Nz=Nz,
                    bc=rng.choice(["", "D", "N"]))
    if kind == "convolve":
        Nx, Ny, Nz = _shape3(rng, 16, 128, 400_000)
        return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, bc=bc)
    return dict(kind=kind, n=_logint(rng, 16, 1024), hi_x=rng.choice([128, 256, 512]),
                hi_y=rng.choice([64, 128, 256]), bc=bc, mode=rng.choice(["wide", "persistent"]),
                sizes_seed=rng.randrange(1000))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _randc(shape, g):
    return torch.complex(torch.randn(shape, generator=g, device=DEV, dtype=torch.float64),
                         torch.randn(shape, generator=g, device=DEV, dtype=torch.float64))


def _freq(n):
    return torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=DEV)


def _poly_nodes(family, N):
    """(x_j, w_j): Chebyshev-Gauss or Legendre-Gauss nodes and weights."""
    if family == "chebyshev":
        th = np.pi * (2 * np.arange(N) + 1) / (2 * N)
        return np.cos(th), np.full(N, np.pi / N)
    # roots of P_N by Newton's iteration, the last steps in extended precision
    x = np.cos(np.pi * (np.arange(N, 0, -1) - 0.25) / (N + 0.5))
    for step in range(5):
        x = x.astype(np.longdouble) if step == 3 else x
        p0, p1 = np.ones_like(x), x
        for k in range(1, N):
            p0, p1 = p1, ((2 * k + 1) * x * p1 - k * p0) / (k + 1)
        dp = N * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / dp
    return x.astype(np.float64), (2 / ((1 - x * x) * dp * dp)).astype(np.float64)


def _vander(family, N, n):
    """P_k(x_j), k < n, at the N nodes of the family."""
    if family == "chebyshev":
        # angles reduced in integers, so that cos sees at most 2 pi
        m = ((2 * np.arange(N)[:, None] + 1) * np.arange(n)[None, :]) % (4 * N)
        return torch.from_numpy(np.cos(np.pi * m / (2 * N))).to(DEV)
    return torch.from_numpy(np.polynomial.legendre.legvander(_poly_nodes(family, N)[0], n - 1)).to(DEV)


def _matmul0(M, x):
    """M contracted with the first axis of a real or complex array."""
    sh = x.shape
    if x.is_complex():
        y = M @ torch.view_as_real(x.contiguous()).reshape(sh[0], -1)
        return torch.view_as_complex(y.reshape(M.shape[0], -1, 2)).reshape((M.shape[0],) + sh[1:])
    return (M @ x.reshape(sh[0], -1)).reshape((M.shape[0],) + sh[1:])


def _field(family, Nx, Ny, Nz, dim, g):
    """Smooth random field on the grid: coefficients N(0, 1) / (1 + |k|^2)^p,
    p = 2 in 3D and 1 below, shape (Nx[, Ny][, Nz])."""
    kx = torch.arange(Nx, dtype=torch.float64, device=DEV)
    if dim == 1:
        c = torch.randn(Nx, generator=g, device=DEV, dtype=torch.float64) / (1 + kx * kx)
        return _vander(family, Nx, Nx) @ c
    kz = torch.arange(Nz // 2 + 1, dtype=torch.float64, device=DEV)
    if dim == 2:
        c = _randc((Nx, kz.numel()), g) / (1 + kx[:, None] ** 2 + kz[None, :] ** 2)
        return torch.fft.irfft(_matmul0(_vander(family, Nx, Nx), c), n=Nz, dim=1, norm="forward")
    k2 = kx[:, None, None] ** 2 + _freq(Ny)[None, :, None] ** 2 + kz[None, None, :] ** 2
    c = _randc((Nx, Ny, kz.numel()), g) / (1 + k2) ** 2
    h = torch.fft.irfftn(c, s=(Ny, Nz), dim=(1, 2), norm="forward")
    return _matmul0(_vander(family, Nx, Nx), h).contiguous()


def _batch_sizes(case):
    """Even sizes log-uniform in [32, hi], alphas uniform in [0.5, 100]."""
    r = np.random.default_rng(case["sizes_seed"])
    n = case["n"]
    nx = 2 * np.round(np.exp(r.uniform(np.log(32), np.log(case["hi_x"]), n)) / 2).astype(np.int64)
    ny = 2 * np.round(np.exp(r.uniform(np.log(32), np.log(case["hi_y"]), n)) / 2).astype(np.int64)
    return nx, ny, r.uniform(0.5, 100.0, n)


def _batch_fields(case, seed):
    """One smooth field per problem, from its lowest 24 x 12 modes."""
    nx, ny, _ = _batch_sizes(case)
    g = _gen(seed)
    mx, my = 24, 12
    kx = torch.arange(mx, dtype=torch.float64, device=DEV)
    ky = torch.arange(my, dtype=torch.float64, device=DEV)
    c = _randc((case["n"], mx, my), g) / (1 + kx[:, None] ** 2 + ky[None, :] ** 2)
    V, E, out = {}, {}, []
    for i, (a, b) in enumerate(zip(nx.tolist(), ny.tolist())):
        if a not in V:
            x = torch.from_numpy(_poly_nodes("legendre", a)[0])
            p = [torch.ones_like(x), x]
            for k in range(1, mx - 1):
                p.append(((2 * k + 1) * x * p[k] - k * p[k - 1]) / (k + 1))
            V[a] = torch.stack(p, 1).to(DEV)
        if b not in E:
            t = torch.arange(b, dtype=torch.float64, device=DEV) * (2 * math.pi / b)
            E[b] = (torch.cos(ky[:, None] * t[None, :]), torch.sin(ky[:, None] * t[None, :]))
        out.append(V[a] @ (c[i].real @ E[b][0] - c[i].imag @ E[b][1]))
    return out


def _dealias_inputs(case, seed):
    """Coefficients of two smooth functions of the space, Nyquist modes and
    boundary slots zero."""
    g = _gen(seed)
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    out = []
    for _ in range(2):
        f = _field("chebyshev", Nx, Ny, Nz, 3, g)
        c = _forward_exact(f, "chebyshev", case["bc"], 3)
        if Ny % 2 == 0:
            c[:, Ny // 2] = 0
        c[:, :, Nz // 2] = 0
        out.append(c.contiguous())
    return out


def _bc(b):
    return {"": None, "D": (0, 0), "N": "Neumann"}[b]


def _space(case):
    bx = sfa.FunctionSpace(case["Nx"], case.get("family", "chebyshev"), bc=_bc(case["bc"]))
    dim = case.get("dim", 3)
    if dim == 1:
        return bx
    bases = [bx, sfa.FunctionSpace(case["Nz"], "F", dtype="d")]
    if dim == 3:
        bases.insert(1, sfa.FunctionSpace(case["Ny"], "F", dtype="D"))
    return sfa.TensorProductSpace(None, tuple(bases))


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.kind = case["kind"]
    if s.kind == "batch2d":
        nx, ny, al = _batch_sizes(case)
        s.H = sfa.BatchedHelmholtz2D(nx, ny, al, case["bc"], mode=case["mode"])
        s.f = s.H.pack(_batch_fields(case, seed))
        s.u = torch.empty_like(s.f)
        return s
    T = s.T = _space(case)
    if s.kind == "convolve":
        s.P = T.get_dealiased(1.5)
        s.a, s.b = _dealias_inputs(case, seed)
        s.c = sfa.Function(T)
        return s
    dim = case.get("dim", 3)
    s.f = _field(case.get("family", "chebyshev"), case["Nx"], case["Ny"], case["Nz"], dim, _gen(seed))
    s.u = torch.empty_like(s.f)
    if s.kind == "solve3d":
        s.H = sfa.HelmholtzSolver3D(T, case["alpha"], precision=case["precision"])
        return s
    s.fh, s.uh = sfa.Function(T), sfa.Function(T)
    if s.kind == "chain":
        if dim == 1:
            A, B = sfa.stiffness_matrix(T), sfa.mass_matrix(T)
            if case["family"] == "chebyshev":
                s.H = sfa.la.Helmholtz(A, B, -1.0, case["alpha"])
            else:
                M = A + B * case["alpha"]
                s.H = M.get_solver()(M)
        else:
            mats = sfa.helmholtz_tpmatrices(T, case["alpha"])
            s.H = (sfa.la.Helmholtz(*mats) if case["family"] == "chebyshev"
                   else sfa.la.SolverGeneric1ND(mats))
    return s


def run(s):
    if s.kind == "solve3d" or s.kind == "batch2d":
        return {"u": s.H(s.f, s.u)}
    if s.kind == "convolve":
        return {"ab_hat": s.P.convolve(s.a, s.b, s.c)}
    if s.kind == "chain":
        fh = s.T.scalar_product(s.f, s.fh)
        uh = s.H(fh, s.uh)
        return {"u_hat": uh, "u": s.T.backward(uh, s.u)}
    fh = s.T.forward(s.f, s.fh)
    return {"f_hat": fh, "f": s.T.backward(fh, s.u)}


# ------------------------------------------------------------------ work
def work(case):
    if case["kind"] == "batch2d":
        nx, ny, _ = _batch_sizes(case)
        x, y = nx.astype(float), ny.astype(float)
        flops = np.sum(4 * (x - 2) * x * (y + 2) + 5 * x * y * np.log2(y) + 12 * x * (y + 2))
        return {"bytes": float(16 * np.sum(x * y)), "flops": float(flops)}
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    dim = case.get("dim", 3)
    Nzh = Nz // 2 + 1 if dim > 1 else 0.5  # 0.5: one real line
    phys = 8.0 * Nx * Ny * Nz
    spec = 16.0 * Nx * Ny * Nzh
    if case["kind"] == "convolve":
        # two spectral inputs and one output; three transforms on the 3/2 grid
        Mx, My, Mz = (int(1.5 * n) for n in (Nx, Ny, Nz))
        fft = 2.5 * Mx * My * Mz * (math.log2(Mx) + math.log2(My) + math.log2(Mz))
        return {"bytes": 3 * spec, "flops": 3 * fft + Mx * My * Mz}
    fourier = (2.5 * Nx * Ny * Nz * math.log2(max(2, Nz)) if dim > 1 else 0.0) + \
        (5.0 * Nx * Ny * Nzh * math.log2(max(2, Ny)) if dim > 2 else 0.0)
    if case.get("family") == "legendre":
        poly = 4.0 * Nx * Nx * Ny * Nzh
    else:
        poly = 5.0 * Nx * math.log2(Nx) * Ny * Nzh
    flops = 2 * (fourier + poly) + 24.0 * Nx * Ny * Nzh
    if case["kind"] == "solve3d":
        return {"bytes": 2 * phys, "flops": flops}
    return {"bytes": 2 * phys + spec, "flops": flops}


# ------------------------------------------------------------------ float64 restatement
def _stencil(family, bc, n):
    """c_k of phi_k = P_k - c_k P_{k+2}, k < n."""
    k = torch.arange(n, dtype=torch.float64, device=DEV)
    if bc == "D":
        return torch.ones_like(k)
    if family == "chebyshev":
        return (k / (k + 2)) ** 2
    return k * (k + 1) / ((k + 2) * (k + 3))


def _norms(family, n):
    k = torch.arange(n, dtype=torch.float64, device=DEV)
    if family == "legendre":
        return 2 / (2 * k + 1)
    h = torch.full_like(k, math.pi / 2)
    h[0] = math.pi
    return h


def _phi(V, c):
    """Basis functions at the nodes from the polynomials' values V (nodes, N)."""
    return V[:, :-2] - V[:, 2:] * c


def _galerkin_solve(family, bc, N, b, a_scale, beta):
    """x of (a_scale K + beta B) x = b along axis 0 (N - 2 rows): B the
    weighted mass matrix and K_kj = -(phi_j'', phi_k)_w.  beta: broadcastable
    against b[0].  Elimination of the one lower band of each parity chain;
    K's upper triangle is g_k w_j, kept as its two factors."""
    M = N - 2
    c, h = _stencil(family, bc, N), _norms(family, N + 2)
    k = torch.arange(N, dtype=torch.float64, device=DEV)
    B0 = h[:N] + c * c * h[2:N + 2]
    B2 = -c * h[2:N + 2]  # (phi_{k+2}, phi_k)
    w = torch.ones_like(k)
    if family == "legendre":
        K0 = 2 * (2 * k + 3) * c  # c = 1: 4k + 6
        g = torch.zeros_like(k)
    elif bc == "D":
        K0 = 2 * math.pi * (k + 1) * (k + 2)
        g = 4 * math.pi * (k + 1)
    else:
        K0 = 2 * math.pi * k * k * (k + 1) / (k + 2)
        g = 4 * math.pi * (k + 1) / (k + 2) ** 2
        w = k * k
    K0, g = (a_scale * K0).tolist(), (a_scale * g).tolist()
    B0, B2, w = B0.tolist(), B2.tolist(), w.tolist()
    beta = torch.as_tensor(beta, dtype=torch.float64, device=DEV).expand(b.shape[1:])
    x = torch.zeros_like(b)
    x[:M] = b[:M]
    for p in (0, 1):
        rows = list(range(p, M, 2))
        D, G, F = {}, {}, {}
        for i in rows:
            d = K0[i] + beta * B0[i]
            e = g[i] * w[i + 2] + beta * B2[i] if i + 2 < M else torch.zeros_like(beta)
            f = torch.full_like(beta, g[i])
            if i > p:
                r = beta * B2[i - 2] / D[i - 2]
                d = d - r * G[i - 2]
                if i + 2 < M:
                    e = e - r * F[i - 2] * w[i + 2]
                f = f - r * F[i - 2]
                x[i] -= r * x[i - 2]
            D[i], G[i], F[i] = d, e, f
        S = torch.zeros_like(x[0])
        for i in reversed(rows):
            v = x[i]
            if i + 2 < M:
                v = v - G[i] * x[i + 2]
            if i + 4 < M:
                S = S + w[i + 4] * x[i + 4]
                v = v - F[i] * S
            x[i] = v / D[i]
            del D[i], G[i], F[i]
    return x


def _fourier_forward(f, dim, norm="forward"):
    if dim == 1:
        return f
    c = torch.fft.rfft(f, dim=-1, norm=norm)
    return torch.fft.fft(c, dim=1, norm=norm) if dim == 3 else c


def _fourier_backward(c, dim, n):
    if dim == 1:
        return c
    if dim == 3:
        c = torch.fft.ifft(c, dim=1, norm="forward")
    return torch.fft.irfft(c, n=n, dim=-1, norm="forward")


def _beta(case_alpha, Ny, Nz, dim):
    if dim == 1:
        return torch.tensor(case_alpha, dtype=torch.float64, device=DEV)
    kz = torch.arange(Nz // 2 + 1, dtype=torch.float64, device=DEV)
    if dim == 2:
        return case_alpha + kz ** 2
    return case_alpha + _freq(Ny)[:, None] ** 2 + kz[None, :] ** 2


def _forward_exact(f, family, bc, dim):
    """Coefficients of the projection of f on the space."""
    N = f.shape[0]
    c = _fourier_forward(f, dim)
    _, w = _poly_nodes(family, N)
    V = _vander(family, N, N)
    w = torch.from_numpy(np.ascontiguousarray(w)).to(DEV)
    if not bc:
        h = _norms(family, N)
        return _matmul0((V * w[:, None]).T.contiguous() / h[:, None], c)
    P = _phi(V, _stencil(family, bc, N - 2))
    s = torch.zeros_like(c)
    s[:N - 2] = _matmul0((P * w[:, None]).T.contiguous(), c)
    return _galerkin_solve(family, bc, N, s, 0.0, 1.0)


def _backward_exact(c, family, bc, dim, Nz):
    N = c.shape[0]
    V = _vander(family, N, N)
    if not bc:
        h = _matmul0(V, c)
    else:
        h = _matmul0(_phi(V, _stencil(family, bc, N - 2)), c[:N - 2])
    return _fourier_backward(h, dim, Nz)


def _solve_exact(f, family, bc, dim, alpha):
    """(u_hat, u) of (alpha - lap) u = f."""
    N, Nz = f.shape[0], f.shape[-1]
    Ny = f.shape[1] if dim == 3 else 1
    c = _fourier_forward(f, dim)
    V = _vander(family, N, N)
    w = torch.from_numpy(np.ascontiguousarray(_poly_nodes(family, N)[1])).to(DEV)
    P = _phi(V, _stencil(family, bc, N - 2))
    s = torch.zeros_like(c)
    s[:N - 2] = _matmul0((P * w[:, None]).T.contiguous(), c)
    uh = _galerkin_solve(family, bc, N, s, 1.0, _beta(alpha, Ny, Nz, dim))
    if family == "legendre":  # those solvers leave the right-hand side's last two rows in place
        uh[N - 2:] = _matmul0((V[:, N - 2:] * w[:, None]).T.contiguous(), c)
    return uh, _fourier_backward(_matmul0(P, uh[:N - 2]), dim, Nz)


def _pad_fourier(c, axis, N, M):
    """Coefficients in fft order along axis, N -> M (Nyquist mode zero)."""
    h = (N - 1) // 2
    shp = list(c.shape)
    shp[axis] = M
    out = torch.zeros(shp, dtype=c.dtype, device=c.device)
    out.narrow(axis, 0, h + 1).copy_(c.narrow(axis, 0, h + 1))
    out.narrow(axis, M - h, h).copy_(c.narrow(axis, N - h, h))
    return out


def _convolve_exact(case, seed):
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    Mx, My, Mz = (int(math.floor(1.5 * n)) for n in (Nx, Ny, Nz))
    V = _vander("chebyshev", Mx, Nx)
    P = _phi(V, _stencil("chebyshev", case["bc"], Nx - 2))
    vals = []
    for c in _dealias_inputs(case, seed):
        h = _pad_fourier(_matmul0(P, c[:Nx - 2]), 1, Ny, My)
        h = torch.fft.ifft(h, dim=1, norm="forward")
        vals.append(torch.fft.irfft(h, n=Mz, dim=2, norm="forward"))
    c = torch.fft.rfft(vals[0] * vals[1], dim=2, norm="forward")[:, :, :Nz // 2 + 1].clone()
    # a Nyquist coefficient of the unpadded space takes both of its aliases
    c[:, :, Nz // 2] = 2 * c[:, :, Nz // 2].real
    c = torch.fft.fft(c, dim=1, norm="forward")
    h = Ny // 2
    t = torch.zeros((Mx, Ny, Nz // 2 + 1), dtype=c.dtype, device=DEV)
    t[:, :h + 1] = c[:, :h + 1]
    if h:
        t[:, Ny - h:] += c[:, My - h:]
    s = torch.zeros((Nx, Ny, Nz // 2 + 1), dtype=c.dtype, device=DEV)
    s[:Nx - 2] = _matmul0(P.T.contiguous() * (math.pi / Mx), t)
    return {"ab_hat": _galerkin_solve("chebyshev", case["bc"], Nx, s, 0.0, 1.0)}


def _dft(n):
    """exp(-2 pi i j k / n) / n, j < n, k <= n/2."""
    m = (np.arange(n)[:, None] * np.arange(n // 2 + 1)[None, :]) % n
    return torch.from_numpy(np.exp(-2j * np.pi * m / n) / n).to(DEV)


def _batch_exact(case, seed):
    """All problems' (mode, parity) systems by one elimination over the lines
    of the whole batch, padded to the longest with unit rows."""
    nx, ny, al = _batch_sizes(case)
    fs = _batch_fields(case, seed)
    bc, top = case["bc"], int(nx.max())
    cols, beta, length, basis = [], [], [], {}
    for f, a, b, alpha in zip(fs, nx.tolist(), ny.tolist(), al.tolist()):
        if a not in basis:
            _, w = _poly_nodes("legendre", a)
            P = _phi(_vander("legendre", a, a), _stencil("legendre", bc, a - 2))
            basis[a] = (P, (P * torch.from_numpy(w).to(DEV)[:, None]).T.contiguous())
        s = torch.zeros((top, b // 2 + 1), dtype=torch.complex128, device=DEV)
        s[:a - 2] = basis[a][1].to(s.dtype) @ (f.to(s.dtype) @ _dft(b))
        cols.append(s)
        beta.append(alpha + torch.arange(b // 2 + 1, dtype=torch.float64, device=DEV) ** 2)
        length += [a - 2] * (b // 2 + 1)
    x, beta = torch.cat(cols, 1), torch.cat(beta)
    m = torch.tensor(length, device=DEV)
    c, h = _stencil("legendre", bc, top), _norms("legendre", top + 2)
    k = torch.arange(top, dtype=torch.float64, device=DEV)
    K0 = 2 * (2 * k + 3) * c
    B0, B2 = h[:top] + c * c * h[2:top + 2], -c * h[2:top + 2]
    for p in (0, 1):
        D, E = {}, {}
        rows = list(range(p, top - 2, 2))
        for i in rows:
            inside = i < m
            d = torch.where(inside, K0[i] + beta * B0[i], 1.0)
            E[i] = torch.where(i + 2 < m, beta * B2[i], 0.0)
            if i > p:
                r = E[i - 2] / D[i - 2]
                d = d - r * E[i - 2]
                x[i] -= r * x[i - 2]
            D[i] = d
        for i in reversed(rows):
            x[i] = (x[i] - E[i] * x[i + 2]) / D[i] if i + 2 < top - 2 else x[i] / D[i]
    out, o = [], 0
    for a, b in zip(nx.tolist(), ny.tolist()):
        uh = x[:a - 2, o:o + b // 2 + 1]
        o += b // 2 + 1
        weight = torch.full((b // 2 + 1,), 2.0 * b, dtype=torch.float64, device=DEV)
        weight[0] = weight[-1] = b
        h = basis[a][0].to(uh.dtype) @ uh
        out.append(((h * weight) @ _dft(b).mH).real.reshape(-1))
    return {"u": torch.cat(out)}


def exact(case, seed):
    if case["kind"] == "batch2d":
        return _batch_exact(case, seed)
    if case["kind"] == "convolve":
        return _convolve_exact(case, seed)
    dim, family = case.get("dim", 3), case.get("family", "chebyshev")
    f = _field(family, case["Nx"], case["Ny"], case["Nz"], dim, _gen(seed))
    if case["kind"] == "transform":
        c = _forward_exact(f, family, case["bc"], dim)
        return {"f_hat": c, "f": _backward_exact(c, family, case["bc"], dim, f.shape[-1])}
    uh, u = _solve_exact(f, family, case["bc"], dim, case["alpha"])
    return {"u": u} if case["kind"] == "solve3d" else {"u_hat": uh, "u": u}
