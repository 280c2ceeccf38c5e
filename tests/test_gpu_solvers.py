"""GPU parity: banded solvers and the Chebyshev Helmholtz solver vs the FP64 oracle."""
import numpy as np
import pytest
import torch

from oracle import spectral as S

pytestmark = pytest.mark.gpu
TOL = 1e-12


def rel(a, b):
    a = a.cpu().numpy() if isinstance(a, torch.Tensor) else a
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.fixture(scope="module")
def sfa():
    import shenfun_amd
    return shenfun_amd


# tests/test_la.py:8-15 of the reference (N = 10 matrices: DiagMA, TwoDMA,
# TDMA_O, TDMA, FDMA, PDMA), plus ThreeDMA and HeptaDMA systems
N10 = 10
MATS = [
    {0: np.arange(N10) + 1.0},
    {0: -2.0, 2: 1.0},
    {-1: 1.0, 0: -2.0, 1: 1.0},
    {-2: 1.0, 0: -2.0, 2: 1.0},
    {-2: 1.0, 0: -2.0, 2: 1.0, 4: 0.1},
    {-4: 0.1, -2: 1.0, 0: -2.0, 2: 1.0, 4: 0.1},
    {0: -2.0, 2: 1.0, 4: 0.3},
    {-4: 0.1, -2: 0.5, 0: -4.0, 2: 1.0, 4: 0.3, 6: -0.2, 8: 0.1},
]

# pattern -> (offsets, oracle LU, oracle solve, C-ABI LU, C-ABI solve)
BANDS = {
    "twodma": ((0, 2), None, "twodma_solve", None, "sfa_twodma_solve"),
    "tdma_o": ((-1, 0, 1), "tdma_o_lu", "tdma_o_solve", "sfa_tdma_o_lu", "sfa_tdma_o_solve"),
    "threedma": ((0, 2, 4), None, "threedma_solve", None, "sfa_threedma_solve"),
    "fdma": ((-2, 0, 2, 4), "fdma_lu", "fdma_solve", "sfa_fdma_lu", "sfa_fdma_solve"),
    "heptadma": ((-4, -2, 0, 2, 4, 6, 8), "heptadma_lu", "heptadma_solve", "sfa_heptadma_lu",
                 "sfa_heptadma_solve"),
}


def _rand_bands(rng, offs, n):
    d = {o: rng.uniform(0.2, 1.0, n - abs(o)) * (1 if o % 4 else -1) for o in offs}
    d[0] = rng.uniform(4.0, 5.0, n)
    return d


@pytest.mark.parametrize("kind", sorted(BANDS))
@pytest.mark.parametrize("n", [8, 9, 64, 255])
def test_band_patterns_per_line_factors(sfa, kind, n):
    """Per-line factors (data_line_stride) and skip_lines through the C ABI, LU
    on the device for all lines at once, against the oracle per line; the
    space axis is strided (axis 1 of (lines, n, 3))."""
    from shenfun_amd import _lib
    print(f"[band {kind} n={n}]", flush=True)
    offs, olu, osol, clu, csol = BANDS[kind]
    rng = np.random.default_rng(n + len(offs))
    nl = 5
    mats = [_rand_bands(rng, offs, n) for _ in range(nl * 3)]
    data = np.stack([S.band_dia(d, n, offs) for d in mats])  # (lines, rows, n)
    dd = dev(data)
    if clu is not None:
        _lib.call(clu, _lib.ptr(dd), n, nl * 3, _lib.stream_ptr())
    b = rng.standard_normal((nl, n, 3)) + 1j * rng.standard_normal((nl, n, 3))
    u = dev(b)
    _lib.call(csol, _lib.ptr(u), _lib.C128, 3, _lib.arr(u.shape), _lib.arr(u.stride()), 1,
              _lib.ptr(dd), n, data.shape[1] * n, 1, _lib.stream_ptr())
    got = u.cpu().numpy()
    assert np.array_equal(got[0, :, 0], b[0, :, 0])  # line 0 skipped
    for i in range(nl):
        for j in range(3):
            L = i * 3 + j
            if L == 0:
                continue
            ld = getattr(S, olu)(data[L]) if olu else data[L]
            if olu:
                assert rel(dd[L], ld) < 1e-13
            ref = getattr(S, osol)(b[i, :, j], ld, 0)
            assert rel(got[i, :, j], ref) < TOL
            assert rel(got[i, :, j], np.linalg.solve(S.dense(mats[L], n), b[i, :, j])) < 1e-11


@pytest.mark.parametrize("kind", sorted(BANDS))
def test_band_patterns_constraint_row0(sfa, kind):
    """apply_constraints((0, val)): row 0 becomes the unit row and b[0] = val
    (la.py:575-586, 628-637, 674-684, 724-741)."""
    offs = BANDS[kind][0]
    n = 14
    rng = np.random.default_rng(7)
    d = _rand_bands(rng, offs, n)
    if kind == "tdma_o":
        d[1] = d[-1]  # get_solver takes TDMA_O for symmetric (-1, 0, 1) only
    M = sfa.SparseMatrix(d, (n, n))
    sol = sfa.la.Solver(M)
    assert type(sol).__name__.lower() == kind
    b = rng.standard_normal((n, 4))
    u = sol(dev(b), axis=0, constraints=((0, 0.25),))
    D = S.dense(d, n)
    D[0, :] = 0.0
    D[0, 0] = 1.0
    bb = b.copy()
    bb[0] = 0.25
    assert rel(u, np.linalg.solve(D, bb)) < 1e-11


@pytest.mark.parametrize("di", MATS)
@pytest.mark.parametrize("cplx", [False, True])
def test_xdma(sfa, di, cplx):
    print(f"[xdma {sorted(di)} cplx={cplx}]", flush=True)
    M = sfa.SparseMatrix(di, (N10, N10))
    sol = sfa.la.Solver(M)
    dense = S.dense(di, N10)
    rng = np.random.default_rng(0)
    b = rng.standard_normal(N10) + (1j * rng.standard_normal(N10) if cplx else 0)
    u = sol(dev(b))
    assert rel(u, np.linalg.solve(dense, b)) < TOL
    bh = rng.standard_normal((N10, N10, 3)) + (1j * rng.standard_normal((N10, N10, 3)) if cplx else 0)
    for axis in (0, 1):
        uh = sol(dev(bh), axis=axis)
        ref = np.moveaxis(np.linalg.solve(dense, np.moveaxis(bh, axis, 0).reshape(N10, -1))
                          .reshape(np.moveaxis(bh, axis, 0).shape), 0, axis)
        assert rel(uh, ref) < TOL


@pytest.mark.parametrize("n", [6, 7, 64, 255])
def test_tdma_pdma_vs_oracle(sfa, n):
    rng = np.random.default_rng(n)
    d3 = {-2: rng.uniform(0.1, 1, n - 2), 0: rng.uniform(3, 4, n), 2: rng.uniform(0.1, 1, n - 2)}
    d5 = {-4: rng.uniform(0.1, .3, n - 4), -2: rng.uniform(0.1, 1, n - 2), 0: rng.uniform(4, 5, n),
          2: rng.uniform(0.1, 1, n - 2), 4: rng.uniform(0.1, .3, n - 4)}
    b = rng.standard_normal((n, 9)) + 1j * rng.standard_normal((n, 9))
    u3 = sfa.la.TDMA(sfa.SparseMatrix(d3, (n, n)))(dev(b), axis=0)
    assert rel(u3, S.tdma_solve(b, S.tdma_lu(S.tdma_dia(d3, n)), 0)) < TOL
    u5 = sfa.la.PDMA(sfa.SparseMatrix(d5, (n, n)))(dev(b), axis=0)
    assert rel(u5, S.pdma_solve(b, S.pdma_lu(S.pdma_dia(d5, n)), 0)) < TOL


@pytest.mark.parametrize("bc", ["D", "N"])
@pytest.mark.parametrize("shape,axis", [((20,), 0), ((32, 7, 5), 0), ((6, 40, 5), 1), ((4, 5, 66), 2),
                                        ((256, 16, 9), 0), ((1024,), 0), ((4096, 3), 0), ((2, 2050), 1)])
def test_helmholtz(sfa, bc, shape, axis):
    """Chebyshev Helmholtz LU/solve/matvec vs the oracle; N >= 514 with few
    lines takes the LDS-staged long-chain solve."""
    print(f"[helmholtz {bc} {shape} axis={axis}]", flush=True)
    N = shape[axis]
    rng = np.random.default_rng(N)
    mshape = list(shape)
    mshape[axis] = 1
    alfa = -np.ones(mshape) * rng.uniform(0.5, 2)
    beta = rng.uniform(0.5, 50, mshape)
    if bc == "N":
        beta.flat[0] = 0.0  # the k = 0 Neumann gauge
    V = sfa.FunctionSpace(N, "chebyshev", bc=bc)
    V.axis = axis

    class _T:  # minimal tensor-product stand-in carrying the shape
        def __init__(self, s):
            self._s = s

        def shape(self, fo=True):
            return tuple(self._s)

    A = sfa.stiffness_matrix(V)
    B = sfa.mass_matrix(V)
    if len(shape) > 1:
        V.tensorproductspace = _T(shape)
    H = sfa.la.Helmholtz(A, B, alfa, beta)
    b = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    u = H(dev(b), torch.zeros(shape, dtype=torch.complex128, device="cuda"))
    d0, d1, d2, L = S.helmholtz_lu(bc, N, np.moveaxis(alfa, axis, 0)[0], np.moveaxis(beta, axis, 0)[0])
    uref = S.helmholtz_solve(np.moveaxis(b, axis, 0), d0, d1, d2, L, neumann=(bc == "N"))
    uref = np.moveaxis(uref, 0, axis)
    assert rel(u, uref) < TOL
    # factors match the reference LU (la.pyx:717-763)
    for got, ref in zip((H.u0, H.u1, H.u2, H.L), (d0, d1, d2, L)):
        assert rel(torch.movedim(got, axis, 0), ref) < TOL
    # matvec of the solution reproduces b on the unknowns (except the gauge row)
    c = H.matvec(u, torch.zeros_like(u))
    cref = S.helmholtz_matvec(uref, np.moveaxis(alfa, axis, 0)[0] if len(shape) > 1 else alfa,
                              np.moveaxis(beta, axis, 0)[0] if len(shape) > 1 else beta, bc, axis)
    assert rel(c, cref) < TOL


@pytest.mark.parametrize("N", [8, 64, 255])
def test_poisson_add(sfa, N):
    V = sfa.FunctionSpace(N, "chebyshev", bc="D")
    A = sfa.stiffness_matrix(V)
    rng = np.random.default_rng(5)
    b = rng.standard_normal((N, 4)) + 1j * rng.standard_normal((N, 4))
    u = sfa.la.ADDSolver(A)(dev(b), torch.zeros(N, 4, dtype=torch.complex128, device="cuda"))
    ref = S.poisson_add_solve(b, N)
    assert rel(u[:N - 2], ref[:N - 2]) < TOL
    dense = S.dense(S.cheb_A_SD(N), N - 2)
    assert rel(u[:N - 2], np.linalg.solve(dense, b[:N - 2])) < 1e-11


@pytest.mark.parametrize("di", MATS)
@pytest.mark.parametrize("axis", [0, 1])
def test_sparse_matvec(sfa, di, axis):
    """SparseMatrix.matvec (matrixbase.py:87-144) along an axis vs numpy."""
    print(f"[matvec {sorted(di)} axis={axis}]", flush=True)
    M = sfa.SparseMatrix(di, (N10, N10), scale=1.5)
    rng = np.random.default_rng(3)
    shp = [12, 4, 3]
    shp[axis] = N10 + 2  # the vector is longer than the matrix: rows >= N come out zero
    v = rng.standard_normal(shp) + 1j * rng.standard_normal(shp)
    c = torch.full(shp, 7.0 + 1j, dtype=torch.complex128, device="cuda")
    M.matvec(dev(v), c, axis=axis)
    vm = np.moveaxis(v, axis, 0)
    ref = np.zeros_like(vm)
    ref[:N10] = np.tensordot(1.5 * S.dense(di, N10), vm[:N10], axes=(1, 0))
    assert rel(c, np.moveaxis(ref, 0, axis)) < 1e-14


def test_matvec_dense_tail_and_tpmatrix(sfa):
    """The Chebyshev stiffness matrix (N/2 diagonals) and TPMatrix.matvec with
    its per-mode scale (matrixbase.py:1437-1449)."""
    SD = sfa.FunctionSpace(40, "C", bc="D")
    K = sfa.FunctionSpace(8, "F", dtype="d")
    T = sfa.TensorProductSpace(None, (SD, K))
    A, B = sfa.helmholtz_tpmatrices(T, 2.0)
    rng = np.random.default_rng(4)
    shp = T.shape(True)
    u = rng.standard_normal(shp) + 1j * rng.standard_normal(shp)
    u[38:] = 0
    c = torch.zeros(shp, dtype=torch.complex128, device="cuda")
    B.matvec(dev(u), c)
    A.matvec(dev(u), c, accumulate=True)
    ref = np.zeros_like(u)
    for m in range(shp[1]):
        Mm = A.scale.reshape(-1)[0] * A.pmat.todense() * float(A.pmat.scale) + \
            B.scale.reshape(-1)[m] * B.pmat.todense() * float(B.pmat.scale)
        ref[:38, m] = Mm @ u[:38, m]
    assert rel(c, ref) < 1e-13


@pytest.mark.parametrize("case", ["legendre", "pg", "bc"])
def test_solver_generic_matvec_roundtrip(sfa, case):
    """SolverGeneric1ND.matvec then the solve returns u (the reference's
    G.matvec check, tests/test_matrices.py:594-621)."""
    print(f"[generic matvec {case}]", flush=True)
    bc = (0.5, -1.0) if case == "bc" else (0, 0)
    fam = "L" if case != "pg" else "C"
    SD = sfa.FunctionSpace(24, fam, bc=bc)
    T = sfa.TensorProductSpace(None, (SD, sfa.FunctionSpace(12, "F", dtype="d")))
    test = T.get_testspace("PG") if case == "pg" else None
    G = sfa.la.SolverGeneric1ND(sfa.helmholtz_tpmatrices(T, 1.5, test=test))
    rng = np.random.default_rng(5)
    shp = T.shape(True)
    u = rng.standard_normal(shp) + 1j * rng.standard_normal(shp)
    u[22:] = 0
    ud = dev(u)
    if case == "bc":
        SD.set_boundary_dofs(ud, final=True)
    c = torch.zeros(shp, dtype=torch.complex128, device="cuda")
    G.matvec(ud, c)
    uc = G(c, sfa.Function(T))
    assert rel(uc, ud.cpu().numpy()) < 1e-11


@pytest.mark.parametrize("shape,axis", [((3,), 0), ((257, 40, 52), 0), ((261, 2, 1030), 0), ((516, 17, 31), 0),
                                        ((1030, 130, 4), 0), ((513, 5), 0), ((4105, 3), 0), ((3, 4105), 1),
                                        ((2, 70, 1100), 1)])
@pytest.mark.parametrize("cplx", [False, True])
def test_chain_scan_shapes(sfa, shape, axis, cplx):
    """The segmented TDMA and Helmholtz solves at the edges of their splits
    (16, 4 or 1 lines per workgroup; one chunk of rows or several; a chain one
    row short of, at and beyond a segment boundary), one set of factors and
    one per line, vs the oracle."""
    print(f"[chain scan {shape} axis={axis} cplx={cplx}]", flush=True)
    from shenfun_amd import _lib
    rng = np.random.default_rng(sum(shape))
    N = shape[axis]
    b = rng.standard_normal(shape) + (1j * rng.standard_normal(shape) if cplx else 0.0)
    d3 = {0: rng.uniform(2, 3, N), -2: rng.uniform(0.1, 1, N - 2), 2: rng.uniform(0.1, 1, N - 2)}
    lu = S.tdma_lu(S.tdma_dia(d3, N))
    assert rel(sfa.la.TDMA(sfa.SparseMatrix(d3, (N, N)))(dev(b), axis=axis),
               S.tdma_solve(b, lu, axis)) < TOL
    nl = b.size // N
    if nl <= 2048:  # factors per line, the first line skipped
        sc = rng.uniform(0.5, 2.0, nl)
        data = dev(sc[:, None, None] * S.tdma_dia(d3, N)[None])
        _lib.call("sfa_tdma_lu", _lib.ptr(data), N, nl, _lib.stream_ptr())
        u = dev(b)
        _lib.call("sfa_tdma_solve", _lib.ptr(u), _lib.C128 if cplx else _lib.F64, u.dim(),
                  _lib.arr(u.shape), _lib.arr(u.stride()), axis, _lib.ptr(data), N, 3 * N, 1,
                  _lib.stream_ptr())
        ref = np.moveaxis(S.tdma_solve(b, lu, axis), axis, -1).reshape(nl, N) / sc[:, None]
        ref[0] = np.moveaxis(b, axis, -1).reshape(nl, N)[0]
        assert rel(np.moveaxis(u.cpu().numpy(), axis, -1).reshape(nl, N), ref) < TOL
    if N < 8:
        return
    ab = [1 if i == axis else n for i, n in enumerate(shape)]
    beta = rng.uniform(0.5, 50, ab)
    for bc in ("D", "N"):
        V = sfa.FunctionSpace(N, "chebyshev", bc=bc)
        V.axis = axis
        if len(shape) > 1:
            class _T:
                def shape(self, fo=True):
                    return tuple(shape)
            V.tensorproductspace = _T()
        H = sfa.la.Helmholtz(sfa.stiffness_matrix(V), sfa.mass_matrix(V), -np.ones(ab), beta)
        bd = dev(b)
        got = H(bd, torch.zeros_like(bd))
        f = S.helmholtz_lu(bc, N, np.moveaxis(-np.ones(ab), axis, 0)[0], np.moveaxis(beta, axis, 0)[0])
        ref = np.moveaxis(S.helmholtz_solve(np.moveaxis(b, axis, 0), *f, neumann=(bc == "N")), 0, axis)
        assert rel(got, ref) < TOL
        # in place (u = b) the rows of the system are the same
        assert torch.equal(H(bd).narrow(axis, 0, N - 2), got.narrow(axis, 0, N - 2))


def test_chain_scan_zero_lines(sfa):
    """Lines of zeros stay zero where the product of a chain's multipliers
    overflows (multipliers above 1 over 1,000 rows), as row by row."""
    n = 2000
    d3 = {0: np.full(n, 1.0), -2: np.full(n - 2, 99.0), 2: np.full(n - 2, 1e-4)}
    b = np.zeros((n, 3))
    u = sfa.la.TDMA(sfa.SparseMatrix(d3, (n, n)))(dev(b), axis=0)
    assert torch.equal(u, torch.zeros_like(u))


@pytest.mark.parametrize("shape,axis", [((12,), 0), ((9, 40, 60), 0), ((5, 33, 7), 1), ((3, 700), 1)])
def test_tdma_mass_solve(sfa, shape, axis):
    """sfa_tdma_mass_solve: the solve's bits, the rows after the system zero, a
    system that would not fit its line refused."""
    from shenfun_amd import _lib
    rng = np.random.default_rng(shape[axis])
    N = shape[axis]
    n = N - 2
    d3 = {0: rng.uniform(2, 3, n), -2: rng.uniform(0.1, 1, n - 2), 2: rng.uniform(0.1, 1, n - 2)}
    lu = dev(S.tdma_lu(S.tdma_dia(d3, n)))
    b = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    u, v = dev(b), dev(b)
    args = lambda t: (_lib.ptr(t), _lib.C128, t.dim(), _lib.arr(t.shape), _lib.arr(t.stride()), axis,  # noqa: E731
                      _lib.ptr(lu))
    _lib.call("sfa_tdma_solve", *args(u), n, 0, 0, _lib.stream_ptr())
    _lib.call("sfa_tdma_mass_solve", *args(v), n, 2, _lib.stream_ptr())
    assert torch.equal(v.narrow(axis, 0, n), u.narrow(axis, 0, n))
    assert not bool(v.narrow(axis, n, 2).any())
    with pytest.raises(RuntimeError):
        _lib.call("sfa_tdma_mass_solve", *args(v), n, 3, _lib.stream_ptr())


@pytest.mark.parametrize("kind", ["TDMA", "Helmholtz", "DiagMA"])
def test_solve_line_counts_past_one_grid(sfa, kind):
    """Many short contiguous lines: more workgroups (or, for the elementwise
    solve, threads) than one dimension of a launch may hold.  The lines repeat
    64 different ones, so every block of 64 has their solution."""
    print(f"[line counts past one grid: {kind}]", flush=True)
    from shenfun_amd import _lib
    N, reps = 8, (1 << 23 if kind == "DiagMA" else 1 << 21) + 1
    if torch.cuda.mem_get_info()[0] < 3 * 64 * reps * N * 8:
        pytest.skip("needs three arrays of the size")
    rng = np.random.default_rng(5)
    b = rng.standard_normal((64, N))
    u = dev(b).repeat(reps, 1)
    if kind == "Helmholtz":
        f = S.helmholtz_lu("D", N, -np.ones(1), np.full(1, 3.0))
        ref = S.helmholtz_solve(b.T.copy(), *f, neumann=False).T
        fd = [dev(np.ascontiguousarray(x.reshape(-1))) for x in f]
        _lib.call("sfa_helmholtz_solve", _lib.ptr(u), _lib.ptr(u), _lib.F64, 2, _lib.arr(u.shape),
                  _lib.arr(u.stride()), _lib.arr(u.stride()), 1, 0, *[_lib.ptr(x) for x in fd],
                  _lib.arr((0, 1)), _lib.stream_ptr())
    else:
        d = {0: rng.uniform(2, 3, N)}
        if kind == "TDMA":
            d.update({-2: rng.uniform(0.1, 1, N - 2), 2: rng.uniform(0.1, 1, N - 2)})
            ref = S.tdma_solve(b, S.tdma_lu(S.tdma_dia(d, N)), 1)
        else:
            ref = b / d[0]
        getattr(sfa.la, kind)(sfa.SparseMatrix(d, (N, N)))(u, axis=1)
    n = N - 2 if kind == "Helmholtz" else N
    u = u.view(reps, 64, N)[:, :, :n]
    r = dev(np.ascontiguousarray(ref[:, :n]))
    assert float((u - r).abs_().amax()) < TOL * float(r.abs().max())


@pytest.mark.parametrize("lines,axis", [(1, 0), (600, 0), (2050, 0), (5, 1), (2050, 1)])
@pytest.mark.parametrize("solver", ["tdma", "helmholtz"])
@pytest.mark.parametrize("sweep", ["forward", "backward"])
def test_chain_scan_range(sfa, lines, axis, solver, sweep):
    """One value per chain carried over 1,000 rows by multipliers whose product
    over a wave's rows (256, 128 or 32 of them) leaves the range of a double in
    either direction, while the values never do.  All of it is powers of two,
    so the result is exact row by row."""
    print(f"[chain range {solver} {sweep} lines={lines} axis={axis}]", flush=True)
    from shenfun_amd import _lib
    n = 2000
    K = n // 2
    for g, sign in ((4, 1), (8, 1), (33, 1), (4, -1), (8, -1), (33, -1)):
        # x_m = -2^steps[m-1] x_{m-1} along the sweep: level, 2^2000 up (or
        # down) from the first row of a wave on, level
        m0 = 255 if sweep == "forward" else 231
        steps = np.zeros(K - 1, dtype=int)
        steps[m0:m0 + 2000 // g] = g * sign
        ex = -1000 * sign + np.concatenate([[0], np.cumsum(steps)])
        x = np.ldexp((-1.0) ** np.arange(K), ex)
        mult = np.ldexp(1.0, steps)
        if sweep == "backward":
            x, mult = x[::-1], mult[::-1]
        start = 0 if sweep == "forward" else K - 1
        ref, rhs = np.repeat(x, 2)[None, :], np.zeros((1, n))  # rows 2 m and 2 m + 1 alike
        rhs[0, [2 * start, 2 * start + 1]] = x[start]
        sc = np.ldexp(1.0, np.arange(lines) % 4)[:, None]
        ref, rhs = sc * ref, sc * rhs
        m2 = np.repeat(mult, 2)
        z = np.zeros(n)
        lo, hi = (m2, 0 * m2) if sweep == "forward" else (0 * m2, m2)
        N = n + 2 if solver == "helmholtz" else n
        b = np.zeros((lines, N))
        b[:, :n] = rhs
        u = dev(b if axis == 1 else b.T)
        shp, st = _lib.arr(u.shape), _lib.arr(u.stride())
        if solver == "tdma":
            d = dev(np.stack([np.append(lo, [0, 0]), np.ones(n), np.append([0, 0], hi)]))
            _lib.call("sfa_tdma_solve", _lib.ptr(u), _lib.F64, 2, shp, st, axis, _lib.ptr(d), n, 0, 0,
                      _lib.stream_ptr())
        else:
            f = [dev(np.append(v, np.zeros(N - v.size))) for v in (np.ones(N), hi, z, lo)]
            _lib.call("sfa_helmholtz_solve", _lib.ptr(u), _lib.ptr(u), _lib.F64, 2, shp, st, st, axis, 0,
                      *[_lib.ptr(v) for v in f], _lib.arr((0, 1) if axis == 1 else (1, 0)), _lib.stream_ptr())
        got = u.cpu().numpy() if axis == 1 else u.cpu().numpy().T
        assert np.max(np.abs(got[:, :n] / ref - 1.0)) < 1e-12


@pytest.mark.parametrize("N,lines,axis", [
    (10, 300, 0), (18, 8201, 0), (19, 8192, 0), (34, 8250, 0), (35, 2050, 0), (66, 8201, 0),  # 64, 16
    (67, 1030, 0), (130, 1500, 0), (131, 600, 0), (194, 2050, 0), (196, 2049, 0), (258, 2100, 0),  # 8, 4, 16
    (260, 1100, 0), (386, 2048, 0), (388, 2050, 0), (514, 2050, 0), (516, 130, 0), (516, 2050, 0),  # 8, 16 (reals), 4
    (260, 65540, 0), (516, 65600, 0),  # 64, several chunks
    (10, 2051, 1), (18, 40, 1), (34, 2050, 1), (66, 2050, 1), (67, 129, 1), (67, 128, 1), (130, 2050, 1),
    (258, 2050, 1), (514, 2050, 1), (516, 2050, 1)])
@pytest.mark.parametrize("cplx", [False, True])
def test_chain_scan_lines_per_workgroup(sfa, N, lines, axis, cplx):
    """Every number of lines per workgroup and rows per thread that the solves
    choose between, at and one past the limits of rows (K = (N - 1) // 2 for a
    system of N - 2) and lines, across and along memory; 32 different lines,
    repeated, vs the oracle."""
    print(f"[chain lines N={N} lines={lines} axis={axis} cplx={cplx}]", flush=True)
    from shenfun_amd import _lib
    rng = np.random.default_rng(N + lines)
    n = N - 2
    b = rng.standard_normal((N, 32)) + (1j * rng.standard_normal((N, 32)) if cplx else 0.0)
    d3 = {0: rng.uniform(2, 3, n), -2: rng.uniform(0.1, 1, n - 2), 2: rng.uniform(0.1, 1, n - 2)}
    lu = S.tdma_lu(S.tdma_dia(d3, n))
    fac = S.helmholtz_lu("D", N, -np.ones(1), np.full(1, 7.0))
    idx = torch.arange(lines, device="cuda") % 32
    code = _lib.C128 if cplx else _lib.F64
    for kind in ("tdma", "helmholtz"):
        u = dev(b)[:, idx].contiguous() if axis == 0 else dev(b.T)[idx].contiguous()
        geom = (code, 2, _lib.arr(u.shape), _lib.arr(u.stride()))
        if kind == "tdma":
            ref = S.tdma_solve(b[:n], lu, 0)
            lud = dev(lu)
            _lib.call("sfa_tdma_mass_solve", _lib.ptr(u), *geom, axis, _lib.ptr(lud), n, 2, _lib.stream_ptr())
        else:
            ref = S.helmholtz_solve(b, *fac, neumann=False)[:n]
            fd = [dev(x.reshape(-1)) for x in fac]
            _lib.call("sfa_helmholtz_solve", _lib.ptr(u), _lib.ptr(u), *geom, _lib.arr(u.stride()), axis, 0,
                      *[_lib.ptr(x) for x in fd], _lib.arr((1, 0) if axis == 0 else (0, 1)), _lib.stream_ptr())
        got = u if axis == 0 else u.T
        r = dev(ref)
        assert float((got[:n] - r[:, idx]).abs().amax()) < TOL * float(r.abs().max())
        if kind == "tdma":
            assert not bool(got[n:].any())


@pytest.mark.parametrize("N,lines,axis", [(34, 8201, 0), (35, 8200, 0), (386, 1100, 0), (388, 300, 0),
                                          (66, 2050, 1), (386, 300, 1), (388, 300, 1), (514, 300, 1)])
def test_chain_scan_own_factors(sfa, N, lines, axis):
    """TDMA factors of each line's own where the lines per workgroup depend on
    it (chains of 16, 17, 192, 193 and 256 rows), vs the oracle's solve with one
    set, each line's matrix a multiple of it."""
    print(f"[chain own factors N={N} lines={lines} axis={axis}]", flush=True)
    from shenfun_amd import _lib
    rng = np.random.default_rng(N)
    n = N - 2
    b = rng.standard_normal((32, N)) + 1j * rng.standard_normal((32, N))
    d3 = {0: rng.uniform(2, 3, n), -2: rng.uniform(0.1, 1, n - 2), 2: rng.uniform(0.1, 1, n - 2)}
    dia = S.tdma_dia(d3, n)
    ref = dev(S.tdma_solve(b[:, :n], S.tdma_lu(dia.copy()), 1))
    sc = dev(rng.uniform(0.5, 2.0, lines))
    data = sc[:, None, None] * dev(dia)[None]
    _lib.call("sfa_tdma_lu", _lib.ptr(data), n, lines, _lib.stream_ptr())
    idx = torch.arange(lines, device="cuda") % 32
    u = dev(b)[idx].contiguous() if axis == 1 else dev(b)[idx].T.contiguous()
    _lib.call("sfa_tdma_solve", _lib.ptr(u), _lib.C128, 2, _lib.arr(u.shape), _lib.arr(u.stride()), axis,
              _lib.ptr(data), n, 3 * n, 0, _lib.stream_ptr())
    got = (u if axis == 1 else u.T)[:, :n]
    want = ref[idx] / sc[:, None]
    assert float((got - want).abs().amax()) < TOL * float(want.abs().max())
