"""GPU batched tridiagonal kernel (the S-line / v-line solver in isolation) against the oracle's Thomas LU.

Systems: a, c ~ U[-1, 0], b = 2.5 + |a| + |c|, d ~ N(0, 1), seed 1; a[0] and c[n-1] ignored
(Neumann(0) folding reduces the reference's Thomas LU to the plain algorithm).  Tolerance 1e-13
relative (FP64), 1e-5 (FP32).
"""
import numpy as np
import pytest

import linear_system_solvers_amd as L

pytestmark = pytest.mark.gpu


def _systems(B, n, dt, seed=1):
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1, 0, (B, n))
    c = rng.uniform(-1, 0, (B, n))
    b = 2.5 + np.abs(a) + np.abs(c)
    d = rng.standard_normal((B, n))
    return [v.astype(dt) for v in (a, b, c, d)]


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout", [L.LAYOUT_CONTIGUOUS, L.LAYOUT_STRIDED])
@pytest.mark.parametrize("B,n", [(1, 4), (37, 5), (1000, 256), (65536, 256)])
def test_tridiag_matches_oracle(oracle, fp, layout, B, n):
    torch = pytest.importorskip("torch")
    dt = L.np_dtype(fp)
    a, b, c, d = _systems(B, n, dt)
    if layout == L.LAYOUT_STRIDED:
        a, b, c, d = (np.ascontiguousarray(v.T) for v in (a, b, c, d))
    ta, tb, tc, td = (torch.from_numpy(v).cuda() for v in (a, b, c, d))
    tx = torch.empty_like(td)
    L.tridiag_batched(fp, layout, B, n, ta.data_ptr(), tb.data_ptr(), tc.data_ptr(), td.data_ptr(), tx.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x = tx.cpu().numpy()
    ref = oracle.thomas_batched(a, b, c, d, B, n, strided=(layout == L.LAYOUT_STRIDED),
                                fp="f64" if fp == L.FP64 else "f32").reshape(x.shape)
    err = np.abs(x.astype(np.float64) - ref).max() / np.abs(ref).max()
    print(f"B={B} n={n} layout={layout} fp={fp}: err {err:.2e} bit-identical {np.array_equal(x, ref)}", flush=True)
    assert err <= (1e-13 if fp == L.FP64 else 1e-5)


# ---------------------------------------------------------------------------------------------
# End conditions (lss_tridiag_batched_bc): the reference's known answers for u'' = -2 on [0, 1]
# (unit_tests/sparse_solvers/lss_thomas_lu_solver_t.hpp:12-243; central differences are exact for
# quadratics) and the oracle's thomas_lu with the same folding on random systems.
# ---------------------------------------------------------------------------------------------
def _solve_bc(fp, layout, a, b, c, d, lower, upper):
    torch = pytest.importorskip("torch")
    B, n = a.shape
    if layout == L.LAYOUT_STRIDED:
        a, b, c, d = (np.ascontiguousarray(v.T) for v in (a, b, c, d))
    ta, tb, tc, td = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (a, b, c, d))
    tx = torch.full_like(td, float("nan"))
    L.tridiag_batched_bc(fp, layout, B, n, ta.data_ptr(), tb.data_ptr(), tc.data_ptr(), td.data_ptr(), tx.data_ptr(),
                         lower, upper, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x = tx.cpu().numpy().astype(np.float64)
    return x.T if layout == L.LAYOUT_STRIDED else x


KAT = [  # (n, lower, upper, exact(t), f64 tolerance)
    (100, (L.BC_DIRICHLET, 0.0), (L.BC_DIRICHLET, 0.0), lambda t: t * (1 - t), 1e-10),
    (100, (L.BC_DIRICHLET, 1.0), (L.BC_ROBIN, 1.0, 0.0), lambda t: -t * t + t + 1, 1e-10),
    (1000, (L.BC_NEUMANN, -1.0), (L.BC_ROBIN, 2.0, 0.0), lambda t: -t * t + t + 0.5, 1e-8),
    (2000, (L.BC_NEUMANN, -1.0), (L.BC_ROBIN, 2.0, 0.0), lambda t: -t * t + t + 0.5, 1e-7),
]


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout", [L.LAYOUT_CONTIGUOUS, L.LAYOUT_STRIDED])
@pytest.mark.parametrize("case", range(len(KAT)))
def test_end_conditions_reproduce_the_known_answers(fp, layout, case):
    n, lower, upper, exact, tol = KAT[case]
    dt = L.np_dtype(fp)
    B = 3
    h = dt(1.0) / dt(n - 1)
    a = np.ones((B, n), dt)
    b = np.full((B, n), -2.0, dt)
    c = np.ones((B, n), dt)
    d = np.full((B, n), dt(-2.0) * h * h, dt)
    x = _solve_bc(fp, layout, a, b, c, d, lower, upper)
    t = np.arange(n) / (n - 1)
    err = np.abs(x - exact(t)[None, :]).max()
    print(f"n={n} {lower} {upper} layout={layout} fp={fp}: max err {err:.2e}", flush=True)
    assert err <= (tol if fp == L.FP64 else 2e-1 if n >= 1000 else 2e-3)


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout", [L.LAYOUT_CONTIGUOUS, L.LAYOUT_STRIDED])
@pytest.mark.parametrize("n", [5, 17, 256, 1500])
def test_end_conditions_match_the_oracle(oracle, fp, layout, n):
    rng = np.random.default_rng(n)
    dt = L.np_dtype(fp)
    ends = [((L.BC_DIRICHLET, 0.7), (L.BC_DIRICHLET, -0.3)), ((L.BC_NEUMANN, 0.4), (L.BC_ROBIN, 1.5, -0.2)),
            ((L.BC_ROBIN, 0.8, 0.1), (L.BC_NEUMANN, -0.6)), ((L.BC_DIRICHLET, 1.1), (L.BC_ROBIN, 0.5, 0.3))]
    ofp = "f64" if fp == L.FP64 else "f32"
    for lower, upper in ends:
        a, b, c, d = _systems(40, n, dt, seed=n + 1)
        x = _solve_bc(fp, layout, a, b, c, d, lower, upper)
        lo = (lower[0], lower[1] if len(lower) == 3 else 0.0, lower[-1])
        hi = (upper[0], upper[1] if len(upper) == 3 else 0.0, upper[-1])
        ref = np.stack([oracle.thomas_lu(a[k], b[k], c[k], d[k], lo, hi, ofp) for k in range(a.shape[0])])
        err = np.abs(x - ref).max() / np.abs(ref).max()
        print(f"n={n} {lower} {upper} layout={layout} fp={fp}: err {err:.2e}", flush=True)
        assert np.isfinite(x).all()
        assert err <= (1e-13 if fp == L.FP64 else 1e-5)


def test_end_condition_type_is_checked():
    torch = pytest.importorskip("torch")
    t = torch.zeros((2, 8), dtype=torch.float64, device="cuda")
    with pytest.raises(L.LssError):
        L.tridiag_batched_bc(L.FP64, L.LAYOUT_CONTIGUOUS, 2, 8, t.data_ptr(), t.data_ptr(), t.data_ptr(),
                             t.data_ptr(), t.data_ptr(), (7, 0.0), (L.BC_DIRICHLET, 0.0))


# ---------------------------------------------------------------------------------------------
# Edges of the kernels' size ranges: one wavefront per system up to 512 (f64) / 1024 (f32) contiguous
# unknowns, one workgroup up to 7168 / 8192, one lane beyond; interleaved systems change their tile
# at 64, 128, 256, 512, 1024 and 2048.  B is odd and not a multiple of any tile.
# Tolerance as above: the rows dominate (|a| + |c| <= 2 against b >= 2.5 + |a| + |c|), so neither
# elimination amplifies rounding and both stay within tens of eps of the exact solution.
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout,n", [(L.LAYOUT_CONTIGUOUS, n) for n in (512, 513, 1024, 1025, 1537, 2048, 2049, 4099,
                                                                       7168, 7169, 8192, 8193)] +
                         [(L.LAYOUT_STRIDED, n) for n in (64, 65, 129, 257, 512, 513, 1024, 1025, 2047, 2048, 2049)])
@pytest.mark.parametrize("in_place", [False, True])
def test_edges_of_the_size_ranges(oracle, fp, layout, n, in_place):
    torch = pytest.importorskip("torch")
    dt, B = L.np_dtype(fp), 35
    a, b, c, d = _systems(B, n, dt, seed=n)
    ref = oracle.thomas_batched(a, b, c, d, B, n, strided=False, fp="f64" if fp == L.FP64 else "f32").reshape(B, n)
    if layout == L.LAYOUT_STRIDED:
        a, b, c, d = (np.ascontiguousarray(v.T) for v in (a, b, c, d))
    ta, tb, tc, td = (torch.from_numpy(v).cuda() for v in (a, b, c, d))
    tx = td if in_place else torch.full_like(td, float("nan"))
    L.tridiag_batched(fp, layout, B, n, ta.data_ptr(), tb.data_ptr(), tc.data_ptr(), td.data_ptr(), tx.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x = tx.cpu().numpy().astype(np.float64)
    x = x.T if layout == L.LAYOUT_STRIDED else x
    err = np.abs(x - ref).max() / np.abs(ref).max()
    print(f"n={n} layout={layout} fp={fp} in place {in_place}: err {err:.2e}", flush=True)
    assert err <= (1e-13 if fp == L.FP64 else 1e-5)


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout", [L.LAYOUT_CONTIGUOUS, L.LAYOUT_STRIDED])
@pytest.mark.parametrize("n", [513, 1026, 2050])
def test_end_conditions_of_long_systems_match_the_oracle(oracle, fp, layout, n):
    # (with two Dirichlet ends 1026 and 2050 points hold 1024 and 2048 unknowns)
    test_end_conditions_match_the_oracle(oracle, fp, layout, n)


# ---------------------------------------------------------------------------------------------
# Long systems (contiguous: 513..7168 unknowns in fp64, 1025..8192 in fp32; interleaved: 1025..2048) whose rows do not
# dominate, or whose diagonals have no reciprocal in the normal range, are swept in the reference's order: bit for bit
# the oracle's values, beside dominant systems of the same batch, which keep the tolerance above.
# ---------------------------------------------------------------------------------------------
LONG = [(L.FP64, L.LAYOUT_CONTIGUOUS, 513), (L.FP64, L.LAYOUT_CONTIGUOUS, 600), (L.FP64, L.LAYOUT_CONTIGUOUS, 2048),
        (L.FP64, L.LAYOUT_CONTIGUOUS, 4100), (L.FP64, L.LAYOUT_CONTIGUOUS, 7168), (L.FP32, L.LAYOUT_CONTIGUOUS, 1025),
        (L.FP32, L.LAYOUT_CONTIGUOUS, 2047), (L.FP32, L.LAYOUT_CONTIGUOUS, 8192), (L.FP64, L.LAYOUT_STRIDED, 1025),
        (L.FP64, L.LAYOUT_STRIDED, 2048), (L.FP32, L.LAYOUT_STRIDED, 1031), (L.FP32, L.LAYOUT_STRIDED, 2048)]


def _solve_plain(fp, layout, a, b, c, d, in_place=False):
    torch = pytest.importorskip("torch")
    B, n = a.shape
    if layout == L.LAYOUT_STRIDED:
        a, b, c, d = (np.ascontiguousarray(v.T) for v in (a, b, c, d))
    ta, tb, tc, td = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (a, b, c, d))
    tx = td if in_place else torch.full_like(td, float("nan"))
    L.tridiag_batched(fp, layout, B, n, ta.data_ptr(), tb.data_ptr(), tc.data_ptr(), td.data_ptr(), tx.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x = tx.cpu().numpy()
    return x.T if layout == L.LAYOUT_STRIDED else x


@pytest.mark.parametrize("fp,layout,n", LONG)
@pytest.mark.parametrize("in_place", [False, True])
def test_long_systems_that_do_not_dominate_equal_the_oracle(oracle, fp, layout, n, in_place):
    dt, B = L.np_dtype(fp), 13
    a, b, c, d = _systems(B, n, dt, seed=n)
    for k, kind in ((1, "zero"), (2, "weaker"), (4, "weak"), (5, "one row"), (7, "tiny"), (8, "huge"), (11, "last row")):
        if kind == "zero":  # only the first diagonal is not zero: beta = -a gamma
            b[k, 1:] = 0.0
            a[k], c[k] = -1.0, 1.0
        elif kind == "weaker":
            b[k] = (0.95 * (np.abs(a[k]) + np.abs(c[k])) + 0.01).astype(dt)
        elif kind == "weak":  # (still dominates: the off-diagonals' sum is below 2)
            b[k] = (0.9 * (np.abs(a[k]) + np.abs(c[k])) + 0.3).astype(dt)
        elif kind == "one row":
            b[k, n // 2] = 0.0
        elif kind == "tiny":  # (c stays: the solution does not overflow)
            s = dt(1e-38 if fp == L.FP32 else 1e-305)
            a[k], b[k], c[k], d[k] = (v * s for v in (a[k], b[k], c[k], d[k]))
        elif kind == "huge":
            s = dt(1e36 if fp == L.FP32 else 1e305)
            a[k], b[k], c[k], d[k] = (v * s for v in (a[k], b[k], c[k], d[k]))
        else:
            a[k, n - 1] = 9.0
    other = np.zeros(B, bool)
    other[[1, 2, 5, 7, 8, 11]] = True
    with np.errstate(all="ignore"):
        ref = oracle.thomas_batched(a, b, c, d, B, n, strided=False, fp="f64" if fp == L.FP64 else "f32").reshape(B, n)
    assert np.isfinite(ref).all()
    x = _solve_plain(fp, layout, a, b, c, d, in_place)
    assert np.isfinite(x).all()
    for k in range(B):
        if other[k]:
            assert np.array_equal(x[k], ref[k]), k
        else:
            assert np.abs(x[k].astype(np.float64) - ref[k]).max() <= (1e-13 if fp == L.FP64 else 1e-5) * np.abs(ref[k]).max()
    # a system's values do not depend on its neighbours
    keep = ~other
    assert np.array_equal(_solve_plain(fp, layout, a[keep], b[keep], c[keep], d[keep]), x[keep])


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("layout", [L.LAYOUT_CONTIGUOUS, L.LAYOUT_STRIDED])
def test_long_systems_with_ends_that_do_not_dominate_equal_the_oracle(oracle, fp, layout):
    # a Robin end whose weight takes away from the diagonal, on Poisson rows (|b| = |a| + |c|)
    dt, B, n = L.np_dtype(fp), 5, 1300
    a, b, c = np.full((B, n), -1.0, dt), np.full((B, n), 2.0, dt), np.full((B, n), -1.0, dt)
    d = np.random.default_rng(5).standard_normal((B, n)).astype(dt)
    for lower, upper in (((L.BC_ROBIN, 2.0, 0.1), (L.BC_DIRICHLET, 0.4)), ((L.BC_DIRICHLET, 0.4), (L.BC_ROBIN, -2.0, 0.1))):
        x = _solve_bc(fp, layout, a, b, c, d, lower, upper)
        lo = (lower[0], lower[1] if len(lower) == 3 else 0.0, lower[-1])
        hi = (upper[0], upper[1] if len(upper) == 3 else 0.0, upper[-1])
        ref = np.stack([oracle.thomas_lu(a[k], b[k], c[k], d[k], lo, hi, "f64" if fp == L.FP64 else "f32") for k in range(B)])
        assert np.isfinite(ref).all() and np.array_equal(x, ref.astype(np.float64))


@pytest.mark.parametrize("fp,layout,n", LONG)
def test_long_systems_are_as_accurate_as_the_sequential_sweep(oracle, fp, layout, n):
    """Error against a longer format, root mean square over the batch, of the rows that the module's tests use: no larger
    than the sequential sweep's in the same precision (host emulation: 0.9 of it)."""
    dt, B = L.np_dtype(fp), 48
    wide = np.longdouble if fp == L.FP64 else np.float64
    a, b, c, d = _systems(B, n, dt, seed=n + 7)
    seq = oracle.thomas_batched(a, b, c, d, B, n, strided=False, fp="f64" if fp == L.FP64 else "f32").reshape(B, n)
    wa, wb, wc, wd = (v.astype(wide) for v in (a, b, c, d))
    g, exact = np.zeros((B, n), wide), np.zeros((B, n), wide)
    g[:, 0], exact[:, 0] = wc[:, 0] / wb[:, 0], wd[:, 0] / wb[:, 0]
    for i in range(1, n):
        beta = wb[:, i] - wa[:, i] * g[:, i - 1]
        g[:, i], exact[:, i] = wc[:, i] / beta, (wd[:, i] - wa[:, i] * exact[:, i - 1]) / beta
    for i in range(n - 2, -1, -1):
        exact[:, i] -= g[:, i] * exact[:, i + 1]
    err = [float(np.sqrt(np.mean((v.astype(wide) - exact) ** 2))) for v in (_solve_plain(fp, layout, a, b, c, d), seq)]
    print(f"n={n} layout={layout} fp={fp}: rms error {err[0]:.2e}, sequential {err[1]:.2e}", flush=True)
    assert err[0] <= err[1]
