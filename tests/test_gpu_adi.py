"""GPU parity of the ADI stepper (through the C-ABI) against the CPU oracle and the reference's surfaces.

Tolerances (FP64): the FIELDS plan reproduces the reference's rounding operation by operation, so it is
held to 1e-13 (it is expected to be bit-identical; the test reports it); the SEPARABLE plan forms the
coefficients from 1-D factors (a few ulp per coefficient): it is held to the 1e-12 stated for the
single problem on that problem (config0 below) and to the batched tolerance 1e-10 on the reference's
stiffer surfaces (199 steps on clustered grids), whose largest relative deviations sit in column
ny-2 next to v_max, where the reference's own surface oscillates through small negative values.  FP32 runs are compared with the FP32 oracle (same index maps, same quirks) at 1e-5.
Error measure: max |g - c| / max(|c|, 1e-8 ||c||_inf).
"""
import numpy as np
import pytest

import linear_system_solvers_amd as L
from tests.golden import reference_outputs as R
from tests.helpers import config0, model_from_case, oracle_solve, rel_err

pytestmark = pytest.mark.gpu


def _solve(m, fp=L.FP64, graph=None):
    plan = L.Plan.from_models([m], fp)
    out = plan.run_host()[0]
    plan.close()
    return out


@pytest.mark.parametrize("case", R.CASES, ids=[c["stem"] for c in R.CASES])
def test_fields_f64_matches_oracle_and_reference_surface(oracle, case):
    m = model_from_case(case)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    err = rel_err(g, c)
    print(f"{case['stem']}: rel err vs oracle {err:.3e}, bit-identical {np.array_equal(g, c)}", flush=True)
    assert err <= 1e-13
    _, _, vals = R.load(case["stem"], "f64")
    assert np.all(np.abs(g - vals) <= 5.01e-6 * np.abs(vals) + 1e-12 * np.abs(vals).max())


@pytest.mark.parametrize("case", [c for c in R.CASES if c["floats"]], ids=[c["stem"] for c in R.CASES if c["floats"]])
def test_fields_f32_matches_oracle(oracle, case):
    m = model_from_case(case)
    g = _solve(m, L.FP32)
    c = oracle_solve(oracle, m, "f32")
    err = float(np.abs(g.astype(np.float64) - c).max() / np.abs(c).max())
    print(f"{case['stem']} f32: normwise err vs f32 oracle {err:.3e}, bit-identical {np.array_equal(g, c)}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("case", R.CASES, ids=[c["stem"] for c in R.CASES])
def test_separable_f64_matches_oracle(oracle, case):
    m = model_from_case(case, coeff_mode=L.COEFF_SEPARABLE)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    err = rel_err(g, c)
    at = np.unravel_index(np.argmax(np.abs(g - c) / np.maximum(np.abs(c), 1e-8 * np.abs(c).max())), c.shape)
    print(f"{case['stem']} separable: rel err {err:.3e} at {at} (value {c[at]:.3e}, max {np.abs(c).max():.3e})",
          flush=True)
    assert err <= 1e-10


@pytest.mark.parametrize("mode", [L.COEFF_FIELDS, L.COEFF_SEPARABLE])
def test_config0_heston_dr_within_1e12(oracle, mode):
    m = config0(coeff_mode=mode)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    err = rel_err(g, c)
    print(f"config0 mode {mode}: rel err {err:.3e} price-surface max {np.abs(c).max():.3f}", flush=True)
    assert err <= 1e-12


@pytest.mark.parametrize("splitting", [0, 1, 2, 3])
@pytest.mark.parametrize("tri", [L.THOMAS_LU, L.DOUBLE_SWEEP])
@pytest.mark.parametrize("direction", [L.FORWARD, L.BACKWARD])
def test_every_scheme_solver_and_direction(oracle, splitting, tri, direction):
    m = config0(nx=37, ny=21, nt=23, grid=L.NONUNIFORM, accumulation_point=100.0, alpha_scale=3.0,
                splitting=splitting, weighting=0.3, implicit_scheme=L.THETA_80, tridiagonal=tri, direction=direction)
    g = _solve(m)
    err = rel_err(g, oracle_solve(oracle, m))
    assert err <= 1e-13, err


def test_sabr_time_dependent_coefficients(oracle):
    m = L.Model(kind=L.MODEL_SABR, strike=100.0, rate=0.05, sig_sig=0.3, rho=-0.4, beta=0.5, maturity=2.0,
                x_lo=20.0, x_hi=250.0, y_lo=0.0, y_hi=1.0, t_hi=2.0, nx=40, ny=24, nt=41, grid=L.NONUNIFORM,
                accumulation_point=100.0, splitting=L.HUNDSDORFER_VERWER, tridiagonal=L.DOUBLE_SWEEP)
    for mode, tol in ((L.COEFF_FIELDS, 1e-13), (L.COEFF_SEPARABLE, 1e-12)):
        m.coeff_mode = mode
        assert rel_err(_solve(m), oracle_solve(oracle, m)) <= tol


def test_book_of_mixed_problems_matches_each_oracle_solve(oracle):
    # problems of different sizes, step counts and schemes stepped together in one plan: each must
    # equal its own oracle solve (FIELDS problems bit for bit; SEPARABLE ones to the batched
    # tolerance, normwise, see test_separable_errors_are_normwise_small)
    rng = np.random.default_rng(7)
    models = []
    for q in range(9):
        models.append(config0(nx=int(rng.integers(8, 60)), ny=int(rng.integers(6, 40)), nt=int(rng.integers(3, 40)),
                              splitting=q % 4, strike=float(rng.uniform(60, 140)), rho=float(rng.uniform(-0.9, 0.0)),
                              sig_kappa=float(rng.uniform(0.5, 5.0)), grid=L.NONUNIFORM, accumulation_point=100.0,
                              coeff_mode=L.COEFF_SEPARABLE if q % 2 else L.COEFF_FIELDS))
    plan = L.Plan.from_models(models)
    outs = plan.run_host()
    for q, (m, g) in enumerate(zip(models, outs)):
        c = oracle_solve(oracle, m)
        norm = float(np.abs(g - c).max() / np.abs(c).max())
        print(f"book problem {q}: {m.nx}x{m.ny}x{m.steps} scheme {m.splitting} mode {m.coeff_mode}: "
              f"per-value {rel_err(g, c):.2e} normwise {norm:.2e} bit-identical {np.array_equal(g, c)}", flush=True)
        if m.coeff_mode == L.COEFF_FIELDS:
            assert np.array_equal(g, c)
        else:
            assert norm <= 1e-12


def test_graph_replay_equals_direct_launches():
    torch = pytest.importorskip("torch")
    m = config0(nx=64, ny=32, nt=31, splitting=L.MODIFIED_CRAIG_SNEYD, weighting=0.3)
    plan = L.Plan.from_models([m])
    u0 = torch.from_numpy(plan.initial(0)).cuda()
    outs = [torch.empty_like(u0) for _ in range(4)]
    st = torch.cuda.current_stream().cuda_stream
    plan.run_dev([u0.data_ptr()], [outs[0].data_ptr()], st, graph=False)
    for k in range(1, 4):  # replays, with eager work and synchronisation in between
        plan.run_dev([u0.data_ptr()], [outs[k].data_ptr()], st, graph=True)
        torch.cuda.synchronize()
        _ = (u0 * 2).sum().item()
    ref = outs[0].cpu().numpy()
    for k in range(1, 4):
        assert np.array_equal(outs[k].cpu().numpy(), ref)
    plan.close()


# ---------------------------------------------------------------------------------------------
# Partitioned line solver: the same per-point arithmetic, a different elimination order for the
# line solves, so it is held to tolerances, normwise per problem (max |g - c| / ||c||_inf).
# ---------------------------------------------------------------------------------------------
def _normwise(g, c):
    return float(np.abs(np.asarray(g, np.float64) - c).max() / np.abs(c).max())


@pytest.mark.parametrize("case", R.CASES, ids=[c["stem"] for c in R.CASES])
@pytest.mark.parametrize("mode", [L.COEFF_FIELDS, L.COEFF_SEPARABLE])
def test_partitioned_matches_oracle(oracle, case, mode):
    m = model_from_case(case, coeff_mode=mode, line_solver=L.LINE_PARTITIONED)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    print(f"{case['stem']} partitioned mode {mode}: normwise {_normwise(g, c):.2e} per-value {rel_err(g, c):.2e}",
          flush=True)
    assert _normwise(g, c) <= 1e-12


def _stable(nx, ny, steps=10, fac=1.5, **kw):
    """Heston DR/CS/MCS/HV problem whose time step keeps the reference's explicit v = 0 row stable
    (3 nu E <= 2 with the uniform-hints v map: k <= 1.5 h2 for kappa = 3, theta_v = 0.2).  MCS with
    zeta != theta is unstable in the reference at moderate sizes (its "- P" correction term amplifies),
    so the sweeps below run MCS at zeta = theta and test the (zeta - theta) term separately."""
    k = min(0.01, fac / (ny - 1))
    return config0(nx=nx, ny=ny, nt=steps + 1, t_hi=k * steps, **kw)


def _assert_stable(c, m):
    assert np.isfinite(c).all() and np.abs(c).max() <= 2.0 * m.x_hi, "test problem is not stable"


@pytest.mark.parametrize("nx,ny", [(4, 4), (6, 5), (9, 7), (66, 66), (67, 130), (131, 200), (300, 140), (514, 258),
                                   (1026, 70), (70, 1026)])
@pytest.mark.parametrize("splitting", [0, 1, 2, 3])
def test_partitioned_sizes_and_schemes(oracle, nx, ny, splitting):
    m = _stable(nx, ny, splitting=splitting, weighting=0.5 if splitting >= 2 else 0.3, coeff_mode=L.COEFF_SEPARABLE,
                line_solver=L.LINE_PARTITIONED)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    _assert_stable(c, m)
    assert _normwise(g, c) <= 1e-12


@pytest.mark.parametrize("nx,ny", [(4, 4), (6, 5), (9, 7), (66, 66), (67, 130)])
@pytest.mark.parametrize("splitting", [2, 3])
def test_partitioned_zeta_terms(oracle, nx, ny, splitting):
    """MCS and HV with zeta != theta (MCS's (zeta - theta) correction with its "- P"; HV's zero-border
    Y2 rows) at time steps where the reference scheme stays bounded."""
    m = _stable(nx, ny, fac=0.2, splitting=splitting, weighting=0.3, coeff_mode=L.COEFF_SEPARABLE,
                line_solver=L.LINE_PARTITIONED)
    g = _solve(m)
    c = oracle_solve(oracle, m)
    _assert_stable(c, m)
    assert _normwise(g, c) <= 1e-12


@pytest.mark.parametrize("fp,tol", [(L.FP64, 1e-13), (L.FP32, 1e-5)])
def test_partitioned_agrees_with_exact_sweeps_on_gpu(oracle, fp, tol):
    for splitting in range(4):
        m = _stable(150, 60, steps=50, splitting=splitting, weighting=0.5 if splitting >= 2 else 0.4,
                    coeff_mode=L.COEFF_FIELDS)
        ex = _solve(m, fp)
        _assert_stable(ex.astype(np.float64), m)
        m.line_solver = L.LINE_PARTITIONED
        pa = _solve(m, fp)
        assert _normwise(pa, ex.astype(np.float64)) <= tol


def test_partitioned_book_matches_oracle(oracle):
    rng = np.random.default_rng(11)
    models = [_stable(int(rng.integers(5, 300)), int(rng.integers(5, 150)), steps=int(rng.integers(1, 30)),
                      splitting=q % 4, strike=float(rng.uniform(60, 140)), coeff_mode=L.COEFF_SEPARABLE,
                      line_solver=L.LINE_PARTITIONED)
              for q in range(16)]
    outs = L.Plan.from_models(models).run_host()
    for m, g in zip(models, outs):
        c = oracle_solve(oracle, m)
        _assert_stable(c, m)
        assert _normwise(g, c) <= 1e-12


def test_every_tile_mapping_gives_identical_results():
    """The autotuner's candidate tile/lane mappings change only the work distribution."""
    rng = np.random.default_rng(21)
    models = [_stable(int(rng.integers(5, 300)), int(rng.integers(5, 150)), steps=int(rng.integers(1, 12)),
                      splitting=q % 4, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)
              for q in range(12)]
    plan = L.Plan.from_models(models)
    chosen = plan.autotune()
    assert chosen[0] in (16, 8, 4) and chosen[1] in (4, 16) and chosen[2] in (0, 1)
    ref = None
    for z in (0, 1):
        for x in (16, 8, 4):
            for v in (4, 16):
                plan.set_mapping(x, v, z)
                outs = plan.run_host()
                if ref is None:
                    ref = outs
                for a, b in zip(ref, outs):
                    np.testing.assert_array_equal(a, b)
    with pytest.raises(L.LssError):
        plan.set_mapping(32, 4)


def test_long_s_lines_take_at_most_8_per_workgroup_and_every_mapping_agrees(oracle):
    """S-lines of more than 512 points use 128 chunks; 16 lines per workgroup is refused."""
    m = _stable(700, 40, steps=4, splitting=2, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)
    plan = L.Plan.from_models([m])
    assert plan.autotune()[0] in (8, 4)
    with pytest.raises(L.LssError):
        plan.set_mapping(16, 4)
    ref = None
    for x in (8, 4):
        for v in (4, 16):
            plan.set_mapping(x, v, 1)
            out = plan.run_host()[0]
            if ref is None:
                ref = out
            np.testing.assert_array_equal(out, ref)
    c = oracle_solve(oracle, m)
    print(f"700x40 long S-lines: normwise {_normwise(ref, c):.2e}", flush=True)
    assert _normwise(ref, c) <= 1e-12


def test_reference_models_use_the_specialized_factor_patterns():
    """Heston (r != 0) and SABR (r = 0) separable data match the compile-time patterns exactly."""
    h = L.Plan.from_models([_stable(40, 20, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)])
    assert h.kernel_config()["factor_pattern"] == 1
    sabr = L.Model(kind=L.MODEL_SABR, strike=0.03, rate=0.0, sig_sig=0.5, rho=-0.3, beta=0.6, x_lo=0.0, x_hi=0.15,
                   y_lo=0.0, y_hi=0.25, nx=40, ny=24, nt=5, t_hi=0.01, grid=L.NONUNIFORM, accumulation_point=0.03,
                   alpha_scale=10.0, beta_scale=50.0, splitting=L.HUNDSDORFER_VERWER,
                   coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)
    s = L.Plan.from_models([sabr])
    assert s.kernel_config()["factor_pattern"] == 2
    mixed = L.Plan.from_models([_stable(40, 20, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED), sabr])
    assert mixed.kernel_config()["factor_pattern"] == 0


def test_book_problems_unstable_in_the_reference_match_it_on_the_exact_path(oracle):
    """Problems of the 2048-problem book (seed 3) that the scheme itself makes unstable at their drawn
    step counts (the oracle's values grow past 10 S_max) still match the oracle bit for bit on the
    exact path, stepped in one plan with stable ones; the stable ones also match on the fast path
    to 1e-10 normwise.  The smallest such problems of the book are used."""
    import dataclasses
    import bench
    book = bench.book_models(2048, coeff_mode=L.COEFF_FIELDS, line_solver=L.LINE_EXACT)
    order = sorted(range(len(book)), key=lambda q: book[q].nx * book[q].ny * book[q].steps)
    unstable, stable, ref = [], [], {}
    for q in order:
        c = oracle_solve(oracle, book[q])
        blown = (not np.isfinite(c).all()) or np.abs(c).max() > 10.0 * book[q].x_hi
        group = unstable if blown else stable
        if len(group) < 4:
            group.append(q)
            ref[q] = c
        if len(unstable) == 4 and len(stable) == 4:
            break
    assert len(unstable) == 4 and len(stable) == 4
    picked = unstable + stable
    exact = L.Plan.from_models([book[q] for q in picked]).run_host()
    fast = L.Plan.from_models([dataclasses.replace(book[q], coeff_mode=L.COEFF_SEPARABLE,
                                                   line_solver=L.LINE_PARTITIONED) for q in stable]).run_host()
    for q, g in zip(picked, exact):
        c = ref[q]
        print(f"book problem {q}: {book[q].nx}x{book[q].ny}x{book[q].steps} scheme {book[q].splitting}, oracle max "
              f"{np.abs(c).max():.3e}, exact path bit-identical {np.array_equal(g, c, equal_nan=True)}", flush=True)
        assert np.array_equal(g, c, equal_nan=True)
    for q, g in zip(stable, fast):
        c = ref[q]
        assert float(np.abs(g - c).max() / np.abs(c).max()) <= 1e-10


def test_graph_groups_of_a_large_plan_equal_direct_launches(oracle):
    """A plan of two or more problems replays its time loop as two graphs on two streams (problems
    alternate between the groups); every replay must equal the direct launches bit for bit, with
    the caller's stream ordered around them, and the problems must match their oracle solves."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(31)
    models = [_stable(int(rng.integers(5, 30)), int(rng.integers(5, 20)), steps=int(rng.integers(1, 14)),
                      splitting=q % 4, strike=float(rng.uniform(60, 140)), coeff_mode=L.COEFF_SEPARABLE,
                      line_solver=L.LINE_PARTITIONED)
              for q in range(520)]
    plan = L.Plan.from_models(models)
    assert plan.kernel_config()["graph_groups"] == 2
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(plan.count)]
    st = torch.cuda.current_stream().cuda_stream
    res = []
    for graph in (False, True, True, True):
        outs = [torch.full_like(u, float("nan")) for u in ins]
        plan.run_dev([u.data_ptr() for u in ins], [o.data_ptr() for o in outs], st, graph=graph)
        got = [(o * 1.0).cpu().numpy() for o in outs]  # stream-ordered work right after the replay
        torch.cuda.synchronize()
        res.append(got)
    for k in range(1, 4):
        assert all(np.array_equal(a, b) for a, b in zip(res[0], res[k]))
    for q in range(0, 520, 37):
        c = oracle_solve(oracle, models[q])
        assert _normwise(res[1][q], c) <= 1e-12
    plan.close()


# ---------------------------------------------------------------------------------------------
# The exact sweeps take lines in groups of 16 points and tiles of 16 lines, and divide by known divisors
# without an IEEE division where the exponents allow it.  Sizes around those edges, both operation orders, both
# coefficient forms side by side, and initial surfaces whose values are huge, tiny, negative zero or subnormal:
# every bit (signs of zeros included) must be the oracle's.
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("nx,ny", [(4, 4), (17, 18), (18, 19), (19, 34), (34, 35), (50, 17), (35, 66)])
def test_exact_sweeps_equal_the_oracle_at_their_edges(oracle, fp, nx, ny):
    ofp = "f64" if fp == L.FP64 else "f32"
    models = [config0(nx=nx, ny=ny, nt=5, splitting=s, tridiagonal=tri, implicit_scheme=L.THETA_80, weighting=0.3)
              for s in range(4) for tri in (L.THOMAS_LU, L.DOUBLE_SWEEP)]
    plan = L.Plan.from_models(models, fp)
    outs = plan.run_host()
    for m, g in zip(models, outs):
        c = oracle_solve(oracle, m, ofp)
        assert np.array_equal(g, c) and np.array_equal(np.signbit(g), np.signbit(c)), (m.splitting, m.tridiagonal)
    plan.close()


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("scale", [1.0, 0.0, -0.0, 1e-30, 1e-300, 1e-310, 1e30, 1e300])
def test_exact_sweeps_keep_the_rounding_at_any_magnitude(oracle, fp, scale):
    # the two operation orders and two tile positions of the same problem step the same surface: the loop is linear
    # and its coefficients do not see the scale, so the sweeps of both halves of the book must agree with a plan that
    # forms gamma anew (fresh) in every step, i.e. one step per run, bit for bit
    dt = L.np_dtype(fp)
    m = config0(nx=37, ny=21, nt=4, splitting=L.CRAIG_SNEYD)
    one = config0(nx=37, ny=21, nt=2, splitting=L.CRAIG_SNEYD, t_hi=1.0 / 3.0, maturity=1.0)
    plan, single = L.Plan.from_models([m], fp), L.Plan.from_models([one], fp)
    rng = np.random.default_rng(3)
    with np.errstate(over="ignore", under="ignore"):
        u = (rng.standard_normal((37, 21)) * scale).astype(dt)
    levels = plan.run_levels_host([u])[0]
    for s in range(3):
        nxt = single.run_host([levels[s]])[0]
        assert np.array_equal(nxt, levels[s + 1], equal_nan=True)
    plan.close()
    single.close()


# A book whose state exceeds the last-level cache is stepped as consecutive slices of problems (3 here: 210 problems
# of about 3.0 or 1.8 MB), each slice ending at its own most steps.  Every problem takes the arithmetic of its own
# plan: no tolerance.
@pytest.mark.parametrize("line", [L.LINE_EXACT, L.LINE_PARTITIONED])
def test_a_book_larger_than_the_cache_equals_its_problems_solved_alone(line):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(41)
    models = [_stable(int(rng.integers(290, 311)), int(rng.integers(240, 261)), steps=int(rng.integers(1, 9)),
                      splitting=q % 4, strike=float(rng.uniform(60, 140)), coeff_mode=L.COEFF_SEPARABLE,
                      line_solver=line)
              for q in range(210)]
    plan = L.Plan.from_models(models)
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(plan.count)]
    st = torch.cuda.current_stream().cuda_stream
    res = []
    for graph in (False, True, True):
        outs = [torch.full_like(u, float("nan")) for u in ins]
        plan.run_dev([u.data_ptr() for u in ins], [o.data_ptr() for o in outs], st, graph=graph)
        res.append([(o * 1.0).cpu().numpy() for o in outs])
        torch.cuda.synchronize()
    plan.close()
    for k in (1, 2):
        assert all(np.array_equal(a, b) for a, b in zip(res[0], res[k]))
    for q in range(0, 210, 13):
        assert np.array_equal(_solve(models[q]), res[0][q]), q


# ---------------------------------------------------------------------------------------------
# Plans of small problems run their whole loop in one launch, a workgroup per problem, 16 chunks of 1 to 7 points per
# line: sizes around the chunk lengths' edges, the smallest and the longest lines, the sizes that only a book of 64
# takes.  Every scheme against the oracle (1e-12 of its largest value, the partitioned solver's tolerance above; fp32
# 1e-5, as above); every level and the checkpointing forward equal the plain run, which runs the same loop.
# ---------------------------------------------------------------------------------------------
def _sabr_small(nx, ny, steps, splitting):
    K = 0.03
    return L.Model(kind=L.MODEL_SABR, strike=K, rate=0.0, sig_sig=0.5, rho=-0.3, beta=0.6, maturity=1.0,
                   x_lo=0.0, x_hi=5 * K, y_lo=0.0, y_hi=0.25, nx=nx, ny=ny, nt=steps + 1, t_hi=0.002 * steps,
                   accumulation_point=K, alpha_scale=10.0, beta_scale=50.0, grid=L.NONUNIFORM, splitting=splitting,
                   weighting=0.5, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("model", ["heston", "sabr"])
@pytest.mark.parametrize("nx,ny,count", [(4, 4, 4), (18, 19, 4), (19, 18, 4), (35, 51, 4), (66, 67, 4), (114, 43, 4),
                                         (43, 114, 4), (101, 60, 64)])
def test_resident_loop_matches_the_oracle(oracle, fp, model, nx, ny, count):
    torch = pytest.importorskip("torch")
    if model == "heston":
        models = [_stable(nx, ny, steps=5 + q % 3, splitting=q % 4, coeff_mode=L.COEFF_SEPARABLE,
                          line_solver=L.LINE_PARTITIONED) for q in range(count)]
    else:
        models = [_sabr_small(nx, ny, 5 + q % 3, q % 4) for q in range(count)]
    plan = L.Plan.from_models(models, fp)
    assert plan.kernel_config()["factor_pattern"] > 0
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(count)]
    pin = [u.data_ptr() for u in ins]
    outs, fwd = ([torch.full_like(u, float("nan")) for u in ins] for _ in range(2))
    levels = [torch.full((plan.shape(p)[2] + 1, nx, ny), float("nan"), dtype=ins[p].dtype, device="cuda")
              for p in range(count)]
    plan.run_dev(pin, [o.data_ptr() for o in outs])
    plan.run_levels_dev(pin, [v.data_ptr() for v in levels])
    plan.forward(pin, [o.data_ptr() for o in fwd], 2)
    torch.cuda.synchronize()
    tol = 1e-12 if fp == L.FP64 else 1e-5
    for p in range(count):
        assert torch.equal(outs[p], levels[p][-1]) and torch.equal(outs[p], fwd[p])
        assert torch.equal(levels[p][0], ins[p])
        if p < 4:
            c = oracle_solve(oracle, models[p], "f64" if fp == L.FP64 else "f32").astype(np.float64)
            assert _normwise(outs[p].cpu().numpy().astype(np.float64), c) <= tol
            short = L.Plan.from_models([models[p]], fp).run_levels_host([plan.initial(p)])[0]
            assert _normwise(levels[p].cpu().numpy().astype(np.float64), short.astype(np.float64)) <= tol
    plan.close()


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("nx,ny", [(4, 4), (5, 70), (6, 130), (19, 34), (131, 66), (150, 260)])
def test_boundary_stage_in_the_last_v_sweep_equals_its_own_launch(fp, nx, ny):
    """Plans of few points evaluate boundary stage B in the step's last v-sweep; a profiled run keeps its launch.  The
    same kernels otherwise: within the partitioned solver's tolerance (1e-12, fp32 1e-5 of the largest value).  The
    150 x 40 problem keeps the plan off the resident loop."""
    torch = pytest.importorskip("torch")
    models = [_stable(nx, ny, steps=3 + q, splitting=q % 4, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)
              for q in range(4)] + [_stable(150, 40, steps=4, coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)]
    plan = L.Plan.from_models(models, fp)
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(plan.count)]
    outs, own = ([torch.full_like(u, float("nan")) for u in ins] for _ in range(2))
    pin = [u.data_ptr() for u in ins]
    plan.run_dev(pin, [o.data_ptr() for o in outs])
    L.run_profiled(plan, pin, [o.data_ptr() for o in own], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    tol = 1e-12 if fp == L.FP64 else 1e-5
    for a, b in zip(outs, own):
        assert _normwise(a.cpu().numpy().astype(np.float64), b.cpu().numpy().astype(np.float64)) <= tol
    plan.close()


# ---------------------------------------------------------------------------------------------
# The exact sweeps against the oracle where they divide by a known divisor and where they must not.
# ---------------------------------------------------------------------------------------------
def _divisors(m, direction, line):
    """Divisors of S-line (0) or v-line (1) `line` of a Heston plan on a uniform grid, for one Euler step, in double."""
    k, h1, h2 = (m.t_hi - m.t_lo) / (m.nt - 1), 1.0 / (m.nx - 1), 1.0 / (m.ny - 1)
    span, y, pt = m.x_hi - m.x_lo, m.y_hi - m.y_lo, m.accumulation_point
    w = np.arcsinh(1.0) * (np.arange(1, m.ny - 1) if direction else line) * h2
    v, dv, ddv = m.y_lo + y * np.sinh(w), y * np.arcsinh(1.0) * np.cosh(w), y * np.arcsinh(1.0) ** 2 * np.sinh(w)
    if direction == 0:
        z = np.arange(1, m.nx - 1) * h1
        c0, c1 = np.arcsinh((m.x_hi - pt) / span), np.arcsinh((m.x_lo - pt) / span)
        w = c0 * z + c1 * (1 - z)
        x, dx, ddx = pt + span * np.sinh(w), span * (c0 - c1) * np.cosh(w), span * (c0 - c1) ** 2 * np.sinh(w)
        diff = 0.5 * v * x * x
        second, first = k / h1 ** 2 * diff / dx ** 2, k / (2 * h1) * (m.rate * x / dx - diff * ddx / dx ** 3)
    else:
        diff = 0.5 * m.sig_sig ** 2 * v
        second = k / h2 ** 2 * diff / dv ** 2
        first = k / (2 * h2) * (m.sig_kappa * (m.sig_theta - v) / dv - diff * ddv / dv ** 3)
    a, b, c = -(second - first), 1.0 + 2.0 * second + 0.5 * k * m.rate, -(second + first)
    beta = [b[0]]
    for t in range(1, len(b)):
        beta.append(b[t] - a[t] * c[t - 1] / beta[-1])
    return np.array(beta)


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("direction", [0, 1])
@pytest.mark.parametrize("splitting", range(4))
def test_a_divisor_out_of_range_in_the_last_row_of_a_line(oracle, fp, direction, splitting):
    # lines of 16 k interior points whose divisors grow past 2^21 (fp64: 2^101) at the last row only; the S-line with
    # the largest v, and every v-line
    ofp, limit = ("f64", 2.0 ** 101) if fp == L.FP64 else ("f32", 2.0 ** 21)
    over = dict(nx=18, ny=34, nt=3 if splitting == 0 else 2, splitting=splitting, implicit_scheme=L.EULER)
    line = 32 if direction == 0 else 8
    ref = _divisors(config0(**over, t_hi=1e12), direction, line)
    t_hi = 1e12 * limit / np.sqrt(ref[-1] * ref[-2])  # (the divisors grow in proportion to the step)
    for tri in (L.THOMAS_LU, L.DOUBLE_SWEEP):
        m = config0(**over, t_hi=t_hi, tridiagonal=tri)
        beta = _divisors(m, direction, line)
        assert beta[-1] > limit * 1.003 and (beta[:-1] < limit * 0.997).all()
        c = oracle_solve(oracle, m, ofp)
        g = _solve(m, fp)
        assert np.isfinite(c).all()
        assert np.array_equal(g, c) and np.array_equal(np.signbit(g), np.signbit(c))


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("rate", [0.02, -9.0])
@pytest.mark.parametrize("scale", [1.0, 0.0, -0.0, 1e-25, 1e-30, 1e-42, 1e-280, 1e-310, 1e25, 1e30, 1e290])
def test_exact_sweeps_round_like_the_oracle_at_any_magnitude(oracle, fp, rate, scale):
    # one step of surfaces whose values are huge, tiny, subnormal or zeros of either sign, also mixed with ordinary
    # values (rate -9: negative diagonals too); every bit must be the oracle's
    from tests.helpers import oracle_cfg, oracle_pde
    dt, ofp = L.np_dtype(fp), "f64" if fp == L.FP64 else "f32"
    rng = np.random.default_rng(3)
    for z in range(8):
        m = config0(nx=37, ny=21, nt=2, rate=rate, splitting=z % 4, tridiagonal=(L.THOMAS_LU, L.DOUBLE_SWEEP)[z // 4],
                    implicit_scheme=L.EULER if z % 2 else L.THETA_80, weighting=0.3)
        with np.errstate(over="ignore", under="ignore"):
            u = (rng.standard_normal((37, 21)) * scale).astype(dt)
            if z % 3 == 0:
                u = np.where(rng.uniform(size=u.shape) < 0.3, rng.standard_normal(u.shape).astype(dt), u)
        plan = L.Plan.from_models([m], fp)
        g = plan.run_host([u])[0]
        plan.close()
        with np.errstate(all="ignore"):
            c = oracle.step(oracle_pde(oracle, m), oracle_cfg(oracle, m), u, 0.0, ofp)  # (its data do not see the time)
        assert np.array_equal(g, c, equal_nan=True) and np.array_equal(np.signbit(g[g == 0]), np.signbit(c[c == 0])), z


def test_an_exact_book_of_sampled_coefficients_equals_its_problems_solved_alone():
    """Exact plans run in slices of problems only if every problem has FIELDS coefficients (2 slices here: 200 problems of
    about 3.0 or 1.8 MB of state); no tolerance."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(43)
    models = [_stable(int(rng.integers(290, 311)), int(rng.integers(240, 261)), steps=int(rng.integers(1, 6)),
                      splitting=q % 4, strike=float(rng.uniform(60, 140)), coeff_mode=L.COEFF_FIELDS,
                      line_solver=L.LINE_EXACT) for q in range(200)]
    plan = L.Plan.from_models(models)
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(plan.count)]
    st = torch.cuda.current_stream().cuda_stream
    res = []
    for graph in (False, True):
        outs = [torch.full_like(u, float("nan")) for u in ins]
        plan.run_dev([u.data_ptr() for u in ins], [o.data_ptr() for o in outs], st, graph=graph)
        res.append([(o * 1.0).cpu().numpy() for o in outs])
        torch.cuda.synchronize()
    plan.close()
    assert all(np.array_equal(a, b) for a, b in zip(*res))
    for q in range(0, 200, 23):
        assert np.array_equal(_solve(models[q]), res[0][q]), q


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("model", ["heston", "sabr"])
@pytest.mark.parametrize("nx,ny,count", [(4, 4, 4), (19, 18, 4), (35, 51, 4), (66, 67, 4), (101, 60, 64)])
def test_resident_loop_steps_like_the_step_by_step_kernels(fp, model, nx, ny, count):
    """Every level of the resident loop against a profiled run of as many steps, which is stepped launch by launch (within
    the partitioned solver's tolerance above).  That the loop was resident shows in the autotuner, which runs before a
    step-by-step plan's first solve and never for a resident one."""
    torch = pytest.importorskip("torch")
    steps = 5

    def problems(n):
        if model == "heston":
            return [_stable(nx, ny, steps=n, splitting=q % 4, coeff_mode=L.COEFF_SEPARABLE,
                            line_solver=L.LINE_PARTITIONED) for q in range(count)]
        return [_sabr_small(nx, ny, n, q % 4) for q in range(count)]

    plan = L.Plan.from_models(problems(steps), fp)
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(count)]
    pin = [u.data_ptr() for u in ins]
    outs = [torch.full_like(u, float("nan")) for u in ins]
    levels = [torch.full((steps + 1, nx, ny), float("nan"), dtype=u.dtype, device="cuda") for u in ins]
    plan.run_levels_dev(pin, [v.data_ptr() for v in levels])
    plan.run_dev(pin, [o.data_ptr() for o in outs])
    torch.cuda.synchronize()
    assert plan.kernel_config()["tuned"] == 0
    plan.close()
    tol = 1e-12 if fp == L.FP64 else 1e-5
    for n in range(1, steps + 1):
        short = L.Plan.from_models(problems(n), fp)
        own = [torch.full_like(u, float("nan")) for u in ins]
        L.run_profiled(short, pin, [o.data_ptr() for o in own], torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        short.close()
        for p in range(count):
            e = _normwise(levels[p][n].cpu().numpy().astype(np.float64), own[p].cpu().numpy().astype(np.float64))
            assert e <= tol, (n, p, e)
