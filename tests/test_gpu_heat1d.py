"""GPU 1-D implicit heat / Black-Scholes solver (include/lss_heat1d.h) against the oracle.

* The exact kernel (four lanes per problem, the reference's Thomas LU / double-sweep order, no
  contraction) equals the oracle's restatement of the reference's host solver bit for bit, final level
  and every level, fp64 and fp32, Euler and Crank-Nicolson, Forward and Backward, both grids.
* The partitioned kernel (one wavefront per problem, the whole loop in registers, fused multiply-adds)
  stays within 1e-12 normwise of the oracle in fp64 and 1e-5 in fp32, for line lengths that take
  every chunk length 1..16.
* Books of mixed problems in one launch give each problem its single-problem result.
* On fine grids the GPU solution converges to black_scholes_exact (common/lss_utility.hpp:70-110).
"""
import numpy as np
import pytest

import linear_system_solvers_amd as L
from linear_system_solvers_amd import heat1d as H

pytestmark = pytest.mark.gpu


def _oracle(O, m: H.BsModel, fp="f64", surfaces=False):
    cfg = O.Heat1dCfg(x_lo=m.x_lo, x_hi=m.x_hi, n=m.n, nt=m.nt, t_lo=m.t_lo, t_hi=m.t_hi,
                      accumulation_point=m.accumulation_point, alpha_scale=m.alpha_scale,
                      nonuniform=m.grid == L.NONUNIFORM, implicit_scheme=m.implicit_scheme,
                      tridiagonal=O.DOUBLE_SWEEP if m.tridiagonal == L.DOUBLE_SWEEP else O.THOMAS_LU,
                      direction=m.direction)
    return O.heat1d_solve(O.bs_heat1d_pde(m.strike, m.rate, m.sig, m.maturity, m.x_hi), cfg, fp, surfaces=surfaces)


def _normwise(g, c):
    return float(np.abs(np.asarray(g, np.float64) - c).max() / np.abs(c).max())


CASES = [
    dict(),                                                                   # print test :209 (CN, default hints)
    dict(implicit_scheme=L.EULER),                                            # :105
    dict(implicit_scheme=L.EULER, accumulation_point=10.0),                   # :327
    dict(accumulation_point=10.0, grid=L.NONUNIFORM),                         # :439
    dict(direction=L.FORWARD, tridiagonal=L.DOUBLE_SWEEP),
    dict(n=37, nt=11, grid=L.NONUNIFORM, accumulation_point=10.0, tridiagonal=L.DOUBLE_SWEEP),
]


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_exact_kernel_is_bit_identical_to_the_oracle(oracle, fp, case):
    m = H.BsModel(**CASES[case])
    plan = H.Heat1dPlan.from_bs_models([m], fp)
    outs, surf = plan.run_host(surfaces=True)
    o, osurf = _oracle(oracle, m, "f64" if fp == L.FP64 else "f32", surfaces=True)
    print(f"case {case} fp {fp}: max |gpu - oracle| {np.abs(outs[0] - o).max():.3e}", flush=True)
    assert np.array_equal(outs[0], o)
    assert np.array_equal(surf[0], osurf)
    np.testing.assert_array_equal(plan.grid(0), oracle.heat1d_grid(
        oracle.Heat1dCfg(x_lo=m.x_lo, x_hi=m.x_hi, n=m.n, nt=m.nt, accumulation_point=m.accumulation_point,
                         alpha_scale=m.alpha_scale, nonuniform=m.grid == L.NONUNIFORM),
        "f64" if fp == L.FP64 else "f32")[0])
    plan.close()


@pytest.mark.parametrize("fp,tol", [(L.FP64, 1e-12), (L.FP32, 1e-5)])
@pytest.mark.parametrize("n", [10, 66, 100, 130, 152, 300, 514, 702, 1026])
def test_partitioned_kernel_within_tolerance(oracle, fp, tol, n):
    """f64: within 1e-12 of the oracle.  f32: the partitioned elimination rounds differently from the
    sequential Thomas sweep, and Crank-Nicolson carries that difference through the loop undamped; the
    bar is 1e-5 or the f32 oracle's own distance from the f64 oracle, whichever is larger, and the GPU's
    distance from the f64 oracle within 1.5 times the f32 oracle's (as accurate as the reference's f32)."""
    # unknowns n - 2 take chunk lengths 1, 1, 2, 2, 3, 6, 8, 16, 16
    for extra in (dict(), dict(implicit_scheme=L.EULER, grid=L.NONUNIFORM, accumulation_point=10.0,
                               direction=L.FORWARD)):
        m = H.BsModel(n=n, nt=60, line_solver=L.LINE_PARTITIONED, **extra)
        plan = H.Heat1dPlan.from_bs_models([m], fp)
        outs, surf = plan.run_host(surfaces=True)
        o, osurf = _oracle(oracle, m, "f64" if fp == L.FP64 else "f32", surfaces=True)
        e, es = _normwise(outs[0], o), _normwise(surf[0], osurf)
        bar, extra_msg = tol, ""
        if fp == L.FP32:
            o64, osurf64 = _oracle(oracle, m, "f64", surfaces=True)
            own = max(_normwise(o, o64), _normwise(osurf, osurf64))
            g64 = max(_normwise(outs[0], o64), _normwise(surf[0], osurf64))
            bar = max(tol, own)
            extra_msg = f"; f32 oracle vs f64 oracle {own:.3e}, partitioned vs f64 oracle {g64:.3e}"
            assert g64 <= 1.5 * own + tol
        print(f"n {n} {extra}: partitioned vs oracle {e:.3e} (surface {es:.3e}){extra_msg}", flush=True)
        assert e <= bar and es <= bar
        plan.close()


def test_book_of_mixed_problems_gives_each_its_single_result(oracle):
    rng = np.random.default_rng(11)
    models = []
    for q in range(300):
        models.append(H.BsModel(strike=float(rng.uniform(5, 15)), rate=float(rng.uniform(0, 0.1)),
                                sig=float(rng.uniform(0.1, 0.6)), maturity=1.0, n=int(rng.integers(8, 600)),
                                nt=int(rng.integers(2, 120)), accumulation_point=float(rng.uniform(5, 15)),
                                grid=L.NONUNIFORM if q % 2 else L.UNIFORM,
                                implicit_scheme=L.EULER if q % 3 == 0 else L.CRANK_NICOLSON,
                                tridiagonal=L.DOUBLE_SWEEP if q % 5 == 0 else L.THOMAS_LU,
                                direction=L.FORWARD if q % 7 == 0 else L.BACKWARD))
    for solver in (L.LINE_EXACT, L.LINE_PARTITIONED):
        for m in models:
            m.line_solver = solver
        plan = H.Heat1dPlan.from_bs_models(models, L.FP64)
        outs = plan.run_host()
        worst = 0.0
        for q in range(0, len(models), 7):
            o = _oracle(oracle, models[q])
            if solver == L.LINE_EXACT:
                assert np.array_equal(outs[q], o), q
            else:
                worst = max(worst, _normwise(outs[q], o))
        print(f"book of {len(models)}, line solver {solver}: worst normwise {worst:.3e}", flush=True)
        assert worst <= 1e-12
        plan.close()


def test_device_run_with_surfaces_equals_host_run():
    torch = pytest.importorskip("torch")
    models = [H.BsModel(n=200, nt=50, line_solver=L.LINE_PARTITIONED, strike=8.0 + q) for q in range(5)]
    plan = H.Heat1dPlan.from_bs_models(models, L.FP64)
    host_out, host_surf = plan.run_host(surfaces=True)
    ins = [torch.from_numpy(plan.initial(p)).cuda() for p in range(plan.count)]
    outs = [torch.empty_like(u) for u in ins]
    surfs = [torch.empty((50, 200), dtype=torch.float64, device="cuda") for _ in ins]
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(2):  # the second run reuses the device pointer table
        plan.run_dev([u.data_ptr() for u in ins], [u.data_ptr() for u in outs], [s.data_ptr() for s in surfs], stream)
    torch.cuda.synchronize()
    for p in range(plan.count):
        assert np.array_equal(outs[p].cpu().numpy(), host_out[p])
        assert np.array_equal(surfs[p].cpu().numpy(), host_surf[p])
    plan.close()


def test_gpu_converges_to_black_scholes_exact():
    from scipy.stats import norm
    errs = []
    for n in (200, 400, 800):
        m = H.BsModel(n=n, nt=n, grid=L.NONUNIFORM, accumulation_point=10.0, line_solver=L.LINE_PARTITIONED)
        plan = H.Heat1dPlan.from_bs_models([m], L.FP64)
        u = plan.run_host()[0]
        x = plan.grid(0)
        sel = (x > 5) & (x < 15)
        xs = x[sel]
        d1 = (np.log(xs / 10.0) + (0.2 + 0.5 * 0.25 ** 2)) / 0.25
        exact = norm.cdf(d1) * xs - norm.cdf(d1 - 0.25) * 10.0 * np.exp(-0.2)
        errs.append(np.abs(u[sel] - exact).max())
        plan.close()
    print("errors vs black_scholes_exact", errs, flush=True)
    assert errs[2] < errs[1] < errs[0] < 5e-3
    assert errs[1] / errs[2] > 3.0


def test_invalid_descriptions_are_rejected():
    with pytest.raises(L.LssError):
        H.Heat1dPlan.from_bs_models([H.BsModel(n=3)])
    with pytest.raises(L.LssError):
        H.Heat1dPlan.from_bs_models([H.BsModel(implicit_scheme=L.THETA_30)])
    with pytest.raises(L.LssError):
        H.Heat1dPlan.from_bs_models([H.BsModel(n=1100, line_solver=L.LINE_PARTITIONED)])
    plan = H.Heat1dPlan.from_bs_models([H.BsModel()])
    with pytest.raises(L.LssError):
        plan.run_host([np.zeros(99)])
    plan.close()


# ---------------------------------------------------------------------------------------------
# Every form of a described problem through the exact kernel: both sweeps, the nine end pairs, coefficients
# and boundaries fixed or changing in time, with and without a source, lines that end anywhere in a group of
# 16 points, problems of different forms and lengths side by side in a wavefront, levels in LDS (every line
# of the plan at most 512 points) and in the workspace.  The oracle steps the same rows one by one; the
# kernel keeps its order of operations, so equality is exact.
# ---------------------------------------------------------------------------------------------
def _descr(ctypes, fp, n, steps, tri, lo, hi, direction, tdep_c, tdep_b, source, theta, rng):
    dt = L.np_dtype(fp)
    cs, bs = (steps if tdep_c else 1), (steps if tdep_b else 1)
    A = rng.uniform(0.1, 2.0, (cs, n)).astype(dt)
    D = rng.uniform(0.1, 2.0, (cs, n)).astype(dt)
    B = ((A + D) / dt(2) + rng.uniform(0.0, 0.2, (cs, n)).astype(dt)).astype(dt)
    return dict(fp=fp, n=n, steps=steps, tri=tri, lo=lo, hi=hi, direction=direction, theta=theta, k=dt(0.01),
                coeff=np.ascontiguousarray(np.stack([A, B, D], 1)), bnd=rng.uniform(-0.5, 0.5, (bs, 4)).astype(dt),
                src=rng.uniform(-1.0, 1.0, (steps, 2, n)).astype(dt) if source else None,
                u0=rng.uniform(-1.0, 1.0, n).astype(dt))


def _stepped(O, q):
    dt, n, N = L.np_dtype(q["fp"]), q["n"], q["n"] - 1
    one, two, th, k = dt(1), dt(2), dt(q["theta"]), dt(q["k"])
    om, h = one - th, one / dt(n - 1)
    u, levels = q["u0"].copy(), [q["u0"]]
    solve = O.double_sweep if q["tri"] == L.DOUBLE_SWEEP else O.thomas_lu
    for s in range(q["steps"]):
        A, B, D = q["coeff"][s if len(q["coeff"]) > 1 else 0]
        ll, lv, hl, hv = q["bnd"][s if len(q["bnd"]) > 1 else 0]
        f = np.zeros(n, dt)
        f[1:N] = (D[1:N] * om * u[2:]) + ((one - two * B[1:N] * om) * u[1:N]) + (A[1:N] * om * u[:N - 1])
        if q["lo"] != L.BC_DIRICHLET:
            beta = two * h * lv
            mid = (one - two * om * B[0]) if q["lo"] == L.BC_NEUMANN else (one - om * (two * B[0] - two * h * ll * A[0]))
            f[0] = om * beta * A[0] + mid * u[0] + om * (A[0] + D[0]) * u[1]
        if q["hi"] != L.BC_DIRICHLET:
            delta = two * h * hv
            mid = (one - two * om * B[N]) if q["hi"] == L.BC_NEUMANN else (one - om * (two * B[N] + two * h * hl * D[N]))
            f[N] = om * (A[N] + D[N]) * u[N - 1] + mid * u[N] - om * delta * D[N]
        if q["src"] is not None:
            F, Fn = q["src"][s]
            f[1:N] = f[1:N] + k * (th * Fn[1:N] + om * F[1:N])
            for e, t in ((0, q["lo"]), (N, q["hi"])):
                if t != L.BC_DIRICHLET:
                    f[e] = f[e] + th * k * Fn[e] + om * k * F[e]
        u = solve(-th * A, one + two * th * B, -th * D, f, (q["lo"], ll, lv), (q["hi"], hl, hv),
                  "f64" if q["fp"] == L.FP64 else "f32")
        levels.append(u)
    return np.stack(levels if q["direction"] == L.FORWARD else levels[::-1]), u


def _described_plan(ctypes, descr, line_solver):
    class D(ctypes.Structure):
        _fields_ = [*[(f, ctypes.c_int32) for f in ("fp", "tridiagonal", "line_solver", "lo_type", "hi_type", "direction")],
                    ("n", ctypes.c_int64), ("steps", ctypes.c_int64), ("theta", ctypes.c_double), ("k", ctypes.c_double),
                    ("coeff_sets", ctypes.c_int64), ("coeff", ctypes.c_void_p), ("bnd_sets", ctypes.c_int64),
                    ("bnd", ctypes.c_void_p), ("source", ctypes.c_void_p)]
    arr = (D * len(descr))(*[D(q["fp"], q["tri"], line_solver, q["lo"], q["hi"], q["direction"], q["n"], q["steps"],
                               q["theta"], float(q["k"]), len(q["coeff"]), q["coeff"].ctypes.data, len(q["bnd"]),
                               q["bnd"].ctypes.data, None if q["src"] is None else q["src"].ctypes.data) for q in descr])
    h = ctypes.c_void_p()
    lib = H._lib()
    assert lib.lss_heat1d_plan_create(arr, ctypes.c_int64(len(descr)), ctypes.byref(h)) == 0, L.lib().lss_last_error()
    return H.Heat1dPlan(h.value, descr[0]["fp"], len(descr))


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("sizes", [(4, 5, 15, 16, 17, 18, 31, 32, 33, 48, 49, 70), (16, 17, 600, 513, 4, 530)])
def test_every_form_of_the_exact_kernel_equals_the_oracle(oracle, fp, sizes):
    import ctypes
    import itertools
    rng = np.random.default_rng(len(sizes))
    ends = (L.BC_DIRICHLET, L.BC_NEUMANN, L.BC_ROBIN)
    descr = []
    for z, (tri, lo, hi, tc, tb, src) in enumerate(itertools.product((L.THOMAS_LU, L.DOUBLE_SWEEP), ends, ends, (0, 1), (0, 1),
                                                                     (0, 1))):
        descr.append(_descr(ctypes, fp, sizes[(z * 5 + z // 7) % len(sizes)], 3 + z % 3, tri, lo, hi,
                            L.FORWARD if z % 2 else L.BACKWARD, tc, tb, src, 1.0 if z % 4 == 3 else 0.5, rng))
    plan = _described_plan(ctypes, descr, L.LINE_EXACT)
    for _ in range(2):  # the second solve finds the first one's workspace
        outs, surfs = plan.run_host([q["u0"] for q in descr], surfaces=True)
        for z, q in enumerate(descr):
            surf, out = _stepped(oracle, q)
            assert np.array_equal(outs[z], out), (z, q["n"], q["tri"], q["lo"], q["hi"])
            assert np.array_equal(surfs[z], surf), (z, q["n"])
    plan.close()


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-25, 1e-42, 1e-280, 1e-305, 1e-318, 1e30, 1e295])
def test_exact_kernel_rounds_like_the_oracle_at_any_magnitude(oracle, fp, scale):
    # the sweep divides by known divisors without an IEEE division where the exponents allow it; zeros of either
    # sign, subnormal, tiny and huge levels (each also mixed with ordinary values) take every way out of that
    import ctypes
    rng = np.random.default_rng(17)
    dt, descr = L.np_dtype(fp), []
    for z in range(24):
        q = _descr(ctypes, fp, 20 + 3 * z, 3, (L.THOMAS_LU, L.DOUBLE_SWEEP)[z % 2], z % 3, (z // 3) % 3, L.FORWARD, 0, 0, 0,
                   0.5, rng)
        with np.errstate(over="ignore", under="ignore"):
            keep = rng.uniform(size=q["n"]) < (0.0 if z % 4 else 0.3)
            q["u0"] = np.where(keep, q["u0"], (q["u0"].astype(np.float64) * scale).astype(dt)).astype(dt)
            q["bnd"] = (q["bnd"].astype(np.float64) * (scale if z % 5 else 1.0)).astype(dt)
        descr.append(q)
    plan = _described_plan(ctypes, descr, L.LINE_EXACT)
    outs = plan.run_host([q["u0"] for q in descr])
    for z, q in enumerate(descr):
        with np.errstate(all="ignore"):
            out = _stepped(oracle, q)[1]
        assert np.array_equal(outs[z], out, equal_nan=True), (z, q["n"])
    plan.close()


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("n", [4, 20, 65, 66, 67, 130, 190, 258, 390, 514, 600, 1024])
def test_every_form_of_the_partitioned_kernels(oracle, fp, n):
    # the nine end pairs, with and without a source, boundaries fixed or changing in time, the matrix fixed (one plan)
    # or changing in time (another): 1..16 points per lane, lines that end on a lane's last point and before it.
    # Tolerance: the rows dominate by at least 1 of at most 5 (b = 1 + theta 2 B, |a| + |c| = theta (A + D) <= theta 2 B),
    # so a step's few tens of roundings grow at most fivefold; 256 eps a step covers both sides.
    import ctypes
    import itertools
    rng = np.random.default_rng(n)
    ends = (L.BC_DIRICHLET, L.BC_NEUMANN, L.BC_ROBIN)
    for tc in (0, 1):
        descr = [_descr(ctypes, fp, n, 6, L.THOMAS_LU, lo, hi, L.FORWARD if src else L.BACKWARD, tc,
                        tb and (tc or L.BC_ROBIN not in (lo, hi)), src, 0.5, rng)
                 for lo, hi, src, tb in itertools.product(ends, ends, (0, 1), (0, 1))]
        plan = _described_plan(ctypes, descr, L.LINE_PARTITIONED)
        outs, surfs = plan.run_host([q["u0"] for q in descr], surfaces=True)
        for z, q in enumerate(descr):
            surf, out = _stepped(oracle, q)
            tol = 256 * q["steps"] * np.finfo(L.np_dtype(fp)).eps
            e, es = _normwise(outs[z], out), _normwise(surfs[z], surf)
            assert e <= tol and es <= tol, (tc, z, q["lo"], q["hi"], e, es)
        plan.close()


# ---------------------------------------------------------------------------------------------
# Divisors outside the range in which the exact kernel divides by a known divisor (2^-20 .. 2^21 in fp32, 2^-100 ..
# 2^101 in fp64): one such row in a line, at each of the 16 positions of a group, or in the line's last row.  A
# wavefront holds 16 problems and takes the division as soon as one of them asks for it, so the 16 problems of a block
# have their row at the same position.  The oracle divides every row; equality is exact, signs of zeros included.
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
@pytest.mark.parametrize("tdep", [0, 1])
@pytest.mark.parametrize("kind", ["large", "small"])
def test_one_divisor_out_of_range_at_every_position(oracle, fp, kind, tdep):
    import ctypes
    rng = np.random.default_rng(23)
    dt, descr = L.np_dtype(fp), []
    bits = 22 if fp == L.FP32 else 102
    for row in [*range(16, 32), -1]:
        for z in range(16):
            lo, hi = z % 3, (z // 3) % 3
            if row < 0 and hi == L.BC_DIRICHLET:
                hi = L.BC_ROBIN  # (the last row has a divisor of its own)
            q = _descr(ctypes, fp, 48 if row < 0 else 33 + 2 * z, 3, (L.THOMAS_LU, L.DOUBLE_SWEEP)[z % 2], lo, hi,
                       L.FORWARD, tdep, 0, 0, 0.5, rng)
            A, B, D = q["coeff"][:, 0], q["coeff"][:, 1], q["coeff"][:, 2]
            if kind == "large":  # diagonal 1 + B
                B[:, row] = 2.0 ** bits
            else:  # diagonal 0: the divisor is what elimination leaves
                B[:, row] = -1.0
                A[:, row] *= dt(2.0 ** -bits)
                if row < 0:
                    D[:, row] = 0.0
                    q["bnd"][:, 2] = 0.0
            descr.append(q)
    plan = _described_plan(ctypes, descr, L.LINE_EXACT)
    outs = plan.run_host([q["u0"] for q in descr])
    for z, q in enumerate(descr):
        out = _stepped(oracle, q)[1]
        assert np.isfinite(out).all()
        assert np.array_equal(outs[z], out) and np.array_equal(np.signbit(outs[z]), np.signbit(out)), (z // 16, z % 16)
    plan.close()


@pytest.mark.parametrize("n,sig", [(8001, 0.41), (10000, 0.46)])
def test_a_fine_fp32_line_whose_diagonal_grows_past_the_range(oracle, n, sig):
    m = H.BsModel(n=n, nt=2, rate=0.05, sig=sig, implicit_scheme=L.EULER)
    plan = H.Heat1dPlan.from_bs_models([m], L.FP32)
    out = plan.run_host()[0]
    plan.close()
    assert np.isfinite(out).all()
    assert np.array_equal(out, _oracle(oracle, m, "f32"))


@pytest.mark.parametrize("fp", [L.FP64, L.FP32])
def test_negative_divisors_keep_the_sign_of_zero(oracle, fp):
    # zero levels and negative diagonals: the quotients are zeros whose signs are the divisors'
    import ctypes
    rng = np.random.default_rng(29)
    dt, descr = L.np_dtype(fp), []
    for z in range(64):
        q = _descr(ctypes, fp, 17 + z, 3, (L.THOMAS_LU, L.DOUBLE_SWEEP)[z % 2], z % 3, (z // 3) % 3, L.FORWARD, 0, 0, 0, 1.0,
                   rng)
        q["coeff"][:, 1] = -rng.uniform(1.1, 4.0, q["coeff"][:, 1].shape).astype(dt)  # diagonal 1 + 2 B < 0
        q["coeff"][:, (0, 2)] *= dt(0.1)
        keep = rng.uniform(size=q["n"]) < 0.2 * (z % 2)
        q["u0"] = np.where(keep, q["u0"], dt(0.0)).astype(dt)
        q["bnd"][:] = 0.0
        descr.append(q)
    plan = _described_plan(ctypes, descr, L.LINE_EXACT)
    outs, surfs = plan.run_host([q["u0"] for q in descr], surfaces=True)
    for z, q in enumerate(descr):
        surf, out = _stepped(oracle, q)
        assert np.array_equal(outs[z], out) and np.array_equal(surfs[z], surf)
        assert np.array_equal(np.signbit(surfs[z]), np.signbit(surf)), (z, q["n"])
    plan.close()
