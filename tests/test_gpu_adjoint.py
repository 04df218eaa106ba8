"""GPU tests of the hand-written adjoint (lss_adi_forward / lss_adi_backward) through the C-ABI.

The reference has no derivatives, so the adjoint is pinned by what the mathematics fixes:
  * the time loop is affine in the initial surface, so <dJ/du_in, d> must equal J(u_in + d) - J(u_in)
    to rounding for any direction d (the transposed-operator identity, exact for every stage);
  * parameter gradients must match central finite differences (h = 1e-6 relative) of the GPU forward
    solve and of the oracle (the CPU reference gradient);
  * a batched plan must give every problem the gradients of its single-problem plan.
Test problems keep the reference's explicit v = 0 row stable (k <= 1.5 h2).
"""
import numpy as np
import pytest

import linear_system_solvers_amd as L
from helpers import config0, oracle_solve

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _heston(splitting, nx=34, ny=20, steps=14, **kw):
    k = min(0.01, 1.5 / (ny - 1))
    base = dict(nx=nx, ny=ny, nt=steps + 1, t_hi=k * steps, splitting=splitting, weighting=0.3,
                coeff_mode=L.COEFF_SEPARABLE, line_solver=L.LINE_PARTITIONED)
    base.update(kw)
    return config0(**base)


def _sabr(nx=40, ny=24, steps=12, **kw):
    K = 0.03
    m = L.Model(kind=L.MODEL_SABR, strike=K, rate=0.0, sig_sig=0.5, rho=-0.3, beta=0.6, maturity=1.0,
                x_lo=0.0, x_hi=5 * K, y_lo=0.0, y_hi=0.25, nx=nx, ny=ny, nt=steps + 1, t_hi=0.002 * steps,
                accumulation_point=K, alpha_scale=10.0, beta_scale=50.0, grid=L.NONUNIFORM,
                splitting=L.HUNDSDORFER_VERWER, weighting=0.5, coeff_mode=L.COEFF_SEPARABLE,
                line_solver=L.LINE_PARTITIONED)
    for k, v in kw.items():
        setattr(m, k, v)
    return m


def _dev(a, fp=L.FP64):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=L.np_dtype(fp))).cuda()


def _run(plan, u0s):
    """Plain GPU solve (graph off) from host surfaces."""
    ins = [_dev(u, plan.fp) for u in u0s]
    outs = [torch.empty_like(d) for d in ins]
    plan.run_dev([d.data_ptr() for d in ins], [o.data_ptr() for o in outs], graph=False)
    torch.cuda.synchronize()
    return [o.cpu().numpy().astype(np.float64) for o in outs]


def _grad(plan, u0s, ws, ckpt=4):
    ins = [_dev(u, plan.fp) for u in u0s]
    outs = [torch.empty_like(d) for d in ins]
    plan.forward([d.data_ptr() for d in ins], [o.data_ptr() for o in outs], ckpt_every=ckpt)
    lo = [_dev(w, plan.fp) for w in ws]
    li = [torch.empty_like(d) for d in ins]
    dp = plan.backward([d.data_ptr() for d in lo], [d.data_ptr() for d in li])
    torch.cuda.synchronize()
    return ([o.cpu().numpy().astype(np.float64) for o in outs], [g.cpu().numpy().astype(np.float64) for g in li],
            dp)


def _price_weights(plan, p, x0, y0):
    xs, ys = plan.grid(p)
    return L.bilinear_weights(xs.astype(np.float64), ys.astype(np.float64), x0, y0)


@pytest.mark.parametrize("splitting", [0, 1, 2, 3])
@pytest.mark.parametrize("mode,solver", [(L.COEFF_SEPARABLE, L.LINE_PARTITIONED), (L.COEFF_FIELDS, L.LINE_EXACT)])
@pytest.mark.parametrize("ckpt", [4, 32])
def test_initial_surface_gradient_is_the_transpose(splitting, mode, solver, ckpt):
    m = _heston(splitting, coeff_mode=mode, line_solver=solver)
    plan = L.Plan.from_models([m])
    u0 = plan.initial(0)
    rng = np.random.default_rng(5 + splitting)
    w = rng.standard_normal(u0.shape)
    d = rng.standard_normal(u0.shape)
    out, gin, _ = _grad(plan, [u0], [w], ckpt)
    U0 = _run(plan, [u0])[0]
    U1 = _run(plan, [u0 + d])[0]
    np.testing.assert_array_equal(out[0], U0)  # the checkpointing forward is the plain forward
    lhs = float(np.sum(w * (U1 - U0)))
    rhs = float(np.sum(gin[0] * d))
    scale = float(np.sum(np.abs(w)) * max(np.abs(U0).max(), np.abs(U1).max()) + np.sum(np.abs(gin[0] * d)))
    print(f"split {splitting} mode {mode} ckpt {ckpt}: lhs {lhs:.12e} rhs {rhs:.12e} scale {scale:.2e}", flush=True)
    assert abs(lhs - rhs) <= 1e-12 * scale


def _fd(models_fn, name, value, x0, y0, rel=1e-6):
    h = rel * abs(value)
    vals = []
    for sgn in (1.0, -1.0):
        m = models_fn(**{name: value + sgn * h})
        plan = L.Plan.from_models([m])
        w = _price_weights(plan, 0, x0, y0)
        vals.append(float(np.sum(w * _run(plan, [plan.initial(0)])[0])))
    return (vals[0] - vals[1]) / (2 * h)


HESTON_ATTR = {"kappa": "sig_kappa", "theta_v": "sig_theta", "sigma": "sig_sig", "rho": "rho", "r": "rate"}


@pytest.mark.parametrize("splitting", [0, 1, 2, 3])
def test_heston_parameter_gradients_match_finite_differences(splitting):
    m = _heston(splitting, nx=40, ny=24, steps=12, grid=L.NONUNIFORM, accumulation_point=100.0, alpha_scale=3.0)
    plan = L.Plan.from_models([m])
    assert plan.param_count(0) == 5
    w = _price_weights(plan, 0, 100.0, 0.04)
    _, _, dp = _grad(plan, [plan.initial(0)], [w], ckpt=4)
    for k, name in enumerate(L.HESTON_PARAMS):
        attr = HESTON_ATTR[name]
        fd = _fd(lambda **o: _heston(splitting, nx=40, ny=24, steps=12, grid=L.NONUNIFORM, accumulation_point=100.0,
                                     alpha_scale=3.0, **o), attr, getattr(m, attr), 100.0, 0.04)
        print(f"split {splitting} {name}: adjoint {dp[0, k]:.10e} fd {fd:.10e}", flush=True)
        assert abs(dp[0, k] - fd) <= 1e-6 * abs(fd) + 1e-7


def test_heston_gradients_match_the_oracle_finite_differences(oracle):
    """CPU reference gradient: central differences of the oracle's solve (the reference's host path)."""
    mk = lambda **o: _heston(2, nx=36, ny=20, steps=10, **o)  # noqa: E731
    m = mk()
    plan = L.Plan.from_models([m])
    w = _price_weights(plan, 0, 100.0, 0.04)
    _, _, dp = _grad(plan, [plan.initial(0)], [w], ckpt=4)
    for k, name in enumerate(L.HESTON_PARAMS):
        attr = HESTON_ATTR[name]
        v = getattr(m, attr)
        h = 1e-6 * abs(v)
        jp = float(np.sum(w * oracle_solve(oracle, mk(**{attr: v + h}))))
        jm = float(np.sum(w * oracle_solve(oracle, mk(**{attr: v - h}))))
        fd = (jp - jm) / (2 * h)
        print(f"{name}: adjoint {dp[0, k]:.10e} oracle fd {fd:.10e}", flush=True)
        assert abs(dp[0, k] - fd) <= 1e-6 * abs(fd) + 1e-7


def test_sabr_parameter_gradients_match_finite_differences():
    m = _sabr()
    plan = L.Plan.from_models([m])
    assert plan.param_count(0) == 4
    x0, y0 = 0.03, 0.05
    w = _price_weights(plan, 0, x0, y0)
    _, _, dp = _grad(plan, [plan.initial(0)], [w], ckpt=4)
    for k, (name, attr) in enumerate(zip(L.SABR_PARAMS, ("sig_sig", "rho", "beta"))):
        fd = _fd(lambda **o: _sabr(**o), attr, getattr(m, attr), x0, y0)
        print(f"sabr {name}: adjoint {dp[0, k]:.10e} fd {fd:.10e}", flush=True)
        assert abs(dp[0, k] - fd) <= 1e-6 * abs(fd) + 1e-9
    # the alpha axis: y_hi and the price point scaled together by lam = 1 +- h
    h, vals = 1e-6, []
    for sgn in (1.0, -1.0):
        lam = 1.0 + sgn * h
        pq = L.Plan.from_models([_sabr(y_hi=m.y_hi * lam)])
        vals.append(float(np.sum(_price_weights(pq, 0, x0, y0 * lam) * _run(pq, [pq.initial(0)])[0])))
    fd = (vals[0] - vals[1]) / (2 * h)
    print(f"sabr alpha axis: adjoint {dp[0, 3]:.10e} fd {fd:.10e}", flush=True)
    assert abs(dp[0, 3] - fd) <= 1e-6 * abs(fd) + 1e-9


def test_sabr_alpha_axis_gradient_with_a_raised_lower_end():
    """With y_lo > 0 the alpha-axis terms of b and e do not vanish (generic adjoint tables); the price is
    read at a fixed eta, i.e. at y_lo + lam (y0 - y_lo)."""
    mk = lambda **o: _sabr(y_lo=0.01, **o)  # noqa: E731
    m = mk()
    plan = L.Plan.from_models([m])
    x0, y0 = 0.03, 0.05
    w = _price_weights(plan, 0, x0, y0)
    _, _, dp = _grad(plan, [plan.initial(0)], [w], ckpt=4)
    assert plan.kernel_config()["adjoint_pattern"] == 0
    h, vals = 1e-6, []
    for sgn in (1.0, -1.0):
        lam = 1.0 + sgn * h
        pq = L.Plan.from_models([mk(y_hi=m.y_lo + (m.y_hi - m.y_lo) * lam)])
        vals.append(float(np.sum(_price_weights(pq, 0, x0, m.y_lo + (y0 - m.y_lo) * lam) *
                                 _run(pq, [pq.initial(0)])[0])))
    fd = (vals[0] - vals[1]) / (2 * h)
    print(f"sabr alpha axis (y_lo 0.01): adjoint {dp[0, 3]:.10e} fd {fd:.10e}", flush=True)
    assert abs(dp[0, 3] - fd) <= 1e-6 * abs(fd) + 1e-9


def test_batched_adjoint_equals_single_problem_adjoints():
    rng = np.random.default_rng(3)
    models = []
    for q in range(6):
        nx, ny = int(rng.integers(10, 70)), int(rng.integers(8, 40))
        models.append(_heston(q % 4, nx=nx, ny=ny, steps=int(rng.integers(3, 15)),
                              sig_kappa=float(rng.uniform(1, 4)), rho=float(rng.uniform(-0.8, 0.2))))
    plan = L.Plan.from_models(models)
    u0s = [plan.initial(p) for p in range(len(models))]
    ws = [rng.standard_normal(u.shape) for u in u0s]
    _, gb, db = _grad(plan, u0s, ws, ckpt=4)
    for p, m in enumerate(models):
        single = L.Plan.from_models([m])
        _, gs, ds = _grad(single, [u0s[p]], [ws[p]], ckpt=4)
        np.testing.assert_allclose(gb[p], gs[0], rtol=0, atol=1e-14 * np.abs(gs[0]).max())
        np.testing.assert_allclose(db[p], ds[0], rtol=1e-13, atol=1e-300)


def test_fp32_adjoint_tracks_fp64():
    m = _heston(3, nx=40, ny=24, steps=12)
    p64 = L.Plan.from_models([m], fp=L.FP64)
    p32 = L.Plan.from_models([m], fp=L.FP32)
    w = _price_weights(p64, 0, 100.0, 0.04)
    _, g64, d64 = _grad(p64, [p64.initial(0)], [w])
    _, g32, d32 = _grad(p32, [p32.initial(0)], [w])
    err_g = np.abs(g32[0] - g64[0]).max() / np.abs(g64[0]).max()
    err_p = np.abs(d32[0, :5] - d64[0, :5]).max() / np.abs(d64[0, :5]).max()
    print(f"fp32 vs fp64: initial-surface gradient {err_g:.2e}, parameters {err_p:.2e}", flush=True)
    assert err_g <= 1e-4 and err_p <= 1e-3


def test_backward_without_forward_is_an_error():
    plan = L.Plan.from_models([_heston(0)])
    lo = _dev(np.zeros((34, 20)))
    with pytest.raises(L.LssError):
        plan.backward([lo.data_ptr()])


@pytest.mark.parametrize("model", ["heston", "sabr"])
def test_specialized_adjoint_kernels_match_the_generic_ones(model):
    """Separable Heston / SABR plans run the adjoint kernels with compile-time factor and derivative-term
    tables; the same problem with FIELDS coefficients runs the generic kernels (tables read at run time).
    Both must give the same gradients, up to the rounding of the two coefficient forms."""
    if model == "heston":
        mk, x0, y0, want = (lambda **o: _heston(2, nx=40, ny=24, steps=12, **o)), 100.0, 0.04, 1
    else:
        mk, x0, y0, want = (lambda **o: _sabr(**o)), 0.03, 0.05, 2
    res = {}
    for mode in (L.COEFF_SEPARABLE, L.COEFF_FIELDS):
        plan = L.Plan.from_models([mk(coeff_mode=mode)])
        assert plan.kernel_config()["adjoint_pattern"] == -1  # not set up before the first forward()
        w = _price_weights(plan, 0, x0, y0)
        _, g, dp = _grad(plan, [plan.initial(0)], [w])
        res[mode] = (plan.kernel_config()["adjoint_pattern"], g[0], dp[0])
    assert res[L.COEFF_SEPARABLE][0] == want and res[L.COEFF_FIELDS][0] == 0
    gs, gf = res[L.COEFF_SEPARABLE][1], res[L.COEFF_FIELDS][1]
    ds, df = res[L.COEFF_SEPARABLE][2], res[L.COEFF_FIELDS][2]
    print(f"{model}: surface gradient diff {np.abs(gs - gf).max() / np.abs(gf).max():.2e}, "
          f"parameters {ds[:5]} vs {df[:5]}", flush=True)
    assert np.abs(gs - gf).max() <= 1e-9 * np.abs(gf).max()
    np.testing.assert_allclose(ds, df, rtol=1e-8, atol=1e-12 * np.abs(df).max())


def test_overlapped_backward_matches_the_single_stream_one():
    """With a second segment store the backward pass recomputes segment c - 1 on a second stream
    while the adjoint of segment c runs; without it both run on the caller's stream.  The gradients
    must not depend on the schedule (600 x 460 MCS, theta 0.5, 300 steps, segments of 32)."""
    m = _heston(2, nx=600, ny=460, steps=300, weighting=0.5)
    plan = L.Plan.from_models([m])
    u0 = plan.initial(0)
    w = _price_weights(plan, 0, 100.0, 0.04)
    res = {}
    for mode in (0, 1):
        plan.set_adjoint_overlap(mode)
        out, g, dp = _grad(plan, [u0], [w], ckpt=32)
        res[mode] = (plan.kernel_config()["adjoint_overlap"], out[0], g[0], dp[0])
    assert res[0][0] == 0 and res[1][0] == 1
    assert np.isfinite(res[0][2]).all() and np.isfinite(res[0][3]).all()
    np.testing.assert_array_equal(res[0][1], res[1][1])
    gd = np.abs(res[0][2] - res[1][2]).max() / np.abs(res[0][2]).max()
    print(f"overlapped vs single-stream backward: surface gradient {gd:.2e}, parameters {res[1][3][:5]} vs "
          f"{res[0][3][:5]}", flush=True)
    assert gd <= 1e-13
    np.testing.assert_allclose(res[1][3], res[0][3], rtol=1e-12, atol=1e-14 * np.abs(res[0][3]).max())
    plan.set_adjoint_overlap(-1)  # automatic: this plan's 0.28 GB second store is under 2 GiB
    _grad(plan, [u0], [w], ckpt=32)
    assert plan.kernel_config()["adjoint_overlap"] == 1
    with pytest.raises(L.LssError):
        plan.set_adjoint_overlap(2)


@pytest.mark.parametrize("solver", [L.LINE_PARTITIONED, L.LINE_EXACT])
@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("steps", [(7,), (8,), (9, 3, 12, 8)])
def test_a_second_backward_of_one_forward_gives_the_same_gradients(solver, overlap, steps):
    """The forward pass leaves the last segment's stages for the first backward pass; a second one recomputes them
    from the checkpoint.  The same kernels on the same values: no tolerance.  Steps around the segment length (4),
    problems that end in earlier segments, and sizes that no resident loop takes."""
    mode = L.COEFF_SEPARABLE if solver == L.LINE_PARTITIONED else L.COEFF_FIELDS
    models = [_heston((2 + q) % 4, nx=150 + q, ny=40 + q, steps=n, coeff_mode=mode, line_solver=solver)
              for q, n in enumerate(steps)]
    plan = L.Plan.from_models(models)
    plan.set_adjoint_overlap(overlap)
    u0s = [plan.initial(p) for p in range(plan.count)]
    ins = [_dev(u) for u in u0s]
    outs = [torch.empty_like(d) for d in ins]
    plan.forward([d.data_ptr() for d in ins], [o.data_ptr() for o in outs], ckpt_every=4)
    lo = [_dev(np.random.default_rng(7 + p).standard_normal(u.shape)) for p, u in enumerate(u0s)]
    res = []
    for _ in range(2):
        li = [torch.empty_like(d) for d in ins]
        dp = plan.backward([d.data_ptr() for d in lo], [d.data_ptr() for d in li])
        torch.cuda.synchronize()
        res.append((dp, [g.cpu().numpy() for g in li]))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    for a, b in zip(res[0][1], res[1][1]):
        np.testing.assert_array_equal(a, b)
    for o, u in zip(outs, _run(plan, u0s)):
        np.testing.assert_array_equal(o.cpu().numpy(), u)
    plan.close()
