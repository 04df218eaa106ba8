// lss_heat1d_wave.hip -- the 1-D implicit heat / Black-Scholes time loop with one wavefront per
// problem and the whole loop in registers.
//
// k_h1_wave steps any problem, k_h1_wave_fixed (below) those whose matrix does not change in time.
// Lane l holds the C consecutive unknowns of its chunk of the line (the partition of
// lss_adi_chunk.hpp), the level's values and, for coefficients that do not change in time, A, B, D of
// its points.  Each step forms the theta scheme's right-hand side from the lane's values and its
// neighbours' (one shuffle each way), folds the boundary pair into the end rows, and solves the
// tridiagonal system by the register-resident partitioned elimination with cyclic reduction of the
// chunk interfaces.  HBM traffic per problem is the first level, the last level (and every level when
// the caller asks for the surface) plus the coefficient and boundary sets that vary in time.
//
// The arithmetic of each row follows implicit_heat_scheme::rhs / rhs_source and
// heat_implicit_solver_method::split (pde_solvers/one_dimensional/heat_type/solver_method/
// lss_heat_implicit_solver_method.hpp:36-171, 200-210) and thomas_lu_solver_boundary's folding of the
// end rows (sparse_solvers/tridiagonal/thomas_lu_solver/lss_thomas_lu_boundary.hpp:114-205); multiply-
// adds may be fused here and the elimination order differs from the sequential Thomas sweep.
#pragma clang fp contract(fast)
#include "lss_adi_chunk.hpp"
#include "lss_heat1d_device.hpp"

namespace lssamd {

template <typename T, int M>
__global__ void __launch_bounds__(64 * H1_WAVES) k_h1_wave(const H1Prob<T> *__restrict__ probs, int count,
                                                           const T *const *__restrict__ uin,
                                                           T *const *__restrict__ uout, T *const *__restrict__ surf)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int p = blockIdx.x * H1_WAVES + wave;
    if (p >= count)
        return;  // uniform over the wavefront
    const H1Prob<T> &P = probs[p];
    const int n = P.n, N = n - 1, steps = P.steps;
    const int gs = P.lo_type == BC_DIRICHLET ? 1 : 0, ge = P.hi_type == BC_DIRICHLET ? n - 2 : n - 1;
    const int Nu = ge - gs + 1;  // unknowns of the folded system
    const T one = (T)1, two = (T)2, theta = P.theta, omt = one - theta, k = P.k, h2 = two * P.step;
    const bool has_src = P.src != nullptr;
    const T *in = uin[p];
    T *out = uout[p];
    T *sf = surf ? surf[p] : nullptr;
    with_chunk_len<M>(chunk_len(Nu), [&](auto cc) {
        constexpr int C = decltype(cc)::value;
        const int s0 = 1 + lane * C;  // first unknown (1-based) of the lane's chunk
        // grid index of the lane's t-th point; points past the line read its last point (discarded)
        auto gidx = [&](int t) { return min(gs + s0 + t - 1, N); };
        T u[C], cA[C], cB[C], cD[C];
#pragma unroll
        for (int t = 0; t < C; ++t)
            u[t] = in[gidx(t)];
        T ulo = in[0], uhi = in[N];  // the level's end values (used where the ends are Dirichlet)
        auto load_coeff = [&](int st) {
            const T *cs = P.coeff + (size_t)(P.coeff_sets > 1 ? st : 0) * 3 * (size_t)P.ld;
#pragma unroll
            for (int t = 0; t < C; ++t) {
                const int g = gidx(t);
                cA[t] = cs[g];
                cB[t] = cs[P.ld + g];
                cD[t] = cs[2 * P.ld + g];
            }
        };
        auto store_level = [&](T *row) {
#pragma unroll
            for (int t = 0; t < C; ++t)
                if (s0 + t <= Nu)
                    row[gs + s0 + t - 1] = u[t];
            if (lane == 0) {
                if (gs == 1)
                    row[0] = ulo;
                if (ge == n - 2)
                    row[N] = uhi;
            }
        };
        load_coeff(0);
        const bool fwd = P.direction == H1_FORWARD;
        if (sf)
            store_level(sf + (size_t)(fwd ? 0 : steps) * n);
        for (int st = 0; st < steps; ++st) {
            if (st > 0 && P.coeff_sets > 1)
                load_coeff(st);
            const T *bs = P.bnd + (P.bnd_sets > 1 ? st : 0) * 4;
            LineBC<T> bc;
            bc.lo = P.lo_type;
            bc.hi = P.hi_type;
            bc.lo_lin = bs[0];
            bc.lo_val = bs[1];
            bc.hi_lin = bs[2];
            bc.hi_val = bs[3];
            bc.h2 = h2;
            T sr[C], srn[C];
            if (has_src) {
                const T *q = P.src + (size_t)st * 2 * (size_t)n;
#pragma unroll
                for (int t = 0; t < C; ++t) {
                    sr[t] = q[gidx(t)];
                    srn[t] = q[n + gidx(t)];
                }
            }
            const T left0 = __shfl_up(u[C - 1], 1), rightC = __shfl_down(u[0], 1);
            auto eq = [&](int t, int kk) -> Eq<T> {
                const int g = gs + kk - 1;
                const T mid = u[t], A = cA[t], B = cB[t], D = cD[t];
                T left = t > 0 ? u[t - 1] : left0;
                T right = t < C - 1 ? u[t + 1] : rightC;
                if (kk == 1)
                    left = ulo;  // read only when the lower end is Dirichlet (g = 1)
                if (kk == Nu)
                    right = uhi;  // read only when the upper end is Dirichlet (g = N - 1)
                T r;
                if (g == 0) {  // Neumann / Robin lower row (lss_heat_implicit_solver_method.hpp:52-67)
                    const T beta = h2 * bc.lo_val;
                    if (P.lo_type == BC_NEUMANN)
                        r = omt * beta * A + (one - two * omt * B) * mid + omt * (A + D) * right;
                    else
                        r = omt * beta * A + (one - omt * (two * B - h2 * bc.lo_lin * A)) * mid + omt * (A + D) * right;
                    if (has_src)
                        r = r + theta * k * srn[t] + omt * k * sr[t];
                } else if (g == N) {  // Neumann / Robin upper row (:70-86)
                    const T delta = h2 * bc.hi_val;
                    if (P.hi_type == BC_NEUMANN)
                        r = omt * (A + D) * left + (one - two * omt * B) * mid - omt * delta * D;
                    else
                        r = omt * (A + D) * left + (one - omt * (two * B + h2 * bc.hi_lin * D)) * mid -
                            omt * delta * D;
                    if (has_src)
                        r = r + theta * k * srn[t] + omt * k * sr[t];
                } else {  // interior (:88-94)
                    r = (D * omt * right) + ((one - two * B * omt) * mid) + (A * omt * left);
                    if (has_src)
                        r = r + k * (theta * srn[t] + omt * sr[t]);
                }
                Eq<T> e;
                e.a = (-theta * A);
                e.b = (one + two * theta * B);
                e.c = (-theta * D);
                e.r = r;
                bc.fold(kk == 1, kk >= Nu, e.a, e.b, e.c, e.r);  // (c = 0 on the padding past the end too)
                return e;
            };
            T nu[C];
            // (the padding past the end restarts from zero every step, so that it stays finite)
            wave_solve_c<T, C, true>(Nu, lane, eq, [&](int t, int kk, T x) { nu[t] = kk <= Nu ? x : (T)0; });
#pragma unroll
            for (int t = 0; t < C; ++t)
                u[t] = nu[t];
            if (P.lo_type == BC_DIRICHLET)
                ulo = bc.lo_val;
            if (P.hi_type == BC_DIRICHLET)
                uhi = bc.hi_val;
            if (sf)
                store_level(sf + (size_t)(fwd ? st + 1 : steps - 1 - st) * n);
        }
        store_level(out);
    });
}

// -------------------------------------------------------------------------------------------------
// The same loop for problems whose matrix does not change in time (one coefficient set, and end conditions
// whose weights are fixed: no Robin end, or one boundary set).  The elimination of the chunks and of the
// interface system is then done once, before the loop: every step applies its multipliers to the right-hand
// side only.  A step of the general kernel is bound by the LDS pipe, which carries its shuffles (80 a step: three
// values, two words each, both ways in six reduction steps) beside 273 VALU instructions; this one shuffles one
// value, the neighbours at distance 1 by DPP.  fp64: 16384 problems x 256 points x 1000 steps 4.4 ms against 16.4;
// 4000 x 500 x 500 0.70 against 4.74; 4000 x 1026 x 240 0.93 against 3.63 (16 points a lane: part of the multipliers
// in accumulation registers).  fp32: 2.3 against 8.6 for the first.
// -------------------------------------------------------------------------------------------------
// lane i takes lane i - 1's (DOWN: i + 1's) value; the first (last) lane keeps its own
template <bool DOWN> __device__ __forceinline__ int wave_next(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, DOWN ? 0x130 : 0x138, 0xf, 0xf, false);
}
template <bool DOWN> __device__ __forceinline__ float wave_next(float v)
{
    return __int_as_float(wave_next<DOWN>(__float_as_int(v)));
}
template <bool DOWN> __device__ __forceinline__ double wave_next(double v)
{
    return __hiloint2double(wave_next<DOWN>(__double2hiint(v)), wave_next<DOWN>(__double2loint(v)));
}

template <typename T, int M>
__global__ void __launch_bounds__(64 * H1_WAVES) k_h1_wave_fixed(const H1Prob<T> *__restrict__ probs, int count,
                                                                 const T *const *__restrict__ uin,
                                                                 T *const *__restrict__ uout,
                                                                 T *const *__restrict__ surf)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int p = __builtin_amdgcn_readfirstlane(blockIdx.x * H1_WAVES + wave);
    if (p >= count)
        return;  // uniform over the wavefront
    const H1Prob<T> &P = probs[p];
    const int n = P.n, N = n - 1, steps = P.steps, ld = P.ld;
    const bool dlo = P.lo_type == BC_DIRICHLET, dhi = P.hi_type == BC_DIRICHLET;
    const int gs = dlo ? 1 : 0, Nu = (dhi ? n - 2 : n - 1) - gs + 1;  // unknowns of the folded system
    const T one = (T)1, two = (T)2, theta = P.theta, omt = one - theta, k = P.k, h2 = two * P.step;
    const bool has_src = P.src != nullptr, fwd = P.direction == H1_FORWARD;
    const gptr<const T> in = G(uin[p]), src = G(P.src), bnd = G(P.bnd), cs = G(P.coeff);
    const gptr<T> out = G(uout[p]);
    T *const sf0 = surf ? surf[p] : nullptr;
    const gptr<T> sf = G(sf0);
    with_chunk_len<M>(chunk_len(Nu), [&](auto cc) {
        constexpr int C = decltype(cc)::value, I = C > 1 ? C - 1 : 1;
        const int s0 = 1 + lane * C;  // first unknown (1-based) of the lane's chunk
        auto gidx = [&](int t) { return min(gs + s0 + t - 1, N); };
        // Right-hand side of unknown kk: am left + bm mid + dm right (+ source) + kl lo_val (kk = 1) + ke hi_val
        // (kk = Nu).  Row Nu + 1 of a Dirichlet end is the end value itself (ke = 1), so that row Nu finds it as its
        // right neighbour; the other rows past the line are zero.
        T am[C], bm[C], dm[C], ke[C], kl = (T)0, u[C];
        // multipliers of the chunk: p_u = r_u rb_u - e_u p_{u-1}; p_u -= g_u p_{u+1}; x_u = p_u + q_u xl + w_u xr
        T rb[I], e[I], g[I], q[I], w[I], ae, be, ce;
#pragma unroll
        for (int t = 0; t < C; ++t) {
            const int kk = s0 + t, gc = gidx(t);
            const T A = cs[gc], B = cs[ld + gc], D = cs[2 * ld + gc];
            T a = -theta * A, b = one + two * theta * B, c = -theta * D;
            am[t] = A * omt;
            bm[t] = one - two * B * omt;
            dm[t] = D * omt;
            ke[t] = (T)0;
            u[t] = in[gc];
            if (kk <= Nu) {  // end rows: lss_heat_implicit_solver_method.hpp:52-86, lss_thomas_lu_boundary.hpp:114-205
                if (kk == 1) {
                    if (dlo) {
                        kl = -a;
                    } else {
                        const T lin = P.lo_type == BC_ROBIN ? h2 * bnd[0] : (T)0;
                        kl = h2 * (omt * A - a);
                        bm[t] = one - omt * (two * B - lin * A);
                        dm[t] = omt * (A + D);
                        am[t] = (T)0;
                        b = b + a * lin;
                        c = a + c;
                    }
                    a = (T)0;
                }
                if (kk == Nu) {
                    if (dhi) {
                        ke[t] = -c;
                    } else {
                        const T lin = P.hi_type == BC_ROBIN ? h2 * bnd[2] : (T)0;
                        ke[t] = h2 * (c - omt * D);
                        bm[t] = one - omt * (two * B + lin * D);
                        am[t] = omt * (A + D);
                        dm[t] = (T)0;
                        b = b - c * lin;
                        a = a + c;
                    }
                    c = (T)0;
                }
            } else {
                a = c = am[t] = bm[t] = dm[t] = (T)0;
                b = one;
                if (dhi && kk == Nu + 1) {
                    ke[t] = one;
                    u[t] = in[N];
                } else {
                    u[t] = (T)0;
                }
            }
            if (t == C - 1) {
                ae = a, be = b, ce = c;
            } else {
                rb[t] = fast_rcp(t == 0 ? b : b - a * g[t > 0 ? t - 1 : 0]);
                g[t] = c * rb[t];
                e[t] = a * rb[t];
                q[t] = t == 0 ? -e[t] : -e[t] * q[t > 0 ? t - 1 : 0];
            }
        }
        T ql = one, wl = (T)0, QF = (T)0, WF = one;  // relations of the last and first interior points
        if constexpr (C >= 2) {
            w[C - 2] = -g[C - 2];
#pragma unroll
            for (int t = C - 3; t >= 0; --t) {
                w[t] = -g[t] * w[t + 1];
                q[t] = q[t] - g[t] * q[t + 1];
            }
            ql = q[C - 2], wl = w[C - 2], QF = q[0], WF = w[0];
        }
        // the interface system's reduction, multipliers only (ka: of the row at distance d below, kc: above)
        T ka[6], kc[6], inv;
        {
            const T nQF = __shfl_down(QF, 1), nWF = __shfl_down(WF, 1);
            T a = ae * ql, b = ae * wl + be + ce * nQF, c = ce * nWF;
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                const int d = 1 << s;
                const T r = fast_rcp(b);
                ka[s] = a * __shfl_up(r, d);
                kc[s] = c * __shfl_down(r, d);
                const T la = __shfl_up(a, d), lc = __shfl_up(c, d), ha = __shfl_down(a, d), hc = __shfl_down(c, d);
                b = b - ka[s] * lc - kc[s] * ha;
                a = -ka[s] * la;
                c = -kc[s] * hc;
            }
            inv = fast_rcp(b);
        }
        T ulo = in[0], uhi = in[N];
        auto store_level = [&](gptr<T> row) {
#pragma unroll
            for (int t = 0; t < C; ++t)
                if (s0 + t <= Nu)
                    row[gs + s0 + t - 1] = u[t];
            if (lane == 0) {
                if (dlo)
                    row[0] = ulo;
                if (dhi)
                    row[N] = uhi;
            }
        };
        if (sf0)
            store_level(sf + (size_t)(fwd ? 0 : steps) * n);
        for (int st = 0; st < steps; ++st) {
            const gptr<const T> bs = bnd + (P.bnd_sets > 1 ? st : 0) * 4;
            const T lo_val = bs[1], hi_val = bs[3];
            T left = wave_next<false>(u[C - 1]), right = wave_next<true>(u[0]);
            left = lane == 0 ? ulo : left;
            right = lane == 63 ? uhi : right;
            T r[C], z[I];
#pragma unroll
            for (int t = 0; t < C; ++t)
                r[t] = am[t] * (t > 0 ? u[t > 0 ? t - 1 : 0] : left) + bm[t] * u[t] +
                       dm[t] * (t < C - 1 ? u[t < C - 1 ? t + 1 : 0] : right) + ke[t] * hi_val;
            r[0] = r[0] + (lane == 0 ? kl : (T)0) * lo_val;
            if (has_src) {
                const gptr<const T> f = src + (size_t)st * 2 * (size_t)n;
#pragma unroll
                for (int t = 0; t < C; ++t)
                    if (s0 + t <= Nu)
                        r[t] = r[t] + k * (theta * f[n + gidx(t)] + omt * f[gidx(t)]);
            }
            T R = r[C - 1];
            if constexpr (C >= 2) {
                z[0] = r[0] * rb[0];
#pragma unroll
                for (int t = 1; t < C - 1; ++t)
                    z[t] = r[t] * rb[t] - e[t] * z[t - 1];
#pragma unroll
                for (int t = C - 3; t >= 0; --t)
                    z[t] = z[t] - g[t] * z[t + 1];
                R = R - ae * z[C - 2] - ce * wave_next<true>(z[0]);
            }
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                const int d = 1 << s;
                const T lo = d == 1 ? wave_next<false>(R) : __shfl_up(R, d), hi = d == 1 ? wave_next<true>(R) : __shfl_down(R, d);
                R = R - ka[s] * lo - kc[s] * hi;
            }
            const T xi = R * inv, xl = wave_next<false>(xi);
            if constexpr (C >= 2) {
#pragma unroll
                for (int t = 0; t < C - 1; ++t)
                    u[t] = z[t] + q[t] * xl + w[t] * xi;
            }
            u[C - 1] = xi;
            if (dlo)
                ulo = lo_val;
            if (dhi)
                uhi = hi_val;
            if (sf0)
                store_level(sf + (size_t)(fwd ? st + 1 : steps - 1 - st) * n);
        }
        store_level(out);
    });
}

#define LSS_INST_H1W(T, M)                                                                                    \
    template __global__ void k_h1_wave<T, M>(const H1Prob<T> *, int, const T *const *, T *const *, T *const *);
LSS_INST_H1W(double, 1)
LSS_INST_H1W(double, 2)
LSS_INST_H1W(double, 4)
LSS_INST_H1W(double, 8)
LSS_INST_H1W(double, 16)
LSS_INST_H1W(float, 1)
LSS_INST_H1W(float, 2)
LSS_INST_H1W(float, 4)
LSS_INST_H1W(float, 8)
LSS_INST_H1W(float, 16)
#undef LSS_INST_H1W
#define LSS_INST_H1F(T, M)                                                                                         \
    template __global__ void k_h1_wave_fixed<T, M>(const H1Prob<T> *, int, const T *const *, T *const *, T *const *);
LSS_INST_H1F(double, 1)
LSS_INST_H1F(double, 2)
LSS_INST_H1F(double, 4)
LSS_INST_H1F(double, 8)
LSS_INST_H1F(double, 16)
LSS_INST_H1F(float, 1)
LSS_INST_H1F(float, 2)
LSS_INST_H1F(float, 4)
LSS_INST_H1F(float, 8)
LSS_INST_H1F(float, 16)
#undef LSS_INST_H1F

}  // namespace lssamd
