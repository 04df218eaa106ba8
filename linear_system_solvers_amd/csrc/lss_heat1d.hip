// lss_heat1d.hip -- the 1-D implicit heat / Black-Scholes solver: the exact kernel (four lanes per problem,
// the reference's sequential Thomas LU / double-sweep order), the host plan and the C-ABI of
// include/lss_heat1d.h.
//
// The exact kernel runs a problem's whole time loop in four lanes: per step it forms each row of the
// theta scheme (implicit_heat_scheme::rhs / rhs_source and heat_implicit_solver_method::split,
// pde_solvers/one_dimensional/heat_type/solver_method/lss_heat_implicit_solver_method.hpp:36-210) and
// sweeps it as thomas_lu_solver (lss_thomas_lu_solver.hpp:125-191 with lss_thomas_lu_boundary.hpp:
// 114-205) or double_sweep_solver (lss_double_sweep_solver.hpp:112-155 with
// lss_double_sweep_boundary.hpp:88-190) does, every operation in the reference's order (this
// translation unit is compiled without contraction), so the result equals the reference's host
// result bit for bit.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "lss/lss_heat1d_sampler.hpp"
#include "lss_capi_common.hpp"
#include "lss_heat1d.h"
#include "lss_heat1d_device.hpp"
#include "lss_quad.hpp"

namespace lssamd {

template <typename T, int M>
__global__ void k_h1_wave(const H1Prob<T> *, int, const T *const *, T *const *, T *const *);
template <typename T, int M>
__global__ void k_h1_wave_fixed(const H1Prob<T> *, int, const T *const *, T *const *, T *const *);

template <typename T> struct H1Vec {
    typedef T v2 __attribute__((ext_vector_type(2)));
};

// Row N after the chain, among the lane's points t0 .. t0 + 3 (x the intermediate solution, gm gamma, gp
// gamma of the point before, sp the intermediate solution before x[0]): a Dirichlet end is the end value;
// the double sweep's Neumann / Robin end is lss_double_sweep_boundary.hpp:140-190 (L = -gamma).
template <typename T>
__device__ __forceinline__ void finish_end(T (&x)[4], const T (&gm)[4], const T (&gp)[4], T sp, int t0, int N, bool dhi,
                                           bool dsweep, int hi_type, T h, T hi_lin, T hi_val)
{
    const T one = (T)1.0, two = (T)2.0;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
        if (t0 + j != N)
            continue;
        if (dhi) {
            x[j] = hi_val;
        } else if (dsweep) {
            const T LN = -gm[j], L1 = -gp[j], K1 = j > 0 ? x[j > 0 ? j - 1 : 0] : sp;
            const T cst = two * h * hi_val;
            if (hi_type == BC_NEUMANN) {
                x[j] = (LN * (K1 - cst) + x[j]) / (one - LN * L1);
            } else {
                const T lin = two * h * hi_lin;
                x[j] = (LN * (K1 - cst) + x[j]) / (one - LN * (L1 - lin));
            }
        }
    }
}

// -------------------------------------------------------------------------------------------------
// The exact kernel: four lanes (a quad) per problem, 16 problems per wavefront, the whole time loop in one
// launch.  A line goes through the quad in groups of 16 points; lane q holds points 4q .. 4q + 3 of the
// group.  Everything that does not depend on the previous point -- the loads, the rows of the theta scheme
// and, once gamma is known, the divisors -- is formed by the four lanes at once; the recurrence of the
// sweep then passes from lane to lane by DPP, each lane running its four points in the reference's order.
// What bounds a wavefront is the number of instructions of that chain and of the rows (it issues one every four to
// five cycles), and a large book also the 40 bytes of A, B, D and gamma (twice) that each point of each step reads
// from the last-level cache: 16384 problems x 256 points x 1000 steps in fp64 take 26.4 ms (29.4 with an IEEE
// division per point), 6.4 TB/s.  With one lane per problem, each access in a cache line of its own, they took 304 ms.
// Four lanes make 1024 wavefronts of that book, one per SIMD.
//
// Layouts: a problem's A, B and D are padded to whole groups (16-byte aligned), so a quad reads whole
// 128-byte lines; the level u (LDS when it fits, else the workspace) and gamma (workspace) are kept by lane,
// so no lane ever reads another's memory.  The coefficients and gamma of the group after next are loaded
// while a group's chain runs.
//
// Coefficients and boundary weights that do not change in time give the same gamma every step: it is
// computed in the first step of a solve and read afterwards, which takes one of the two divisions out of
// the chain.  The double sweep is the Thomas sweep with L = -gamma (b + a L = b - a gamma,
// -c / beta = -(c / beta), L x + K = K - gamma x: negation is exact), so both run the same recurrence and
// differ in the end rows only.
// -------------------------------------------------------------------------------------------------
template <typename T, bool LDSU>
__global__ void __launch_bounds__(64) k_h1_exact(const H1Prob<T> *__restrict__ probs, int count,
                                                 const T *const *__restrict__ uin, T *const *__restrict__ uout,
                                                 T *const *__restrict__ surf)
{
    typedef typename H1Vec<T>::v2 v2;
    extern __shared__ unsigned char h1_lds[];
    const int lane = (int)threadIdx.x, ql = lane & 3;
    const int p = (int)blockIdx.x * H1_EXACT_PROBS + (lane >> 2);
    if (p >= count)
        return;  // whole quads; there is no barrier
    const H1Prob<T> &P = probs[p];
    const int n = P.n, N = n - 1, steps = P.steps, ng = (n + 15) / 16, ld = P.ld;
    const T one = (T)1.0, two = (T)2.0, theta = P.theta, k = P.k, h = P.step, omt = one - theta;
    const bool dlo = P.lo_type == BC_DIRICHLET, dhi = P.hi_type == BC_DIRICHLET, dsweep = P.tri == TRI_DSWEEP;
    const bool fwd = P.direction == H1_FORWARD, has_src = P.src != nullptr;
    const bool const_gamma =
        P.coeff_sets == 1 && (P.bnd_sets == 1 || (P.lo_type != BC_ROBIN && P.hi_type != BC_ROBIN));
    const gptr<T> gbase = G(P.gamma), ubase = G(P.level);
    lptr<v2> ush = (lptr<v2>)h1_lds;
    // four own values of group g in the lane-ordered workspace / the level
    auto ld4 = [&](gptr<T> b, int g, T(&v)[4]) {
        const v2 x = *(gptr<const v2>)(b + ((size_t)(2 * g) * 64 + lane) * 2),
                 y = *(gptr<const v2>)(b + ((size_t)(2 * g + 1) * 64 + lane) * 2);
        v[0] = x.x, v[1] = x.y, v[2] = y.x, v[3] = y.y;
    };
    auto st4 = [&](gptr<T> b, int g, const T(&v)[4]) {
        *(gptr<v2>)(b + ((size_t)(2 * g) * 64 + lane) * 2) = v2{v[0], v[1]};
        *(gptr<v2>)(b + ((size_t)(2 * g + 1) * 64 + lane) * 2) = v2{v[2], v[3]};
    };
    auto uget = [&](int g, T(&v)[4]) {
        if constexpr (LDSU) {
            const v2 p0 = ush[(2 * g) * 64 + lane], p1 = ush[(2 * g + 1) * 64 + lane];
            v[0] = p0.x, v[1] = p0.y, v[2] = p1.x, v[3] = p1.y;
        } else {
            ld4(ubase, g, v);
        }
    };
    auto uput = [&](int g, const T(&v)[4]) {
        if constexpr (LDSU) {
            ush[(2 * g) * 64 + lane] = v2{v[0], v[1]};
            ush[(2 * g + 1) * 64 + lane] = v2{v[2], v[3]};
        } else {
            st4(ubase, g, v);
        }
    };
    auto store_level = [&](gptr<T> row, int g, const T(&v)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (16 * g + 4 * ql + j < n)
                row[16 * g + 4 * ql + j] = v[j];
    };
    T *const sf0 = surf ? surf[p] : nullptr;
    const gptr<T> sf = G(sf0), out = G(uout[p]);
    {
        const gptr<const T> in = G(uin[p]);
        for (int g = 0; g < ng; ++g) {
            T v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = in[min(16 * g + 4 * ql + j, N)];
            uput(g, v);
            if (sf0)
                store_level(sf + (size_t)(fwd ? 0 : steps) * n, g, v);
        }
    }
    struct Stage {
        T A[4], B[4], D[4], G[4], u[4];
    };
    struct Back {
        T G[4], s[4];
    };
    for (int st = 0; st < steps; ++st) {
        const gptr<const T> cs = G(P.coeff) + (size_t)(P.coeff_sets > 1 ? st : 0) * 3 * (size_t)ld;
        const gptr<const T> bs = G(P.bnd) + (P.bnd_sets > 1 ? st : 0) * 4;
        const T lo_lin = bs[0], lo_val = bs[1], hi_lin = bs[2], hi_val = bs[3];
        const gptr<const T> src = G(P.src) + (size_t)st * 2 * (size_t)n;
        const bool reuse = const_gamma && st > 0;  // gamma of this problem is in the workspace
        auto load = [&](int g, Stage &s) {
            const int o = 16 * g + 4 * ql;
            auto two_of = [&](gptr<const T> b, T(&v)[4]) {
                const v2 x = *(gptr<const v2>)(b + o), y = *(gptr<const v2>)(b + o + 2);
                v[0] = x.x, v[1] = x.y, v[2] = y.x, v[3] = y.y;
            };
            two_of(cs, s.A);
            two_of(cs + ld, s.B);
            two_of(cs + 2 * ld, s.D);
            if (reuse)
                ld4(gbase, g, s.G);
            uget(g, s.u);
        };
        // ---- forward sweep: rows (a, b, c, f), gamma and the intermediate solution, which replaces the level
        T ulast = (T)0, glast = (T)0, scar = (T)0;
        auto forward = [&](int g, Stage &s0) {
            T un[4];
            uget(min(g + 1, ng - 1), un);
            T left = quad_perm<QUAD_UP>(s0.u[3]), right = quad_perm<QUAD_DOWN>(s0.u[0]);
            const T nfirst = quad_perm<QUAD_BCAST<0>>(un[0]);
            left = ql == 0 ? ulast : left;
            right = ql == 3 ? nfirst : right;
            T a[4], b[4], c[4], f[4], gp[4], x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const T A = s0.A[j], B = s0.B[j], D = s0.D[j];
                const T um = j > 0 ? s0.u[j - 1] : left, up = j < 3 ? s0.u[j + 1] : right;
                // rows of split (:200-210): low = -theta A, diag = 1 + 2 theta B, high = -theta D; interior
                // right-hand side (:88-94)
                a[j] = (-theta * A);
                b[j] = (one + two * theta * B);
                c[j] = (-theta * D);
                f[j] = (D * omt * up) + ((one - two * B * omt) * s0.u[j]) + (A * omt * um);
            }
            const bool edge = g == 0 || 16 * g + 16 >= N;  // holds row 0, N - 1, N or points past the line
            if (edge || has_src) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int t = 16 * g + 4 * ql + j;
                    const T A = s0.A[j], B = s0.B[j], D = s0.D[j];
                    const T um = j > 0 ? s0.u[j - 1] : left, up = j < 3 ? s0.u[j + 1] : right;
                    const T sr = has_src ? src[min(t, N)] : (T)0, srn = has_src ? src[n + min(t, N)] : (T)0;
                    if (t == 0) {
                        if (dlo) {  // the end value; row 1 then folds it as f - a lo
                            a[j] = c[j] = (T)0;
                            b[j] = one;
                            f[j] = lo_val;
                        } else {  // Neumann / Robin lower row (:52-67) and its folding
                            const T beta = two * h * lo_val;
                            T r;
                            if (P.lo_type == BC_NEUMANN) {
                                r = omt * beta * A + (one - two * omt * B) * s0.u[j] + omt * (A + D) * up;
                            } else {
                                const T alpha = two * h * lo_lin;
                                r = omt * beta * A + (one - omt * (two * B - alpha * A)) * s0.u[j] + omt * (A + D) * up;
                            }
                            if (has_src)
                                r = r + theta * k * srn + omt * k * sr;
                            const T ra = a[j];
                            if (dsweep) {  // lss_double_sweep_boundary.hpp:88-190
                                if (P.lo_type == BC_ROBIN)
                                    b[j] = b[j] + ra * h * two * lo_lin;
                                f[j] = r - ra * h * two * lo_val;
                            } else {  // lss_thomas_lu_boundary.hpp:114-205
                                if (P.lo_type == BC_ROBIN)
                                    b[j] = b[j] + ra * (two * h * lo_lin);
                                f[j] = r - ra * (two * h * lo_val);
                            }
                            c[j] = ra + c[j];
                            a[j] = (T)0;
                        }
                    } else if (t == N) {
                        if (dhi) {
                            a[j] = c[j] = f[j] = (T)0;
                            b[j] = one;
                        } else {  // Neumann / Robin upper row (:70-86)
                            const T delta = two * h * hi_val;
                            T r;
                            if (P.hi_type == BC_NEUMANN) {
                                r = omt * (A + D) * um + (one - two * omt * B) * s0.u[j] - omt * delta * D;
                            } else {
                                const T gamma = two * h * hi_lin;
                                r = omt * (A + D) * um + (one - omt * (two * B + gamma * D)) * s0.u[j] -
                                    omt * delta * D;
                            }
                            if (has_src)
                                r = r + theta * k * srn + omt * k * sr;
                            f[j] = r;
                            if (!dsweep) {
                                const T ra = a[j], rc = c[j];
                                a[j] = ra + rc;
                                if (P.hi_type == BC_ROBIN)
                                    b[j] = b[j] - rc * (two * h * hi_lin);
                                f[j] = r + rc * (two * h * hi_val);
                            }
                        }
                    } else if (t > N) {
                        a[j] = c[j] = f[j] = (T)0;
                        b[j] = one;
                    } else {
                        if (has_src)
                            f[j] = f[j] + k * (theta * srn + omt * sr);
                        if (t == N - 1 && dhi && !dsweep)
                            f[j] = f[j] - c[j] * hi_val;
                    }
                }
            }
            // gamma = c / beta and beta = b - a gamma, then the chain s = (f - a s) / beta
            T beta[4], gm[4], y[4];
            if (reuse) {
                const T gup = quad_perm<QUAD_UP>(s0.G[3]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    gm[j] = s0.G[j];
                    gp[j] = j > 0 ? s0.G[j > 0 ? j - 1 : 0] : (ql == 0 ? glast : gup);
                    beta[j] = b[j] - (a[j] * gp[j]);
                }
                glast = quad_perm<QUAD_BCAST<3>>(s0.G[3]);
            } else {
                const T gnext = quad_gamma(a, b, c, glast, beta, gm);
                const T gup = quad_perm<QUAD_UP>(gm[3]);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    gp[j] = j > 0 ? gm[j > 0 ? j - 1 : 0] : (ql == 0 ? glast : gup);
                glast = gnext;
                st4(gbase, g, gm);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                y[j] = quick_rcp(beta[j]);
            const T sprev = scar;
            SeenNum seen;
            scar = quad_forward<true>(a, f, beta, y, sprev, x, seen);
            if (__builtin_amdgcn_ballot_w64(!seen_ok(seen, sprev)))
                scar = quad_forward<false>(a, f, beta, y, sprev, x, seen);
            if (edge) {
                const T xup = quad_perm<QUAD_UP>(x[3]);
                finish_end(x, gm, gp, ql == 0 ? sprev : xup, 16 * g + 4 * ql, N, dhi, dsweep, P.hi_type, h, hi_lin, hi_val);
            }
            uput(g, x);
            ulast = quad_perm<QUAD_BCAST<3>>(s0.u[3]);
        };
        quad_stages<Stage>(0, ng, 1, load, forward);
        // ---- back substitution x = s - gamma x, from the last group down
        const gptr<T> lv = sf + (size_t)(fwd ? st + 1 : steps - 1 - st) * n;
        T xcar = (T)0;
        auto loadb = [&](int g, Back &b) {
            ld4(gbase, g, b.G);
            uget(g, b.s);
        };
        auto backward = [&](int g, Back &b) {
            T x[4];
            if (g == 0 || 16 * g + 16 >= N)
                // the forward sweep left the value itself at row N, at a Dirichlet row 0 and at the Thomas sweep's
                // last row before a Dirichlet end
                xcar = quad_backward_ends(
                    b.G, b.s, xcar, x,
                    [&](int j) {
                        const int t = 16 * g + 4 * ql + j;
                        return t >= N || (t == 0 && dlo) || (t == N - 1 && dhi && !dsweep);
                    },
                    [](int) { return false; });
            else
                xcar = quad_backward(b.G, b.s, xcar, x);
            uput(g, x);
            if (sf0)
                store_level(lv, g, x);
            if (st == steps - 1)
                store_level(out, g, x);
        };
        quad_stages<Back>(ng - 1, ng, -1, loadb, backward);
    }
}

#define LSS_INST_H1E(T)                                                                                             \
    template __global__ void k_h1_exact<T, true>(const H1Prob<T> *, int, const T *const *, T *const *, T *const *); \
    template __global__ void k_h1_exact<T, false>(const H1Prob<T> *, int, const T *const *, T *const *, T *const *);
LSS_INST_H1E(double)
LSS_INST_H1E(float)
#undef LSS_INST_H1E

}  // namespace lssamd

using namespace lssamd;
using namespace lssamd_host;

struct lss_heat1d_plan {
    virtual ~lss_heat1d_plan() = default;
    int fp = LSS_FP64;
    int64_t count = 0;
    std::vector<int64_t> n, steps;
    std::vector<std::vector<char>> init_host, grid_host;  // model plans only
    virtual void run(const void *const *u_in, void *const *u_out, void *const *surf, hipStream_t st, bool host) = 0;
};

namespace {

template <typename T> struct H1Plan final : lss_heat1d_plan {
    std::vector<H1Prob<T>> probs;
    dev_buffer mem, probs_dev, table_dev;
    dev_buffer ws_dev;  // exact plans: gamma (and levels that do not fit LDS) of each wavefront, by lane
    int line_solver = LSS_LINE_EXACT;
    int ngmax = 0;           // groups of 16 points of the longest line
    bool lds_level = false;  // the level of every problem stays in LDS
    int pm = 1;  // chunk bound of the partitioned kernel
    bool fixed = true;  // no problem's matrix changes in time
    std::vector<const void *> table;  // u_in, u_out, surfaces pointers of the last device run
    bool table_valid = false;

    static void validate(const lss_heat1d_desc &d)
    {
        require(d.fp == (sizeof(T) == 8 ? LSS_FP64 : LSS_FP32), "all problems of a plan share fp");
        require(d.n >= 4 && d.n <= (1 << 24), "n must be in [4, 2^24]");
        require(d.steps >= 1 && d.steps < (1 << 30), "steps must be >= 1");
        require(d.coeff_sets == 1 || d.coeff_sets == d.steps, "coeff_sets must be 1 or steps");
        require(d.bnd_sets == 1 || d.bnd_sets == d.steps, "bnd_sets must be 1 or steps");
        require(d.coeff && d.bnd, "null coefficient or boundary array");
        for (int t : {d.lo_type, d.hi_type})
            require(t == LSS_BC_DIRICHLET || t == LSS_BC_NEUMANN || t == LSS_BC_ROBIN,
                    "boundary type must be LSS_BC_DIRICHLET, LSS_BC_NEUMANN or LSS_BC_ROBIN");
        require(d.direction == LSS_FORWARD || d.direction == LSS_BACKWARD, "direction must be Forward or Backward");
        require(d.line_solver == LSS_LINE_EXACT || d.line_solver == LSS_LINE_PARTITIONED, "unknown line_solver");
        if (d.line_solver == LSS_LINE_PARTITIONED) {
            const int64_t nu = d.n - (d.lo_type == LSS_BC_DIRICHLET) - (d.hi_type == LSS_BC_DIRICHLET);
            require(nu <= 64 * 16, "the partitioned 1-D solver takes at most 1024 unknowns per line");
        }
    }

    void build(const lss_heat1d_desc *d, int64_t cnt)
    {
        require(cnt >= 1 && cnt < (1 << 30), "count must be in [1, 2^30)");
        count = cnt;
        line_solver = d[0].line_solver;
        size_t total = 0;
        std::vector<size_t> off(cnt);
        auto round = [](size_t x) { return (x + 63) / 64 * 64; };
        for (int64_t q = 0; q < cnt; ++q) {
            validate(d[q]);
            require(d[q].line_solver == line_solver, "all problems of a plan share line_solver");
            const size_t nq = (size_t)d[q].n;
            const size_t ldq = (nq + 15) / 16 * 16;
            off[q] = total;
            total += round(3 * ldq * (size_t)d[q].coeff_sets) + round(4 * (size_t)d[q].bnd_sets) +
                     (d[q].source ? round(2 * nq * (size_t)d[q].steps) : 0);
            ngmax = std::max(ngmax, (int)(ldq / 16));
            const int64_t nu = d[q].n - (d[q].lo_type == LSS_BC_DIRICHLET) - (d[q].hi_type == LSS_BC_DIRICHLET);
            while (pm * 64 < nu && pm < 16)
                pm *= 2;
            const bool robin = d[q].lo_type == LSS_BC_ROBIN || d[q].hi_type == LSS_BC_ROBIN;
            fixed = fixed && d[q].coeff_sets == 1 && (d[q].bnd_sets == 1 || !robin);
        }
        mem.alloc(total * sizeof(T));
        probs.resize(cnt);
        n.resize(cnt);
        steps.resize(cnt);
        T *base = (T *)mem.p;
        std::vector<T> padded;
        for (int64_t q = 0; q < cnt; ++q) {
            const lss_heat1d_desc &e = d[q];
            const size_t nq = (size_t)e.n;
            H1Prob<T> &P = probs[q];
            std::memset(&P, 0, sizeof(P));
            P.n = (int32_t)e.n;
            P.steps = (int32_t)e.steps;
            P.tri = e.tridiagonal == LSS_DOUBLE_SWEEP ? TRI_DSWEEP : TRI_THOMAS;
            P.lo_type = e.lo_type;
            P.hi_type = e.hi_type;
            P.direction = e.direction == LSS_FORWARD ? H1_FORWARD : H1_BACKWARD;
            P.coeff_sets = (int32_t)e.coeff_sets;
            P.bnd_sets = (int32_t)e.bnd_sets;
            P.theta = (T)e.theta;
            P.k = (T)e.k;
            P.step = (T)1 / (T)(e.n - 1);  // grid_config<One>: one / (n - 1)
            T *o = base + off[q];
            T *c = o;
            const size_t ldq = (nq + 15) / 16 * 16, rows = 3 * (size_t)e.coeff_sets;
            P.ld = (int32_t)ldq;
            o += round(ldq * rows);
            T *b = o;
            o += round(4 * (size_t)e.bnd_sets);
            padded.assign(ldq * rows, (T)0);
            for (size_t r = 0; r < rows; ++r)
                std::memcpy(padded.data() + r * ldq, (const T *)e.coeff + r * nq, nq * sizeof(T));
            LSS_HIPCHK(hipMemcpy(c, padded.data(), padded.size() * sizeof(T), hipMemcpyHostToDevice));
            LSS_HIPCHK(hipMemcpy(b, e.bnd, 4 * (size_t)e.bnd_sets * sizeof(T), hipMemcpyHostToDevice));
            P.coeff = c;
            P.bnd = b;
            if (e.source) {
                LSS_HIPCHK(hipMemcpy(o, e.source, 2 * nq * (size_t)e.steps * sizeof(T), hipMemcpyHostToDevice));
                P.src = o;
                o += round(2 * nq * (size_t)e.steps);
            }
            n[q] = e.n;
            steps[q] = e.steps;
        }
        if (line_solver == LSS_LINE_EXACT) {  // each wavefront's workspace follows its longest line
            lds_level = level_bytes() <= 65536;
            std::vector<size_t> first(1, 0);
            for (int64_t q = 0; q < cnt; q += H1_EXACT_PROBS) {
                size_t ngw = 0;
                for (int64_t z = q; z < std::min(cnt, q + H1_EXACT_PROBS); ++z)
                    ngw = std::max(ngw, (size_t)probs[z].ld / 16);
                first.push_back(first.back() + ngw * 256);
            }
            ws_dev.alloc(first.back() * (lds_level ? 1 : 2) * sizeof(T));
            for (int64_t q = 0; q < cnt; ++q) {
                probs[q].gamma = (T *)ws_dev.p + first[q / H1_EXACT_PROBS];
                probs[q].level = lds_level ? nullptr : probs[q].gamma + first.back();
            }
        }
        probs_dev.alloc(cnt * sizeof(H1Prob<T>));
        LSS_HIPCHK(hipMemcpy(probs_dev.p, probs.data(), cnt * sizeof(H1Prob<T>), hipMemcpyHostToDevice));
        table_dev.alloc(3 * cnt * sizeof(void *));
    }

    size_t level_bytes() const { return (size_t)ngmax * 256 * sizeof(T); }  // levels of a wavefront's problems

    template <int M> void launch_wave(hipStream_t st, const T *const *ui, T *const *uo, T *const *sf)
    {
        const unsigned blocks = (unsigned)((count + H1_WAVES - 1) / H1_WAVES);
        if (fixed) {
            hipLaunchKernelGGL((k_h1_wave_fixed<T, M>), dim3(blocks), dim3(64 * H1_WAVES), 0, st,
                               (const H1Prob<T> *)probs_dev.p, (int)count, ui, uo, sf);
            return;
        }
        hipLaunchKernelGGL((k_h1_wave<T, M>), dim3(blocks), dim3(64 * H1_WAVES), 0, st,
                           (const H1Prob<T> *)probs_dev.p, (int)count, ui, uo, sf);
    }

    void launch(hipStream_t st, bool with_surf)
    {
        void **tb = (void **)table_dev.p;
        const T *const *ui = (const T *const *)tb;
        T *const *uo = (T *const *)(tb + count);
        T *const *sf = with_surf ? (T *const *)(tb + 2 * count) : nullptr;
        if (line_solver == LSS_LINE_EXACT) {
            const unsigned blocks = (unsigned)((count + H1_EXACT_PROBS - 1) / H1_EXACT_PROBS);
            if (lds_level)
                hipLaunchKernelGGL((k_h1_exact<T, true>), dim3(blocks), dim3(64), (unsigned)level_bytes(), st,
                                   (const H1Prob<T> *)probs_dev.p, (int)count, ui, uo, sf);
            else
                hipLaunchKernelGGL((k_h1_exact<T, false>), dim3(blocks), dim3(64), 0, st,
                                   (const H1Prob<T> *)probs_dev.p, (int)count, ui, uo, sf);
        } else {
            switch (pm) {
            case 1: launch_wave<1>(st, ui, uo, sf); break;
            case 2: launch_wave<2>(st, ui, uo, sf); break;
            case 4: launch_wave<4>(st, ui, uo, sf); break;
            case 8: launch_wave<8>(st, ui, uo, sf); break;
            default: launch_wave<16>(st, ui, uo, sf); break;
            }
        }
        LSS_HIPCHK(hipGetLastError());
    }

    // the pointer table (u_in, u_out, surfaces) on the device; rewritten only when it changes
    void set_table(const void *const *u_in, void *const *u_out, void *const *surf, hipStream_t st)
    {
        std::vector<const void *> t(3 * count, nullptr);
        for (int64_t q = 0; q < count; ++q) {
            t[q] = u_in[q];
            t[count + q] = u_out[q];
            t[2 * count + q] = surf ? surf[q] : nullptr;
        }
        if (table_valid && t == table)
            return;
        LSS_HIPCHK(hipStreamSynchronize(st));  // an earlier launch may still read the old table
        LSS_HIPCHK(hipMemcpy(table_dev.p, t.data(), t.size() * sizeof(void *), hipMemcpyHostToDevice));
        table = std::move(t);
        table_valid = true;
    }

    void run(const void *const *u_in, void *const *u_out, void *const *surf, hipStream_t st, bool host) override
    {
        require(u_in && u_out, "null u_in / u_out array");
        for (int64_t q = 0; q < count; ++q)
            require(u_in[q] && u_out[q], "null surface pointer");
        bool with_surf = false;
        if (surf)
            for (int64_t q = 0; q < count; ++q)
                with_surf = with_surf || surf[q] != nullptr;
        if (!host) {
            set_table(u_in, u_out, with_surf ? surf : nullptr, st);
            launch(st, with_surf);
            return;
        }
        // host pointers: stage everything through one device allocation
        size_t tot = 0;
        std::vector<size_t> oi(count), oo(count), os(count, 0);
        for (int64_t q = 0; q < count; ++q) {
            oi[q] = tot;
            tot += (size_t)n[q];
            oo[q] = tot;
            tot += (size_t)n[q];
            if (with_surf && surf[q]) {
                os[q] = tot;
                tot += (size_t)n[q] * (size_t)(steps[q] + 1);
            }
        }
        dev_buffer stage;
        stage.alloc(tot * sizeof(T));
        T *sb = (T *)stage.p;
        std::vector<const void *> di(count);
        std::vector<void *> dout(count), ds(count, nullptr);
        for (int64_t q = 0; q < count; ++q) {
            LSS_HIPCHK(hipMemcpy(sb + oi[q], u_in[q], (size_t)n[q] * sizeof(T), hipMemcpyHostToDevice));
            di[q] = sb + oi[q];
            dout[q] = sb + oo[q];
            if (with_surf && surf[q])
                ds[q] = sb + os[q];
        }
        set_table(di.data(), dout.data(), with_surf ? ds.data() : nullptr, nullptr);
        launch(nullptr, with_surf);
        LSS_HIPCHK(hipDeviceSynchronize());
        table_valid = false;  // the staging buffer goes away
        for (int64_t q = 0; q < count; ++q) {
            LSS_HIPCHK(hipMemcpy(u_out[q], sb + oo[q], (size_t)n[q] * sizeof(T), hipMemcpyDeviceToHost));
            if (with_surf && surf[q])
                LSS_HIPCHK(hipMemcpy(surf[q], sb + os[q], (size_t)n[q] * (size_t)(steps[q] + 1) * sizeof(T),
                                     hipMemcpyDeviceToHost));
        }
    }
};

lss_heat1d_plan *make_plan(const lss_heat1d_desc *d, int64_t cnt)
{
    if (d[0].fp == LSS_FP64) {
        auto *p = new H1Plan<double>();
        p->fp = LSS_FP64;
        try {
            p->build(d, cnt);
        } catch (...) {
            delete p;
            throw;
        }
        return p;
    }
    require(d[0].fp == LSS_FP32, "fp must be LSS_FP64 or LSS_FP32");
    auto *p = new H1Plan<float>();
    p->fp = LSS_FP32;
    try {
        p->build(d, cnt);
    } catch (...) {
        delete p;
        throw;
    }
    return p;
}

// Black-Scholes data of the reference's 1-D tests (lss_black_scholes_equation_t.hpp:66-80): the
// captured constants are double, each closure computes in double and rounds on return.
template <typename T> lss_amd_detail::heat1d_data<T> bs_data(const lss_bs_model &m)
{
    lss_amd_detail::heat1d_data<T> u;
    const double K = m.strike, r = m.rate, sig = m.sig, mat = m.maturity, xh = m.x_hi;
    u.a = [=](T, T x) { return (T)(0.5 * sig * sig * x * x); };
    u.b = [=](T, T x) { return (T)(r * x); };
    u.c = [=](T, T) { return (T)(-r); };
    u.init = [=](T x) { return std::max<T>((T)0.0, (T)(x - K)); };
    u.lo_type = LSS_BC_DIRICHLET;
    u.hi_type = LSS_BC_DIRICHLET;
    u.lo_val = [](T) { return (T)0.0; };
    u.hi_val = [=](T t) { return (T)(xh - K * std::exp(-r * (mat - t))); };
    return u;
}

template <typename T> lss_heat1d_plan *bs_plan(const lss_bs_model *models, int64_t cnt)
{
    std::vector<lss_amd_detail::heat1d_sampled<T>> s(cnt);
    std::vector<lss_heat1d_desc> d(cnt);
    for (int64_t q = 0; q < cnt; ++q) {
        const lss_bs_model &m = models[q];
        require(m.n >= 4 && m.nt >= 2, "model grid too small");
        require(m.implicit_scheme == LSS_EULER || m.implicit_scheme == LSS_CRANK_NICOLSON,
                "the 1-D solver takes the Euler or Crank-Nicolson scheme");
        lss_amd_detail::heat1d_spec<T> g;
        g.x_lo = (T)m.x_lo;
        g.x_hi = (T)m.x_hi;
        g.t_lo = (T)m.t_lo;
        g.t_hi = (T)m.t_hi;
        g.n = (size_t)m.n;
        g.nt = (size_t)m.nt;
        g.accumulation_point = (T)m.accumulation_point;
        g.alpha_scale = (T)m.alpha_scale;
        g.nonuniform = m.grid == LSS_GRID_NONUNIFORM;
        g.implicit_scheme = m.implicit_scheme;
        g.tridiagonal = m.tridiagonal;
        g.direction = m.direction;
        lss_amd_detail::sample_heat1d(bs_data<T>(m), g, s[q], lss_amd_detail::TIME_INDEPENDENT,
                                      lss_amd_detail::TIME_DEPENDENT);
        d[q] = s[q].desc(m.line_solver);
    }
    lss_heat1d_plan *plan = make_plan(d.data(), cnt);
    plan->init_host.resize(cnt);
    plan->grid_host.resize(cnt);
    for (int64_t q = 0; q < cnt; ++q) {
        plan->init_host[q].resize(s[q].init.size() * sizeof(T));
        std::memcpy(plan->init_host[q].data(), s[q].init.data(), plan->init_host[q].size());
        plan->grid_host[q].resize(s[q].xs.size() * sizeof(T));
        std::memcpy(plan->grid_host[q].data(), s[q].xs.data(), plan->grid_host[q].size());
    }
    return plan;
}

}  // namespace

extern "C" {

int lss_heat1d_plan_create(const lss_heat1d_desc *descs, int64_t count, lss_heat1d_plan **plan)
{
    return guarded([&] {
        require(descs && plan && count >= 1, "null descriptor/plan pointer or count < 1");
        *plan = nullptr;
        *plan = make_plan(descs, count);
    });
}

int lss_heat1d_plan_destroy(lss_heat1d_plan *plan)
{
    return guarded([&] { delete plan; });
}

int lss_heat1d_run_dev(lss_heat1d_plan *plan, const void *const *u_in, void *const *u_out, void *const *surfaces,
                       void *stream)
{
    return guarded([&] {
        require(plan != nullptr, "null plan");
        plan->run(u_in, u_out, surfaces, (hipStream_t)stream, false);
    });
}

int lss_heat1d_run_host(lss_heat1d_plan *plan, const void *const *u_in, void *const *u_out, void *const *surfaces)
{
    return guarded([&] {
        require(plan != nullptr, "null plan");
        plan->run(u_in, u_out, surfaces, nullptr, true);
    });
}

int lss_heat1d_problem_shape(const lss_heat1d_plan *plan, int64_t p, int64_t *n, int64_t *steps)
{
    return guarded([&] {
        require(plan != nullptr, "null plan");
        require(p >= 0 && p < plan->count, "problem index out of range");
        if (n)
            *n = plan->n[p];
        if (steps)
            *steps = plan->steps[p];
    });
}

int lss_bs_plan_create(const lss_bs_model *models, int64_t count, int32_t fp, lss_heat1d_plan **plan)
{
    return guarded([&] {
        require(models && plan && count >= 1, "null model/plan pointer or count < 1");
        *plan = nullptr;
        if (fp == LSS_FP64)
            *plan = bs_plan<double>(models, count);
        else if (fp == LSS_FP32)
            *plan = bs_plan<float>(models, count);
        else
            throw lss_error(LSS_ERR_INVALID, "fp must be LSS_FP64 or LSS_FP32");
    });
}

int lss_heat1d_initial(const lss_heat1d_plan *plan, int64_t p, void *u0_host)
{
    return guarded([&] {
        require(plan && u0_host, "null pointer");
        require(p >= 0 && p < plan->count, "problem index out of range");
        require((int64_t)plan->init_host.size() == plan->count, "plan was not created from models");
        std::memcpy(u0_host, plan->init_host[p].data(), plan->init_host[p].size());
    });
}

int lss_heat1d_grid(const lss_heat1d_plan *plan, int64_t p, void *xs_host)
{
    return guarded([&] {
        require(plan && xs_host, "null pointer");
        require(p >= 0 && p < plan->count, "problem index out of range");
        require((int64_t)plan->grid_host.size() == plan->count, "plan was not created from models");
        std::memcpy(xs_host, plan->grid_host[p].data(), plan->grid_host[p].size());
    });
}

}  // extern "C"
