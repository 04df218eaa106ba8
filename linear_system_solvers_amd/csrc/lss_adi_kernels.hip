// lss_adi_kernels.hip -- HIP kernels of the ADI time step for gfx950 (MI355X).
//
// One time step of every scheme is the same program of launches (the reference's loop body,
// pde_solvers/two_dimensional/heat_type/lss_2d_general_heston_equation_implicit_kernel.hpp:177-184):
//   xsweep  stage 1: S-lines j = 1..ny-2, rhs_intermed_1 of u, implicit solve along S  -> Y1; with it boundary
//           stage A: v = 0 column (explicit degenerate row) and v = v_max column
//           (lss_2d_general_heston_equation_explicit_boundary.hpp:181-200, :39-84)
//   vsweep  stage 1: v-lines i = 1..nx-2, v-direction rhs, implicit solve along v     -> Y2 (DR: next)
//   xsweep  stage 2: CS/MCS rhs_intermed_3 -> Y3; HV rhs_intermed_4 -> Y4, its explicit stage Y3 evaluated in place
//   vsweep  stage 2: v-direction rhs of (u, Y3) or (Y2, Y4)                          -> next
//   bnd_b   boundary stage B: S_min row and S_max Neumann extrapolation (explicit_boundary.hpp:202-238)
//           (exact lines: evaluated by the step's last v-sweep)
// The explicit Euler solver's step is one launch of k_euler (interior and both boundary stages).
// Kernels are compiled with -ffp-contract=off and keep the reference's operand order, so with
// FIELDS coefficients every value is rounded exactly as the reference's host code rounds it.

#include "lss_adi_stencil.hpp"
#include "lss_quad.hpp"

#include <type_traits>

namespace lssamd {

template <typename T>
__global__ void __launch_bounds__(TILE) k_bnd_b(const Prob<T> *__restrict__ probs, const Tile *__restrict__ tiles,
                                                int step)
{
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    if (step >= p.steps || (int)threadIdx.x >= tl.count)
        return;
    bnd_b_col(p, step, tl.first + (int)threadIdx.x);
}

// -------------------------------------------------------------------------------------------------
// Exact line sweeps.  DIR 0: S-lines (line l = column, point t = row), DIR 1: v-lines (line = row, point =
// column).  A tile of EXL lines is swept in phases:
//   exact_rhs     every thread forms right-hand sides of the tile's points (independent of each other), the
//                 Dirichlet ends folded, into the workspace;
//   exact_factor  a, beta = b - a gamma, 1 / beta and gamma = c / beta of the tile's rows, which do not depend on
//                 the right-hand sides: in a loop's first step (fresh) for coefficients that do not change in time,
//                 for both stages of every step, else in every step's first stage;
//   exact_sweep   the recurrence s = (f - a s) / beta and the back substitution x = s - gamma x, four lanes (a quad)
//                 per line, one wavefront per tile.
// The last two take a line through the quad in groups of 16 points, lane q holding points 4q .. 4q + 3 of the group,
// and pass the recurrence between the lanes in the reference's order, so every value is rounded as the reference
// rounds it.  The double sweep is the same recurrence with L = -gamma (b + a L = b - a gamma, L x + K = K - gamma x:
// negation is exact); the two differ in the last row only.
// A wavefront issues an instruction every four to five cycles whatever it depends on, and one wavefront sweeps a
// tile, so what bounds a sweep is the number of instructions of the recurrence: everything else is done by other
// wavefronts (exact_rhs) or once per loop (exact_factor), and the workspace is laid out by lane, in 16-byte pieces at
// fixed offsets, so that a group costs no addresses.  Measured in fp64 (one lane per line with the rows formed in the
// sweep before): 100 x 50, 100 steps DR 8.8 -> 1.96 ms (the S-sweep 58.8 -> 12, the v-sweep 24.5 -> 8 us); 512 x 256
// HV 1134 -> 157 us a step; 256 mixed problems of up to 512 x 256 points 149 -> 40 ms.
//
// Workspace (Prob::scr): the S-lines' tiles, then the v-lines'; of each tile its groups, of each group EX_ARRAYS
// arrays of 256 values as [half][lane][2]: the right-hand sides, the intermediate solution, a, beta, 1 / beta, gamma.
// -------------------------------------------------------------------------------------------------
constexpr int EXT = 256;  // threads per tile
constexpr int EXU = 3;    // points a thread forms at a time
enum { EX_F = 0, EX_S = 1, EX_A = 2, EX_BETA = 3, EX_Y = 4, EX_G = 5 };

// groups of 16 points of a line and block of array `arr` of (tile, group); the S-lines' tiles number the v-lines'
// groups and the other way round
template <typename T, int DIR> __device__ __forceinline__ int ex_groups(const Prob<T> &p)
{
    return ((DIR == 0 ? p.nx : p.ny) - 2 + 15) / 16;
}
template <typename T, int DIR> __device__ __forceinline__ gptr<T> ex_tile(const Prob<T> &p, int tile)
{
    const size_t nb = (size_t)ex_groups<T, 0>(p) * (size_t)ex_groups<T, 1>(p);
    return G(p.scr) + ((size_t)DIR * nb + (size_t)tile * ex_groups<T, DIR>(p)) * (EX_ARRAYS * 256);
}
// point accessor at a 32-bit offset from a scalar base
template <typename T> struct PAt32 {
    gptr<const T> b;
    uint32_t q, ny;
    __device__ __forceinline__ T operator()(int di, int dj) const
    {
        return ldg(b, q + (uint32_t)di * ny + (uint32_t)dj);
    }
};
template <typename T> struct Pair {
    typedef T v2 __attribute__((ext_vector_type(2)));
};
template <typename T> __device__ __forceinline__ void ex_load(gptr<T> b, int g, int arr, int lane, T (&v)[4])
{
    typedef typename Pair<T>::v2 v2;
    const gptr<const v2> q = (gptr<const v2>)(b + (size_t)g * (EX_ARRAYS * 256) + lane * 2) + arr * 128;
    const v2 x = q[0], y = q[64];
    v[0] = x.x, v[1] = x.y, v[2] = y.x, v[3] = y.y;
}
template <typename T> __device__ __forceinline__ void ex_store(gptr<T> b, int g, int arr, int lane, const T (&v)[4])
{
    typedef typename Pair<T>::v2 v2;
    const gptr<v2> q = (gptr<v2>)(b + (size_t)g * (EX_ARRAYS * 256) + lane * 2) + arr * 128;
    q[0] = v2{v[0], v[1]};
    q[64] = v2{v[2], v[3]};
}

// Right-hand sides.  KIND: 0 stage-1 S-lines (every scheme); 1 CS, 2 MCS, 3 HV stage-2 S-lines (HV evaluates its
// explicit stage Y3 in place); 4 v-lines (of in, inh).  Dirichlet ends of line l: lo(l), hi(l).
template <typename T, int PAT, int KIND, typename LoF, typename HiF>
__device__ __forceinline__ void exact_rhs(const Prob<T> &p, int step, int l0, int cnt, gptr<const T> in,
                                          gptr<const T> inh, LoF &&lo, HiF &&hi, int tid)
{
    constexpr int DIR = KIND == 4 ? 1 : 0;
    const int nx = p.nx, ny = p.ny, N = (DIR ? ny : nx) - 2;
    constexpr int RP = EXT / EXL;  // points of a line formed side by side
    const int c = DIR ? tid / RP : tid % EXL, r = DIR ? tid % RP : tid / EXL;
    if (c >= cnt)
        return;
    const int l = l0 + c;
    const gptr<const T> cs = coeff_set(p, step);
    const gptr<T> ws = ex_tile<T, DIR>(p, (l0 + EXL - 2) / EXL);
    const gptr<const T> u = G((const T *)((step & 1) ? p.b : p.a)), y1 = G((const T *)p.y1), y2 = G((const T *)p.y2);
    const T one = (T)1.0, theta = p.theta;
    const T *sp = KIND == 0 ? src_set(p, step) : nullptr;
    const int64_t nxy = (int64_t)nx * ny;
    const bool thomas = p.tri == TRI_THOMAS;
    auto at = [&](gptr<const T> b, uint32_t q) { return PAt32<T>{b, q, (uint32_t)ny}; };
    auto point = [&](int t) -> T {
        const int i = DIR ? l : t, j = DIR ? t : l;
        const uint32_t q = (uint32_t)i * (uint32_t)ny + (uint32_t)j;
        const Stencil<T> s = stencil_at<T, PAT>(p, cs, i, j);
        T v;
        if constexpr (KIND == 0) {
            v = rhs_intermed_1(p, s, at(u, q));
            // rhs_intermed_1_source (lss_heat_douglas_rachford_method.hpp:70-104)
            if (sp)
                v = v + (theta * p.rho * sp[nxy + q]) + ((one - theta) * p.rho * sp[q]);
        } else if constexpr (KIND == 1) {
            v = rhs_intermed_3<T, false>(p, s, at(u, q), at(y1, q), at(y2, q));
        } else if constexpr (KIND == 2) {
            v = rhs_intermed_3<T, true>(p, s, at(u, q), at(y1, q), at(y2, q));
        } else if constexpr (KIND == 3) {  // rhs_intermed_4 (lss_heat_hundsdorfer_verwer_method.hpp:174-194)
            const T y3 = hv_y3_at(p, s, at(u, q), at(y1, q), at(y2, q));
            const auto y2q = at(y2, q);
            v = (-theta * s.M * y2q(-1, 0)) + (theta * s.Z * y2q(0, 0)) - (theta * s.P * y2q(1, 0)) + y3;
        } else {
            v = rhs_v(p, s, GAt<T>{in, q}, GAt<T>{inh, q});
        }
        // the folded ends (thomas_lu_boundary.hpp:127-135, double_sweep_boundary.hpp:100-106)
        if (t == 1)
            v = v - (-theta * (DIR ? s.Mt : s.M)) * lo(l);
        if (t == N && thomas)
            v = v - (-theta * (DIR ? s.Pt : s.P)) * hi(l);
        return v;
    };
    auto put = [&](int t, T v) {
        const int g = (t - 1) >> 4, k = (t - 1) & 15, ln = c * 4 + (k >> 2);
        ws[(size_t)g * (EX_ARRAYS * 256) + EX_F * 256 + ((k >> 1) & 1) * 128 + ln * 2 + (k & 1)] = v;
    };
    // EXU points at a time, loaded before the first store
    for (int t = 1 + r; t <= N; t += RP * EXU) {
        T v[EXU];
#pragma unroll
        for (int k = 0; k < EXU; ++k)
            v[k] = point(min(t + RP * k, N));
#pragma unroll
        for (int k = 0; k < EXU; ++k)
            if (t + RP * k <= N)
                put(t + RP * k, v[k]);
    }
}

// a, beta, 1 / beta and gamma of the rows of a tile's lines (identity rows past a line's end and for lines past the
// tile's count, so that the sweep needs no conditions)
template <typename T, int PAT, int DIR> __device__ __forceinline__ void exact_factor(const Prob<T> &p, int step, int l0, int cnt)
{
    const int lane = (int)threadIdx.x & 63, ql = lane & 3, end = (DIR == 0 ? p.nx : p.ny) - 2, ng = (end + 15) / 16;
    const bool live = (lane >> 2) < cnt;
    const int l = l0 + (live ? lane >> 2 : 0);
    const gptr<const T> cs = coeff_set(p, step);
    const gptr<T> ws = ex_tile<T, DIR>(p, (l0 + EXL - 2) / EXL);
    const T one = (T)1.0, theta = p.theta;
    struct Stage {
        T M[4], Z[4], P[4];
    };
    auto load = [&](int g, Stage &s) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = min(1 + 16 * g + 4 * ql + j, end);
            const Stencil<T> st = stencil_at<T, PAT>(p, cs, DIR == 0 ? t : l, DIR == 0 ? l : t);
            s.M[j] = DIR == 0 ? st.M : st.Mt;
            s.Z[j] = DIR == 0 ? st.Z : st.W;
            s.P[j] = DIR == 0 ? st.P : st.Pt;
        }
    };
    T gcar = (T)0;
    auto body = [&](int g, Stage &s) {
        T a[4], b[4], c[4], beta[4], gm[4], y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = 1 + 16 * g + 4 * ql + j;
            const bool row = live && t <= end;
            a[j] = (row && t > 1) ? (-theta * s.M[j]) : (T)0;  // (the first row's end is folded)
            b[j] = row ? (one + theta * s.Z[j]) : one;
            c[j] = row ? (-theta * s.P[j]) : (T)0;
        }
        gcar = quad_gamma(a, b, c, gcar, beta, gm);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            y[j] = quick_rcp(beta[j]);
        ex_store(ws, g, EX_A, lane, a);
        ex_store(ws, g, EX_BETA, lane, beta);
        ex_store(ws, g, EX_Y, lane, y);
        ex_store(ws, g, EX_G, lane, gm);
    };
    quad_stages<Stage>(0, ng, 1, load, body);
}

// forward recurrence and back substitution of a tile's lines; out: the solution's array, lo and hi: the lane's line's
// end values
template <typename T, int DIR>
__device__ __forceinline__ void exact_sweep(const Prob<T> &p, int l0, int cnt, gptr<T> out, T lo, T hi)
{
    const int lane = (int)threadIdx.x & 63, ql = lane & 3, ny = p.ny, end = (DIR == 0 ? p.nx : ny) - 2, ng = (end + 15) / 16;
    const bool live = (lane >> 2) < cnt;
    const gptr<T> ws = ex_tile<T, DIR>(p, (l0 + EXL - 2) / EXL);
    const bool thomas = p.tri == TRI_THOMAS;
    struct Stage {
        T a[4], beta[4], y[4], f[4];
    };
    auto load = [&](int g, Stage &s) {
        ex_load(ws, g, EX_A, lane, s.a);
        ex_load(ws, g, EX_BETA, lane, s.beta);
        ex_load(ws, g, EX_Y, lane, s.y);
        ex_load(ws, g, EX_F, lane, s.f);
    };
    SeenNum seen;
    T scar = (T)0;
    quad_stages<Stage>(0, ng, 1, load, [&](int g, Stage &s) {
        T x[4];
        scar = quad_forward<true>(s.a, s.f, s.beta, s.y, scar, x, seen);
        ex_store(ws, g, EX_S, lane, x);
    });
    if (__builtin_amdgcn_ballot_w64(!seen_ok(seen, scar))) {  // a numerator outside quick_div's range
        scar = (T)0;
#pragma unroll 1
        for (int g = 0; g < ng; ++g) {
            Stage s;
            T x[4];
            load(g, s);
            scar = quad_forward<false>(s.a, s.f, s.beta, s.y, scar, x, seen);
            ex_store(ws, g, EX_S, lane, x);
        }
    }
    struct Back {
        T G[4], s[4];
    };
    auto loadb = [&](int g, Back &b) {
        ex_load(ws, g, EX_G, lane, b.G);
        ex_load(ws, g, EX_S, lane, b.s);
    };
    const uint32_t l = (uint32_t)(l0 + (live ? lane >> 2 : 0));
    const uint32_t base = DIR == 0 ? l : l * (uint32_t)ny, str = DIR == 0 ? (uint32_t)ny : 1u;
    T xcar = hi;
    quad_stages<Back>(ng - 1, ng, -1, loadb, [&](int g, Back &b) {
        const int t0 = 1 + 16 * g + 4 * ql;
        T x[4];
        if (g == ng - 1) {  // the Thomas sweep's last point is s itself
            xcar = quad_backward_ends(
                b.G, b.s, xcar, x, [&](int j) { return t0 + j == end && thomas; }, [&](int j) { return t0 + j > end; });
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (live && t0 + j <= end)
                    stg(out, base + (uint32_t)(t0 + j) * str, x[j]);
        } else {
            xcar = quad_backward(b.G, b.s, xcar, x);
            if (live) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    stg(out, base + (uint32_t)(t0 + j) * str, x[j]);
            }
        }
    });
    if (live && ql == 0) {
        stg(out, base, lo);
        stg(out, base + (uint32_t)(end + 1) * str, hi);
    }
}

// S-line sweep of tile (l0, cnt).  stage 1: rhs_intermed_1(u) -> Y1.  stage 2: CS/MCS rhs_intermed_3(u, Y1, Y2)
// -> Y3; HV rhs_intermed_4(Y2, Y3) -> Y4.  Dirichlet ends u(0, idx2[j]), u(nx-1, idx2[j])
// (implicit_kernel.hpp:86-101, old time level).
template <typename T, int PAT>
__device__ __forceinline__ void xsweep_rhs(const Prob<T> &p, int step, int stage, int l0, int cnt, int tid)
{
    const gptr<const T> u = G((const T *)((step & 1) ? p.b : p.a)), none = nullptr;
    auto lo = [&](int j) { return ldg(u, p.idx2[j]); };
    auto hi = [&](int j) { return ldg(u, (uint32_t)(p.nx - 1) * (uint32_t)p.ny + p.idx2[j]); };
    if (stage == 1)
        exact_rhs<T, PAT, 0>(p, step, l0, cnt, none, none, lo, hi, tid);
    else if (p.scheme == SCHEME_CS)
        exact_rhs<T, PAT, 1>(p, step, l0, cnt, none, none, lo, hi, tid);
    else if (p.scheme == SCHEME_MCS)
        exact_rhs<T, PAT, 2>(p, step, l0, cnt, none, none, lo, hi, tid);
    else
        exact_rhs<T, PAT, 3>(p, step, l0, cnt, none, none, lo, hi, tid);
}
template <typename T, int PAT>
__device__ __forceinline__ void xsweep_solve(const Prob<T> &p, int step, int stage, bool fresh, int l0, int cnt)
{
    const int lane = (int)threadIdx.x & 63;
    if (fresh)
        exact_factor<T, PAT, 0>(p, step, l0, cnt);
    const gptr<const T> u = G((const T *)((step & 1) ? p.b : p.a));
    const uint32_t jj = p.idx2[l0 + min(lane >> 2, cnt - 1)];
    exact_sweep<T, 0>(p, l0, cnt, G(stage == 1 ? p.y1 : (p.scheme == SCHEME_HV ? p.y4 : p.y3)), ldg(u, jj),
                      ldg(u, (uint32_t)(p.nx - 1) * (uint32_t)p.ny + jj));
}

// v-line sweep of tile (l0, cnt).  stage 1: rhs_v(u, Y1) -> Y2 (DR: next).  stage 2: CS/MCS rhs_v(u, Y3) -> next;
// HV rhs_v(Y2, Y4) -> next.  Dirichlet ends colA0/colA1[idx1[i]]: the copy of `next` the vertical lambdas
// captured after boundary stage A (implicit_kernel.hpp:69-84).
template <typename T, int PAT>
__device__ __forceinline__ void vsweep_rhs(const Prob<T> &p, int step, int stage, int l0, int cnt, int tid)
{
    const T *u = (step & 1) ? p.b : p.a;
    const bool hv2 = stage == 2 && p.scheme == SCHEME_HV;
    const gptr<const T> cA = G((const T *)p.colA0), cB = G((const T *)p.colA1);
    exact_rhs<T, PAT, 4>(p, step, l0, cnt, G(hv2 ? (const T *)p.y2 : u),
                    G((const T *)(stage == 1 ? p.y1 : (hv2 ? p.y4 : p.y3))), [&](int i) { return ldg(cA, p.idx1[i]); },
                    [&](int i) { return ldg(cB, p.idx1[i]); }, tid);
}
template <typename T, int PAT>
__device__ __forceinline__ void vsweep_solve(const Prob<T> &p, int step, int stage, bool fresh, int l0, int cnt)
{
    const int lane = (int)threadIdx.x & 63;
    if (fresh)
        exact_factor<T, PAT, 1>(p, step, l0, cnt);
    const uint32_t ii = p.idx1[l0 + min(lane >> 2, cnt - 1)];
    exact_sweep<T, 1>(p, l0, cnt, G((stage == 1 && p.scheme != SCHEME_DR) ? p.y2 : ((step & 1) ? p.a : p.b)),
                      ldg((gptr<const T>)G(p.colA0), ii), ldg((gptr<const T>)G(p.colA1), ii));
}

// One tile per workgroup: its threads form the right-hand sides, its first wavefront sweeps; in
// stage 1 of the S-sweep the other wavefronts evaluate the tile's share of boundary stage A meanwhile (the v-sweeps
// read it), and in the step's last v-sweep the tile that holds rows nx - 2 and nx - 3 (the plan lays v-line tiles out
// from the last row) evaluates boundary stage B.  Workgroups of 1024 threads, for fewer rounds of loads in the
// right-hand sides, were slower also for one small problem (100 x 50 x 100 steps: 2.29 ms against 1.96), and a loop
// that keeps the whole problem in one workgroup was as well (2.92 ms: the loads of the right-hand sides then go
// through one CU's L1).
template <typename T, int PAT>
__global__ void __launch_bounds__(EXT) k_xsweep(const Prob<T> *__restrict__ probs, const Tile *__restrict__ tiles,
                                               int step, int stage, int fresh)
{
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    if (step >= p.steps || (stage == 2 && p.scheme == SCHEME_DR))
        return;  // uniform over the workgroup
    const int tid = (int)threadIdx.x;
    xsweep_rhs<T, PAT>(p, step, stage, tl.first, tl.count, tid);
    __syncthreads();
    if (tid < 64) {
        xsweep_solve<T, PAT>(p, step, stage, stage == 1 && (fresh || p.coeff_sets > 1), tl.first, tl.count);
    } else if (stage == 1) {
        const int ntl = (p.ny - 2 + EXL - 1) / EXL, k = (tl.first - 1) / EXL;
        for (int i = k * (EXT - 64) + tid - 64; i < p.nx; i += ntl * (EXT - 64))
            bnd_a_row(p, step, i);
    }
}

template <typename T, int PAT>
__global__ void __launch_bounds__(EXT) k_vsweep(const Prob<T> *__restrict__ probs, const Tile *__restrict__ tiles,
                                               int step, int stage, int fresh)
{
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    if (step >= p.steps || (stage == 2 && p.scheme == SCHEME_DR))
        return;  // uniform over the workgroup
    const int tid = (int)threadIdx.x;
    vsweep_rhs<T, PAT>(p, step, stage, tl.first, tl.count, tid);
    __syncthreads();
    if (tid < 64)
        vsweep_solve<T, PAT>(p, step, stage, stage == 1 && (fresh || p.coeff_sets > 1), tl.first, tl.count);
    if ((stage == 2 || p.scheme == SCHEME_DR) && tl.first + tl.count == p.nx - 1) {  // uniform
        __syncthreads();
        for (int j = tid; j < p.ny; j += EXT)
            bnd_b_col(p, step, j);
    }
}

// -------------------------------------------------------------------------------------------------
// Explicit Euler step of the explicit solver in one launch (lss_heston_euler_solver_scheme.hpp:63-67,
// 78-83: the interior, boundary stage A, boundary stage B, each from the level before):
//   interior  explicit_heston_scheme::rhs (lss_heston_euler_solver_method.hpp:26-52), whose C is
//             gamma * c (lss_heston_euler_coefficients.hpp:50-51);
//   column 0 and ny - 1  boundary stage A (explicit_boundary.hpp:39-84, 181-200), which writes them
//             for every row;
//   row 0 and nx - 1     boundary stage B (explicit_boundary.hpp:202-238); its S_max extrapolation
//             reads rows nx - 2 and nx - 3 of the new level through idx2, and the thread recomputes
//             those two values from u with the same arithmetic instead of waiting for them.
// Every value is rounded as the reference rounds it (this file is compiled without contraction), so
// with FIELDS coefficients the step is bit-identical to the three stages run one after another.
// PAT selects compile-time factor patterns of SEPARABLE plans.  Two-dimensional tiles of GTR * ERPT
// rows x GTC columns; a thread takes ERPT consecutive rows of one column (lanes along the contiguous v
// direction) and reads the rows of its three columns once.
// -------------------------------------------------------------------------------------------------
template <typename T, int PAT>
__global__ void __launch_bounds__(GTR *GTC) k_euler(const Prob<T> *__restrict__ probs,
                                                    const Tile *__restrict__ tiles, int step)
{
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    if (step >= p.steps)
        return;
    const int tg = threadIdx.x / GTC, tc = threadIdx.x % GTC;
    const int j = tl.col + tc;
    const int nx = p.nx, ny = p.ny;
    const int r0 = tl.first + tg * ERPT;               // this thread's rows r0 .. r0 + rn - 1
    const int rn = min(ERPT, tl.first + tl.count - r0);
    if (j >= ny || rn <= 0)
        return;
    const gptr<const T> u = G((const T *)((step & 1) ? p.b : p.a));
    const gptr<T> nxt = G((step & 1) ? p.a : p.b);
    const gptr<const T> cs = coeff_set(p, step);
    const gptr<const T> bs = bnd_set(p, step);
    const T one = (T)1.0, two = (T)2.0, three = (T)3.0, four = (T)4.0;
    // the value stages "interior" and A give point (r, c), 1 <= r <= nx - 2, from direct loads
    auto level = [&](int r, int c) -> T {
        const gptr<const T> w = u + ((int64_t)r * ny + c);
        if (c == ny - 1)
            return bs[r];  // v_upper(t, X(zeta_r))
        if (c == 0) {      // the degenerate v = 0 row
            T D, E, F;
            def_row0<T, PAT>(p, cs, r, D, E, F);
            const T delta = p.delta, ni = p.ni, rho = p.rho;
            return (-delta * D * w[-ny]) + ((one - three * ni * E + rho * F) * w[0]) + (delta * D * w[ny]) -
                   (ni * E * w[2]) + (four * ni * E * w[1]);
        }
        const Stencil<T> s = stencil_at<T, PAT>(p, cs, r, c);
        const T C = p.gamma * s.C;
        return C * w[-ny - 1] + s.M * w[-ny] - C * w[-ny + 1] + s.Mt * w[-1] + (one - s.Z - s.W) * w[0] +
               s.Pt * w[1] - C * w[ny - 1] + s.P * w[ny] + C * w[ny + 1];
    };
    // rows r0 - 1 .. r0 + ERPT of columns j - 1, j, j + 1 (clamped into the grid), all loaded before
    // the first store, so that each value is read once and the interior points share them
    const int jm = max(j - 1, 0), jp = min(j + 1, ny - 1);
    T w[ERPT + 2][3];
#pragma unroll
    for (int t = 0; t < ERPT + 2; ++t) {
        const gptr<const T> row = u + (int64_t)min(max(r0 - 1 + t, 0), nx - 1) * ny;
        w[t][0] = row[jm];
        w[t][1] = row[j];
        w[t][2] = row[jp];
    }
    T out[ERPT];
#pragma unroll
    for (int t = 0; t < ERPT; ++t) {
        const int i = r0 + t;
        T v = (T)0;
        if (t < rn) {
            if (i == 0) {
                v = bs[nx + j];  // h_lower(t, Y(eta_j))
            } else if (i == nx - 1) {
                const int jj = (int)p.idx2[j];
                v = (((four * level(nx - 2, jj)) - level(nx - 3, jj) - (two * p.h1 * bs[nx + ny + j])) / three);
            } else if (j == 0 || j == ny - 1) {
                v = level(i, j);
            } else {
                const Stencil<T> s = stencil_at<T, PAT>(p, cs, i, j);
                const T C = p.gamma * s.C;
                v = C * w[t][0] + s.M * w[t][1] - C * w[t][2] + s.Mt * w[t + 1][0] + (one - s.Z - s.W) * w[t + 1][1] +
                    s.Pt * w[t + 1][2] - C * w[t + 2][0] + s.P * w[t + 2][1] + C * w[t + 2][2];
            }
        }
        out[t] = v;
    }
#pragma unroll
    for (int t = 0; t < ERPT; ++t)
        if (t < rn)
            nxt[(int64_t)(r0 + t) * ny + j] = out[t];
}

// -------------------------------------------------------------------------------------------------
// The whole explicit Euler time loop of one small problem in one workgroup of ERES_T threads, its two
// time levels resident in LDS (lss_heston_euler_solver_scheme.hpp:63-67, 78-83).  Per step: the
// interior and boundary stage A from the old level into the new one; a barrier; boundary stage B (row 0,
// and row nx - 1 extrapolated from rows nx - 2 and nx - 3 of the new level, as the reference reads
// them); a barrier.  Every value takes the arithmetic of k_euler in the same order.
//
// A thread holds a strip of K consecutive rows of one column: its stencil weights, formed once (one coefficient
// set and one boundary set), and its column's values stay in registers, so that per strip and step it reads
// 2 K + 6 values from LDS and writes K (K = 6: 4 accesses a point; a thread per point, scattered, takes 10, which
// bound the loop by LDS bandwidth: 1024 problems 50 x 30, 7999 steps in fp64 19.0 ms at 52 TB/s against 11.0 ms at 36
// with strips; the v = 0 weights in LDS instead of registers: 11.4 ms).  Strips of columns
// with at least K interior rows overlap at the bottom instead of ending early (both compute the same values);
// shorter columns mask.  Values that do not change from step to step (row 0, column ny - 1) are written in the
// first two steps only.  For problems of at most ERES_POINTS points with nx >= 4 and ny <= ERES_T: then some K of 6,
// 8 and 10 gives every strip a thread.  HBM is read once and written once.
// -------------------------------------------------------------------------------------------------
template <typename T, int PAT, int K>
__global__ void __launch_bounds__(ERES_T) __attribute__((amdgpu_waves_per_eu(K <= 6 ? 4 : 2)))
k_euler_res(const Prob<T> *__restrict__ probs, const Tile *__restrict__ tiles)
{
    __shared__ T lv[2][ERES_POINTS];
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    const int nx = p.nx, ny = p.ny, n = nx * ny, steps = p.steps, tid = (int)threadIdx.x;
    const T one = (T)1.0, two = (T)2.0, three = (T)3.0, four = (T)4.0;
    {
        const gptr<const T> a = G((const T *)p.a);
        for (int q = tid; q < n; q += ERES_T)
            lv[0][q] = a[q];
    }
    const gptr<const T> cs = coeff_set(p, 0);
    const gptr<const T> bs = bnd_set(p, 0);
    // the thread's strip: rows r0 .. r0 + nv - 1 of column c
    const int cols = ny - 2, rows = nx - 2, nst = (rows + K - 1) / K;
    const bool strip = tid < nst * cols;
    const int c = strip ? 1 + tid % cols : 1, sr = strip ? tid / cols : 0;
    const int nv = min(K, rows), r0 = 1 + min(sr * K, rows - nv), o0 = r0 * ny + c;
    T wt[K][6];  // C, M, M~, 1 - Z - W, P~, P (C = gamma c)
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const Stencil<T> st = stencil_at<T, PAT>(p, cs, min(r0 + j, nx - 2), c);
        wt[j][0] = p.gamma * st.C;
        wt[j][1] = st.M;
        wt[j][2] = st.Mt;
        wt[j][3] = one - st.Z - st.W;
        wt[j][4] = st.Pt;
        wt[j][5] = st.P;
    }
    // the v = 0 points of rows 1 + k, from the last thread down: -delta D, 1 - 3 ni E + rho F, delta D, ni E, 4 ni E
    constexpr int NV0 = (ERES_POINTS / 4 + ERES_T - 1) / ERES_T;
    T w0[NV0][5];
#pragma unroll
    for (int k = 0; k < NV0; ++k) {
        T D, E, F;
        def_row0<T, PAT>(p, cs, min(1 + ERES_T - 1 - tid + k * ERES_T, nx - 2), D, E, F);
        const T delta = p.delta, ni = p.ni, rho = p.rho;
        w0[k][0] = -delta * D;
        w0[k][1] = one - three * ni * E + rho * F;
        w0[k][2] = delta * D;
        w0[k][3] = ni * E;
        w0[k][4] = four * ni * E;
    }
    T lo_j = (T)0, hup_j = (T)0;  // boundary stage B of column tid: h_lower and 2 h_1 h_upper X'(1)
    int jj = 0;
    if (tid < ny) {
        lo_j = bs[nx + tid];  // h_lower(t, Y(eta_j))
        hup_j = two * p.h1 * bs[nx + ny + tid];
        jj = (int)p.idx2[tid];
    }
    __syncthreads();
    T own[K];
#pragma unroll
    for (int j = 0; j < K; ++j)
        own[j] = lv[0][o0 + min(j, nv - 1) * ny];
    auto loop = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;  // the strip has K rows
        for (int s = 0; s < steps; ++s) {
            const T *u = lv[s & 1];
            T *w = lv[(s & 1) ^ 1];
            if (strip) {
                const T *q = u + o0;
                const T bot = q[nv * ny];
                // column above, at and below the current row, and its neighbours' values
                T um = q[-ny], lm = q[-ny - 1], rm = q[-ny + 1], l0 = q[-1], r0v = q[1];
                T nw[K];
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const int jd = FULL ? j + 1 : min(j + 1, nv);
                    const T lp = q[jd * ny - 1], rp = q[jd * ny + 1];
                    const T up = FULL ? (j + 1 < K ? own[j + 1 < K ? j + 1 : 0] : bot)
                                      : (j + 1 < nv ? own[j + 1 < K ? j + 1 : 0] : bot);
                    const T C = wt[j][0];
                    nw[j] = C * lm + wt[j][1] * um - C * rm + wt[j][2] * l0 + wt[j][3] * own[j] + wt[j][4] * r0v - C * lp +
                            wt[j][5] * up + C * rp;
                    um = own[j];
                    lm = l0;
                    rm = r0v;
                    l0 = lp;
                    r0v = rp;
                }
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    if (FULL || j < nv)
                        w[o0 + j * ny] = nw[j];
                    own[j] = nw[j];
                }
            }
#pragma unroll
            for (int k = 0; k < NV0; ++k) {
                const int r = 1 + ERES_T - 1 - tid + k * ERES_T;
                if (r <= nx - 2) {
                    const T *q = u + r * ny;
                    w[r * ny] = (w0[k][0] * q[-ny]) + (w0[k][1] * q[0]) + (w0[k][2] * q[ny]) - (w0[k][3] * q[2]) +
                                (w0[k][4] * q[1]);
                }
            }
            if (s < 2) {
                for (int r = 1 + tid; r <= nx - 2; r += ERES_T)
                    w[r * ny + ny - 1] = bs[r];  // v_upper(t, X(zeta_r))
                if (tid < ny)
                    w[tid] = lo_j;
            }
            __syncthreads();
            if (tid < ny)
                w[(nx - 1) * ny + tid] = (((four * w[(nx - 2) * ny + jj]) - w[(nx - 3) * ny + jj] - hup_j) / three);
            __syncthreads();
        }
    };
    if (rows >= K)
        loop(std::true_type{});
    else
        loop(std::false_type{});
    const gptr<T> out = G((steps & 1) ? p.b : p.a);
    for (int q = tid; q < n; q += ERES_T)
        out[q] = lv[steps & 1][q];
}

// -------------------------------------------------------------------------------------------------
// Batched tridiagonal systems (one lane per system), the reference's Thomas LU in its operation
// order with the end rows folded by `bc` (LineBC; PLAIN ignores a[0] and c[n-1]).
// Layout: contiguous x[k*n + i] (strided == 0) or interleaved x[i*B + k] (strided == 1).
// -------------------------------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_tridiag_lane(int64_t B, int n, int strided, const T *__restrict__ a,
                                                      const T *__restrict__ b, const T *__restrict__ c,
                                                      const T *__restrict__ d, T *__restrict__ x, T *__restrict__ scr,
                                                      LineBC<T> bc)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= B)
        return;
    const int64_t base = strided ? k : k * n, st = strided ? B : 1;
    const int s0 = bc.start(), e0 = bc.end(n);
    // row t with its end folded (thomas_lu_solver.hpp:125-191, thomas_lu_boundary.hpp:114-205)
    auto row = [&](int t, T &at, T &bt, T &ct, T &rt) {
        const int64_t q = base + t * st;
        at = a[q];
        bt = b[q];
        ct = c[q];
        rt = d[q];
        bc.fold(t == s0, t == e0, at, bt, ct, rt);
    };
    T at, bt, ct, rt;
    row(s0, at, bt, ct, rt);
    T beta = bt;
    T g = ct / beta;
    T s = rt / beta;
    scr[base + s0 * st] = g;
    x[base + s0 * st] = s;
    for (int t = s0 + 1; t <= e0; ++t) {
        row(t, at, bt, ct, rt);
        beta = bt - (at * g);
        g = ct / beta;
        s = (rt - (at * s)) / beta;
        scr[base + t * st] = g;
        x[base + t * st] = s;
    }
    T xv = s;
    for (int t = e0 - 1; t >= s0; --t) {
        const int64_t q = base + t * st;
        xv = x[q] - (scr[q] * xv);
        x[q] = xv;
    }
    if (bc.lo == BC_DIRICHLET)
        x[base] = bc.lo_val;
    if (bc.hi == BC_DIRICHLET)
        x[base + (int64_t)(n - 1) * st] = bc.hi_val;
}

// -------------------------------------------------------------------------------------------------
// explicit instantiations
// -------------------------------------------------------------------------------------------------
#define LSS_INST_EX(T, PAT)                                                                                   \
    template __global__ void k_xsweep<T, PAT>(const Prob<T> *, const Tile *, int, int, int);                  \
    template __global__ void k_vsweep<T, PAT>(const Prob<T> *, const Tile *, int, int, int);
#define LSS_INST_ERES(T, PAT)                                                                                 \
    template __global__ void k_euler_res<T, PAT, 6>(const Prob<T> *, const Tile *);                           \
    template __global__ void k_euler_res<T, PAT, 8>(const Prob<T> *, const Tile *);                           \
    template __global__ void k_euler_res<T, PAT, 10>(const Prob<T> *, const Tile *);
#define LSS_INST(T)                                                                                           \
    template __global__ void k_bnd_b<T>(const Prob<T> *, const Tile *, int);                                  \
    LSS_INST_EX(T, PAT_GENERIC) LSS_INST_EX(T, PAT_FIELDS)                                                    \
    LSS_INST_ERES(T, PAT_GENERIC) LSS_INST_ERES(T, PAT_HESTON) LSS_INST_ERES(T, PAT_SABR0)                    \
    template __global__ void k_euler<T, PAT_GENERIC>(const Prob<T> *, const Tile *, int);                     \
    template __global__ void k_euler<T, PAT_HESTON>(const Prob<T> *, const Tile *, int);                      \
    template __global__ void k_euler<T, PAT_SABR0>(const Prob<T> *, const Tile *, int);                       \
    template __global__ void k_tridiag_lane<T>(int64_t, int, int, const T *, const T *, const T *, const T *, \
                                               T *, T *, LineBC<T>);
LSS_INST(double)
LSS_INST(float)
#undef LSS_INST
#undef LSS_INST_EX
#undef LSS_INST_ERES

}  // namespace lssamd
