// lss_adi_resident.hpp -- the whole time loop of a small ADI problem in one launch: a workgroup per problem, its
// levels and intermediates resident in LDS.
//
// Step by step, such a plan is bound by its launches: 64 problems of 100 x 50 in fp64 take 18.5 us a DR step for 1 us of
// traffic, 22 us when every level is copied out.  Here a stage ends at a barrier of its workgroup: 7.4 us a step (8.3
// with the levels, which the S-sweep's phase stores while it reads them), for 1 to 256 problems; 1024 problems 11.8 ->
// 3.0 ms for 100 steps, one problem 1.08 -> 0.74 ms, 200 MCS problems of 40 x 20 2.84 -> 0.79 ms; fp32 64 problems 1.58
// -> 0.53 ms.
// What bounds a step is the issue of its instructions (a point's equation is formed and eliminated in about 75, and a
// SIMD has four wavefronts), so the partition wastes few of them: a line takes 16 lanes, whose chunks are as short as
// its length allows (any length up to ARES_C, not only those of wave_solve), and the 16 interface equations are
// reduced in registers by DPP row shifts (wave_solve's 64 chunks would need twice as many reduction steps, on four
// times the lanes, through the LDS pipe).  The stages and equations are those of the partitioned sweeps
// (lss_adi_partitioned.hpp); DR works in two buffers, the v-sweep over Y1, the other schemes in three.
// Only compile-time factor patterns: with run-time codes every body spills.
#pragma once
#pragma clang fp contract(fast)
#include "lss_adi_chunk.hpp"
#include "lss_adi_stencil.hpp"

namespace lssamd {

// Lane l of a row of 16 lanes takes lane l - D's / l + D's value, its own where there is none (DPP row shifts).
template <int CTRL> __device__ __forceinline__ int row_mov(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL> __device__ __forceinline__ float row_shift(float v)
{
    return __int_as_float(row_mov<CTRL>(__float_as_int(v)));
}
template <int CTRL> __device__ __forceinline__ double row_shift(double v)
{
    return __hiloint2double(row_mov<CTRL>(__double2hiint(v)), row_mov<CTRL>(__double2loint(v)));
}
template <int D, typename T> __device__ __forceinline__ T row_up(T v) { return row_shift<0x110 + D>(v); }
template <int D, typename T> __device__ __forceinline__ T row_down(T v) { return row_shift<0x100 + D>(v); }

template <int D, typename T> __device__ __forceinline__ Eq<T> row_pcr(const Eq<T> &e)
{
    const NEq<T> m = normalized(e);
    const NEq<T> l{row_up<D>(m.a), row_up<D>(m.c), row_up<D>(m.r)};
    const NEq<T> h{row_down<D>(m.a), row_down<D>(m.c), row_down<D>(m.r)};
    return pcr_step(e, l, h);
}

// wave_solve_c with one line per row of 16 lanes, chunks of C points (16 C >= N), any C: every exchange stays in
// registers.
template <typename T, int C, typename EqF, typename PutF>
__device__ __forceinline__ void row_solve(int N, int ll, EqF &&eq, PutF &&put)
{
    const int s = 1 + ll * C;
    Chunk<T, C> ch;
    if (s <= N) {
#pragma unroll
        for (int t = 0; t < C; ++t)
            ch.put(t, eq(t, s + t));
        ch.bwd();
    } else {
        ch.set_identity();
    }
    T PF, QF, RF;
    ch.first_rel(PF, QF, RF);
    Eq<T> e = ch.interface_eq(row_down<1>(PF), row_down<1>(QF), row_down<1>(RF));
    e = row_pcr<1>(e);
    e = row_pcr<2>(e);
    e = row_pcr<4>(e);
    e = row_pcr<8>(e);
    const T xi = e.r * fast_rcp(e.b);
    const T xl = row_up<1>(xi);
#pragma unroll
    for (int t = 0; t < C; ++t)
        if (s + t <= N)
            put(t, ch.value(t, xl, xi));
}

// A value that the compiler knows nothing of: the bodies of a step, one per chunk length, share registers with what it
// would otherwise compute once for all of them before the loop over steps (and spill).
__device__ __forceinline__ int opaque_lane(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int opaque_uniform(int v)
{
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
    return v;
}

// f(std::integral_constant<int, c>), 1 <= c <= ARES_C (uniform)
template <int C = 1, typename F> __device__ __forceinline__ void with_length(int c, F &&f)
{
    if constexpr (C < ARES_C) {
        if (c > C) {
            with_length<C + 1>(c, f);
            return;
        }
    }
    f(std::integral_constant<int, C>{});
}

// a problem's arrays in LDS
template <typename T> struct ResMem {
    lptr<T> u, y1, y2;         // old level; Y1, then Y3 / Y4, then the new level; Y2.  Row stride ld
    LArr<T> xf, yf;            // factor vectors (compile-time patterns)
    lptr<T> cA0, cA1, bn;      // boundary stage A's columns, the boundary set
    lptr<const int> idx1, idx2;
    GArr<T> cs;                // the coefficient set (run-time pattern)
    int ld;
};
// point accessor through the row pointers of a chunk
template <typename T, int R> struct ResAt {
    lptr<const T> (&r)[R];
    int t;
    int off;  // from the array the row pointers point into
    __device__ __forceinline__ T operator()(int di, int dj) const { return r[t + 1 + di][off + dj]; }
};
template <typename T> struct ResRow {
    lptr<const T> l, c, r;
    int off;
    __device__ __forceinline__ T operator[](int d) const { return (d < 0 ? l : d > 0 ? r : c)[off]; }
};

template <typename T, int PAT> __device__ __forceinline__ Stencil<T> res_stencil(const Prob<T> &p, const ResMem<T> &m, int i, int j)
{
    if constexpr (PAT != PAT_GENERIC)
        return stencil_xy<T, PAT>(p, m.xf, m.yf, i, j);
    else
        return stencil_at<T, PAT>(p, m.cs, i, j);
}

// S-line sweep (XLine's equations): KIND 0: u -> Y1; 1, 2, 3: CS, MCS, HV from (u, Y1, Y2) over Y1
template <typename T, int KIND, int PAT, int C>
__device__ __forceinline__ void res_xsweep(const Prob<T> *__restrict__ probs, int prob, const ResMem<T> &m)
{
    const Prob<T> &p = probs[opaque_uniform(prob)];
    const int tid = opaque_lane((int)threadIdx.x), wave = opaque_uniform(tid >> 6), sub = (tid & 63) >> 4, ll = tid & 15;
    const int N = p.nx - 2, lines = p.ny - 2, s = 1 + ll * C, kmax = N + 1, ld = m.ld;
    const T one = (T)1.0, theta = p.theta;
    for (int g = 4 * wave; g < lines; g += ARES_T / 16) {
        const int j = 1 + min(g + sub, lines - 1);
        const bool own = g + sub < lines;  // (a row of lanes without a line repeats its neighbour's)
        const int jj = m.idx2[j];
        const T lo = m.u[jj], hi = m.u[(N + 1) * ld + jj];
        lptr<const T> r[C + 2];  // rows s - 1 .. s + C, past the line's end row N + 1
        const int left = (kmax - (s - 1)) * ld;
#pragma unroll
        for (int t = 0; t < C + 2; ++t)
            r[t] = m.u + ((s - 1) * ld + j) + min(t * ld, left);
        const int o1 = (int)(m.y1 - m.u), o2 = KIND ? (int)(m.y2 - m.u) : 0;
        auto eq = [&](int t, int k) -> Eq<T> {
            const Stencil<T> st = res_stencil<T, PAT>(p, m, min(k, kmax), j);
            Eq<T> e;
            e.a = (-theta * st.M);
            e.b = (one + theta * st.Z);
            e.c = (-theta * st.P);
            typedef ResAt<T, C + 2> At;
            const At uq{r, t, 0}, y1q{r, t, o1}, y2q{r, t, o2};
            if constexpr (KIND == 0)
                e.r = rhs_intermed_1(p, st, uq);
            else if constexpr (KIND == 1)
                e.r = rhs_intermed_3<T, false>(p, st, uq, y1q, y2q);
            else if constexpr (KIND == 2)
                e.r = rhs_intermed_3<T, true>(p, st, uq, y1q, y2q);
            else
                e.r = (-theta * st.M * y2q(-1, 0)) + (theta * st.Z * y2q(0, 0)) - (theta * st.P * y2q(1, 0)) +
                      hv_y3_at(p, st, uq, y1q, y2q);
            if (k == 1) {
                e.r = e.r - e.a * lo;
                e.a = (T)0;
            }
            if (k >= N) {
                e.r = e.r - e.c * hi;
                e.c = (T)0;
            }
            return e;
        };
        lptr<T> out = m.y1 + (s * ld + j);
        row_solve<T, C>(N, ll, eq, [&](int t, T x) {
            if (own)
                out[t * ld] = x;
        });
        if (ll == 0 && own) {
            m.y1[j] = lo;
            m.y1[(N + 1) * ld + j] = hi;
        }
    }
}

// v-line sweep (vsweep_lines' equations): in and Y1 -> out
template <typename T, int PAT, int C>
__device__ __forceinline__ void res_vsweep(const Prob<T> *__restrict__ probs, int prob, const ResMem<T> &m,
                                           lptr<const T> in, lptr<T> out)
{
    const Prob<T> &p = probs[opaque_uniform(prob)];
    const int tid = opaque_lane((int)threadIdx.x), wave = opaque_uniform(tid >> 6), sub = (tid & 63) >> 4, ll = tid & 15;
    const int N = p.ny - 2, lines = p.nx - 2, s = 1 + ll * C, jmax = N + 1, ld = m.ld;
    const T one = (T)1.0, theta = p.theta;
    for (int g = 4 * wave; g < lines; g += ARES_T / 16) {
        const int i = 1 + min(g + sub, lines - 1);
        const bool own = g + sub < lines;
        const int ii = m.idx1[i];
        const T lo = m.cA0[ii], hi = m.cA1[ii];
        lptr<const T> r[C + 2];  // points s - 1 .. s + C, past the line's end point N + 1
#pragma unroll
        for (int t = 0; t < C + 2; ++t)
            r[t] = in + (i * ld + s - 1) + min(t, jmax - (s - 1));
        const int o1 = (int)(m.y1 - in);
        auto eq = [&](int t, int k) -> Eq<T> {
            const Stencil<T> st = res_stencil<T, PAT>(p, m, i, min(k, jmax));
            Eq<T> e;
            e.a = (-theta * st.Mt);
            e.b = (one + theta * st.W);
            e.c = (-theta * st.Pt);
            e.r = rhs_v(p, st, ResRow<T>{r[t], r[t + 1], r[t + 2], 0}, ResRow<T>{r[t], r[t + 1], r[t + 2], o1});
            if (k == 1) {
                e.r = e.r - e.a * lo;
                e.a = (T)0;
            }
            if (k >= N) {
                e.r = e.r - e.c * hi;
                e.c = (T)0;
            }
            return e;
        };
        lptr<T> o = out + (i * ld + s);
        row_solve<T, C>(N, ll, eq, [&](int t, T x) {
            if (own)
                o[t] = x;
        });
        if (ll == 0 && own) {
            out[i * ld] = lo;
            out[i * ld + N + 1] = hi;
        }
    }
}

// The v-lines' matrix, eliminated once: with the compile-time patterns b, e and f have no X factor, so it is the same
// for every line, and for every step when the coefficients do not change in time.  vt: per point the equation (a, b - 1,
// c) and rb = 1 / b', zq and g of Chunk; vc: per chunk a, c and 1 / b of the interface row before each reduction step, and
// the last 1 / b.  (Per step a v-sweep then costs its right-hand sides: 100 x 50 in fp64
// 8.7 -> 7.4 us a DR step.)
template <typename T, int PAT> constexpr bool res_same_vlines()
{
    if constexpr (PAT == PAT_GENERIC) {
        return false;
    } else {
        bool same = true;
        for (int q : {1, 4, 5})
            same = same && FPat<PAT>::c[2 * q] < 0 && FPat<PAT>::c[2 * q + 1] < 0;
        return same;
    }
}
template <typename T> struct VTab {
    lptr<T> vt, vc;
    int n;  // points: 16 chunks
    __device__ __forceinline__ lptr<T> at(int arr, int q) const { return vt + arr * n + q; }
    __device__ __forceinline__ lptr<T> level(int k, int ll) const { return vc + k * 16 + ll; }
};
template <typename T, int D> __device__ __forceinline__ Eq<T> res_vlevel(const VTab<T> &v, int k, int ll, bool st, const Eq<T> &e)
{
    if (st) {
        *v.level(3 * k, ll) = e.a;
        *v.level(3 * k + 1, ll) = e.c;
        *v.level(3 * k + 2, ll) = fast_rcp(e.b);
    }
    return row_pcr<D>(e);
}
// by the first wavefront
template <typename T, int PAT, int C>
__device__ __forceinline__ void res_vtable(const Prob<T> *__restrict__ probs, int prob, const ResMem<T> &m, const VTab<T> &v)
{
    const Prob<T> &p = probs[opaque_uniform(prob)];
    const int tid = opaque_lane((int)threadIdx.x), ll = tid & 15, N = p.ny - 2, s = 1 + ll * C;
    if (tid >= 64)
        return;
    const bool st = tid < 16;  // (the four rows of lanes do the same)
    const T one = (T)1.0, theta = p.theta;
    T g[C], zq[C], ae = (T)0, be = one, ce = (T)0;
#pragma unroll
    for (int t = 0; t < C; ++t) {
        const Stencil<T> sc = res_stencil<T, PAT>(p, m, 0, min(s + t, N + 1));
        T a = (-theta * sc.Mt), b = theta * sc.W, c = (-theta * sc.Pt);
        if (st) {
            *v.at(0, s - 1 + t) = a;
            *v.at(1, s - 1 + t) = b;
            *v.at(2, s - 1 + t) = c;
        }
        b = one + b;
        if (s > N)  // a chunk wholly past the end: identity rows
            a = c = (T)0, b = one;
        a = s + t == 1 ? (T)0 : a;
        c = s + t >= N ? (T)0 : c;
        if (t == C - 1) {
            ae = a, be = b, ce = c;
        } else {
            const T rb = fast_rcp(t == 0 ? b : b - a * g[t > 0 ? t - 1 : 0]);
            g[t] = c * rb;
            zq[t] = (t == 0 ? -a : -a * zq[t > 0 ? t - 1 : 0]) * rb;
            if (st)
                *v.at(3, s - 1 + t) = rb;
        }
    }
    T ql = one, rl = (T)0, QF = (T)0, RF = one;
    if constexpr (C >= 2) {
        g[C - 2] = -g[C - 2];
#pragma unroll
        for (int u = C - 3; u >= 0; --u) {
            const T gu = g[u];
            g[u] = -gu * g[u + 1];
            zq[u] = zq[u] - gu * zq[u + 1];
        }
        ql = zq[C - 2], rl = g[C - 2], QF = zq[0], RF = g[0];
        if (st) {
#pragma unroll
            for (int t = 0; t < C - 1; ++t) {
                *v.at(4, s - 1 + t) = zq[t];
                *v.at(5, s - 1 + t) = g[t];
            }
        }
    }
    Eq<T> e{ae * ql, (T)0, (T)0, (T)0};
    const T nQF = row_down<1>(QF), nRF = row_down<1>(RF);
    e.b = ae * rl + be + ce * nQF;
    e.c = ce * nRF;
    e = res_vlevel<T, 1>(v, 0, ll, st, e);
    e = res_vlevel<T, 2>(v, 1, ll, st, e);
    e = res_vlevel<T, 4>(v, 2, ll, st, e);
    e = res_vlevel<T, 8>(v, 3, ll, st, e);
    if (st)
        *v.level(12, ll) = fast_rcp(e.b);
}
template <typename T, int D> __device__ __forceinline__ T res_vreduce(const VTab<T> &v, int k, int ll, T r)
{
    const T a = *v.level(3 * k, ll), c = *v.level(3 * k + 1, ll), n = r * *v.level(3 * k + 2, ll);
    return r - a * row_up<D>(n) - c * row_down<D>(n);
}
// res_vsweep with the eliminated matrix
template <typename T, int C>
__device__ __forceinline__ void res_vsweep_tab(const Prob<T> *__restrict__ probs, int prob, const ResMem<T> &m, const VTab<T> &v,
                                               lptr<const T> in, lptr<T> out)
{
    const Prob<T> &p = probs[opaque_uniform(prob)];
    const int tid = opaque_lane((int)threadIdx.x), wave = opaque_uniform(tid >> 6), sub = (tid & 63) >> 4, ll = tid & 15;
    const int N = p.ny - 2, lines = p.nx - 2, s = 1 + ll * C, jmax = N + 1, ld = m.ld;
    for (int g = 4 * wave; g < lines; g += ARES_T / 16) {
        const int i = 1 + min(g + sub, lines - 1);
        const bool own = g + sub < lines;
        const int ii = m.idx1[i];
        const T lo = m.cA0[ii], hi = m.cA1[ii];
        const int o1 = (int)(m.y1 - in);
        T zp[C], re = (T)0, ae = (T)0, ce = (T)0;
        if (s <= N) {
            lptr<const T> q = in + (i * ld + s - 1);
            T left = q[0], mid = q[min(1, jmax - (s - 1))];
            T g0[C];
#pragma unroll
            for (int t = 0; t < C; ++t) {
                const int k = s + t;
                const T right = q[min(t + 2, jmax - (s - 1))];
                const T a = *v.at(0, k - 1), c = *v.at(2, k - 1);
                T r = (a * left) + (*v.at(1, k - 1) * mid) + (c * right) + q[o1 + min(t + 1, jmax - (s - 1))];
                if (k == 1)
                    r = r - a * lo;
                if (k >= N)
                    r = r - c * hi;
                const T cf = k >= N ? (T)0 : c;
                if (t == C - 1) {
                    re = r, ae = a, ce = cf;
                } else {
                    const T rb = *v.at(3, k - 1);
                    g0[t] = cf * rb;
                    zp[t] = (t == 0 ? r : r - a * zp[t > 0 ? t - 1 : 0]) * rb;
                }
                left = mid;
                mid = right;
            }
#pragma unroll
            for (int u = C - 3; u >= 0; --u)
                zp[u] = zp[u] - g0[u] * zp[u + 1];
        } else {
#pragma unroll
            for (int t = 0; t < C; ++t)
                zp[t] = (T)0;
        }
        const T pl = C >= 2 ? zp[C >= 2 ? C - 2 : 0] : (T)0, PF = C >= 2 ? zp[0] : (T)0;
        T r = re - ae * pl - ce * row_down<1>(PF);
        r = res_vreduce<T, 1>(v, 0, ll, r);
        r = res_vreduce<T, 2>(v, 1, ll, r);
        r = res_vreduce<T, 4>(v, 2, ll, r);
        r = res_vreduce<T, 8>(v, 3, ll, r);
        const T xi = r * *v.level(12, ll);
        const T xl = row_up<1>(xi);
        lptr<T> o = out + (i * ld + s);
        if (own) {
#pragma unroll
            for (int t = 0; t < C; ++t)
                if (s + t <= N)
                    o[t] = t == C - 1 ? xi : zp[t] + *v.at(4, s - 1 + t) * xl + *v.at(5, s - 1 + t) * xi;
            if (ll == 0) {
                out[i * ld] = lo;
                out[i * ld + N + 1] = hi;
            }
        }
    }
}

// the surface in LDS to or from HBM, a wavefront per row
template <typename T> __device__ __forceinline__ void res_store(gptr<T> dst, lptr<const T> u, int nx, int ny, int ld)
{
    for (int i = (int)threadIdx.x >> 6; i < nx; i += ARES_T / 64)
        for (int j = (int)threadIdx.x & 63; j < ny; j += 64)
            dst[i * ny + j] = u[i * ld + j];
}

// levels: null, or per problem where level s goes, for the s < steps that are multiples of `every`, one after the
// other; out: null (the last level stays where the step-by-step loop leaves it) or per problem where it goes.
// TWO: some problem has the second pair of stages.
template <typename T, int PAT, bool TWO>
__global__ void __launch_bounds__(ARES_T) k_adi_res(const Prob<T> *__restrict__ probs, const Tile *__restrict__ tiles,
                                                    const CopyJob *__restrict__ levels, int every,
                                                    const CopyJob *__restrict__ out)
{
    __shared__ T mem[ARES_BYTES / sizeof(T)];
    const Tile tl = tiles[blockIdx.x];
    const Prob<T> &p = probs[tl.prob];
    const int nx = p.nx, ny = p.ny, steps = p.steps, tid = (int)threadIdx.x, ld = ares_ld(nx, ny);
    const bool two = TWO && p.scheme != SCHEME_DR;
    constexpr int NVX = fpat_nvec<PAT>(0), NVY = fpat_nvec<PAT>(12);
    ResMem<T> m;
    m.ld = ld;
    lptr<T> at = (lptr<T>)mem;
    auto take = [&](int n) {
        const lptr<T> q = at;
        at += n;
        return q;
    };
    m.u = take(nx * ld);
    m.y1 = take(nx * ld);
    m.y2 = two ? take(nx * ld) : m.u;
    const lptr<T> xf = take(NVX * nx), yf = take(NVY * ny);
    m.xf = LArr<T>{xf};
    m.yf = LArr<T>{yf};
    m.cA0 = take(nx);
    m.cA1 = take(nx);
    m.bn = take(nx + 2 * ny);
    const VTab<T> v{take(ARES_VT * 16 * ares_chunk(ny)), take(ARES_VC * 16), 16 * ares_chunk(ny)};
    const lptr<int> ix = (lptr<int>)at;
    m.idx1 = ix;
    m.idx2 = ix + nx;
    const int n = nx * ny, cx = ares_chunk(nx), cv = ares_chunk(ny);
    {
        const gptr<const T> a = G((const T *)p.a);
        for (int i = tid >> 6; i < nx; i += ARES_T / 64)
            for (int j = tid & 63; j < ny; j += 64)
                m.u[i * ld + j] = a[i * ny + j];
        for (int i = tid; i < nx; i += ARES_T)
            ix[i] = (int)p.idx1[i];
        for (int j = tid; j < ny; j += ARES_T)
            ix[nx + j] = (int)p.idx2[j];
        // Y2's first and last row stay zero; Y1's end columns are read by the points past a line's end, which have to
        // be finite
        for (int q = tid; q < (two ? 2 : 1) * nx * ld; q += ARES_T)
            m.y1[q] = (T)0;
    }
    const gptr<T> lv = levels ? G((T *)levels[tl.prob].dst) : nullptr;
    auto vsweep = [&](lptr<const T> in, lptr<T> o) {
        if (res_same_vlines<T, PAT>() && p.coeff_sets == 1)
            with_length(cv, [&](auto c) { res_vsweep_tab<T, decltype(c)::value>(probs, tl.prob, m, v, in, o); });
        else
            with_length(cv, [&](auto c) { res_vsweep<T, PAT, decltype(c)::value>(probs, tl.prob, m, in, o); });
    };
    const T two_ = (T)2.0, three = (T)3.0, four = (T)4.0;
    for (int s = 0; s < steps; ++s) {
        m.cs = GArr<T>{coeff_set(p, s)};
        if (s == 0 || p.coeff_sets > 1 || p.bnd_sets > 1) {
            const gptr<const T> bs = bnd_set(p, s);
            for (int q = tid; q < NVX * nx; q += ARES_T)
                xf[q] = m.cs[(uint32_t)q];
            for (int q = tid; q < NVY * ny; q += ARES_T)
                yf[q] = m.cs[(uint32_t)(12 * nx + q)];
            for (int q = tid; q < nx + 2 * ny; q += ARES_T)
                m.bn[q] = bs[q];
            __syncthreads();
            if constexpr (res_same_vlines<T, PAT>()) {  // (read after the S-sweep's barrier)
                if (s == 0 && p.coeff_sets == 1)
                    with_length(cv, [&](auto c) { res_vtable<T, PAT, decltype(c)::value>(probs, tl.prob, m, v); });
            }
        }
        with_length(cx, [&](auto c) { res_xsweep<T, 0, PAT, decltype(c)::value>(probs, tl.prob, m); });
        {  // boundary stage A, from the last thread down
            const int i = ARES_T - 1 - tid;
            if (i < nx) {
                T D, E, F;
                if constexpr (PAT != PAT_GENERIC) {
                    D = sep<T, PAT, 3>(p, m.xf, m.yf, i, 0);
                    E = sep<T, PAT, 4>(p, m.xf, m.yf, i, 0);
                    F = sep<T, PAT, 5>(p, m.xf, m.yf, i, 0);
                } else {
                    def_row0<T, PAT>(p, m.cs, i, D, E, F);
                }
                const lptr<const T> ui = m.u + i * ld;
                m.cA0[i] = bnd_a_value(p, i, D, E, F, [&](int di, int dj) { return ui[di * ld + dj]; }, m.bn[nx],
                                       m.bn[nx + ny]);
                m.cA1[i] = m.bn[i];
            }
        }
        if (lv && s % every == 0)
            res_store<T>(lv + (size_t)(s / every) * n, m.u, nx, ny, ld);
        __syncthreads();
        vsweep(m.u, two ? m.y2 : m.y1);
        __syncthreads();
        if constexpr (TWO) {
            if (two) {
                with_length(cx, [&](auto c) {
                    if (p.scheme == SCHEME_CS)
                        res_xsweep<T, 1, PAT, decltype(c)::value>(probs, tl.prob, m);
                    else if (p.scheme == SCHEME_MCS)
                        res_xsweep<T, 2, PAT, decltype(c)::value>(probs, tl.prob, m);
                    else
                        res_xsweep<T, 3, PAT, decltype(c)::value>(probs, tl.prob, m);
                });
                __syncthreads();
                vsweep(p.scheme == SCHEME_HV ? m.y2 : m.u, m.y1);
                __syncthreads();
            }
        }
        if (tid < ny) {  // boundary stage B
            const lptr<T> w = m.y1;
            const int jj = m.idx2[tid];
            w[(nx - 1) * ld + tid] =
                (((four * w[(nx - 2) * ld + jj]) - w[(nx - 3) * ld + jj] - (two_ * p.h1 * m.bn[nx + ny + tid])) / three);
            w[tid] = m.bn[nx + tid];
        }
        __syncthreads();
        const lptr<T> z = m.u;
        m.u = m.y1;
        m.y1 = z;
    }
    if (lv && every == 1)
        res_store<T>(lv + (size_t)steps * n, m.u, nx, ny, ld);
    else
        res_store<T>(G(out ? (T *)out[tl.prob].dst : (steps & 1) ? p.b : p.a), m.u, nx, ny, ld);
}

}  // namespace lssamd

// Instantiations (one translation unit per precision and coefficient pattern)
#define LSS_INST_RES(T, PAT)                                                                                     \
    namespace lssamd {                                                                                           \
    template __global__ void k_adi_res<T, PAT, false>(const Prob<T> *, const Tile *, const CopyJob *, int,       \
                                                      const CopyJob *);                                          \
    template __global__ void k_adi_res<T, PAT, true>(const Prob<T> *, const Tile *, const CopyJob *, int,        \
                                                     const CopyJob *);                                           \
    }
