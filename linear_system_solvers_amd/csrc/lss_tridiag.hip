// lss_tridiag.hip -- batched plain tridiagonal systems for gfx950 with the register-resident
// partitioned elimination (no scratch arrays in HBM: every input is read once, the solution
// written once).
//
// System k has unknowns x_0..x_{n-1} and rows a_i x_{i-1} + b_i x_i + c_i x_{i+1} = d_i, whose end rows
// are folded with the end conditions `bc` (LineBC: Dirichlet / Neumann / Robin as the reference's
// thomas_lu_boundary.hpp:114-205 folds them, or PLAIN: a_0 and c_{n-1} ignored).  The folded system
// has unknowns start..end; Dirichlet end values are written to x_0 / x_{n-1}.
//   k_tridiag_rows  contiguous layout x[k*n + i]: one wavefront per system; the system is staged
//                   through LDS so that every global access is a coalesced row of the system.
//   k_tridiag_long  contiguous systems too long for one wavefront: one workgroup per system.
//   k_tridiag_cols  strided layout x[i*B + k]: W systems x NC chunks per workgroup, so that each access
//                   reads W consecutive systems of one row.
//   k_tridiag_cols_long  the same for more than 1024 unknowns.
//
// Memory bounds them (5 values moved per unknown), the long ones also the registers of their last pass.  Measured on
// one MI355X, where a 4 + 4 GiB copy reaches 4.8 TB/s: rows 65536 x 256 fp64 5.4 TB/s; long 1000 x 2000 fp64 19.2 us
// (4.2 TB/s; one lane per system took 3380 us), 8388 x 2000 131 us (5.1 TB/s); cols 12289 x 509 fp32 38 us (3.3 TB/s;
// 53 us in launch order).

// The fast path may fuse multiply-adds (the library is built with -ffp-contract=off so that the exact
// line solver keeps the reference's rounding; this translation unit opts back in).
#pragma clang fp contract(fast)
#include "lss_adi_chunk.hpp"

namespace lssamd {

constexpr int TRI_WAVES = 4;  // systems per workgroup of k_tridiag_rows

template <typename T, int M>
__global__ void __launch_bounds__(64 * TRI_WAVES) k_tridiag_rows(int64_t B, int n, const T *__restrict__ a,
                                                                  const T *__restrict__ b, const T *__restrict__ c,
                                                                  const T *__restrict__ d, T *__restrict__ x,
                                                                  LineBC<T> bc)
{
    extern __shared__ unsigned char lds_raw[];
    T *lds = reinterpret_cast<T *>(lds_raw);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t k = (int64_t)blockIdx.x * TRI_WAVES + wave;
    const bool live = k < B;
    T *sa = lds + (size_t)wave * 4 * n, *sb = sa + n, *sc = sb + n, *sd = sc + n;
    if (live) {
        const int64_t base = k * n;
        for (int i = lane; i < n; i += 64) {
            sa[i] = a[base + i];
            sb[i] = b[base + i];
            sc[i] = c[base + i];
            sd[i] = d[base + i];
        }
    }
    __syncthreads();
    const int s0 = bc.start(), e0 = bc.end(n), nf = e0 - s0 + 1;
    if (live) {
        auto eq = [&](int kk) -> Eq<T> {
            const int i = s0 + min(kk, nf) - 1;  // points past the end repeat the last equation
            Eq<T> e;
            e.a = sa[i];
            e.b = sb[i];
            e.c = sc[i];
            e.r = sd[i];
            bc.fold(i == s0, i == e0, e.a, e.b, e.c, e.r);
            return e;
        };
        auto put = [&](int, int kk, T v) { sd[s0 + kk - 1] = v; };  // every eq() has run before the first put()
        wave_solve<T, M>(nf, lane, eq, put);
        if (lane == 0) {
            if (bc.lo == BC_DIRICHLET)
                sd[0] = bc.lo_val;
            if (bc.hi == BC_DIRICHLET)
                sd[n - 1] = bc.hi_val;
        }
    }
    __syncthreads();
    if (live) {
        const int64_t base = k * n;
        for (int i = lane; i < n; i += 64)
            x[base + i] = sd[i];
    }
}

// W systems x NC chunks of at most M points per workgroup.  Neighbouring workgroups share the cache lines at
// the edges of their rows (all of them when B is odd), so each XCD takes a contiguous run of workgroups and
// meets the shared lines in its own L2: 12289 x 509 in fp32 goes from 53 to 38 us by that alone.
template <typename T, int M, int W, int NC>
__global__ void __launch_bounds__(W *NC) k_tridiag_cols(int64_t B, int n, const T *__restrict__ a,
                                                        const T *__restrict__ b, const T *__restrict__ c,
                                                        const T *__restrict__ d, T *__restrict__ x, LineBC<T> bc)
{
    __shared__ T sh[2][4][NC][W];
    const int col = threadIdx.x % W, chn = threadIdx.x / W;
    const int64_t k = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * W + col;
    const bool live = k < B;
    const int s0 = bc.start(), e0 = bc.end(n), nf = e0 - s0 + 1;
    auto eq = [&](int kk) -> Eq<T> {
        const int i = s0 + min(kk, nf) - 1;  // points past the end repeat the last equation
        const int64_t q = (int64_t)i * B + k;
        Eq<T> e;
        e.a = a[q];
        e.b = b[q];
        e.c = c[q];
        e.r = d[q];
        bc.fold(i == s0, i == e0, e.a, e.b, e.c, e.r);
        return e;
    };
    auto put = [&](int, int kk, T v) { x[(int64_t)(s0 + kk - 1) * B + k] = v; };
    block_solve<T, M, W, false, NC>(sh, nf, col, chn, live, eq, put);
    if (live && chn == 0) {
        if (bc.lo == BC_DIRICHLET)
            x[k] = bc.lo_val;
        if (bc.hi == BC_DIRICHLET)
            x[(int64_t)(n - 1) * B + k] = bc.hi_val;
    }
}

// -------------------------------------------------------------------------------------------------
// Long systems: a workgroup holds W systems, position pos of a system (np of them) the C consecutive unknowns from
// pos * C on.  The chunks are eliminated and their interface system (one equation per position) is reduced by cyclic
// reduction in LDS; the solution is then put through every row once more,
//     x_k = (d_k - a_k x_{k-1} - c_k x_{k+1}) / b_k,
// which takes away the rounding error that the chunks' three-term relations leave: with rows of |b| = 2.5 + |a| + |c|
// the root mean square against a longer format is 0.9 of the sequential sweep's (1.2 to 1.3 of it without that pass),
// in both precisions, 513 to 8192 unknowns.  Without the pass 1000 x 2000 in fp64 takes 16.1 us, with it 19.2.
//
// All this is sound while the rows dominate, |a| + |c| <= |b|: then so do the rows that any elimination leaves, in
// whatever order, no multiplier exceeds 1 and the last pass cannot amplify an error.  A system with a row that does not
// dominate, or whose diagonal leaves the range that fast_rcp and a few sums need, is swept as the reference sweeps it
// instead, with divisions, position after position (the result of one lane per system, bit for bit).  The threads
// still share the loads and the other systems' work: 1000 systems of 2000 unknowns in fp64 take 0.50 ms, 8388 of them
// 3.2 ms (one lane per system: 3.5 and 3.7), interleaved 0.27 and 2.1 ms (1.6 and 2.05).
// -------------------------------------------------------------------------------------------------
__device__ __forceinline__ bool dominates(double a, double b, double c)
{
    const double m = fabs(b);
    return (fabs(a) + fabs(c) <= m * (1 + 0x1p-49)) & (m >= 0x1p-900) & (m <= 0x1p900);
}
__device__ __forceinline__ bool dominates(float a, float b, float c)
{
    const float m = fabsf(b);
    return (fabsf(a) + fabsf(c) <= m * (1 + 0x1p-20f)) & (m >= 0x1p-100f) & (m <= 0x1p100f);
}
// the last pass: an unknown from its row and its neighbours
__device__ __forceinline__ double closing(const Eq<double> &e, double left, double right)
{
    const double r = e.r - e.a * left - e.c * right, y = fast_rcp(e.b), q = r * y;
    return __builtin_fma(__builtin_fma(-e.b, q, r), y, q);
}
__device__ __forceinline__ float closing(const Eq<float> &e, float left, float right)
{
    const float r = e.r - e.a * left - e.c * right, y = fast_rcp(e.b), q = r * y;
    return __builtin_fmaf(__builtin_fmaf(-e.b, q, r), y, q);
}

// Zero, of which the compiler does not know: rows at an offset from it are read again (from the caches), not kept in
// registers from the elimination on.
__device__ __forceinline__ int opaque_zero()
{
    int v = 0;
    asm volatile("" : "+s"(v));
    return v;
}

// LDS values of long_solve: six per position and system, and a flag per system, not 0 if it is to be swept
__host__ __device__ constexpr int long_lds(int np, int W) { return (6 * np + 1) * W; }
template <typename T> __device__ __forceinline__ T *long_flag(T *sh, int np, int W) { return sh + 6 * np * W; }

// The sequential sweep of the systems of which `mine` is set (thomas_lu_solver.hpp:125-191)
template <typename T, int C, typename Row>
__device__ __forceinline__ void long_sweep(T *sh, int W, int pos, int col, int nf, bool mine, Row &&row, T (&x)[C])
{
#pragma clang fp contract(off)
    const int npos = (nf + C - 1) / C;
    Eq<T> e[C];  // at hand before the position's turn comes; c becomes gamma
    if (mine) {
#pragma unroll
        for (int j = 0; j < C; ++j)
            e[j] = row(j);
    }
    __syncthreads();
    for (int p = 0; p < npos; ++p) {
        if (mine && pos == p) {
            T gk = p ? sh[col] : (T)0, sk = p ? sh[W + col] : (T)0;
#pragma unroll
            for (int j = 0; j < C; ++j) {
                if (p * C + j >= nf)
                    continue;
                const T beta = e[j].b - (e[j].a * gk);
                e[j].c = gk = e[j].c / beta;
                x[j] = sk = (e[j].r - (e[j].a * sk)) / beta;
            }
            sh[col] = gk;
            sh[W + col] = sk;
        }
        __syncthreads();
    }
    for (int p = npos - 1; p >= 0; --p) {
        if (mine && pos == p) {
            T xk = sh[2 * W + col];
#pragma unroll
            for (int j = C - 1; j >= 0; --j) {
                if (p * C + j >= nf)
                    continue;
                if (p * C + j < nf - 1)
                    x[j] = x[j] - (e[j].c * xk);
                xk = x[j];
            }
            sh[2 * W + col] = xk;
        }
        __syncthreads();
    }
}

// Solves for the unknowns x of position pos, whose rows are row(0) .. row(C - 1) (ends folded, identity rows past the
// end; not asked for where `holds` is not set: a position without rows), and the unknowns to the left and to the right
// of them.  Every thread of the workgroup calls it (it holds barriers); sh may be in use by the caller until then.
// Returns whether some system of the workgroup is flagged.
template <typename T, int C, typename Row>
__device__ __forceinline__ bool long_solve(T *sh, int np, int W, int pos, int col, bool holds, Row &&row, T (&x)[C],
                                           T &left, T &right)
{
    const int st = np * W, at = pos * W + col;
    T *const flag = long_flag(sh, np, W);
    const int prev = pos > 0 ? at - W : at, next = pos + 1 < np ? at + W : at;
    T nPF, nQF, nRF, xl, xi, xr;
    {
        Chunk<T, C> ch;
        bool good = true;
        if (holds) {
#pragma unroll
            for (int j = 0; j < C; ++j) {
                const Eq<T> e = row(j);
                good &= dominates(e.a, e.b, e.c);
                ch.put(j, e);
            }
            ch.bwd();
        } else {
            ch.set_identity();
        }
        T PF, QF, RF;
        ch.first_rel(PF, QF, RF);
        __syncthreads();
        sh[at] = PF;
        sh[st + at] = QF;
        sh[2 * st + at] = RF;
        if (pos == 0)
            flag[col] = (T)0;
        __syncthreads();
        if (!good)
            flag[col] = (T)1;
        // (a position without a neighbour reads its own row: its coupling to that side is exactly zero)
        nPF = sh[next], nQF = sh[st + next], nRF = sh[2 * st + next];
        Eq<T> e = ch.interface_eq(nPF, nQF, nRF);
        T *cur = sh + 3 * st, *oth = sh;
        {
            const NEq<T> m = normalized(e);
            cur[at] = m.a;
            cur[st + at] = m.c;
            cur[2 * st + at] = m.r;
        }
        __syncthreads();
        for (int dd = 1; dd < np; dd <<= 1) {
            const int tl = pos >= dd ? at - dd * W : at, th = pos + dd < np ? at + dd * W : at;
            const NEq<T> l{cur[tl], cur[st + tl], cur[2 * st + tl]}, h{cur[th], cur[st + th], cur[2 * st + th]};
            e = pcr_step(e, l, h);
            T *s = cur;
            cur = oth;
            oth = s;
            const NEq<T> m = normalized(e);
            cur[at] = m.a;
            cur[st + at] = m.c;
            cur[2 * st + at] = m.r;
            __syncthreads();
        }
        xi = e.r * fast_rcp(e.b);
        oth[at] = xi;
        __syncthreads();
        xl = oth[prev];
        xr = oth[next];
#pragma unroll
        for (int j = 0; j < C; ++j)
            x[j] = ch.value(j, xl, xi);
    }
    left = xl;
    right = nPF + nQF * xi + nRF * xr;
    bool any = false;
    for (int w = 0; w < W; ++w)
        any = any || flag[w] != (T)0;
    return any;
}

constexpr int LONG_CLOSE = 4;  // rows that are read again at a time

// Contiguous systems too long for one wavefront: one workgroup per system.  All loads of the four arrays are coalesced
// rows of the workgroup, issued together; each array then passes through LDS once to reach the thread that owns its
// points (positions padded by one per chunk, so that neither side meets a bank conflict), so LDS holds one array and not
// four.  The rows stay in registers for the last pass where that leaves three wavefronts a SIMD (fp64 up to 2048
// unknowns: 21 us against 23 with rows read again, 1000 x 2000 beyond the caches); longer fp64 systems read them again
// (1000 x 4000: 49 us against 85 with spills).
template <typename T, int NTMAX>
__global__ void __launch_bounds__(NTMAX) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && NTMAX <= 256 ? 3 : 1)))
k_tridiag_long(int64_t B, int n, const T *__restrict__ a, const T *__restrict__ b, const T *__restrict__ c,
               const T *__restrict__ d, T *__restrict__ x, LineBC<T> bc)
{
    constexpr int C = TRI_LONG_C;
    extern __shared__ unsigned char lds_raw[];
    T *sh = reinterpret_cast<T *>(lds_raw);  // (C + 1) values per thread
    const int nt = (int)blockDim.x, t = (int)threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * n;
    const int s0 = bc.start(), e0 = bc.end(n), nf = e0 - s0 + 1;
    T va[C], vb[C], vc[C], vd[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int64_t q = base + s0 + min(j * nt + t, nf - 1);  // points past the end repeat the last row
        va[j] = a[q];
        vb[j] = b[q];
        vc[j] = c[q];
        vd[j] = d[q];
    }
    auto spread = [&](T(&v)[C]) {  // row order -> the thread's own points t * C + j
        __syncthreads();
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const int q = j * nt + t;
            sh[q + q / C] = v[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < C; ++j)
            v[j] = sh[t * (C + 1) + j];
    };
    spread(va);
    spread(vb);
    spread(vc);
    spread(vd);
    auto own = [&](int j) {
        const int k = t * C + j;
        Eq<T> e{va[j], vb[j], vc[j], vd[j]};
        bc.fold(k == 0, k == nf - 1, e.a, e.b, e.c, e.r);
        return k < nf ? e : identity_eq<T>();
    };
    T v[C], left, right;
    const bool sweep = long_solve<T, C>(sh, nt, 1, t, 0, t * C < nf, own, v, left, right);
    constexpr bool KEEP = NTMAX <= 256 || sizeof(T) == 4;
    auto again = [&](int k, int64_t from) {
        const int64_t q = from + min(k, nf - 1);
        Eq<T> e{a[q], b[q], c[q], d[q]};
        bc.fold(k == 0, k >= nf - 1, e.a, e.b, e.c, e.r);
        return e;
    };
    if (sweep) {
        if constexpr (KEEP)
            long_sweep<T, C>(sh, 1, t, 0, nf, true, own, v);
        else
            long_sweep<T, C>(sh, 1, t, 0, nf, true, [&](int j) { return again(t * C + j, base + s0 + opaque_zero()); }, v);
    } else if constexpr (KEEP) {
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const T mid = v[j];
            v[j] = closing(own(j), left, j < C - 1 ? v[j < C - 1 ? j + 1 : j] : right);
            left = mid;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C; ++j)
        sh[t * (C + 1) + j] = v[j];
    __syncthreads();
    auto at = [&](int k) { return sh[k + k / C]; };
    const int64_t from = base + s0 + opaque_zero();
#pragma unroll LONG_CLOSE
    for (int j = 0; j < C; ++j) {
        const int q = j * nt + t;
        T z = at(q);
        if constexpr (!KEEP) {
            if (!sweep)
                z = closing(again(q, from), at(max(q - 1, 0)), at(min(q + 1, C * nt - 1)));
        }
        if (q < nf)
            x[base + s0 + q] = z;
    }
    if (t == 0) {
        if (bc.lo == BC_DIRICHLET)
            x[base] = bc.lo_val;
        if (bc.hi == BC_DIRICHLET)
            x[base + n - 1] = bc.hi_val;
    }
}

// Interleaved systems of more than 1024 unknowns: W systems per workgroup, NC positions of C unknowns each.  fp32 keeps
// its rows for the last pass (8388 x 2000: 141 us against 170 with rows read again), fp64 reads them again (320 us; kept
// they spill); without the pass 116 and 210 us.
template <typename T, int C, int W, int NC>
__global__ void __launch_bounds__(W *NC) k_tridiag_cols_long(int64_t B, int n, const T *__restrict__ a,
                                                             const T *__restrict__ b, const T *__restrict__ c,
                                                             const T *__restrict__ d, T *__restrict__ x, LineBC<T> bc)
{
    __shared__ T sh[long_lds(NC, W)];
    const int col = threadIdx.x % W, pos = threadIdx.x / W;
    const int64_t k = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * W + col;
    const bool live = k < B;
    const int s0 = bc.start(), e0 = bc.end(n), nf = e0 - s0 + 1;
    const bool holds = live && pos * C < nf;
    auto load = [&](int j, int64_t at) {
        const int i = pos * C + j;
        const int64_t q = (int64_t)(s0 + min(i, nf - 1)) * B + at;
        Eq<T> e{a[q], b[q], c[q], d[q]};
        bc.fold(i == 0, i >= nf - 1, e.a, e.b, e.c, e.r);  // (past the end the last row again, its c zero too)
        return e;
    };
    constexpr bool KEEP = sizeof(T) == 4;
    Eq<T> rows[KEEP ? C : 1];
    if constexpr (KEEP) {
        if (holds) {
#pragma unroll
            for (int j = 0; j < C; ++j)
                rows[KEEP ? j : 0] = load(j, k);
        }
    }
    auto row = [&](int j, int64_t at) { return KEEP ? rows[KEEP ? j : 0] : load(j, at); };
    T v[C], left, right;
    const bool any = long_solve<T, C>(sh, NC, W, pos, col, holds, [&](int j) { return row(j, k); }, v, left, right);
    const bool mine = holds && long_flag(sh, NC, W)[col] != (T)0;
    if (holds && !mine) {
        const int64_t kz = k + opaque_zero();
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const T mid = v[j];
            v[j] = closing(row(j, kz), left, j < C - 1 ? v[j < C - 1 ? j + 1 : j] : right);
            left = mid;
            if (!KEEP && j % LONG_CLOSE == LONG_CLOSE - 1)
                __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (any)
        long_sweep<T, C>(sh, W, pos, col, nf, mine, [&](int j) { return row(j, k + opaque_zero()); }, v);
    if (!live)
        return;
#pragma unroll
    for (int j = 0; j < C; ++j)
        if (pos * C + j < nf)
            x[(int64_t)(s0 + pos * C + j) * B + k] = v[j];
    if (pos == 0) {
        if (bc.lo == BC_DIRICHLET)
            x[k] = bc.lo_val;
        if (bc.hi == BC_DIRICHLET)
            x[(int64_t)(n - 1) * B + k] = bc.hi_val;
    }
}

#define LSS_INST_R(T, M) \
    template __global__ void k_tridiag_rows<T, M>(int64_t, int, const T *, const T *, const T *, const T *, T *, LineBC<T>);
#define LSS_INST_C(T, M, W, NC)                                                                                     \
    template __global__ void k_tridiag_cols<T, M, W, NC>(int64_t, int, const T *, const T *, const T *, const T *, T *, \
                                                         LineBC<T>);
#define LSS_INST_L(T, NTMAX)                                                                                         \
    template __global__ void k_tridiag_long<T, NTMAX>(int64_t, int, const T *, const T *, const T *, const T *, T *, \
                                                      LineBC<T>);
#define LSS_INST_CL(T, C, W, NC)                                                                                         \
    template __global__ void k_tridiag_cols_long<T, C, W, NC>(int64_t, int, const T *, const T *, const T *, const T *, \
                                                              T *, LineBC<T>);
#define LSS_INST_T(T)                                                                                               \
    LSS_INST_R(T, 1) LSS_INST_R(T, 2) LSS_INST_R(T, 4) LSS_INST_R(T, 8) LSS_INST_R(T, 16) LSS_INST_L(T, 256) \
    LSS_INST_L(T, 1024)
LSS_INST_T(double)
LSS_INST_T(float)
LSS_INST_C(double, 1, 16, 64)
LSS_INST_C(double, 2, 16, 64)
LSS_INST_C(double, 4, 16, 64)
LSS_INST_C(double, 8, 8, 64)
LSS_INST_C(double, 8, 8, 128)
LSS_INST_C(float, 2, 32, 32)
LSS_INST_C(float, 4, 32, 32)
LSS_INST_C(float, 8, 32, 32)
LSS_INST_C(float, 1, 16, 64)
LSS_INST_C(float, 2, 16, 64)
LSS_INST_C(float, 4, 16, 64)
LSS_INST_C(float, 8, 16, 64)
LSS_INST_C(float, 16, 16, 64)
LSS_INST_CL(double, 16, 4, 128)
LSS_INST_CL(float, 16, 8, 128)
#undef LSS_INST_R
#undef LSS_INST_C
#undef LSS_INST_CL
#undef LSS_INST_L
#undef LSS_INST_T

}  // namespace lssamd
