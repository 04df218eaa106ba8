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
//
// Memory bounds all three (5 values moved per unknown).  Measured on one MI355X, where a 4 + 4 GiB copy
// reaches 4.8 TB/s: rows 65536 x 256 fp64 5.4 TB/s; long 1000 x 2000 fp64 16.3 us (4.9 TB/s; one lane per
// system took 3380 us), 8388 x 2000 5.5 TB/s; cols 12289 x 509 fp32 38 us (3.3 TB/s; 53 us in launch
// order).

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

// Contiguous systems too long for one wavefront: one workgroup per system, a thread holds TRI_LONG_C
// consecutive unknowns.  All loads of the four arrays are coalesced rows of the workgroup, issued together;
// each array then passes through LDS once to reach the thread that owns its points (positions padded by one
// per chunk, so that neither side meets a bank conflict), so LDS holds one array and not four.  The interface
// system (one equation per thread) is reduced by cyclic reduction in the same LDS.
template <typename T, int NTMAX>
__global__ void __launch_bounds__(NTMAX) k_tridiag_long(int64_t B, int n, const T *__restrict__ a,
                                                        const T *__restrict__ b, const T *__restrict__ c,
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
    Chunk<T, C> ch;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int k = t * C + j;
        Eq<T> e;
        e.a = va[j];
        e.b = vb[j];
        e.c = vc[j];
        e.r = vd[j];
        bc.fold(k == 0, k == nf - 1, e.a, e.b, e.c, e.r);
        if (k >= nf)
            e = identity_eq<T>();
        ch.put(j, e);
    }
    ch.bwd();
    {
        T PF, QF, RF;
        ch.first_rel(PF, QF, RF);
        __syncthreads();
        sh[t] = PF;
        sh[nt + t] = QF;
        sh[2 * nt + t] = RF;
    }
    __syncthreads();
    // (a thread without a neighbour reads its own row: its coupling to that side is exactly zero)
    const int tn = t + 1 < nt ? t + 1 : t;
    Eq<T> e = ch.interface_eq(sh[tn], sh[nt + tn], sh[2 * nt + tn]);
    T *cur = sh + 3 * nt, *oth = sh;
    {
        const NEq<T> m = normalized(e);
        cur[t] = m.a;
        cur[nt + t] = m.c;
        cur[2 * nt + t] = m.r;
    }
    __syncthreads();
    for (int dd = 1; dd < nt; dd <<= 1) {
        const int tl = t >= dd ? t - dd : t, th = t + dd < nt ? t + dd : t;
        NEq<T> l, h;
        l.a = cur[tl];
        l.c = cur[nt + tl];
        l.r = cur[2 * nt + tl];
        h.a = cur[th];
        h.c = cur[nt + th];
        h.r = cur[2 * nt + th];
        e = pcr_step(e, l, h);
        T *s = cur;
        cur = oth;
        oth = s;
        const NEq<T> m = normalized(e);
        cur[t] = m.a;
        cur[nt + t] = m.c;
        cur[2 * nt + t] = m.r;
        __syncthreads();
    }
    const T xi = e.r * fast_rcp(e.b);
    oth[t] = xi;
    __syncthreads();
    const T xl = oth[t > 0 ? t - 1 : 0];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C; ++j)
        sh[t * (C + 1) + j] = ch.value(j, xl, xi);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int q = j * nt + t;
        if (q < nf)
            x[base + s0 + q] = sh[q + q / C];
    }
    if (t == 0) {
        if (bc.lo == BC_DIRICHLET)
            x[base] = bc.lo_val;
        if (bc.hi == BC_DIRICHLET)
            x[base + n - 1] = bc.hi_val;
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
LSS_INST_C(double, 16, 4, 128)
LSS_INST_C(float, 2, 32, 32)
LSS_INST_C(float, 4, 32, 32)
LSS_INST_C(float, 8, 32, 32)
LSS_INST_C(float, 1, 16, 64)
LSS_INST_C(float, 2, 16, 64)
LSS_INST_C(float, 4, 16, 64)
LSS_INST_C(float, 8, 16, 64)
LSS_INST_C(float, 16, 16, 64)
LSS_INST_C(float, 16, 8, 128)
#undef LSS_INST_R
#undef LSS_INST_C
#undef LSS_INST_L
#undef LSS_INST_T

}  // namespace lssamd
