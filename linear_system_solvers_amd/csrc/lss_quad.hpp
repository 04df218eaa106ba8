// lss_quad.hpp -- exchange inside a quad of lanes, for the kernels that pass a sequential line sweep through
// four lanes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace lssamd {

// Lane i of a quad takes lane (CTRL >> 2i) & 3's value (DPP quad_perm).
template <int CTRL> __device__ __forceinline__ int quad_mov(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL> __device__ __forceinline__ float quad_perm(float v)
{
    return __int_as_float(quad_mov<CTRL>(__float_as_int(v)));
}
template <int CTRL> __device__ __forceinline__ double quad_perm(double v)
{
    return __hiloint2double(quad_mov<CTRL>(__double2hiint(v)), quad_mov<CTRL>(__double2loint(v)));
}
constexpr int QUAD_UP = 0x90, QUAD_DOWN = 0xf9;            // lane q takes lane q - 1's / q + 1's
template <int Q> constexpr int QUAD_BCAST = Q * 0x55;      // every lane takes lane Q's

// -------------------------------------------------------------------------------------------------
// Division by a divisor that is known before its numerator.  With y = RN(1 / b) and z = y (1 - b y), a y + a z is
// a / b to twice the precision, so its rounding q is faithful, and one residual step makes it RN(a / b)
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34,
// 1990: q' = RN(q + r y) with r = a - b q is the correctly rounded quotient when q is faithful and
// y = RN(1 / b)).  Four dependent operations instead of the ten of an IEEE division.  It holds while no
// intermediate value leaves the normal range: the exponents of a and b are bounded so that 1 / b, the quotients
// and the residuals (multiples of ulp(b) ulp(q)) are normal or exact.  A numerator of +0 gives +0, which is right for
// positive divisors (a y = +0, and +0 + a z = +0 for either sign of z); for negative ones it would depend on the sign
// of z, so they take the division, as everything else does.
// -------------------------------------------------------------------------------------------------
// sign and exponent (a negative number lies above every positive one)
__device__ __forceinline__ uint32_t sign_exponent(double x) { return (uint32_t)__double2hiint(x) >> 20; }
__device__ __forceinline__ uint32_t sign_exponent(float x) { return __float_as_uint(x) >> 23; }
// divisors from 2^-100 to below 2^101 (fp32: 2^-20 to below 2^21), numerators from +-2^-900 to below 2^900 (2^-90, 2^90)
// or +0
__device__ __forceinline__ bool quick_div_ok(double b) { return sign_exponent(b) - (1023u - 100u) <= 200u; }
__device__ __forceinline__ bool quick_div_ok(float b) { return sign_exponent(b) - (127u - 20u) <= 40u; }
// y = RN(1 / b) and its correction z = y (1 - b y)
__device__ __forceinline__ double quick_div(double a, double b, double y, double z)
{
    const double q = __builtin_fma(a, y, a * z);
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
__device__ __forceinline__ float quick_div(float a, float b, float y, float z)
{
    const float q = __builtin_fmaf(a, y, a * z);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ double quick_rcp_low(double b, double y) { return y * __builtin_fma(-b, y, 1.0); }
__device__ __forceinline__ float quick_rcp_low(float b, float y) { return y * __builtin_fmaf(-b, y, 1.0f); }

// The sequential sweeps of a quad.  A group is 16 points, four per lane, lane 0 first.  The recurrence runs
// four times in all four lanes at once, each lane starting from its neighbour's last value: after the k-th time
// the first k lanes hold their final values (and keep them: they start from the same value again), so the fourth
// is complete without a branch or a mask, and other work can be scheduled between the dependent operations.
// A value depends on exactly the operations of the sequential sweep, in its order.

// Groups g0, g0 + dg, ... (ng of them) through body(g, stage), each loaded QUAD_AHEAD groups before its turn.
// The stages take turns in place: a stage that moved from variable to variable would have to arrive before it could
// be copied, and a path that skips a group on the way to the loop's head would leave the loads of the next stage
// the youngest; both turn the wait for one stage into a wait for everything in flight.
constexpr int QUAD_AHEAD = 2;
template <typename Stage, typename Load, typename Body>
__device__ __forceinline__ void quad_stages(int g0, int ng, int dg, Load &&load, Body &&body)
{
    auto at = [&](int k) { return g0 + dg * min(k, ng - 1); };
    Stage s0, s1;
    load(at(0), s0);
    load(at(1), s1);
    for (int k = 0;;) {
        body(at(k), s0);
        load(at(k + QUAD_AHEAD), s0);
        if (++k == ng)
            break;
        body(at(k), s1);
        load(at(k + QUAD_AHEAD), s1);
        if (++k == ng)
            break;
    }
}

// s_t = (f_t - a_t s_{t-1}) / beta_t, y = RN(1 / beta) (NaN for a divisor outside quick_div's range), carry = the s
// before the group; returns the group's last s.  `seen` gathers the numerators and each lane's last quotient: while
// seen_ok() every value is the correctly rounded quotient, otherwise the sweep has to run again with QUICK = false
// (divisions) from a carry that was found good.  A divisor outside the range makes its own quotient NaN; inside a lane
// the next point's numerator shows that, and the lane's last quotient has to be looked at itself (the group's last one
// meets no other numerator of the group).
struct SeenNum {
    uint32_t lo = 0xffffffffu, hi = 0;  // range of the high words without their sign (a zero counts in neither)
    int32_t sg = 0;                     // smallest high word as an integer: INT32_MIN means -0
    __device__ __forceinline__ void add(double v)
    {
        add_word((uint32_t)__double2hiint(v), __double2loint(v) == 0 ? 1u : 0u);
    }
    __device__ __forceinline__ void add(float v) { add_word(__float_as_uint(v), 1u); }
    __device__ __forceinline__ void add_word(uint32_t w, uint32_t one)  // one: takes a zero below the smallest number
    {
        const uint32_t m = (w & 0x7fffffffu) - one;
        lo = min(lo, m);
        hi = max(hi, m + 1u);
        sg = min(sg, (int32_t)w);
    }
    // a quotient: only NaN counts (and what lies far above the numerators' range)
    __device__ __forceinline__ void add_quotient(double v) { hi = max(hi, (uint32_t)__double2hiint(v) & 0x7fffffffu); }
    __device__ __forceinline__ void add_quotient(float v) { hi = max(hi, __float_as_uint(v) & 0x7fffffffu); }
};
__device__ __forceinline__ bool seen_ok(const SeenNum &s, double)
{
    return s.lo >= ((1023u - 900u) << 20) - 1u && s.hi < (1023u + 900u) << 20 && s.sg != INT32_MIN;
}
__device__ __forceinline__ bool seen_ok(const SeenNum &s, float)
{
    return s.lo >= ((127u - 90u) << 23) - 1u && s.hi < (127u + 90u) << 23 && s.sg != INT32_MIN;
}
template <bool QUICK, typename T>
__device__ __forceinline__ T quad_forward(const T (&a)[4], const T (&f)[4], const T (&beta)[4], const T (&y)[4], T carry,
                                          T (&x)[4], SeenNum &seen)
{
    const bool first = ((int)threadIdx.x & 3) == 0;
    T c = carry;
    if constexpr (QUICK) {
        T z[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            z[j] = quick_rcp_low(beta[j], y[j]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            T sv = c, num[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                num[j] = f[j] - (a[j] * sv);
                x[j] = sv = quick_div(num[j], beta[j], y[j], z[j]);
            }
            if (k < 3) {
                const T up = quad_perm<QUAD_UP>(x[3]);
                c = first ? carry : up;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    seen.add(num[j]);
                seen.add_quotient(x[3]);
            }
        }
    } else {
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
            T sv = c;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                x[j] = sv = (f[j] - (a[j] * sv)) / beta[j];
            const T up = quad_perm<QUAD_UP>(x[3]);
            c = first ? carry : up;
        }
    }
    return quad_perm<QUAD_BCAST<3>>(x[3]);
}
template <typename T> __device__ __forceinline__ T quick_rcp(T beta)
{
    return quick_div_ok(beta) ? (T)1.0 / beta : (T)__builtin_nanf("");
}

// beta_t = b_t - a_t gamma_{t-1}, gamma_t = c_t / beta_t, carry = the gamma before the group; returns its last gamma
template <typename T>
__device__ __forceinline__ T quad_gamma(const T (&a)[4], const T (&b)[4], const T (&c)[4], T carry, T (&beta)[4], T (&gm)[4])
{
    const bool first = ((int)threadIdx.x & 3) == 0;
    T cg = carry;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        T gv = cg;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            beta[j] = b[j] - (a[j] * gv);
            gm[j] = gv = c[j] / beta[j];
        }
        const T ug = quad_perm<QUAD_UP>(gm[3]);
        cg = first ? carry : ug;
    }
    return quad_perm<QUAD_BCAST<3>>(gm[3]);
}

// x_t = s_t - gamma_t x_{t+1}, carry = the x after the group; own(j): x_t = s_t instead; skip(j): x_t = x_{t+1}
// (points past the line).  Returns the group's first x.
template <typename T> __device__ __forceinline__ T quad_backward(const T (&g)[4], const T (&s)[4], T carry, T (&x)[4])
{
    const bool last = ((int)threadIdx.x & 3) == 3;
    T c = carry;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        T xv = c;
#pragma unroll
        for (int j = 3; j >= 0; --j)
            x[j] = xv = s[j] - (g[j] * xv);
        if (k < 3) {
            const T dn = quad_perm<QUAD_DOWN>(x[0]);
            c = last ? carry : dn;
        }
    }
    return quad_perm<QUAD_BCAST<0>>(x[0]);
}
template <typename T, typename Own, typename Skip>
__device__ __forceinline__ T quad_backward_ends(const T (&g)[4], const T (&s)[4], T carry, T (&x)[4], Own &&own,
                                                Skip &&skip)
{
    const bool last = ((int)threadIdx.x & 3) == 3;
    T c = carry;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        T xv = c;
#pragma unroll
        for (int j = 3; j >= 0; --j) {
            const T v = s[j] - (g[j] * xv);
            xv = skip(j) ? xv : (own(j) ? s[j] : v);
            x[j] = xv;
        }
        const T dn = quad_perm<QUAD_DOWN>(x[0]);
        c = last ? carry : dn;
    }
    return quad_perm<QUAD_BCAST<0>>(x[0]);
}

}  // namespace lssamd
