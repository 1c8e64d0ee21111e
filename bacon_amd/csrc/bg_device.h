// bg_device.h — device-side building blocks of the batched IVP engine:
// Butcher tableaux as compile-time data, registered right-hand sides, and the
// RK step attempt (bacon-sci src/ivp/rk.rs:361-423) for one lane.
//
// Operation order is fixed: every multiply-add is an explicit fma(), zero
// tableau entries are skipped at compile time, and the controller works on
// squared norms with the exact-operation root8() below.
// Add, multiply, divide and fma are correctly rounded on gfx950, so a
// lane's arithmetic is reproducible bit for bit by a CPU that performs the
// same operations in the same order.  The file is compiled with
// -ffp-contract=off so the compiler adds no fusions of its own.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/bacon_gpu.h"

namespace bg {

// ---------------------------------------------------------------------------
// Coefficients as FMA operands.  A VOP2 v_fmac_f64 can take a 32-bit literal
// but overwrites its addend, so a literal coefficient applied to a value
// that stays live (y in Y = y + m K) costs an extra v_mov_b64; a VOP3
// v_fma_f64 cannot encode a literal on gfx950 but takes an SGPR pair.  kc()
// passes a coefficient that is not an inline constant through an SGPR pair
// (an empty asm the optimiser cannot see into), so the three-address form is
// used.  The value is unchanged.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double kc(double v) {
    if (v == 0.5 || v == -0.5 || v == 1.0 || v == -1.0 || v == 2.0 || v == -2.0 || v == 4.0 ||
        v == -4.0)
        return v;
    asm("" : "+s"(v));
    return v;
}

// ---------------------------------------------------------------------------
// Caller buffers reached through a descriptor in device memory are generic
// pointers, so the compiler emits FLAT accesses for them.  A FLAT access
// counts on the LDS counter too: the next LDS read (the root8 table, staged
// observation times) then waits until that global store or load completes.
// gptr() states that the buffer is global memory, so the access is a
// GLOBAL one and LDS waits no longer cover it.  Descriptor buffers are
// always device (global) memory.
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gptr(T *p) {
    return (__attribute__((address_space(1))) T *)p;
}

// ---------------------------------------------------------------------------
// Tableaux.  L is the reference's literal "Row i" data (rk.rs:459-502,
// 580-601).  The reference stores it with Matrix::from_vec, which fills
// column-major, and iterates row_iter, so its stage loop reads L transposed;
// Tableau<_, true> reproduces that, Tableau<_, false> reads rows as rows.
// ---------------------------------------------------------------------------
struct Fehlberg45 {
    static constexpr int S = 6;
    static constexpr double c[6] = {0.0, 1.0 / 4.0, 3.0 / 8.0, 12.0 / 13.0, 1.0, 1.0 / 2.0};
    static constexpr double L[6][6] = {
        {0, 0, 0, 0, 0, 0},
        {1.0 / 4.0, 0, 0, 0, 0, 0},
        {3.0 / 32.0, 9.0 / 32.0, 0, 0, 0, 0},
        {1932.0 / 2197.0, -7200.0 / 2197.0, 7296.0 / 2197.0, 0, 0, 0},
        {439.0 / 216.0, -8.0, 3680.0 / 513.0, -845.0 / 4104.0, 0, 0},
        {-8.0 / 27.0, 2.0, -3544.0 / 2565.0, 1859.0 / 4104.0, -11.0 / 40.0, 0}};
    // 4th-order propagation weights (rk.rs:505-514)
    static constexpr double b[6] = {25.0 / 216.0, 0.0, 1408.0 / 2565.0, 2197.0 / 4104.0,
                                    -(1.0 / 5.0), 0.0};
    // error weights b5 - b4 (rk.rs:516-525)
    static constexpr double e[6] = {1.0 / 360.0, 0.0, -128.0 / 4275.0, -2197.0 / 75240.0,
                                    1.0 / 50.0, 2.0 / 55.0};
};

struct BogackiShampine23 {
    static constexpr int S = 4;
    static constexpr double c[4] = {0.0, 1.0 / 2.0, 3.0 / 4.0, 1.0};
    static constexpr double L[4][4] = {{0, 0, 0, 0},
                                       {1.0 / 2.0, 0, 0, 0},
                                       {0, 3.0 / 4.0, 0, 0},
                                       {2.0 / 9.0, 1.0 / 3.0, 4.0 / 9.0, 0}};
    static constexpr double b[4] = {2.0 / 9.0, 1.0 / 3.0, 4.0 / 9.0, 0.0};
    static constexpr double e[4] = {-5.0 / 72.0, 1.0 / 12.0, 1.0 / 9.0, -(1.0 / 8.0)};
};

template <class Lit, bool AsBuilt>
struct Tableau {
    static constexpr int S = Lit::S;
    static constexpr bool as_built = AsBuilt;
    __host__ __device__ static constexpr double m(int i, int j) {
        return AsBuilt ? Lit::L[j][i] : Lit::L[i][j];
    }
    __host__ __device__ static constexpr double c(int i) { return Lit::c[i]; }
    __host__ __device__ static constexpr double b(int i) { return Lit::b[i]; }
    __host__ __device__ static constexpr double e(int i) { return Lit::e[i]; }
    // index of the first non-zero error weight
    __host__ __device__ static constexpr int e_first() {
        int k = 0;
        while (k < S && Lit::e[k] == 0.0) ++k;
        return k;
    }
};

// ---------------------------------------------------------------------------
// Registered right-hand sides.  eval() returns false for a UserError.
// P = number of per-instance parameters (loaded from a [P][n] SoA array).
// ---------------------------------------------------------------------------
template <int D_>
struct RhsExp {
    static constexpr int D = D_, P = 0;
    __device__ static bool eval(double, const double (&y)[D], const double *, double (&f)[D]) {
#pragma unroll
        for (int i = 0; i < D; ++i) f[i] = y[i];
        return true;
    }
};

template <int D_>
struct RhsNeg {
    static constexpr int D = D_, P = 0;
    __device__ static bool eval(double, const double (&y)[D], const double *, double (&f)[D]) {
#pragma unroll
        for (int i = 0; i < D; ++i) f[i] = -y[i];
        return true;
    }
};

template <int D_>
struct RhsQuadratic {
    static constexpr int D = D_, P = 0;
    __device__ static bool eval(double t, const double (&)[D], const double *, double (&f)[D]) {
#pragma unroll
        for (int i = 0; i < D; ++i) f[i] = -2.0 * t;
        return true;
    }
};

template <int D_>
struct RhsCos {
    static constexpr int D = D_, P = 0;
    __device__ static bool eval(double t, const double (&)[D], const double *, double (&f)[D]) {
        const double c = cos(t);
#pragma unroll
        for (int i = 0; i < D; ++i) f[i] = c;
        return true;
    }
};

template <int D_>
struct RhsFailAfter {
    static constexpr int D = D_, P = 1;
    __device__ static bool eval(double t, const double (&y)[D], const double *p, double (&f)[D]) {
        if (t >= p[0]) return false;
#pragma unroll
        for (int i = 0; i < D; ++i) f[i] = y[i];
        return true;
    }
};

struct RhsLorenz {
    static constexpr int D = 3, P = 3;
    // FLOPs per evaluation (fma = 2): sub+mul, sub+fma, mul+fma
    static constexpr int FLOPS = 8;
    __device__ static bool eval(double, const double (&y)[3], const double *p, double (&f)[3]) {
        const double s = p[0], r = p[1], b = p[2];
        f[0] = s * (y[1] - y[0]);
        f[1] = fma(y[0], r - y[2], -y[1]);
        f[2] = fma(y[0], y[1], -(b * y[2]));
        return true;
    }
    static constexpr int VJP_FLOPS = 21;
    __device__ static void vjp(double, const double (&y)[3], const double *p, const double (&fb)[3],
                               double (&yb)[3], double *pb) {
        const double s = p[0], r = p[1], b = p[2];
        yb[0] = fma(-s, fb[0], fma(r - y[2], fb[1], y[1] * fb[2]));
        yb[1] = fma(s, fb[0], fma(y[0], fb[2], -fb[1]));
        yb[2] = fma(-y[0], fb[1], -(b * fb[2]));
        pb[0] = fma(y[1] - y[0], fb[0], pb[0]);
        pb[1] = fma(y[0], fb[1], pb[1]);
        pb[2] = fma(-y[2], fb[2], pb[2]);
    }
};

struct RhsLotkaVolterra {
    static constexpr int D = 2, P = 4;
    static constexpr int FLOPS = 7;
    static constexpr int VJP_FLOPS = 20;
    __device__ static bool eval(double, const double (&y)[2], const double *p, double (&f)[2]) {
        const double a = p[0], b = p[1], g = p[2], d = p[3];
        const double xy = y[0] * y[1];
        f[0] = fma(a, y[0], -(b * xy));
        f[1] = fma(d, xy, -(g * y[1]));
        return true;
    }
    // yb = (df/dy)^T fb, pb += (df/dp)^T fb
    __device__ static void vjp(double, const double (&y)[2], const double *p, const double (&fb)[2],
                               double (&yb)[2], double *pb) {
        const double a = p[0], b = p[1], g = p[2], d = p[3];
        const double x = y[0], w = y[1], xw = x * w;
        yb[0] = fma(a - b * w, fb[0], (d * w) * fb[1]);
        yb[1] = fma(-(b * x), fb[0], (d * x - g) * fb[1]);
        pb[0] = fma(x, fb[0], pb[0]);
        pb[1] = fma(-xw, fb[0], pb[1]);
        pb[2] = fma(-w, fb[1], pb[2]);
        pb[3] = fma(xw, fb[1], pb[3]);
    }
};

// Robertson's chemical kinetics (stiff): params k1, k2, k3 (classically
// 0.04, 3e7, 1e4); y0' = -k1 y0 + k3 y1 y2, y1' = k1 y0 - k3 y1 y2 - k2 y1^2,
// y2' = k2 y1^2.  Separate products and sums (no fused operations).
struct RhsRobertson {
    static constexpr int D = 3, P = 3;
    static constexpr int FLOPS = 10;
    __device__ static bool eval(double, const double (&y)[3], const double *p, double (&f)[3]) {
        const double a = p[0] * y[0];
        const double b = p[2] * (y[1] * y[2]);
        const double c = p[1] * (y[1] * y[1]);
        f[0] = b - a;
        f[1] = (a - b) - c;
        f[2] = c;
        return true;
    }
};

// Complex state (bacon-sci's N: ComplexField): a two-level system
// c' = (-i H - gamma) c, H = [[hd, ho], [ho, -hd]], params hd, ho, gamma.
// The two complex components are stored as (re, im) pairs, y = (a0, b0, a1,
// b1) with c_k = a_k + i b_k: -i H c = H b - i H a.  With real times and
// step sizes the solver's complex products by real coefficients act on the
// parts separately, so the pairs run as four reals; |c|^2 decays as
// exp(-2 gamma t).
struct RhsTwoLevel {
    static constexpr int D = 4, P = 3;
    __device__ static bool eval(double, const double (&y)[4], const double *p, double (&f)[4]) {
        const double hd = p[0], ho = p[1], g = p[2];
        const double ha0 = fma(hd, y[0], ho * y[2]);
        const double ha1 = fma(ho, y[0], -(hd * y[2]));
        const double hb0 = fma(hd, y[1], ho * y[3]);
        const double hb1 = fma(ho, y[1], -(hd * y[3]));
        f[0] = fma(-g, y[0], hb0);
        f[1] = fma(-g, y[1], -ha0);
        f[2] = fma(-g, y[2], hb1);
        f[3] = fma(-g, y[3], -ha1);
        return true;
    }
};

struct RhsOscillator {
    static constexpr int D = 2, P = 0;
    __device__ static bool eval(double, const double (&y)[2], const double *, double (&f)[2]) {
        f[0] = y[1];
        f[1] = -y[0];
        return true;
    }
};

// ---------------------------------------------------------------------------
// r^(1/8) for r in (1e-8, 65536) from exact operations only (frexp, fma,
// ldexp, products of correctly rounded constants): r = m 2^e, m in [1,2);
// m^(1/8) by a degree-5 polynomial in (m - 1.5) interpolating at Chebyshev
// nodes (relative error below 1.11e-6); 2^(e/8) = 2^floor(e/8) times a product of
// 2^(1/8), 2^(1/4), 2^(1/2) selected by the bits of e mod 8.  NaN in, NaN
// out.  Used as the step-size factor (tol/err)^(1/4); the caller bounds it
// by the tangent at r = 1.
// ---------------------------------------------------------------------------
// 2^((e mod 8)/8) as the product ((s1 s2) s4) of the selected constants,
// rounded exactly as a runtime evaluation would (constexpr arithmetic is
// IEEE round-to-nearest).
__host__ __device__ constexpr double root8_scale(int b) {
    return (((b & 1) ? 1.0905077326652577 : 1.0) * ((b & 2) ? 1.189207115002721 : 1.0)) *
           ((b & 4) ? 1.4142135623730951 : 1.0);
}

// The eight scales in LDS for kernels that call root8_lds(): a per-lane
// table read replaces three select pairs and two products.  r8_init() fills
// it at kernel entry (every thread of the block must call it).  Entry k is
// the scale of the arguments whose biased exponent is k mod 8, times 2^-128
// (a power of two, so every product with it rounds like one with the scale):
// root8_lds() then takes the entry and the final exponent straight from the
// argument's high word.
__shared__ double r8_table[8];
__device__ __forceinline__ void r8_init() {
    // r = m 2^e, m in [1, 2), has the biased exponent e + 1023
    if (threadIdx.x < 8) {
        const int b = (int)((threadIdx.x + 1) & 7);  // e mod 8
        r8_table[threadIdx.x] = root8_scale(b) * (b == 0 ? 0x1p-127 : 0x1p-128);
    }
    __syncthreads();
}

// The polynomial's coefficients, highest degree first.
constexpr double kRoot8Poly[6] = {0.0029682975037312034, -0.005693672682686368,
                                  0.010621966427993313,  -0.025512534910039072,
                                  0.08766623673998887,   1.0519887150881322};

__device__ __forceinline__ double root8_poly(double r, int &e) {
    int ex;
    const double mant = frexp(r, &ex);
    // mant * 2 is exact, so the fused form rounds like mul-then-add
    const double x = fma(mant, 2.0, -1.5);
    e = ex - 1;
    // coefficients through SGPRs: three-address fma, no accumulator copies
    double p = kc(kRoot8Poly[0]);
#pragma unroll
    for (int k = 1; k < 6; ++k) p = fma(p, x, kc(kRoot8Poly[k]));
    return p;
}

__device__ __forceinline__ double root8(double r) {
    int e;
    const double p = root8_poly(r, e);
    return ldexp(p * root8_scale(e & 7), e >> 3);
}

// The same value for r in (1e-8, 65536), the scale read from r8_table: the
// entry by the three low bits of the biased exponent, the final exponent its
// other bits (the -128 in the table brings (e + 1023) >> 3 back to e >> 3,
// the entry that belongs to e mod 8 = 0 one more, because 1023 = 8 * 127 + 7).
// c: kRoot8Poly.  Anything outside that range gives an unused value.
__device__ __forceinline__ double root8_lds(double r, const double (&c)[6]) {
    const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, r) >> 32);
    const double scale =
        *(const double *)((const char *)r8_table + ((hi >> 17) & 0x38u));
    const double x = fma(__builtin_amdgcn_frexp_mant(r), 2.0, -1.5);
    double p = c[0];
#pragma unroll
    for (int k = 1; k < 6; ++k) p = fma(p, x, c[k]);
    return ldexp(p * scale, (int)(hi >> 23));
}

// ---------------------------------------------------------------------------
// IEEE minNum / maxNum on values that are never signalling NaNs (results of
// arithmetic): v_min_f64 / v_max_f64 directly.  fmin/fmax give the same
// values but first quiet each operand the compiler cannot prove quiet (a
// v_max_f64 x, x per operand).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double qmin(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double qmax(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double qmax_one(double a) {
    double r;
    asm("v_max_f64 %0, %1, 1.0" : "=v"(r) : "v"(a));
    return r;
}
// b through an SGPR pair
__device__ __forceinline__ double qmin_s(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "s"(b));
    return r;
}

// Values of the lanes l ^ 16 and l ^ 32 by VALU lane swaps (gfx950):
//   v_permlane16_swap(v, v): [0] = v[32 (l / 32) + l mod 16],
//     [1] = v[32 (l / 32) + 16 + l mod 16]
//   v_permlane32_swap(v, v): [0] = v[l mod 32], [1] = v[32 + l mod 32]
// value of lane l ^ 16
__device__ __forceinline__ uint32_t xor16_u32(uint32_t v) {
    const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (__lane_id() & 16) ? p[0] : p[1];
}
__device__ __forceinline__ double xor16_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = xor16_u32((uint32_t)b), hi = xor16_u32((uint32_t)(b >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// value of lane l ^ 32
__device__ __forceinline__ double xor32_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto hi =
        __builtin_amdgcn_permlane32_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    const bool low = __lane_id() < 32;
    const uint32_t l = low ? lo[1] : lo[0], h = low ? hi[1] : hi[0];
    return __builtin_bit_cast(double, ((uint64_t)h << 32) | l);
}

// The lanes (of those active) for which c holds.
__device__ __forceinline__ uint64_t ballot(bool c) { return __builtin_amdgcn_ballot_w64(c); }

__device__ __forceinline__ bool lane_bit(uint64_t mask) { return (mask >> __lane_id()) & 1; }

// v of the first lane of a non-empty mask, wave-uniform.
__device__ __forceinline__ uint32_t first_of(uint32_t v, uint64_t mask) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, __ffsll((unsigned long long)mask) - 1);
}

// ---------------------------------------------------------------------------
// a / b correctly rounded, where the quotient lies in (1e-8, 65536) and a in
// [kMidLo, kMidHi]: the hardware reciprocal (relative error below 2^-22),
// one cubic refinement (error e^3), the product, its exact residual (a multiple
// of 2^-106 a: no underflow) and one correction (Markstein 1990).  Eight
// operations against the IEEE division's eleven, which also scale for exponents
// that do not occur here.
// ---------------------------------------------------------------------------
constexpr double kMidLo = 0x1p-920, kMidHi = 0x1p900;
__device__ __forceinline__ double div_mid(double a, double b) {
    const double y0 = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, y0, 1.0);
    const double y = fma(y0, fma(e, e, e), y0);
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// The controller's factor before the tangent bound for a quotient r = q2 / ss
// (div_mid's) outside (r_lo, 65536); f0: the root of r.  Either the clamp
// delta >= 4 applies (only the quotient's size matters): the first test, since
// an instance whose steps stay at dt_max is here on every attempt.  Or r_lo is
// +inf, for an instance whose q2 may leave div_mid's range (RkLane::set_range):
// then this attempt's q2 decides whether r and f0 stand.  Or the clamp
// delta <= 0.1 applies (r <= 1e-8), or r is NaN.  What is left takes the IEEE
// division and a root of its own.  1,024 Lorenz-63 instances to t = 10, 1.8 ms,
// take 2.2 with no lower step bound; 2.6 with the division and the second root
// each time.
__device__ __forceinline__ double factor_outside(double q2, double ss, double r_lo, double f0,
                                                 double &r) {
    if (r >= 65536.0 && r_lo < 1.0) return 4.0;
    if (r_lo > 1.0 && q2 >= kMidLo && q2 <= kMidHi) {
        if (r >= 65536.0) return 4.0;
        if (r > 1e-8) return f0;
    }
    r = q2 / ss;
    return r <= 1e-8 ? 0.1 : (r >= 65536.0 ? 4.0 : root8(r));
}

// A time that is zero or at least 2^-200 away from it.  If the start, the end
// and every stop are, and dt_min is not below 2^-200, all of a solve's times and
// steps are multiples of 2^-254: the bounds are, sums and differences of such
// multiples round to such multiples, and a proposed step is not below dt_min.  A
// step is then zero or at least 2^-254, also where it is what is left to a
// target at t = 0.
__device__ __forceinline__ bool time_mid(double t) { return t == 0.0 || fabs(t) >= 0x1p-200; }

// r_lo for an instance: 1e-8 if every quotient of its controller is sure to take
// div_mid, else +inf.
__device__ __forceinline__ double quotient_range(double t0, double end, double tol, double dt_min,
                                                 double dt_max) {
    const bool mid = tol >= 0x1p-200 && tol <= 0x1p200 && dt_min >= 0x1p-200 &&
                     dt_max <= 0x1p200 && time_mid(t0) && time_mid(end);
    return mid ? 1e-8 : __builtin_inf();
}

// Right-hand sides that can report a UserError.
template <class RHS>
inline constexpr bool kRhsFails = false;
template <int D>
inline constexpr bool kRhsFails<RhsFailAfter<D>> = true;

// ---------------------------------------------------------------------------
// One lane's RK state and one call of RungeKuttaSolver::step (rk.rs:361-423),
// in two parts:
//   head(target)  the step size h with the end clamp of rk.rs:366-368 aimed
//                 at `target` and the first stage's right-hand side;
//   attempt()     the stages, the error test, the controller and, if the
//                 step is accepted, the update.
// A loop calls head() for the next attempt right after attempt(): its dozen
// independent operations then cover the latency of the loop's exit test.
//
// What bounds an attempt is the number of instructions it issues: a wave alone
// on its SIMD issues one FP64 operation per ~5 cycles whether or not it
// depends on the one before (measured: 5.2 cycles dependent, 5.1 in four
// chains), two or more waves one per 4, and a branch around a few lanes' work
// costs 30-40 (compare, exec update, jump).  So the ordinary attempt runs
// straight through: the quotient without range scaling (div_mid), the root for
// every lane, and one wave-uniform test that sends the lanes outside its range
// to code off that line.
// ---------------------------------------------------------------------------

// HOIST: the tableau and root coefficients are put through SGPR pairs once,
// where the lane state is declared, rather than at each use (see cm below);
// for the persistent loops and the adjoint's backward replay, whose SGPR
// budgets have room for them (in the adjoint's forward pass they would
// double its SGPR spills).
template <class RHS, class Tab, bool HOIST = false>
struct RkLane {
    static constexpr int D = RHS::D, S = Tab::S;
    double t, dt, end, tol, dt_min, dt_max;
    double y[D];
    double K[S][D];  // half_steps; persists across attempts (read by AS_BUILT)
    double p[RHS::P > 0 ? RHS::P : 1];
    double h;        // the attempt's step size (head)
    double F0[D];    // f(t, y) (head; not for right-hand sides that can fail)
    double r_lo;     // 1e-8, or +inf: see factor_outside
    bool clamped;    // h was cut to reach the target
    // With HOIST, the stage coefficients, the first error weight and the
    // root's polynomial through SGPR pairs (kc), taken once where the lane
    // state is declared, so every attempt reads the pairs directly instead
    // of copying each constant into a fresh pair at its use (25 scalar moves
    // per Lorenz RK45 attempt).  Without, kc at each use, which keeps fewer
    // SGPRs live in kernels that have other uses for them.
    double cm[S][S];
    double ce0;
    double cr[6];
    double c_below_one;  // 1 - 2^-53

    __device__ RkLane() {
        if constexpr (HOIST) {
#pragma unroll
            for (int i = 0; i < S; ++i)
#pragma unroll
                for (int j = 0; j < S; ++j) cm[i][j] = kc(Tab::m(i, j));
            ce0 = kc(Tab::e(Tab::e_first()));
            c_below_one = 0x1.fffffffffffffp-1;
#pragma unroll
            for (int k = 0; k < 6; ++k) cr[k] = kc(kRoot8Poly[k]);
            // one operand of the polynomial's first fma in a VGPR pair: an
            // instruction reads at most one SGPR pair
            asm("" : "+v"(cr[0]));
        }
    }
    __device__ __forceinline__ double coef_m(int i, int j) const {
        if constexpr (HOIST) return cm[i][j];
        return kc(Tab::m(i, j));
    }

    // Called when an instance is loaded: whether every quotient of the
    // controller is sure to take div_mid, q2 = (tol h)^2 in [kMidLo, kMidHi].
    __device__ __forceinline__ void set_range(bool stops_mid = true) {
        r_lo = stops_mid ? quotient_range(t, end, tol, dt_min, dt_max) : __builtin_inf();
    }

    __device__ __forceinline__ void head(double target) {
        clamped = t + dt >= target;
        h = clamped ? target - t : dt;
        if constexpr (!kRhsFails<RHS>) (void)RHS::eval(fma(Tab::c(0), h, t), y, p, F0);
    }

    // The stages of a step of size h from (t, y): rk.rs:370-384.  False if
    // the right-hand side reports an error.  HEAD: the first stage's
    // right-hand side is in F0.
    template <bool HEAD>
    __device__ __forceinline__ bool stages(double hh) {
#pragma unroll
        for (int i = 0; i < S; ++i) {
            double Y[D];
#pragma unroll
            for (int d = 0; d < D; ++d) Y[d] = y[d];
            // the first row of a tableau read as built is not empty: its
            // stage does not start from y
            bool from_y = i == 0;
#pragma unroll
            for (int j = 0; j < S; ++j) {
                const double m = Tab::m(i, j);
                if (m != 0.0) {
                    from_y = false;
#pragma unroll
                    for (int d = 0; d < D; ++d) Y[d] = fma(coef_m(i, j), K[j][d], Y[d]);
                }
            }
            double f[D];
            if (HEAD && !kRhsFails<RHS> && from_y) {
#pragma unroll
                for (int d = 0; d < D; ++d) f[d] = F0[d];
            } else {
                const double ti = fma(Tab::c(i), hh, t);
                if (!RHS::eval(ti, Y, p, f)) return false;
            }
#pragma unroll
            for (int d = 0; d < D; ++d) K[i][d] = f[d] * hh;
        }
        return true;
    }

    // The accepted step's update from the stages: rk.rs:392-398.
    __device__ __forceinline__ void update(double hh) {
        t += hh;
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const double b = Tab::b(j);
            if (b != 0.0) {
#pragma unroll
                for (int d = 0; d < D; ++d) y[d] = fma(b, K[j][d], y[d]);
            }
        }
    }

    // A step of size hh known to be accepted (the replay of a recorded step):
    // the operations of an accepted attempt, so (t, y) come out
    // bit-identical, without the error estimate and the controller.  dt is
    // left as it was.
    __device__ __forceinline__ bool advance(double hh) {
        if (!stages<false>(hh)) return false;
        update(hh);
        return true;
    }

    // One attempt of size h (head).  Returns whether it was accepted, and
    // counts it in nacc then; failed is set if the right-hand side reported an
    // error (then nothing else has changed but K).
    __device__ __forceinline__ bool attempt(bool &failed, uint32_t &nacc) {
        failed = false;
        if (!stages<true>(h)) {
            failed = true;
            return false;
        }
        // rk.rs:386-390
        double E[D];
        constexpr int e0 = Tab::e_first();
#pragma unroll
        for (int d = 0; d < D; ++d) E[d] = (HOIST ? ce0 : kc(Tab::e(e0))) * K[e0][d];
#pragma unroll
        for (int j = e0 + 1; j < S; ++j) {
            const double e = Tab::e(j);
            if (e != 0.0) {
#pragma unroll
                for (int d = 0; d < D; ++d) E[d] = fma(e, K[j][d], E[d]);
            }
        }
        double ss = E[0] * E[0];
#pragma unroll
        for (int d = 1; d < D; ++d) ss = fma(E[d], E[d], ss);
        // rk.rs:390-412 in squared form: err = |E|/dt <= tol  <=>  ss <= q^2
        // with q = tol*dt; delta = (tol/err)^(1/4) = r^(1/8), r = q^2/ss,
        // and the clamps delta <= 0.1 / delta >= 4 become r <= 1e-8 /
        // r >= 65536 (safety factor 100/100 = 1.0, rk.rs:266-268).
        const double q = tol * h;
        const double q2 = q * q;
        const bool accepted = ss <= q2;
        double r = div_mid(q2, ss);
        double f0;
        if constexpr (HOIST) {
            f0 = root8_lds(r, cr);
        } else {
            double c[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) c[k] = kc(kRoot8Poly[k]);
            f0 = root8_lds(r, c);
        }
        const bool outside = !(r > r_lo && r < 65536.0);
        if (__builtin_expect(ballot(outside) != 0, 0)) {
            if (outside) f0 = factor_outside(q2, ss, r_lo, f0, r);
        }
        // near r = 1 the sign of delta - 1 ~ (r - 1)/8 is far below root8's
        // error: bound by the tangent 1 + (r - 1)/8 (r^(1/8) is concave, the
        // tangent is exact to second order at 1), then keep the exact power's
        // side of 1 (a rejection shrinks dt, an acceptance never does).
        // fmin/fmax are IEEE minNum/maxNum: a NaN error estimate (rejected)
        // gets the factor 1 - 2^-53, so dt stays finite and the instance runs
        // into the attempt cap (the reference retries forever).
        const double tang = fma(r - 1.0, 0.125, 1.0);
        const double f = qmin(f0, tang);
        double factor = HOIST ? qmin(f, c_below_one) : qmin_s(f, 0x1.fffffffffffffp-1);
        if (accepted) {
            update(h);
            ++nacc;
            factor = qmax_one(f);
        }
        // dt is never NaN here (factor is finite), so the clamp is a minimum
        dt = qmin(h * factor, dt_max);
        return accepted;
    }
};

// The descriptor, read at the point of use.  The empty asm hides the
// pointer's value from the optimiser, so the loads are not hoisted out of the
// persistent loop (no ~30 descriptor registers live across the attempts)
// while staying ordinary cached loads that issue together under one wait.
// (Volatile reads would be uncached, each waited for in turn.)
template <class DP>
__device__ __forceinline__ DP desc_at_use(DP dv) {
    asm volatile("" : "+s"(dv));
    return dv;
}

// A kernel whose first parameter is the descriptor by value reads it from its
// argument segment (constant memory, scalar loads): no copy in device memory
// and no kernel before it to make one.
typedef const __attribute__((address_space(4))) bg_ensemble_desc *karg_desc;
__device__ __forceinline__ karg_desc kernarg_desc() {
    return (karg_desc)__builtin_amdgcn_kernarg_segment_ptr();
}

template <class DP>
__device__ __forceinline__ bg_ensemble_desc desc_inputs(DP dv_) {
    const DP dv = desc_at_use(dv_);
    bg_ensemble_desc d;
    d.n = dv->n;
    d.order = dv->order;
    d.y0 = dv->y0;
    d.params = dv->params;
    d.t0 = dv->t0;
    d.t_end = dv->t_end;
    d.tol = dv->tol;
    d.dt_min = dv->dt_min;
    d.dt_max = dv->dt_max;
    d.t0_s = dv->t0_s;
    d.t_end_s = dv->t_end_s;
    d.tol_s = dv->tol_s;
    d.dt_min_s = dv->dt_min_s;
    d.dt_max_s = dv->dt_max_s;
    return d;
}

template <class DP>
__device__ __forceinline__ bg_ensemble_desc desc_outputs(DP dv_) {
    const DP dv = desc_at_use(dv_);
    bg_ensemble_desc d;
    d.n = dv->n;
    d.t_out = dv->t_out;
    d.y_out = dv->y_out;
    d.status = dv->status;
    d.counts = dv->counts;
    d.work = dv->work;
    return d;
}

// ---------------------------------------------------------------------------
// The work queue of a persistent launch.  Lane g of the grid starts with
// schedule position g; positions from the number of lanes on are handed out by
// a counter that starts there.  A launch whose positions all have a lane passes
// no counter: nothing to set up before it, and no wave asks for more.
//
// A wave claims a run of positions with one atomicAdd and hands them to its
// lanes as they finish.  One atomicAdd per finished lane made the counter the
// bottleneck of short instances: it serves one request per ~12 ns whatever the
// chip computes (10^6 Lotka-Volterra solves of 350 attempts: 8.5 ms, 1.2 ms
// of it arithmetic; with runs 2.4 ms).  Long instances want the opposite: a
// position that waits in one wave's run is one that no other wave can start
// (2^20 Lorenz-63 solves of 9,000 attempts on two waves per SIMD: 53 ms one at
// a time, 55 ms in runs of up to 64).  So the length of a run follows the time
// the last one took: doubled below 128 loop iterations, halved above 512 (all
// of a few thousand waves claiming every 128 attempts, 50 us, keep the counter
// busy less than half the time), and never more than a quarter to a half of the
// wave's even share of what is left.  With a schedule the run's entries are
// loaded when it is claimed, one per lane, so a refill does not wait for its
// order[] entry.
//
// Every function is called by the whole wave.
// ---------------------------------------------------------------------------
struct WaveQueue {
    uint32_t base, end;   // unassigned positions of the claimed run
    uint32_t first;       // position whose schedule entry lane 0 holds
    int32_t entry;        // schedule entry of position first + lane
    bool open;            // the counter may hold more
    uint32_t run;         // length of the next run
    uint32_t ticks;       // loop iterations since the last claim
    uint32_t waves;       // waves that share the queue

    __device__ __forceinline__ WaveQueue(const uint32_t *counter, uint32_t blocks = gridDim.x)
        : base(0), end(0), first(0), entry(0), open(counter != nullptr), run(1), ticks(0),
          waves(blocks * (blockDim.x >> 6)) {}

    __device__ __forceinline__ bool drained() const { return !open && base >= end; }

    // the instance of the lane's own position, -1 if there is none
    __device__ __forceinline__ int64_t start(uint64_t n, const int32_t *order) const {
        const uint64_t pos = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (pos >= n) return -1;
        return order ? (int64_t)gptr(order)[pos] : (int64_t)pos;
    }

    // the next instance for every lane that wants one, -1 if there is none;
    // pos: its schedule position (the other lanes' stays what it was: they are
    // still at work on theirs)
    __device__ __forceinline__ int64_t next(uint32_t *counter, uint32_t n, const int32_t *order,
                                            bool want, uint32_t &pos) {
        const uint32_t lane = __lane_id();
        const uint64_t need = ballot(want);
        const uint32_t cnt = (uint32_t)__popcll(need);
        const uint32_t rank = (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
        const uint32_t avail = end - base;
        bool have = want && rank < avail;
        uint32_t at = base + rank;
        int32_t idx = order ? __shfl(entry, (int)((at - first) & 63u)) : (int32_t)at;
        if (cnt <= avail) {
            base += cnt;
        } else if (open) {
            const uint32_t lacking = cnt - avail;
            const uint32_t left = n - (end ? end : waves << 6);
            const uint32_t share = left >> (33 - __builtin_clz(waves));
            if (ticks < 128u)
                run = run < 64u ? 2u * run : 64u;
            else if (ticks > 512u)
                run = run > 1u ? run >> 1 : 1u;
            ticks = 0;
            uint32_t size = run < share ? run : share;
            size = size < lacking ? lacking : size;
            uint32_t b = 0;
            if (lane == 0) b = atomicAdd(counter, size);
            b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
            open = b < n && size < n - b;
            b = b < n ? b : n;
            end = open ? b + size : n;
            first = b;
            if (order) entry = b + lane < end ? gptr(order)[b + lane] : 0;
            const uint32_t k = rank - avail;
            const int32_t other = order ? __shfl(entry, (int)(k & 63u)) : (int32_t)(b + k);
            if (want && rank >= avail) {
                at = b + k;
                idx = other;
                have = at < end;
            }
            base = lacking < end - b ? b + lacking : end;
        } else {
            base = end;
        }
        if (want) pos = at;
        return have ? (int64_t)idx : -1;
    }
};

// ---------------------------------------------------------------------------
// Shared stop (observation) times are read at every instance start
// (count_stops) and at every stop.  With OBS_LDS (n_obs <= kObsLds) they are staged in LDS at
// kernel entry: the reads then neither wait on L2 (a serial scan of 20
// global loads per instance start cost microseconds) nor, being known LDS
// accesses, wait for the loop's outstanding stores.  Every thread
// of the block calls it.
static constexpr uint32_t kObsLds = 1024;
template <bool OBS_LDS>
__device__ __forceinline__ const double *stage_obs(double *lds, const double *obs,
                                                   uint32_t n_obs) {
    if constexpr (!OBS_LDS) {
        return obs;
    } else {
        for (uint32_t k = threadIdx.x; k < n_obs; k += blockDim.x) lds[k] = gptr(obs)[k];
        __syncthreads();
        return lds;
    }
}

// Number of times strictly before `end` (those of them after the start become
// stops): a binary search over the increasing times, ~log2(n_obs) dependent
// reads at each instance start instead of one per time before the end.
__device__ __forceinline__ uint32_t count_stops(const double *obs, uint32_t n_obs, double end) {
    uint32_t lo = 0, hi = n_obs;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (obs[mid] < end)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// time_mid of each of the increasing times: those around zero are the last
// below it and the first above it.
__device__ __forceinline__ bool times_mid(const double *obs, uint32_t n_obs) {
    const uint32_t below = count_stops(obs, n_obs, 0.0);
    const uint32_t above = count_stops(obs, n_obs, 0x1p-1074);
    return (below == 0 || time_mid(obs[below - 1])) && (above >= n_obs || time_mid(obs[above]));
}

// The largest value over the wave's lanes, wave-uniform (every lane active).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)v, m);
        v = o > v ? o : v;
    }
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

}  // namespace bg
