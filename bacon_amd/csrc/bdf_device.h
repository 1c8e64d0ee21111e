// bdf_device.h — device side of the batched BDF (BDF6 / BDF2) for gfx950,
// shared by bdf_kernels.hip and bdf_systems.hip.
//
// Hot path: bacon-sci's BDFSolver::step (src/ivp/bdf.rs:495-634) with its
// RK4 bootstrap (bdf.rs:346-387), finite-difference Jacobian (bdf.rs:390-411)
// and Broyden corrector (bdf.rs:414-475), recast as an ensemble.
//
// Layout: one instance per group of W lanes, the power of two W >= D (the
// whole wave for the 32-component Brusselator, split into half rows; one
// lane for scalar problems; W - D padding lanes for small systems such as
// Lorenz-63).  Lane g of a group
// owns component g of every vector (state, guess, residuals, the history of
// the last O accepted values) and row g of the Jacobian inverse, all in VGPRs.
// Group collectives are DPP moves and lane swaps; the column sums of
// the Broyden update u = s^T J^-1 go through an LDS transpose (row stride
// W+1 doubles: conflict-free column reads).  The inverse is Gauss-Jordan with
// partial pivoting on the rows (implicit, no row swaps); its arithmetic type
// is a template parameter (double, or float with the Broyden iteration and
// all residuals in double).  Instances are refilled per group from a global
// work counter, like the RK ensemble kernel.
#pragma once

#include <type_traits>
#include <utility>

#include "bg_device.h"
#include "bg_internal.h"

namespace bg {

constexpr uint32_t kBdfDefaultMaxSteps = 1000000u;


// ---------------------------------------------------------------------------
// cross-lane moves without LDS traffic (gfx950 lane layouts, measured):
//   DPP row_ror:1 (0x121): lane i <- lane (i - 1) mod 16 within its row of 16
//   DPP row_ror:15 (0x12F): lane i <- lane (i + 1) mod 16
//   DPP quad_perm [1,0,3,2] (0xB1): i <- i ^ 1;  [2,3,0,1] (0x4E): i <- i ^ 2
//   DPP row_half_mirror (0x141): i <- 7 - i within 8; row_mirror (0x140):
//     i <- 15 - i within 16
//   ds_swizzle bitmask 0x401F: i <- i ^ 16 within 32
//   v_permlane32_swap(v, v): [0] = v[l mod 32], [1] = v[32 + l mod 32]
//   v_permlane16_swap(v, v): [0] = v[32 (l / 32) + l mod 16],
//     [1] = v[32 (l / 32) + 16 + l mod 16]
// The permlane swaps are VALU operations; ds_swizzle goes through the LDS
// unit and waits for it.
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xF, 0xF, false);
    const uint32_t hi =
        (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// lane l's value, broadcast (l wave-uniform)
__device__ __forceinline__ double readlane_lu(double v, int l) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float readlane_lu(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
// half hk's value in both halves (hk a constant: one of a swap's results)
__device__ __forceinline__ double half_lu(double v, int hk) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
    const auto pl = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto ph = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __builtin_bit_cast(double, ((uint64_t)ph[hk] << 32) | pl[hk]);
}
__device__ __forceinline__ float half_lu(float v, int hk) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto p = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    const uint32_t w = p[hk];  // (a bit cast of the element itself takes element 0)
    return __builtin_bit_cast(float, w);
}

// 1 / a for a pivot of the whole-wave elimination: the hardware reciprocal
// refined by Newton steps (two for double, one for float), within an ulp or
// two of the correctly rounded quotient, in 3-5 instructions instead of the
// IEEE division's ten.  The inverse is an approximation of the Jacobian's
// anyway (the Broyden iteration only needs a nearby matrix); a is never 0
// here (the pivot key rejected zeros).
__device__ __forceinline__ double pivot_recip(double a) {
    double r = __builtin_amdgcn_rcp(a);
    r = fma(r, fma(-a, r, 1.0), r);
    return fma(r, fma(-a, r, 1.0), r);
}
__device__ __forceinline__ float pivot_recip(float a) {
    const float r = __builtin_amdgcn_rcpf(a);
    return fmaf(r, fmaf(-a, r, 1.0f), r);
}

// The compiler does not insert the wait states of lane operations around inline
// assembly.  lane_operand: v as the broadcast operand of fma_newbcast, two wait
// states after the instruction that wrote it; every use of the result comes
// after them, in whatever order the multiply-adds are scheduled (each with a
// wait of its own in one of them, ilp-first schedules put others before it).
// `with`, the other factor, is taken through it too where v comes from memory:
// the wait for v then does not hold up what computes the factor.
template <class T>
__device__ __forceinline__ T lane_operand(T v) {
    asm("s_nop 1" : "+v"(v));
    return v;
}
template <class T>
__device__ __forceinline__ T lane_operand(T v, T &with) {
    asm("s_nop 1" : "+v"(v), "+v"(with));
    return v;
}
// d + row_newbcast(r, C) * f by one fma: lane C of each 16-lane row of r, a
// lane_operand, is an operand modifier of the multiply-add (through the
// intrinsic it would be a move before it).  TO_LANES: the sum may go into a lane
// operation next.
template <int C, bool TO_LANES>
__device__ __forceinline__ double fma_newbcast(double r, double f, double d) {
    if constexpr (TO_LANES)
        asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\ts_nop 1"
            : "+v"(d) : "v"(r), "v"(f), "n"(C));
    else
        asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
            : "+v"(d) : "v"(r), "v"(f), "n"(C));
    return d;
}
template <int C, bool TO_LANES>
__device__ __forceinline__ float fma_newbcast(float r, float f, float d) {
    if constexpr (TO_LANES)
        asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\ts_nop 1"
            : "+v"(d) : "v"(r), "v"(f), "n"(C));
    else
        asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
            : "+v"(d) : "v"(r), "v"(f), "n"(C));
    return d;
}
// f(0), ..., f(N - 1) with constant arguments
template <class F, int... I>
__device__ __forceinline__ void for_ints(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_ints(F &&f) {
    for_ints(f, std::make_integer_sequence<int, N>{});
}

// ---------------------------------------------------------------------------
// group collectives (every lane of the group active)
// ---------------------------------------------------------------------------
// value of the lane M apart (l ^ M), M = 1, 2, 4 or 8, by DPP moves
template <int M>
__device__ __forceinline__ double xor_f64(double v) {
    if constexpr (M == 1) return dpp_f64<0xB1>(v);
    else if constexpr (M == 2) return dpp_f64<0x4E>(v);
    else if constexpr (M == 4) return dpp_f64<0x1B>(dpp_f64<0x141>(v));  // 7 - (l ^ 3)
    else return dpp_f64<0x128>(v);  // rotation by 8 within 16
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int M>
__device__ __forceinline__ uint32_t xor_u32(uint32_t v) {
    if constexpr (M == 1) return dpp_u32<0xB1>(v);
    else if constexpr (M == 2) return dpp_u32<0x4E>(v);
    else if constexpr (M == 4) return dpp_u32<0x1B>(dpp_u32<0x141>(v));
    else return dpp_u32<0x128>(v);
}

template <int W>
struct Grp {
    int g;  // lane index in the group
    __device__ __forceinline__ double bcast(double v, int src) const {
        if constexpr (W == 1) return v;
        return __shfl(v, src, W);
    }
    // lane K's value (K known at compile time: one DPP move per word where
    // the group is within a quad)
    template <int K>
    __device__ __forceinline__ double bcast_at(double v) const {
        if constexpr (W == 1) return v;
        else if constexpr (W == 2) return dpp_f64<K | K << 2 | (2 + K) << 4 | (2 + K) << 6>(v);
        else if constexpr (W == 4) return dpp_f64<K * 0x55>(v);
        else return __shfl(v, K, W);
    }
    // all-reduce sum; symmetric pairings, so every lane gets the same bits
    __device__ __forceinline__ double sum(double v) const {
        if constexpr (W == 32) {
            v += dpp_f64<0xB1>(v);
            v += dpp_f64<0x4E>(v);
            v += dpp_f64<0x141>(v);
            v += dpp_f64<0x140>(v);
            v += xor16_f64(v);
            return v;
        } else {
            if constexpr (W >= 16) v += xor_f64<8>(v);
            if constexpr (W >= 8) v += xor_f64<4>(v);
            if constexpr (W >= 4) v += xor_f64<2>(v);
            if constexpr (W >= 2) v += xor_f64<1>(v);
            return v;
        }
    }
    // all-reduce maximum of unsigned keys (one DPP max per stage)
    __device__ __forceinline__ uint32_t max_u32(uint32_t v) const {
        if constexpr (W == 32) {
            v = __builtin_elementwise_max(v, dpp_u32<0xB1>(v));
            v = __builtin_elementwise_max(v, dpp_u32<0x4E>(v));
            v = __builtin_elementwise_max(v, dpp_u32<0x141>(v));
            v = __builtin_elementwise_max(v, dpp_u32<0x140>(v));
            v = __builtin_elementwise_max(v, xor16_u32(v));
            return v;
        } else {
            if constexpr (W >= 16) v = __builtin_elementwise_max(v, xor_u32<8>(v));
            if constexpr (W >= 8) v = __builtin_elementwise_max(v, xor_u32<4>(v));
            if constexpr (W >= 4) v = __builtin_elementwise_max(v, xor_u32<2>(v));
            if constexpr (W >= 2) v = __builtin_elementwise_max(v, xor_u32<1>(v));
            return v;
        }
    }
    // all-reduce maximum (IEEE maxNum: a NaN operand loses)
    __device__ __forceinline__ double max(double v) const {
        if constexpr (W == 32) {
            v = fmax(v, dpp_f64<0xB1>(v));
            v = fmax(v, dpp_f64<0x4E>(v));
            v = fmax(v, dpp_f64<0x141>(v));
            v = fmax(v, dpp_f64<0x140>(v));
            v = fmax(v, xor16_f64(v));
            return v;
        } else {
            if constexpr (W >= 16) v = fmax(v, xor_f64<8>(v));
            if constexpr (W >= 8) v = fmax(v, xor_f64<4>(v));
            if constexpr (W >= 4) v = fmax(v, xor_f64<2>(v));
            if constexpr (W >= 2) v = fmax(v, xor_f64<1>(v));
            return v;
        }
    }
};

// sqrt(ss) <= bound (OR_EQUAL) or sqrt(ss) < bound, as the rounded square root
// would decide.  SQUARES: away from a positive bound the squares decide (a
// margin of 1e-10 each way, far above their rounding), within it, and for any
// other bound (the square would lose its sign), the root itself.  Not
// in the whole-wave solver, whose registers are full: there the branch cost
// more in spills than the root (27.5 against 26.7 ms, 32,768 instances to t = 2).
template <bool SQUARES, bool OR_EQUAL>
__device__ __forceinline__ bool norm_below(double ss, double bound) {
    if constexpr (SQUARES) {
        const double b2 = bound * bound;
        if (bound > 1e-145) {
            if (ss < b2 * (1.0 - 1e-10)) return true;
            if (ss > b2 * (1.0 + 1e-10)) return false;
        }
    }
    const double nrm = sqrt(ss);
    return OR_EQUAL ? nrm <= bound : nrm < bound;
}

// maximum of unsigned keys over each 16-lane row (one DPP max per stage)
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
    v = __builtin_elementwise_max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
    v = __builtin_elementwise_max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
    v = __builtin_elementwise_max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
    v = __builtin_elementwise_max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));
    return v;
}

// Pivot choice key: |a| with its 5 lowest mantissa bits replaced by 31 - g,
// so the maximum key names the row with the largest |a| and the lowest lane
// among equal ones (ties below 2^-47 relative resolve towards lower lanes).
// Rows not eligible (already pivots, NaN) get key 0.
__device__ __forceinline__ double pivot_key(double a, bool eligible, int g) {
    const double m = fabs(a);
    if (!eligible || !(m == m)) return 0.0;
    const uint64_t b = (__builtin_bit_cast(uint64_t, m) & ~(uint64_t)31) | (uint64_t)(31 - g);
    return __builtin_bit_cast(double, b);
}
__device__ __forceinline__ int pivot_lane(double key) {
    return 31 - (int)(__builtin_bit_cast(uint64_t, key) & 31);
}
__device__ __forceinline__ bool pivot_nonzero(double key) {
    return (__builtin_bit_cast(uint64_t, key) & ~(uint64_t)31) != 0;
}

// The same choice on 32-bit keys: the high word of |a| (sign, exponent and
// 20 mantissa bits) with its 5 lowest bits replaced by 31 - g, reduced by
// one DPP integer max per stage.  The largest |a| wins up to 2^-15
// relative (candidates that close are equally good pivots); ties go to the
// lowest lane.  |a| below 2^-1017 counts as zero (SingularMatrix), as do
// rows already used and NaN.
__device__ __forceinline__ uint32_t pivot_key32(double a, bool eligible, int g) {
    if (!eligible || !(a == a)) return 0u;
    const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, a) >> 32) & 0x7fffffffu;
    return (hi & ~31u) | (uint32_t)(31 - g);
}
// The FP32 inverse's key straight from the float: |a|'s exponent and 23
// mantissa bits, the 5 lowest replaced by 31 - g (the largest |a| wins up
// to 2^-18 relative); |a| below 2^-144 counts as zero.
__device__ __forceinline__ uint32_t pivot_key32(float a, bool eligible, int g) {
    if (!eligible || !(a == a)) return 0u;
    const uint32_t m = __builtin_bit_cast(uint32_t, a) & 0x7fffffffu;
    return (m & ~31u) | (uint32_t)(31 - g);
}
__device__ __forceinline__ int pivot_lane32(uint32_t key) { return 31 - (int)(key & 31u); }
__device__ __forceinline__ bool pivot_nonzero32(uint32_t key) { return (key & ~31u) != 0u; }

// ---------------------------------------------------------------------------
// right-hand sides evaluated cooperatively: lane g returns f_g(t, y)
// ---------------------------------------------------------------------------
template <template <int> class R>
struct ScalarBdf {  // the 1-D reference-test right-hand sides
    static constexpr int D = 1, W = 1, P = R<1>::P;
    template <class G>
    __device__ static bool lane_eval(double t, double y, const double *p, const G &, double &f) {
        double yy[1] = {y}, ff[1];
        const bool ok = R<1>::eval(t, yy, p, ff);
        f = ff[0];
        return ok;
    }
};

// 1-D Brusselator reaction-diffusion, CELLS cells, periodic, dx = 1/CELLS;
// y = [u_0..u_{CELLS-1}, v_0..v_{CELLS-1}], params A, B, alpha.
template <int CELLS>
struct RhsBrusselatorG {
    static constexpr int D = 2 * CELLS, W = D, P = 3;
    template <class G>
    __device__ static bool lane_eval(double, double y, const double *p, const G &grp, double &f) {
        const int g = grp.g;
        const bool isu = g < CELLS;
        const int c = isu ? g : g - CELLS;
        const int base = isu ? 0 : CELLS;
        double left, right, other;
        if constexpr (CELLS == 16) {
            // a species' 16 cells fill one DPP row: periodic neighbours are
            // row rotations, the other species is the lane 16 apart
            left = dpp_f64<0x121>(y);
            right = dpp_f64<0x12F>(y);
            other = xor16_f64(y);
        } else if constexpr (CELLS == 8) {
            // a species' 8 cells fill half a row: a rotation of the row, with
            // the half's wrap from the rotation by 8 more
            const double l1 = dpp_f64<0x121>(y), l9 = dpp_f64<0x129>(y);
            const double r1 = dpp_f64<0x12F>(y), r9 = dpp_f64<0x127>(y);
            left = c == 0 ? l9 : l1;
            right = c == CELLS - 1 ? r9 : r1;
            other = xor_f64<8>(y);
        } else if constexpr (CELLS == 4) {
            left = dpp_f64<0x93>(y);   // quad_perm [3, 0, 1, 2]
            right = dpp_f64<0x39>(y);  // quad_perm [1, 2, 3, 0]
            other = xor_f64<4>(y);
        } else if constexpr (CELLS == 2) {
            left = right = xor_f64<1>(y);
            other = xor_f64<2>(y);
        } else {
            left = grp.bcast(y, base + (c + CELLS - 1) % CELLS);
            right = grp.bcast(y, base + (c + 1) % CELLS);
            other = grp.bcast(y, isu ? g + CELLS : g - CELLS);
        }
        const double u = isu ? y : other, v = isu ? other : y;
        const double A = p[0], B = p[1], alpha = p[2];
        const double dx = 1.0 / CELLS;
        const double cl = alpha / (dx * dx);
        const double uuv = u * u * v;
        const double lap = fma(-2.0, y, left) + right;
        // u: A + u^2 v - (B + 1) u + cl lap;  v: B u - u^2 v + cl lap
        const double react = isu ? fma(-(B + 1.0), u, A + uuv) : fma(B, u, -uuv);
        f = fma(cl, lap, react);
        return true;
    }
    // FLOPs of one full evaluation (all 2*CELLS components)
    static constexpr int FLOPS = CELLS * (6 + 4 + 4 + 5);

    // Column colouring for the finite-difference Jacobian (Curtis, Powell &
    // Reid 1974): row u_i depends on u_{i-1}, u_i, u_{i+1}, v_i and row v_i
    // on v_{i-1}, v_i, v_{i+1}, u_i.  Colour u_j with j mod 4 and v_j with
    // (j + 2) mod 4: the four members of every row's stencil then carry the
    // four colours, so one evaluation per colour (and sign) yields one
    // entry of every row (CELLS divisible by 4 keeps the periodic wrap
    // consistent).
    static constexpr int NC = 4;
    // the column of colour k in row g's stencil
    __device__ static int member(int g, int k) {
        const bool isu = g < CELLS;
        const int i = isu ? g : g - CELLS;
        const int d = (k - i) & 3;
        if (isu) {
            const int c[4] = {g, (i + 1) % CELLS, CELLS + i, (i + CELLS - 1) % CELLS};
            return c[d];
        }
        const int c[4] = {i, CELLS + (i + CELLS - 1) % CELLS, g, CELLS + (i + 1) % CELLS};
        return c[d];
    }
    // row g's stencil in increasing column order
    __device__ static void stencil(int g, int (&s)[4]) {
        const bool isu = g < CELLS;
        const int i = isu ? g : g - CELLS;
        const int base = isu ? 0 : CELLS;
        int a[4] = {base + (i + CELLS - 1) % CELLS, g, base + (i + 1) % CELLS,
                    isu ? CELLS + i : i};
        // sort four (a tiny network; compile-time unrolled)
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
            for (int y = 0; y < 3 - x; ++y)
                if (a[y] > a[y + 1]) {
                    const int tmp = a[y];
                    a[y] = a[y + 1];
                    a[y + 1] = tmp;
                }
#pragma unroll
        for (int x = 0; x < 4; ++x) s[x] = a[x];
    }
    // f_g at the state the reference's column loop (bdf.rs:402-406) holds
    // while it evaluates column c: components j < c already restored
    // (`rest`, x + dt - 2 dt + dt), j > c original (`orig`), c itself
    // perturbed (`pert`: x + dt on half 0, x + dt - 2 dt on half 1).  Every
    // lane supplies its own three candidates; `own` receives the value of
    // the lane's own component in that state.  A c outside the stencil
    // gives the unperturbed state of that column.
    template <class G>
    __device__ static bool lane_eval_state(double t, double orig, double rest, double pert, int c,
                                           const double *p, const G &grp, double &f,
                                           double &own) {
        static_assert(CELLS == 16, "state evaluation uses the DPP row layout of 16 cells");
        const int g = grp.g;
        const bool isu = g < CELLS;
        const int i = isu ? g : g - CELLS;
        const int base = isu ? 0 : CELLS;
        const int jl = base + (i + CELLS - 1) % CELLS, jr = base + (i + 1) % CELLS;
        const int jo = isu ? g + CELLS : g - CELLS;
        auto pick = [&](int j, double o, double r, double q) {
            return j == c ? q : (j < c ? r : o);
        };
        own = pick(g, orig, rest, pert);
        const double left = pick(jl, dpp_f64<0x121>(orig), dpp_f64<0x121>(rest), dpp_f64<0x121>(pert));
        const double right =
            pick(jr, dpp_f64<0x12F>(orig), dpp_f64<0x12F>(rest), dpp_f64<0x12F>(pert));
        const double other = pick(jo, xor16_f64(orig), xor16_f64(rest), xor16_f64(pert));
        const double u = isu ? own : other, v = isu ? other : own;
        const double A = p[0], B = p[1], alpha = p[2];
        const double dx = 1.0 / CELLS;
        const double cl = alpha / (dx * dx);
        const double uuv = u * u * v;
        const double lap = fma(-2.0, own, left) + right;
        const double react = isu ? fma(-(B + 1.0), u, A + uuv) : fma(B, u, -uuv);
        f = fma(cl, lap, react);
        return true;
    }
};

// A small system given as a register right-hand side (bg_device.h: f from
// the whole state): every lane of the group gathers the D components,
// evaluates f and keeps its own component.  The group is the power of two
// W >= D; lanes g >= D are padding that hold 0 in every vector, 0 as f, and
// the identity row and column of the Jacobian, so they never affect a sum,
// a pivot or an update.
template <class R>
struct GatherBdf {
    static constexpr int D = R::D, P = R::P;
    static constexpr int W = D <= 1 ? 1 : D <= 2 ? 2 : D <= 4 ? 4 : D <= 8 ? 8 : D <= 16 ? 16 : 32;
    static_assert(D <= 16, "gathered systems take at most a 16-lane group");
    template <class G, int... K>
    __device__ __forceinline__ static void gather(double y, const G &grp, double (&yy)[D],
                                                  std::integer_sequence<int, K...>) {
        ((yy[K] = grp.template bcast_at<K>(y)), ...);
    }
    template <class G>
    __device__ static bool lane_eval(double t, double y, const double *p, const G &grp, double &f) {
        double yy[D], ff[D];
        gather(y, grp, yy, std::make_integer_sequence<int, D>{});
        const bool ok = R::eval(t, yy, p, ff);
        f = 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) f = grp.g == k ? ff[k] : f;
        return ok;
    }
};

// quirk register as compile-time data (bdf.rs:403-407, 568, 622)
template <bool AsBuilt>
struct BdfSem {
    static constexpr double fd_sign = AsBuilt ? 1.0 : -1.0;  // Q3
    static constexpr bool lower_own_hist = !AsBuilt;         // Q4
    static constexpr double theta = AsBuilt ? 0.0 : 1.0;     // Q5
    static constexpr bool restore_mul = !AsBuilt;            // Q6
};

// BDF coefficients (bdf.rs:646-672, 713-729)
template <int O>
struct BdfCoef;
template <>
struct BdfCoef<7> {
    __device__ static constexpr double hi(int k) {
        constexpr double h = 147.0;
        constexpr double c[7] = {60.0 / h, -360.0 / h, 450.0 / h, -400.0 / h,
                                 225.0 / h, -72.0 / h, 10.0 / h};
        return c[k];
    }
    __device__ static constexpr double lo(int k) {
        constexpr double l = 137.0;
        constexpr double c[7] = {60.0 / l, -300.0 / l, 300.0 / l, -200.0 / l,
                                 75.0 / l, -12.0 / l, 0.0};
        return c[k];
    }
};
template <>
struct BdfCoef<3> {
    __device__ static constexpr double hi(int k) {
        constexpr double c[3] = {2.0 / 3.0, -4.0 / 3.0, 1.0 / 3.0};
        return c[k];
    }
    __device__ static constexpr double lo(int k) {
        constexpr double c[3] = {1.0, -1.0, 0.0};
        return c[k];
    }
};

enum : int { BDF_YIELD = -1, BDF_REDO = -2, BDF_DONE = -3 };

// ---------------------------------------------------------------------------
// one group's BDF solver state (per lane: its component / its row)
// ---------------------------------------------------------------------------
// SPLIT = 1: a group of W = D lanes per instance; lane g owns component g and
// row g of the Jacobian inverse.  SPLIT = 2: the whole wave per instance
// (2 W = 64 lanes): lane (h, g) = h W + g owns component g (both halves hold
// the same component values, computed redundantly) and the half row
// Jinv[g][h W/2 .. h W/2 + W/2 - 1].  The split halves the registers for the
// inverse, runs the FD Jacobian's +dt and -dt evaluations on the two halves
// at once, and leaves no second instance in the wave to diverge from.
template <class RHS, int O, class Sem, class LuT, int SPLIT = 1>
struct BdfLane {
    // D components in a group of W lanes (W = D except for padded gathered
    // systems); SPLIT = 2 only for D = W = 32
    static constexpr int D = RHS::D, W = RHS::W, WJ = W / SPLIT;
    using C = BdfCoef<O>;
    Grp<W> grp;
    int h = 0;    // half of the wave (SPLIT = 2)
    double *lds;  // this group's W x (W+1) transpose buffer, then 2 scalars
    float *prow_f = nullptr;  // SPLIT = 2, FP32 inverse: the pivot row

    // The elimination's pivot row (W entries) in the inverse's arithmetic
    // type: FP64 uses the group's LDS buffer (its row 0, free during the
    // elimination), FP32 a float buffer of its own.  1 / pivot goes from the
    // pivot lane by readlane.
    __device__ __forceinline__ LuT *pivot_row() const {
        if constexpr (sizeof(LuT) == sizeof(double)) return lds;
        else return prow_f;
    }
    // instance scalars (replicated across the group)
    double t, dt, end, tol, dt_min, dt_max;
    int yield_memory;
    bool hist_full;
    double hist_t[O];
    // per-lane component data
    double y, save;
    double hist[O];  // prev_values front..back (own component)
    double jinv[WJ];  // row g of the Jacobian inverse (SPLIT = 2: half row h)
    double p[RHS::P > 0 ? RHS::P : 1];
    // counters
    uint32_t n_newton, n_lu;

    __device__ __forceinline__ bool f(double tt, double yy, double &out) const {
        return RHS::lane_eval(tt, yy, p, grp, out);
    }

    // hist push_back + pop_front on a full deque
    __device__ __forceinline__ void hist_shift(double tt, double yy) {
#pragma unroll
        for (int k = 0; k < O - 1; ++k) {
            hist[k] = hist[k + 1];
            hist_t[k] = hist_t[k + 1];
        }
        hist[O - 1] = yy;
        hist_t[O - 1] = tt;
    }

    // bdf.rs:346-387: classical RK4, `iterations` steps; with fill = true the
    // deque is rebuilt from the states after steps 1..O (O == iterations).
    template <int IT, bool FILL>
    __device__ __forceinline__ int runge_kutta() {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            double k1, k2, k3, k4;
            if (!f(t, y, k1)) return BG_USER_ERROR;
            k1 *= dt;
            if (!f(t + 0.5 * dt, y + k1 * 0.5, k2)) return BG_USER_ERROR;
            k2 *= dt;
            if (!f(t + 0.5 * dt, y + k2 * 0.5, k3)) return BG_USER_ERROR;
            k3 *= dt;
            if (!f(t + dt, y + k3, k4)) return BG_USER_ERROR;
            k4 *= dt;
            if (FILL && i != 0) {
                hist[i - 1] = y;
                hist_t[i - 1] = t;
            }
            y += (k1 + k2 * 2.0 + k3 * 2.0 + k4) * (1.0 / 6.0);
            t += dt;
        }
        if (FILL) {
            hist[IT - 1] = y;
            hist_t[IT - 1] = t;
            hist_full = true;
        }
        return BG_OK;
    }

    // residual closures bdf.rs:548-575 (lane g's component), given
    // fx = f(t_n, x)_g
    template <bool LOWER>
    __device__ __forceinline__ double combine(double fx, double x) const {
        constexpr bool own = LOWER && Sem::lower_own_hist;
        double g = (-fx) * dt * (LOWER ? C::lo(0) : C::hi(0));
#pragma unroll
        for (int ind = 1; ind < O; ++ind) {
            const double c = own ? C::lo(ind) : C::hi(ind);
            if (c != 0.0) g = fma(hist[O - ind], c, g);
        }
        return g + x;
    }

    template <bool LOWER>
    __device__ __forceinline__ bool residual(double tt, double x, double &g) const {
        double fx;
        if (!f(tt, x, fx)) return false;
        g = combine<LOWER>(fx, x);
        return true;
    }

    // every component of x to every lane of a quad or pair
    template <int... K>
    __device__ __forceinline__ void spread(double x, double (&xs)[W],
                                           std::integer_sequence<int, K...>) const {
        ((xs[K] = grp.template bcast_at<K>(x)), ...);
    }

    // SPLIT = 2: component h W/2 + j of v in lane j of each 16-lane row, where
    // multiply-adds take it as their broadcast operand.  32,768 Brusselator
    // instances against 16 values per lane through LDS in each product and
    // update: 82.9 -> 79.4 ms (FP32 inverse 56.2 -> 53.6).
    __device__ __forceinline__ double half_columns(double v) const {
        const double o = xor16_f64(v);
        return (grp.g >> 4) == h ? v : o;
    }

    // y_g = -(Jinv x)_g with x broadcast through LDS (quads: DPP moves; the
    // whole wave: half_columns)
    __device__ __forceinline__ double neg_jinv_times(double x) {
        if constexpr (W <= 4) {
            double xs[W];
            spread(x, xs, std::make_integer_sequence<int, W>{});
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < W; ++j) acc = fma(jinv[j], xs[j], acc);
            return -acc;
        }
        double acc = 0.0;
        if constexpr (SPLIT == 2) {
            const double xs = lane_operand(half_columns(x));
            for_ints<WJ>([&](auto col) {
                constexpr int j = decltype(col)::value;
                acc = fma_newbcast<j, j == WJ - 1>(xs, jinv[j], acc);
            });
            acc += xor32_f64(acc);
        } else {
            lds[grp.g] = x;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < WJ; ++j) acc = fma(jinv[j], lds[j], acc);
            __builtin_amdgcn_wave_barrier();
        }
        return -acc;
    }

    // All-reduce sum of the component values.  SPLIT = 2: both halves hold
    // the same values, so half 0's two 16-lane row sums, added once,
    // replace the cross-row swap (the same bits: r0 + r1 = r1 + r0).
    __device__ __forceinline__ double comp_sum(double v) const {
        if constexpr (SPLIT == 2) {
            v += dpp_f64<0xB1>(v);
            v += dpp_f64<0x4E>(v);
            v += dpp_f64<0x141>(v);
            v += dpp_f64<0x140>(v);
            return readlane_lu(v, 0) + readlane_lu(v, 16);
        } else {
            return grp.sum(v);
        }
    }

    // In-place Gauss-Jordan inversion (exchange steps) of the group matrix
    // whose row g is staged in row g of the LDS buffer, with partial pivoting
    // on rows that are not swapped: column k pivots on the unused row p with
    // the largest |a(p,k)| (pivot_key: lowest lane on ties).  Afterwards lane
    // p holds row col(p) of the inverse with its columns permuted by col(),
    // which one LDS scatter/gather undoes.  Arithmetic in LuT; returns false
    // on a zero (or NaN) pivot.
    __device__ __forceinline__ bool invert() {
        if constexpr (SPLIT == 2) return invert_split();
        else return invert_group();
    }

    // SPLIT = 2: the same exchange steps on half rows.  Column k lives in
    // half k / WJ; the other half fetches a(g, k) across the halves.
    // Normalisation is deferred: the pivot row is published unscaled with
    // 1 / pivot beside it (LDS slot W, the padding column of row 0, unused
    // until the final scatter), the other rows eliminate with
    // f = a(g, k) / pivot, and each row is scaled by its own 1 / pivot once
    // at the end.  A row that has been a pivot row holds pivot times its
    // normalised values, so later updates stay consistent; this saves the
    // per-step scaling of the pivot row.
    //
    // The step was bound by the LDS unit: 64 lanes reading the half row as 8
    // broadcast b128 loads (8 cycles each) beside its 8 stores, for 16
    // multiply-adds.  Lane j of a 16-lane row now reads column j alone, one
    // b64 load, and the multiply-adds take it as their broadcast operand at
    // the full rate (FP32: at half rate, still the shorter way).  What is left
    // is the stores (57 % of the LDS unit's cycles) and the vector issue
    // (60 %).  32,768 Brusselator instances to t = 10: FP64 98.5 -> 83.0 ms,
    // FP32 60.9 -> 56.2.  With the matrix spread over the wave by columns, one
    // store of the pivot row in place of 8, the row's choice at run time cost
    // more than the stores (101 ms).
    __device__ __forceinline__ bool invert_split() {
        LuT b[WJ];
#pragma unroll
        for (int j = 0; j < WJ; ++j) b[j] = (LuT)lds[grp.g * (W + 1) + h * WJ + j];
        __builtin_amdgcn_wave_barrier();
        bool used = false;
        // the smallest key so far: a running minimum, so no column's key
        // stays live until the end of the elimination
        uint32_t key_min = ~0u;
        int my_col = 0;
        LuT my_inv = (LuT)1;
        LuT *const prow = pivot_row();
        for_ints<W>([&](auto column) {
            constexpr int k = decltype(column)::value, hk = k / WJ, kk = k % WJ;
            const LuT mk = b[kk];
            // half hk holds column k in its own lanes: its reduction is the
            // key (the other half reduces another column, unused), and the
            // lane swap for the other half's copy stays off the search
            // (the maxima of its two 16-lane rows, combined in scalars)
            const uint32_t rm = row_max_u32(pivot_key32(mk, !used, grp.g));
            const uint32_t key = __builtin_elementwise_max(
                (uint32_t)__builtin_amdgcn_readlane((int)rm, hk * W),
                (uint32_t)__builtin_amdgcn_readlane((int)rm, hk * W + 16));
            const LuT agk = half_lu(mk, hk);
            key_min = __builtin_elementwise_min(key_min, key);
            const int pl = pivot_lane32(key);
            const bool piv = (pl == grp.g);
            if (piv) {
#pragma unroll
                for (int j = 0; j < WJ; ++j) prow[h * WJ + j] = b[j];
            }
            used = used || piv;
            my_col = piv ? k : my_col;
            __builtin_amdgcn_wave_barrier();
            // lane j of a 16-lane row reads column j of its half
            const LuT from_lds = prow[h * WJ + (grp.g & 15)];
            __builtin_amdgcn_wave_barrier();
            // 1 / pivot in every lane (the pivot is wave-uniform), while the
            // row is on its way through LDS
            const LuT inv = pivot_recip(readlane_lu(mk, hk * W + pl));
            my_inv = piv ? inv : my_inv;
            // here, not deferred to the end of the elimination with all the
            // columns' pivots kept until then
            asm("" : "+v"(my_inv));
            asm("" : "+s"(key_min));
            // Every lane updates, so the next column's pivot search can
            // overlap this step's FMAs.  The pivot row's lanes read back
            // their own row and take factor +0: fma(+0, b, b) = b for every
            // finite b, zeros' signs included (an infinite entry turns into
            // NaN instead of staying infinite: the inverse is not finite
            // either way).
            const LuT f = agk * inv;
            LuT nf = piv ? (LuT)0 : -f;
            // the next column first: its pivot search starts while the others
            // are updated
            constexpr int next = (kk + 1) % WJ;
            const LuT pr = lane_operand(from_lds, nf);
            b[next] = fma_newbcast<next, true>(pr, nf, b[next]);
            for_ints<WJ>([&](auto col) {
                constexpr int j = decltype(col)::value;
                if constexpr (j != next) b[j] = fma_newbcast<j, false>(pr, nf, b[j]);
            });
            // column k of the inverse: pivot * (1 / pivot) on the pivot row,
            // -a(g, k) / pivot elsewhere
            if (h == hk) b[kk] = piv ? (LuT)1 : -f;
            __builtin_amdgcn_wave_barrier();
        });
        const bool ok = pivot_nonzero32(key_min);
#pragma unroll
        for (int j = 0; j < WJ; ++j) b[j] *= my_inv;
#pragma unroll
        for (int c = 0; c < WJ; ++c) lds[my_col * (W + 1) + h * WJ + c] = (double)b[c];
        lds[grp.g * (W + 1) + W] = (double)my_col;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < WJ; ++q) {
            int cq = (int)lds[(h * WJ + q) * (W + 1) + W];
            cq = cq < 0 ? 0 : (cq >= W ? W - 1 : cq);
            jinv[q] = lds[grp.g * (W + 1) + cq];
        }
        __builtin_amdgcn_wave_barrier();
        return ok;
    }

    __device__ __forceinline__ bool invert_group() {
        LuT b[W];
#pragma unroll
        for (int j = 0; j < W; ++j) b[j] = (LuT)lds[grp.g * (W + 1) + j];
        __builtin_amdgcn_wave_barrier();
        return invert_row(b);
    }

    // The elimination on the rows in registers (b: row g).  The pivot row,
    // scaled, goes to the other lanes through LDS, within a pair or quad by
    // lane shuffles.  A padding row is its own column's pivot and changes no
    // other row: its columns are not eliminated.
    __device__ __forceinline__ bool invert_row(LuT (&b)[W]) {
        bool used = grp.g >= D, ok = true;
        int my_col = grp.g >= D ? grp.g : 0;
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const double key = grp.max(pivot_key((double)b[k], !used, grp.g));
            if (!pivot_nonzero(key)) ok = false;
            const int pl = pivot_lane(key);
            const bool piv = (pl == grp.g);
            if constexpr (W == 1) {
                b[0] = (LuT)1 / b[0];
            } else if constexpr (W <= 4) {
                const LuT ip = (LuT)1 / b[k];
                const LuT f = b[k];
                LuT pr[W];
#pragma unroll
                for (int j = 0; j < D; ++j) pr[j] = j == k ? ip : b[j] * ip;
#pragma unroll
                for (int j = 0; j < D; ++j) pr[j] = __shfl(pr[j], pl, W);
#pragma unroll
                for (int j = 0; j < D; ++j) {
                    const LuT other = j == k ? -f * pr[k] : fma(-f, pr[j], b[j]);
                    b[j] = piv ? pr[j] : other;
                }
            } else {
                if (piv) {
                    const LuT ip = (LuT)1 / b[k];
#pragma unroll
                    for (int j = 0; j < W; ++j)
                        if (j != k) b[j] *= ip;
                    b[k] = ip;
#pragma unroll
                    for (int j = 0; j < W; ++j) lds[j] = (double)b[j];
                }
                __builtin_amdgcn_wave_barrier();
                if (!piv) {
                    const LuT f = b[k];
#pragma unroll
                    for (int j = 0; j < W; ++j)
                        if (j != k) b[j] = fma(-f, (LuT)lds[j], b[j]);
                    b[k] = -f * (LuT)lds[k];
                }
                __builtin_amdgcn_wave_barrier();
            }
            if (piv) {
                used = true;
                my_col = k;
            }
        }
        if constexpr (W == 1) {
            jinv[0] = (double)b[0];
            return ok;
        }
        // lane p: row col(p) of the inverse, column c belongs to inverse
        // column q with col(q) = c.  Scatter rows by col(), publish col() in
        // the padding column, gather with the column permutation.
#pragma unroll
        for (int c = 0; c < W; ++c) lds[my_col * (W + 1) + c] = (double)b[c];
        lds[grp.g * (W + 1) + W] = (double)my_col;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < W; ++q) {
            int cq = (int)lds[q * (W + 1) + W];
            cq = cq < 0 ? 0 : (cq >= W ? W - 1 : cq);
            jinv[q] = lds[grp.g * (W + 1) + cq];
        }
        __builtin_amdgcn_wave_barrier();
        return ok;
    }

    // The finite-difference Jacobian's right-hand sides (bdf.rs:396-406) for
    // both of a step's secants: they start from the same guess at the same
    // time, so the derivatives at the perturbed states are the same and only
    // their combination with the history differs.  fx: own component of
    // f(t, x + dt e_c) and f(t, x - dt e_c).
    static constexpr bool kSharedFd = SPLIT == 1 && W <= 8;
    struct FdPoints {
        double f0, above[kSharedFd ? D : 1], below[kSharedFd ? D : 1];
    };
    __device__ __forceinline__ bool fd_points(double tt, FdPoints &fd) const {
        double x = y;
        if (!f(tt, x, fd.f0)) return false;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            const bool mine = (grp.g == c);
            x = mine ? x + dt : x;
            if (!f(tt, x, fd.above[c])) return false;
            x = mine ? x - 2.0 * dt : x;
            if (!f(tt, x, fd.below[c])) return false;
            x = mine ? x + dt : x;
        }
        return true;
    }
    // Row g of the Jacobian from them; leaves the guess as the reference's
    // column loop does.
    template <bool LOWER>
    __device__ __forceinline__ void fd_row(const FdPoints &fd, double denom, double &guess,
                                           LuT (&b)[W]) const {
        guess = y;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            const bool mine = (grp.g == c);
            guess = mine ? guess + dt : guess;
            const double above = combine<LOWER>(fd.above[c], guess);
            guess = mine ? guess - 2.0 * dt : guess;
            const double below = combine<LOWER>(fd.below[c], guess);
            guess = mine ? guess + dt : guess;
            b[c] = (LuT)((above + Sem::fd_sign * below) * denom);
        }
#pragma unroll
        for (int c = D; c < W; ++c) b[c] = grp.g == c ? (LuT)1 : (LuT)0;
        if (grp.g >= D) {
#pragma unroll
            for (int c = 0; c < D; ++c) b[c] = (LuT)0;
        }
    }

    // bdf.rs:390-411 for the whole-wave layout (SPLIT = 2): the
    // finite-difference Jacobian by column colouring.  The reference's loop
    // perturbs one column at a time (x_c + dt, then x_c + dt - 2 dt, then
    // restores x_c as x_c + dt - 2 dt + dt, which may differ from x_c by a
    // rounding), so column c is evaluated at a state whose components
    // before c are restored and after c original.  Entry (g, c) depends only
    // on row g's stencil, so one evaluation per colour (half 0 at + dt,
    // half 1 at - dt) gives every row its entry of that colour, each lane at
    // the state its own column c would see: the same inputs, hence the same
    // bits, as the column loop.  Entries outside the stencil see identical
    // inputs above and below: the central difference (intended) makes them
    // exactly 0; the sum (as built, Q3) makes them (G + G) / (2 dt) at the
    // unperturbed state of their column, which depends only on how many
    // stencil members precede the column (at most five states).  Lane
    // (h, g) writes the entries of its half row h into row g of the LDS
    // buffer.  Returns the guess after the loop (every component restored).
    template <bool LOWER>
    __device__ __forceinline__ bool fd_coloured(double tt, double denom, double &guess) {
        const double orig = guess;
        const double xp = orig + dt, xm = xp - 2.0 * dt;
        const double rest = xm + dt;  // the reference's restore (bdf.rs:405)
        const double pert = h == 0 ? xp : xm;
        const int g = grp.g;
        double *row = lds + g * (W + 1);
        if constexpr (Sem::fd_sign > 0.0) {
            // as built: the dense part, from the unperturbed states
            int s[4];
            RHS::stencil(g, s);
            double Gm[5];
#pragma unroll
            for (int m = 0; m < 5; ++m) {
                // a column with exactly m stencil members before it, if the
                // row has one (otherwise the value is not used)
                const int rep = m == 0 ? 0 : s[m - 1] + 1;
                double fx, own;
                if (!RHS::lane_eval_state(tt, orig, rest, pert, rep, p, grp, fx, own)) return false;
                Gm[m] = combine<LOWER>(fx, own);
            }
#pragma unroll
            for (int j = 0; j < WJ; ++j) {
                const int c = h * WJ + j;
                const int m = (s[0] < c) + (s[1] < c) + (s[2] < c) + (s[3] < c);
                double v = Gm[0];
#pragma unroll
                for (int q = 1; q < 5; ++q) v = m == q ? Gm[q] : v;
                row[c] = (v + Sem::fd_sign * v) * denom;
            }
        } else {
#pragma unroll
            for (int j = 0; j < WJ; ++j) row[h * WJ + j] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < RHS::NC; ++k) {
            const int c = RHS::member(g, k);
            double fx, own;
            if (!RHS::lane_eval_state(tt, orig, rest, pert, c, p, grp, fx, own)) return false;
            const double r = combine<LOWER>(fx, own);
            const double other = xor32_f64(r);
            const double above = h == 0 ? r : other, below = h == 0 ? other : r;
            if (c / WJ == h) row[c] = (above + Sem::fd_sign * below) * denom;
        }
        guess = rest;
        return true;
    }

    // bdf.rs:390-411: the finite-difference Jacobian into the LDS rows,
    // starting from guess = y; leaves the guess as the reference's column
    // loop does.  False on a UserError.
    template <bool LOWER>
    __device__ __forceinline__ bool fd_jacobian(double tt, double denom, double &guess) {
        guess = y;
        if constexpr (SPLIT == 2) {
            if (!fd_coloured<LOWER>(tt, denom, guess)) return false;
        } else {
        // columns (G(x + dt e_c) +/- G(x - dt e_c)) / (2 dt); lane g stores
        // J(g, c) into row g of the group's LDS buffer
#pragma unroll 1
        for (int c = 0; c < W; ++c) {
            if (c >= D) {  // padding column: e_c
                lds[grp.g * (W + 1) + c] = grp.g == c ? 1.0 : 0.0;
                continue;
            }
            const bool mine = (grp.g == c);
            if (mine) guess += dt;
            double above, below;
            if (!residual<LOWER>(tt, guess, above)) return false;
            if (mine) guess -= 2.0 * dt;
            if (!residual<LOWER>(tt, guess, below)) return false;
            if (mine) guess += dt;
            lds[grp.g * (W + 1) + c] = (above + Sem::fd_sign * below) * denom;
        }
        }
        __builtin_amdgcn_wave_barrier();
        return true;
    }

    // ---- the rest of the inverse cascade (bdf.rs:429-444) -----------------
    // nalgebra tries partial-pivot LU, then full-pivot LU, then QR, and
    // reports SingularMatrix only when all three meet an exact zero pivot.
    // The fast path is the partial-pivot elimination above; when it finds
    // no pivot, these two run on the same matrix (rebuilt in the LDS rows by
    // fd_jacobian).  They are rare, so they work in LDS with rolled loops
    // (few registers) and keep their per-lane temporaries in private memory.
    // Both halves of a whole-wave group compute the same values; every lane
    // ends holding its part of row g of the inverse in jinv.
    __device__ __forceinline__ double &mat(int r, int c) const { return lds[r * (W + 1) + c]; }

    // row g of the inverse, given as the matrix M whose row qinv(g) holds
    // row g with column j at position col(j); col(r) is in mat(r, W).
    __device__ __forceinline__ void gather_permuted_row() {
        const int g = grp.g;
        int src = 0;
#pragma unroll 1
        for (int r = 0; r < W; ++r) src = ((int)mat(r, W) == g) ? r : src;
        double row[WJ];
#pragma unroll
        for (int q = 0; q < WJ; ++q) {
            int cq = (int)mat(h * WJ + q, W);
            cq = cq < 0 ? 0 : (cq >= W ? W - 1 : cq);
            row[q] = mat(src, cq);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < WJ; ++q) jinv[q] = row[q];
    }

    // Full-pivot Gauss-Jordan (exchange steps): step k pivots on the largest
    // |a| over the unused rows and columns (first column, then lowest row,
    // on ties) and fails on an exact zero, like FullPivLU's try_inverse.
    __device__ __forceinline__ bool invert_full_pivot() {
        const int g = grp.g;
        bool used = false;
        uint32_t ucols = 0;  // columns already pivoted (the same in every lane)
        int my_col = -1;
#pragma unroll 1
        for (int k = 0; k < W; ++k) {
            double best = -1.0;
            int bc = 0;
            if (!used) {
#pragma unroll 1
                for (int c = 0; c < W; ++c) {
                    const double v = fabs(mat(g, c));
                    if (!((ucols >> c) & 1u) && v > best) {
                        best = v;
                        bc = c;
                    }
                }
            }
            const double gmax = grp.max(best);
            if (!(gmax > 0.0)) return false;
            const uint32_t key = grp.max_u32((!used && best == gmax) ? (uint32_t)(63 - g) : 0u);
            const int p = 63 - (int)key;
            const int q = (int)grp.bcast((double)bc, p);
            const double ip = 1.0 / mat(p, q);
            __builtin_amdgcn_wave_barrier();
            if (g == p) {
#pragma unroll 1
                for (int j = 0; j < W; ++j) mat(p, j) = j == q ? ip : mat(p, j) * ip;
                used = true;
                my_col = q;
            }
            __builtin_amdgcn_wave_barrier();
            if (g != p) {
                const double fq = mat(g, q);
#pragma unroll 1
                for (int j = 0; j < W; ++j)
                    if (j != q) mat(g, j) = fma(-fq, mat(p, j), mat(g, j));
                mat(g, q) = -fq * ip;
            }
            ucols |= 1u << q;
            __builtin_amdgcn_wave_barrier();
        }
        mat(g, W) = (double)my_col;
        __builtin_amdgcn_wave_barrier();
        gather_permuted_row();
        return true;
    }

    // Householder QR (reflections chosen away from cancellation), failing on
    // an exact zero on R's diagonal like QR's try_inverse.  Reflection k is
    // kept below the diagonal of column k, scaled to a unit leading entry,
    // with its factor in mat(k, W).  Row g of the inverse R^-1 Q^T is
    // (Q w)^T with R^T w = e_g, solved by each lane on its own.
    __device__ __forceinline__ bool invert_qr() {
        const int g = grp.g;
#pragma unroll 1
        for (int k = 0; k < W; ++k) {
            const double x = g >= k ? mat(g, k) : 0.0;
            const double nrm = sqrt(grp.sum(x * x));
            const double akk = mat(k, k);
            const double alpha = akk >= 0.0 ? -nrm : nrm;
            const double vk = akk - alpha;
            double v = g > k ? x : (g == k ? vk : 0.0);
            const double vv = grp.sum(v * v);
            const bool skip = nrm == 0.0 || vv == 0.0;
            const double beta = skip ? 0.0 : 2.0 / vv;
#pragma unroll 1
            for (int c = k; c < W; ++c) {
                const double dot = grp.sum(v * mat(g, c));
                __builtin_amdgcn_wave_barrier();
                if (g >= k) mat(g, c) = fma(-(beta * dot), v, mat(g, c));
                __builtin_amdgcn_wave_barrier();
            }
            // unit leading entry: v / vk, factor beta vk^2
            const double sv = skip ? 0.0 : v / vk;
            if (g > k) mat(g, k) = sv;
            if (g == k) mat(k, W) = skip ? 0.0 : beta * vk * vk;
            __builtin_amdgcn_wave_barrier();
        }
        bool ok = true;
#pragma unroll 1
        for (int k = 0; k < W; ++k) ok = ok && mat(k, k) != 0.0;
        if (!ok) return false;
        double w[W];
#pragma unroll 1
        for (int i = 0; i < W; ++i) {  // R^T w = e_g, forward
            double s = i == g ? 1.0 : 0.0;
#pragma unroll 1
            for (int l = 0; l < i; ++l) s = fma(-mat(l, i), w[l], s);
            w[i] = s / mat(i, i);
        }
#pragma unroll 1
        for (int k = W - 1; k >= 0; --k) {  // w <- H_k w, last reflection first
            const double bk = mat(k, W);
            double dot = w[k];
#pragma unroll 1
            for (int i = k + 1; i < W; ++i) dot = fma(mat(i, k), w[i], dot);
            const double sc = bk * dot;
            w[k] -= sc;
#pragma unroll 1
            for (int i = k + 1; i < W; ++i) w[i] = fma(-sc, mat(i, k), w[i]);
        }
#pragma unroll
        for (int q = 0; q < WJ; ++q) jinv[q] = w[h * WJ + q];
        __builtin_amdgcn_wave_barrier();
        return true;
    }

    // bdf.rs:414-475; on success `guess` holds the corrected value.
    template <bool LOWER>
    __device__ __forceinline__ int secant(const FdPoints &fd, double &guess) {
        const double tt = t + Sem::theta * dt;
        const double denom = 1.0 / (2.0 * dt);
        double F;
        guess = y;
        bool inverted;
        if constexpr (kSharedFd) {
            F = combine<LOWER>(fd.f0, guess);
            LuT b[W];
            fd_row<LOWER>(fd, denom, guess, b);
            ++n_lu;
            inverted = invert_row(b);
        } else {
            double fx0;
            if (!f(tt, guess, fx0)) return BG_USER_ERROR;
            F = combine<LOWER>(fx0, guess);
            if (!fd_jacobian<LOWER>(tt, denom, guess)) return BG_USER_ERROR;
            ++n_lu;
            inverted = invert();
        }
        if (!inverted) {
            // bdf.rs:432-441: full-pivot LU, then QR, each on the Jacobian
            // rebuilt from the same evaluations
            if (!fd_jacobian<LOWER>(tt, denom, guess)) return BG_USER_ERROR;
            if (!invert_full_pivot()) {
                if (!fd_jacobian<LOWER>(tt, denom, guess)) return BG_USER_ERROR;
                if (!invert_qr()) return BG_SINGULAR_MATRIX;
            }
        }
        double s = neg_jinv_times(F);
        guess += s;
#pragma unroll 1
        for (int n = 2; n < 1000; ++n) {
            const double Fl = F;
            if (!residual<LOWER>(tt, guess, F)) return BG_USER_ERROR;
            ++n_newton;
            const double adj = neg_jinv_times(F - Fl);
            // p = (-s)^T adj ; u = s^T Jinv (column sums through LDS)
            const double pp = comp_sum(adj * (-s));
#pragma unroll
            for (int j = 0; j < WJ; ++j) lds[grp.g * (W + 1) + h * WJ + j] = jinv[j] * s;
            __builtin_amdgcn_wave_barrier();
            double u = 0.0;
            if constexpr (SPLIT == 2) {
                // column g: rows of half h, then the other half's partial sum
#pragma unroll
                for (int k = 0; k < WJ; ++k) u += lds[(h * WJ + k) * (W + 1) + grp.g];
                u += xor32_f64(u);
            } else {
#pragma unroll
                for (int k = 0; k < W; ++k) u += lds[k * (W + 1) + grp.g];
            }
            __builtin_amdgcn_wave_barrier();
            const double w = (s + adj) / pp;
            if constexpr (W <= 4) {
                double us[W];
                spread(u, us, std::make_integer_sequence<int, W>{});
#pragma unroll
                for (int j = 0; j < W; ++j) jinv[j] = fma(us[j], w, jinv[j]);
            } else if constexpr (SPLIT == 2) {
                const double us = lane_operand(half_columns(u));
                for_ints<WJ>([&](auto col) {
                    constexpr int j = decltype(col)::value;
                    jinv[j] = fma_newbcast<j, false>(us, w, jinv[j]);
                });
            } else {
                lds[grp.g] = u;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int j = 0; j < WJ; ++j) jinv[j] = fma(lds[j], w, jinv[j]);
                __builtin_amdgcn_wave_barrier();
            }
            // s = -Jinv_new F (bdf.rs:464-465) without a second product
            // through LDS: with Jinv_new = Jinv + w u^T and Jinv F = -adj - s
            // (the previous s was -Jinv F_l), -Jinv_new F = adj + s - w (u . F);
            // equal in exact arithmetic, other roundings
            const double uf = comp_sum(u * F);
            s = fma(-w, uf, adj + s);
            guess += s;
            if (norm_below<SPLIT == 1, true>(comp_sum(s * s), tol)) return BG_OK;
        }
        return BG_MAXIMUM_ITERATIONS_EXCEEDED;
    }

    // One call of BDFSolver::step (bdf.rs:495-634).  Returns BDF_YIELD,
    // BDF_REDO, BDF_DONE or an IVPError code.  On a yield, (*yt, *yv) is the
    // yielded value (own component).
    __device__ __forceinline__ int step(double *yt, double *yv, bool *rejected) {
        *rejected = false;
        if (yield_memory > 0 && yield_memory <= O) {  // bdf.rs:500-512
            const int item = O - yield_memory;
            yield_memory -= 1;
            if (yield_memory == 0) yield_memory = O + 2;
            double vt = hist_t[0], vy = hist[0];
#pragma unroll
            for (int k = 1; k < O; ++k)
                if (item == k) {
                    vt = hist_t[k];
                    vy = hist[k];
                }
            *yt = vt;
            *yv = vy;
            return BDF_YIELD;
        }
        if (yield_memory == O + 2) {  // bdf.rs:519-525
            yield_memory = 0;
            hist_shift(t, y);
            *yt = t;
            *yv = y;
            return BDF_YIELD;
        }
        if (t >= end) return BDF_DONE;
        if (t + dt >= end) {  // bdf.rs:531-535
            dt = end - t;
            const int rc = runge_kutta<1, false>();
            if (rc) return rc;
            *yt = t;
            *yv = y;
            return BDF_YIELD;
        }
        if (!hist_full) return bootstrap();
        const int rc = multistep(rejected);
        if (rc == BDF_YIELD) {
            *yt = t;
            *yv = y;
        }
        return rc;
    }

    // bdf.rs:537-546
    __device__ __forceinline__ int bootstrap() {
        save = y;
        if (t + dt * (double)O >= end) dt = (end - t) / (double)O;
        const int rc = runge_kutta<O, true>();
        if (rc) return rc;
        yield_memory = O + 1;
        return BDF_REDO;
    }

    // The step from a full history (bdf.rs:548-633); a yield is the current
    // (t, y)
    __device__ __forceinline__ int multistep(bool *rejected) {
        *rejected = false;
        double hi, lo;
        FdPoints fd;
        if constexpr (kSharedFd) {
            if (!fd_points(t + Sem::theta * dt, fd)) return BG_USER_ERROR;
        }
        int rc = secant<false>(fd, hi);
        if (rc) return rc;
        rc = secant<true>(fd, lo);
        if (rc) return rc;
        const double dlt = hi - lo;
        const double error2 = grp.sum(dlt * dlt);  // the squared error
        if (norm_below<SPLIT == 1, true>(error2, tol)) {  // bdf.rs:583-614
            y = hi;
            t += dt;
            if (yield_memory == O + 1) {
                yield_memory -= 1;
                return BDF_REDO;
            }
            hist_shift(t, y);
            if (norm_below<SPLIT == 1, false>(error2, 0.1 * tol)) {
                dt *= 2.0;
                if (dt > dt_max) dt = dt_max;
                hist_full = false;
            }
            return BDF_YIELD;
        }
        *rejected = true;
        if (yield_memory == O + 1) {  // bdf.rs:620-624
            if (Sem::restore_mul)
                t -= dt * (double)O;
            else
                t -= dt - (double)O;  // Q6
            y = save;
        }
        dt *= 0.5;
        if (dt < dt_min) return BG_MINIMUM_TIME_DELTA_EXCEEDED;
        hist_full = false;
        return BDF_REDO;
    }

    __device__ __forceinline__ void load(const bg_ensemble_desc &d, uint64_t i) {
        const uint64_t n = d.n;
        y = grp.g < D ? d.y0[(uint64_t)grp.g * n + i] : 0.0;
#pragma unroll
        for (int k = 0; k < RHS::P; ++k) p[k] = d.params[(uint64_t)k * n + i];
        t = d.t0 ? d.t0[i] : d.t0_s;
        end = d.t_end ? d.t_end[i] : d.t_end_s;
        tol = d.tol ? d.tol[i] : d.tol_s;
        dt_min = d.dt_min ? d.dt_min[i] : d.dt_min_s;
        dt_max = d.dt_max ? d.dt_max[i] : d.dt_max_s;
        dt = (dt_max + dt_min) * 0.5;  // bdf.rs:302
        yield_memory = 0;
        hist_full = false;
        save = y;
        n_newton = n_lu = 0;
#pragma unroll
        for (int k = 0; k < O; ++k) {
            hist[k] = 0.0;
            hist_t[k] = 0.0;
        }
    }
};

// ---------------------------------------------------------------------------
// persistent ensemble kernels
// ---------------------------------------------------------------------------
// One instance per wave (the 32-component system).
// Four waves per SIMD (the LDS limit) hide each other's waits in the
// elimination, a chain of pivot search, LDS round trip and reciprocal per
// step.  32,768 Brusselator instances, while the Broyden products still went
// through LDS: 82.9 ms with 4 waves and their spills, 85.9 with 3 (up to 20
// instances per CU the 3 win: bdf_kernel).
template <class RHS, int O, class Sem, class LuT, int WAVES>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES, 8)))
    bdf_wave_kernel(const bg_ensemble_desc, uint32_t *__restrict__ counter) {
    constexpr int W = RHS::W;
    static_assert(W == 32, "a whole wave per instance");
    __shared__ double lds_all[W * (W + 1) + 2];
    const karg_desc dv = kernarg_desc();
    const int lane = __lane_id();
    BdfLane<RHS, O, Sem, LuT, 2> L;
    L.grp.g = lane % W;
    L.h = lane / W;
    L.lds = lds_all;
    if constexpr (sizeof(LuT) == sizeof(float)) {
        __shared__ float prow_all[W];
        L.prow_f = prow_all;
    }
    const uint64_t max_att = dv->max_attempts;
    const uint32_t cap =
        (uint32_t)((max_att && max_att < kBdfDefaultMaxSteps) ? max_att : kBdfDefaultMaxSteps);
    // schedule position: the wave's own first, then from the counter
    uint32_t pos = blockIdx.x;
    for (;;) {
        const bg_ensemble_desc di = desc_inputs(dv);
        if (pos >= di.n) break;
        const uint64_t inst = di.order ? (uint64_t)di.order[pos] : (uint64_t)pos;
        L.load(di, inst);
        uint32_t steps = 0, nacc = 0, nrej = 0;
        int st;
        for (;;) {
            if (steps >= cap) {
                st = BG_MAXIMUM_ITERATIONS_EXCEEDED;
                break;
            }
            ++steps;
            double yt, yv;
            bool rej;
            const int r = L.step(&yt, &yv, &rej);
            if (rej) ++nrej;
            if (r == BDF_YIELD) {
                ++nacc;
            } else if (r == BDF_DONE) {
                st = BG_OK;
                break;
            } else if (r != BDF_REDO) {
                st = r;
                break;
            }
        }
        const bg_ensemble_desc d = desc_outputs(dv);
        const uint64_t n = d.n, i = inst;
        if (d.y_out && L.h == 0 && L.grp.g < RHS::D) d.y_out[(uint64_t)L.grp.g * n + i] = L.y;
        if (lane == 0) {
            if (d.t_out) d.t_out[i] = L.t;
            if (d.status) d.status[i] = st;
            if (d.counts) {
                bg_counts c;
                c.n_accepted = nacc;
                c.n_rejected = nrej;
                d.counts[i] = c;
            }
            if (d.work) {
                bg_counts c;
                c.n_accepted = L.n_newton;
                c.n_rejected = L.n_lu;
                d.work[i] = c;
            }
        }
        if (counter == nullptr) break;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(counter, 1u);
        pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    }
}

// One instance per group of W <= 16 lanes.
// A wave alone on its SIMD is bound by its instruction count, so the group
// collectives are DPP moves (a shuffle is two LDS-unit operations and a wait),
// the finite differences' right-hand sides are evaluated once for both
// secants, the bootstrap's yields are settled at once, and the groups take
// their bootstraps before a multistep that all of them share.  Two waves per
// SIMD are enough registers for the shared evaluations (four spilled them).
// 16,384 Robertson instances, 405 yields each: 0.86 -> 0.39 ms; 131,072 3.07 ->
// 1.85; Brusselator with 4 (8, 16) components, 8,192 instances, 0.74 -> 0.31
// (1.04 -> 0.58, 2.40 -> 1.61); Lotka-Volterra 0.76 -> 0.35.
template <class RHS, int O, class Sem, class LuT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8)))
    bdf_ensemble_kernel(const bg_ensemble_desc, uint32_t *__restrict__ counter) {
    constexpr int W = RHS::W;
    constexpr int GPW = 64 / W;  // groups per wave
    __shared__ double lds_all[GPW][W * (W + 1) + 2];
    const karg_desc dv = kernarg_desc();
    const int lane = __lane_id();
    const int grp_id = lane / W;
    BdfLane<RHS, O, Sem, LuT> L;
    L.grp.g = lane % W;
    L.lds = lds_all[grp_id];
    const bool leader = (lane % W == 0);
    const uint64_t max_att = dv->max_attempts;
    const uint32_t cap =
        (uint32_t)((max_att && max_att < kBdfDefaultMaxSteps) ? max_att : kBdfDefaultMaxSteps);
    // schedule position: the group's own first, then from the counter (which
    // starts behind the groups' own; none if every instance has a group)
    uint64_t pos = (uint64_t)blockIdx.x * GPW + grp_id;
    bool idle = false;  // this group has no further instance
    for (;;) {
        int64_t inst = -1;
        if (!idle) {
            const bg_ensemble_desc di = desc_inputs(dv);
            if (pos < di.n) {
                inst = di.order ? (int64_t)di.order[pos] : (int64_t)pos;
                L.load(di, (uint64_t)inst);
            } else {
                idle = true;
            }
        }
        if (inst >= 0) {
            // The groups of a wave go through the calls of step() together:
            // first the final RK4 step or the bootstrap of those that are
            // there, then the multistep of all that have a history, so a
            // group that bootstraps takes its multistep in the same pass as
            // the others.
            uint32_t steps = 0, nacc = 0, nrej = 0;
            int st = -1;
            while (st < 0) {
                int r = BDF_REDO;
                bool called = false;
                if (steps >= cap) {
                    st = BG_MAXIMUM_ITERATIONS_EXCEEDED;
                } else if (L.t >= L.end) {
                    ++steps;
                    st = BG_OK;
                } else if (L.t + L.dt >= L.end) {  // bdf.rs:531-535
                    ++steps;
                    called = true;
                    L.dt = L.end - L.t;
                    r = L.template runge_kutta<1, false>();
                    if (r == BG_OK) ++nacc;
                    else st = r;
                } else if (!L.hist_full) {
                    ++steps;
                    r = L.bootstrap();
                    if (r != BDF_REDO) st = r;
                }
                if (st < 0 && !called && L.hist_full && steps < cap && !(L.t >= L.end) &&
                    !(L.t + L.dt >= L.end)) {
                    ++steps;
                    bool rej;
                    r = L.multistep(&rej);
                    if (rej) ++nrej;
                    if (r == BDF_YIELD) {
                        ++nacc;
                    } else if (r != BDF_REDO) {
                        st = r;
                    } else if (L.yield_memory == O) {
                        // the first step after a bootstrap: the bootstrap's
                        // values and this one are yielded next, one call each
                        // (bdf.rs:500-525), which moves nothing but the history
                        const uint32_t room = cap - steps;
                        const uint32_t k = (uint32_t)O + 1u < room ? (uint32_t)O + 1u : room;
                        steps += k;
                        nacc += k;
                        L.yield_memory = 0;
                        L.hist_shift(L.t, L.y);
                    }
                }
            }
            const bg_ensemble_desc d = desc_outputs(dv);
            const uint64_t n = d.n, i = (uint64_t)inst;
            if (d.y_out && L.grp.g < RHS::D) d.y_out[(uint64_t)L.grp.g * n + i] = L.y;
            if (leader) {
                if (d.t_out) d.t_out[i] = L.t;
                if (d.status) d.status[i] = st;
                if (d.counts) {
                    bg_counts c;
                    c.n_accepted = nacc;
                    c.n_rejected = nrej;
                    d.counts[i] = c;
                }
                if (d.work) {
                    bg_counts c;
                    c.n_accepted = L.n_newton;
                    c.n_rejected = L.n_lu;
                    d.work[i] = c;
                }
            }
        }
        if (counter == nullptr) break;
        const uint64_t need = ballot(leader && !idle);
        if (need == 0) break;
        const int first = __ffsll((unsigned long long)need) - 1;
        uint32_t base = 0;
        if (lane == first) base = atomicAdd(counter, (uint32_t)__popcll(need));
        base = first_of(base, need);
        // rank of my group's leader among the leaders that ask
        pos = (uint64_t)base + (uint64_t)__popcll(need & ((1ull << (grp_id * W)) - 1ull));
    }
}

// Single-instance path production (one group): every yield is written into
// the path buffer; resumable when the buffer is full.
template <class RHS, int O, class Sem, class LuT>
__global__ void __launch_bounds__(64)
    bdf_path_kernel(BdfPathState *__restrict__ st, double *__restrict__ path_t,
                    double *__restrict__ path_y, uint32_t cap) {
    constexpr int D = RHS::D, W = RHS::W;
    __shared__ double lds[W * (W + 1) + 2];
    const int lane = __lane_id();
    if (lane >= W) return;
    BdfLane<RHS, O, Sem, LuT> L;
    L.grp.g = lane;
    L.lds = lds;
    L.t = st->t;
    L.dt = st->dt;
    L.end = st->end;
    L.tol = st->tol;
    L.dt_min = st->dt_min;
    L.dt_max = st->dt_max;
    L.yield_memory = st->yield_memory;
    L.hist_full = st->hist_full != 0;
    L.y = st->y[lane];
    L.save = st->save[lane];
#pragma unroll
    for (int k = 0; k < O; ++k) {
        L.hist[k] = st->hist[k][lane];
        L.hist_t[k] = st->hist_t[k];
    }
#pragma unroll
    for (int k = 0; k < RHS::P; ++k) L.p[k] = st->p[k];
    L.n_newton = st->n_newton;
    L.n_lu = st->n_lu;
    uint32_t count = 0;
    int status = BG_OK, finished = st->finished;
    uint64_t steps = st->steps;
    uint32_t nacc = st->n_accepted, nrej = st->n_rejected;
    while (!finished && count < cap) {
        if (steps >= st->max_steps) {
            status = BG_MAXIMUM_ITERATIONS_EXCEEDED;
            finished = 1;
            break;
        }
        ++steps;
        double yt, yv;
        bool rej;
        const int r = L.step(&yt, &yv, &rej);
        if (rej) ++nrej;
        if (r == BDF_YIELD) {
            ++nacc;
            if (lane == 0) path_t[count] = yt;
            if (lane < D) path_y[(uint64_t)count * D + lane] = yv;
            ++count;
        } else if (r == BDF_DONE) {
            finished = 1;
        } else if (r != BDF_REDO) {
            status = r;
            finished = 1;
        }
    }
    st->y[lane] = L.y;
    st->save[lane] = L.save;
#pragma unroll
    for (int k = 0; k < O; ++k) st->hist[k][lane] = L.hist[k];
    if (lane == 0) {
        st->t = L.t;
        st->dt = L.dt;
        st->yield_memory = L.yield_memory;
        st->hist_full = L.hist_full ? 1 : 0;
#pragma unroll
        for (int k = 0; k < O; ++k) st->hist_t[k] = L.hist_t[k];
        st->steps = steps;
        st->n_accepted = nacc;
        st->n_rejected = nrej;
        st->n_newton = L.n_newton;
        st->n_lu = L.n_lu;
        st->status = status;
        st->finished = finished;
        st->count = count;
    }
}

template <int = 0>
__global__ void bdf_counter_kernel(uint32_t *counter, uint32_t groups) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *counter = groups;
}

// ---------------------------------------------------------------------------
// The corrector's inverse cascade on caller matrices (bg_bdf_inverse_device):
// one matrix per group, W x W row-major in `a`; lane (h, g) stages row g in
// the group's LDS rows, runs partial-pivot Gauss-Jordan, and on failure the
// full-pivot and QR members on the reloaded matrix, exactly as the secant
// does (from member `first` on: 0 the whole cascade, 1 full pivot, 2 QR);
// it writes its part of row g of the inverse and the member that answered
// (0, 1, 2; -1: SingularMatrix).
// ---------------------------------------------------------------------------
template <int W_>
struct InverseOnly {  // a right-hand side in name only: the lane layout of W_
    static constexpr int D = W_, W = W_, P = 0;
};

template <int W, int SPLIT>
__global__ void __launch_bounds__(64)
    bdf_inverse_kernel(const double *__restrict__ a, double *__restrict__ inv,
                       int32_t *__restrict__ branch, uint64_t count, int first) {
    constexpr int GW = W * SPLIT, GPW = 64 / GW;
    __shared__ double lds_all[GPW][W * (W + 1) + 2];
    const int lane = __lane_id();
    const int grp_id = lane / GW;
    BdfLane<InverseOnly<W>, 7, BdfSem<false>, double, SPLIT> L;
    L.grp.g = lane % W;
    L.h = (lane % GW) / W;
    L.lds = lds_all[grp_id];
    const uint64_t m = (uint64_t)blockIdx.x * GPW + grp_id;
    const bool live = m < count;
    const uint64_t mm = live ? m : 0;  // a spare group inverts matrix 0 and writes nothing
    auto stage = [&]() {
        for (int c = 0; c < W; ++c)
            L.lds[L.grp.g * (W + 1) + c] = a[(mm * W + L.grp.g) * W + c];
        __builtin_amdgcn_wave_barrier();
    };
    stage();
    int br = first;
    bool ok = false;
    if (first == 0) ok = L.invert();
    if (!ok && first <= 1) {
        stage();
        br = 1;
        ok = L.invert_full_pivot();
    }
    if (!ok) {
        stage();
        br = 2;
        ok = L.invert_qr();
    }
    if (!ok) br = -1;
    if (!live) return;
#pragma unroll
    for (int q = 0; q < L.WJ; ++q) inv[(mm * W + L.grp.g) * W + L.h * L.WJ + q] = L.jinv[q];
    if (L.grp.g == 0 && L.h == 0) branch[mm] = br;
}

// ---------------------------------------------------------------------------
// launch (each translation unit instantiates its own set of systems)
// ---------------------------------------------------------------------------
template <class T>
struct BTag {
    using type = T;
};

// few: at most five waves per SIMD in all.  The kernel that is limited to three
// resident ones spills less; a second round of a third of them costs less than
// the spills up to there: to t = 10 4096 (5000, 6144, 9000) Brusselator
// instances take 15.8 (18.8, 21.8, 28.3) ms with it against 18.2 (19.2, 22.0,
// 28.0) with four resident; 256 to t = 4 2.8 against 3.1.
template <class R, int O, class S, class F>
static constexpr auto bdf_kernel(bool few) {
    if constexpr (R::W == 32)
        return few ? bdf_wave_kernel<R, O, S, F, 3> : bdf_wave_kernel<R, O, S, F, 4>;
    else return bdf_ensemble_kernel<R, O, S, F>;
}

// Persistent grid (one wave per block, as many as are resident, at most
// cap_per_cu per CU when cap_per_cu > 0) and the launch workspace: the work
// counter.  *occupancy, if given, receives the
// resident blocks per CU before the cap.
template <class R, int O, class S, class F>
static int bdf_launch_shape(const bg_ensemble_desc &d, uint64_t &grid, size_t &bytes, bool &few,
                            uint32_t cap_per_cu = 0, int *occupancy = nullptr) {
    constexpr int W = R::W;
    constexpr int SP = W == 32 ? 2 : 1;  // a 32-component instance takes the whole wave
    constexpr int GPW = 64 / (W * SP);
    int dev = 0;
    BG_HIP_CHECK(hipGetDevice(&dev));
    int per_cu = 0;
    few = d.n <= (uint64_t)(20 * device_cu_count(dev));
    BG_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, bdf_kernel<R, O, S, F>(few), 64, 0));
    if (occupancy) *occupancy = per_cu;
    if (cap_per_cu && (int)cap_per_cu < per_cu) per_cu = (int)cap_per_cu;
    if (per_cu < 1) per_cu = 1;
    grid = (uint64_t)per_cu * (uint64_t)device_cu_count(dev);
    const uint64_t need = (d.n + GPW - 1) / GPW;
    if (grid > need) grid = need;
    bytes = kLaunchWorkspaceBytes;
    return BG_OK;
}

template <class R, int O, class S, class F>
static int bdf_launch_one(const bg_ensemble_desc &d, hipStream_t stream, void *ws_in,
                          size_t ws_bytes, uint32_t cap_per_cu = 0) {
    if (d.n == 0) return BG_OK;
    if (d.n > 0x7fffffffull || !d.y0) return BG_ERR_INVALID_ARGUMENT;
    if (R::P > 0 && (!d.params || d.n_params < (uint32_t)R::P)) return BG_ERR_INVALID_ARGUMENT;
    constexpr int SP = R::W == 32 ? 2 : 1;
    uint64_t grid = 0;
    size_t bytes = 0;
    bool few = false;
    const int rc = bdf_launch_shape<R, O, S, F>(d, grid, bytes, few, cap_per_cu);
    if (rc != BG_OK) return rc;
    if (ws_in && ws_bytes < bytes) return BG_ERR_INVALID_ARGUMENT;
    // a group for every instance: no queue, no workspace
    constexpr int GPW = 64 / (R::W * SP);
    const bool queue = d.n > grid * GPW;
    char *ws = (char *)ws_in;
    if (queue) {
        if (!ws_in) BG_HIP_CHECK(hipMallocAsync((void **)&ws, bytes, stream));
        bdf_counter_kernel<<<1, 64, 0, stream>>>((uint32_t *)ws, (uint32_t)(grid * GPW));
    }
    bdf_kernel<R, O, S, F>(few)<<<(uint32_t)grid, 64, 0, stream>>>(
        d, queue ? (uint32_t *)ws : nullptr);
    const hipError_t launched = hipGetLastError();
    if (queue && !ws_in) BG_HIP_CHECK(hipFreeAsync(ws, stream));
    BG_HIP_CHECK(launched);
    return BG_OK;
}

template <class R, int O, class S, class F>
static int bdf_path_one(BdfPathState *state, double *path_t, double *path_y, uint32_t cap,
                        hipStream_t stream) {
    bdf_path_kernel<R, O, S, F><<<1, 64, 0, stream>>>(state, path_t, path_y, cap);
    BG_HIP_CHECK(hipGetLastError());
    return BG_OK;
}

// Method and semantics dispatch around a per-system visitor `sys(rtag,
// ftag)` of the caller's translation unit.
template <class V>
static int bdf_with_order_sem(int method, int semantics, V &&v) {
    if (semantics != BG_AS_BUILT && semantics != BG_INTENDED) return BG_ERR_INVALID_ARGUMENT;
    auto with_sem = [&](auto otag) -> int {
        return semantics == BG_AS_BUILT ? v(otag, BTag<BdfSem<true>>{})
                                        : v(otag, BTag<BdfSem<false>>{});
    };
    if (method == BG_BDF6) return with_sem(std::integral_constant<int, 7>{});
    if (method == BG_BDF2) return with_sem(std::integral_constant<int, 3>{});
    return BG_ERR_UNSUPPORTED;
}

}  // namespace bg
