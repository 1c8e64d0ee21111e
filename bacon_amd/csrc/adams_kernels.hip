// adams_kernels.hip — batched Adams-Bashforth-Moulton predictor-corrector
// (Adams5 / Adams3) for gfx950.
//
// Reference: bacon-sci's AdamsSolver (src/ivp/adams.rs:336-633): an
// (O-1)-step Adams-Bashforth predictor, an O-coefficient Adams-Moulton
// corrector evaluated once (PECE), the error estimate
// (19/270) / dt * |corrector - predictor|, an RK4 bootstrap of O - 1 steps
// after every step-size change, and the yield bookkeeping of the iterator.
//
// One lane per instance, refilled like the RK ensemble kernel's.  The
// derivative deque holds at most O - 1 entries when the predictor runs, so it
// lives in registers as a shift register (a push that follows a full deque
// drops the oldest entry, which is the reference's push_back + pop_front).
// The value deque only matters through its length here (final states, not the
// path).  Arithmetic follows the oracle's DEVICE profile operation by
// operation (explicit fma, rootn() for the step-size factor), so results are
// bit-identical to it.
//
// Semantics: as built, the derivative of the first Adams step after a
// bootstrap never joins the deque (adams.rs:434-441 pushes the value only),
// leaving the history one step stale; intended pushes it.
#include "bg_device.h"
#include "bg_internal.h"

namespace bg {

static constexpr uint32_t kAdamsDefaultMaxSteps = 10000000u;

// x^(1/N), N = 3 or 5, from exact operations (frexp, fma, ldexp, rounded
// constants): x = m 2^e with m in [1, 2); m^(1/N) by a degree-6 polynomial in
// (m - 1.5) interpolating at Chebyshev nodes (relative error < 2.5e-7);
// 2^(e/N) = 2^floor(e/N) * 2^((e mod N)/N).  0, inf and NaN map to themselves.
template <int N>
__device__ __forceinline__ double rootn(double x) {
    static_assert(N == 3 || N == 5, "rootn: N = 3 or 5");
    if (!(x == x) || x == 0.0 || x == __builtin_inf()) return x;
    int ex;
    const double m = frexp(x, &ex);
    const double u = fma(m, 2.0, -1.5);
    const int e = ex - 1;
    double p;
    if constexpr (N == 3) {
        p = kc(-0.0027033338703399646);
        p = fma(p, u, kc(0.0051666994182390956));
        p = fma(p, u, kc(-0.009260767947395939));
        p = fma(p, u, kc(0.02085714929540036));
        p = fma(p, u, kc(-0.05653050145457822));
        p = fma(p, u, kc(0.254383453864114));
        p = fma(p, u, kc(1.1447142425533323));
    } else {
        p = kc(-0.002242595967870246);
        p = fma(p, u, kc(0.004170036250587015));
        p = fma(p, u, kc(-0.007159250830014004));
        p = fma(p, u, kc(0.015356114792636277));
        p = fma(p, u, kc(-0.038560210159460984));
        p = fma(p, u, kc(0.14459836703782772));
        p = fma(p, u, kc(1.0844717711976986));
    }
    int a = e / N, b = e % N;
    if (b < 0) {
        b += N;
        a -= 1;
    }
    double s;
    if constexpr (N == 3)
        s = b == 0 ? 1.0 : (b == 1 ? 1.2599210498948732 : 1.5874010519681994);
    else
        s = b == 0 ? 1.0
                   : (b == 1 ? 1.148698354997035
                             : (b == 2 ? 1.3195079107728942
                                       : (b == 3 ? 1.515716566510398 : 1.7411011265922482)));
    return ldexp(p * s, a);
}

// adams.rs:568-661
template <int O>
struct AdamsCoef;
template <>
struct AdamsCoef<5> {
    __device__ static constexpr double pred(int k) {
        constexpr double tf = 24.0;
        constexpr double c[5] = {55.0 / tf, -59.0 / tf, 37.0 / tf, -9.0 / tf, 0.0};
        return c[k];
    }
    __device__ static constexpr double corr(int k) {
        constexpr double sh = 720.0;
        constexpr double c[5] = {251.0 / sh, 646.0 / sh, -264.0 / sh, 106.0 / sh, -19.0 / sh};
        return c[k];
    }
};
template <>
struct AdamsCoef<3> {
    __device__ static constexpr double pred(int k) {
        constexpr double c[3] = {1.0 + 1.0 / 2.0, -(1.0 / 2.0), 0.0};
        return c[k];
    }
    __device__ static constexpr double corr(int k) {
        constexpr double c[3] = {5.0 / 12.0, 2.0 / 3.0, -(1.0 / 12.0)};
        return c[k];
    }
};

// The coefficients through SGPR pairs (kc): at each use, or once for a loop.
template <class C>
struct CoefAtUse {
    __device__ __forceinline__ double pred(int k) const { return kc(C::pred(k)); }
    __device__ __forceinline__ double corr(int k) const { return kc(C::corr(k)); }
};
template <class C, int O>
struct CoefOnce {
    double p[O - 1], c[O];
    __device__ __forceinline__ CoefOnce() {
#pragma unroll
        for (int k = 0; k < O - 1; ++k) p[k] = kc(C::pred(k));
#pragma unroll
        for (int k = 0; k < O; ++k) c[k] = kc(C::corr(k));
    }
    __device__ __forceinline__ double pred(int k) const { return p[k]; }
    __device__ __forceinline__ double corr(int k) const { return c[k]; }
};

enum : int { ADAMS_YIELD = -1, ADAMS_REDO = -2, ADAMS_DONE = -3 };

// PATH: also keep the values of the last bootstrap (the value deque's
// entries, oldest first), which the yield_memory countdown of adams.rs:415-428
// yields; `yitem` names what a yield returns: -1 the current (t, y), else
// that entry.  Without PATH both are dead and compile away.
// COLD: the values that only a change of the step size looks at (tolerance,
// step bounds, the state before the bootstrap) lie in LDS, one column of
// kColdStride doubles apart per value, instead of registers: the ensemble
// kernel then holds four waves per SIMD without spills (spilled, each change of
// the step size waited for some fifty scratch reloads: 262,144 Lorenz-63
// instances to t = 10 at tol 1e-6 took 12.8 ms instead of 7.9).
constexpr int kColdStride = 256;
template <class RHS, int O, bool AsBuilt, bool PATH = false, bool COLD = false>
struct AdamsLane {
    static constexpr int D = RHS::D;
    using C = AdamsCoef<O>;
    static constexpr int kCold = 3 + D;
    double t, dt, end;
    double cold_reg[COLD ? 1 : kCold];
    double *cold_lds;  // COLD: this lane's column
    __device__ __forceinline__ double &cold(int k) {
        if constexpr (COLD) return cold_lds[k * kColdStride];
        else return cold_reg[k];
    }
    __device__ __forceinline__ double &tol() { return cold(0); }
    __device__ __forceinline__ double &dt_min() { return cold(1); }
    __device__ __forceinline__ double &dt_max() { return cold(2); }
    __device__ __forceinline__ double &save(int c) { return cold(3 + c); }
    double y[D], impl[D];
    double dq[O - 1][D];  // derivative history, oldest first (shift register)
    double vt[PATH ? O - 1 : 1], vy[PATH ? O - 1 : 1][D];  // value deque (PATH only)
    int vlen;             // length of the value deque
    int ym;               // yield_memory
    int yitem;
    double p[RHS::P > 0 ? RHS::P : 1];
    uint32_t n_rej;

    __device__ __forceinline__ bool f(double tt, const double (&yy)[D], double (&out)[D]) const {
        return RHS::eval(tt, yy, p, out);
    }
    __device__ __forceinline__ void push_d(const double (&v)[D]) {
#pragma unroll
        for (int k = 0; k < O - 2; ++k)
#pragma unroll
            for (int c = 0; c < D; ++c) dq[k][c] = dq[k + 1][c];
#pragma unroll
        for (int c = 0; c < D; ++c) dq[O - 2][c] = v[c];
    }
    // a history whose oldest entry is dq[r] put in order (r differs by lane)
    __device__ __forceinline__ void rotate_history(uint32_t r) {
#pragma unroll
        for (int by = 1; by < O - 1; by <<= 1) {
            double m[O - 1][D];
#pragma unroll
            for (int k = 0; k < O - 1; ++k)
#pragma unroll
                for (int c = 0; c < D; ++c)
                    m[k][c] = (r & (uint32_t)by) ? dq[(k + by) % (O - 1)][c] : dq[k][c];
#pragma unroll
            for (int k = 0; k < O - 1; ++k)
#pragma unroll
                for (int c = 0; c < D; ++c) dq[k][c] = m[k][c];
        }
    }
    // value push at the full deque: push_back + pop_front, as for dq
    __device__ __forceinline__ void push_v() {
        if constexpr (PATH) {
#pragma unroll
            for (int k = 0; k < O - 2; ++k) {
                vt[k] = vt[k + 1];
#pragma unroll
                for (int c = 0; c < D; ++c) vy[k][c] = vy[k + 1][c];
            }
            vt[O - 2] = t;
#pragma unroll
            for (int c = 0; c < D; ++c) vy[O - 2][c] = y[c];
        }
    }

    // adams.rs:344-396
    template <int IT>
    __device__ __forceinline__ int runge_kutta() {
#pragma unroll 1
        for (int it = 0; it < IT; ++it) {
            double k1[D], k2[D], k3[D], k4[D], mid[D];
            if (!f(t, y, k1)) return BG_USER_ERROR;
#pragma unroll
            for (int c = 0; c < D; ++c) k1[c] *= dt;
#pragma unroll
            for (int c = 0; c < D; ++c) mid[c] = fma(k1[c], 0.5, y[c]);
            if (!f(fma(0.5, dt, t), mid, k2)) return BG_USER_ERROR;
#pragma unroll
            for (int c = 0; c < D; ++c) k2[c] *= dt;
#pragma unroll
            for (int c = 0; c < D; ++c) mid[c] = fma(k2[c], 0.5, y[c]);
            if (!f(fma(0.5, dt, t), mid, k3)) return BG_USER_ERROR;
#pragma unroll
            for (int c = 0; c < D; ++c) k3[c] *= dt;
#pragma unroll
            for (int c = 0; c < D; ++c) mid[c] = y[c] + k3[c];
            if (!f(t + dt, mid, k4)) return BG_USER_ERROR;
#pragma unroll
            for (int c = 0; c < D; ++c) k4[c] *= dt;
            if (it != 0) {
                double fd[D];
                if (!f(t, y, fd)) return BG_USER_ERROR;
                push_d(fd);
                push_v();
                ++vlen;
            }
#pragma unroll
            for (int c = 0; c < D; ++c) {
                double sum = fma(k2[c], 2.0, k1[c]);
                sum = fma(k3[c], 2.0, sum);
                sum = sum + k4[c];
                y[c] = fma(sum, kc(1.0 / 6.0), y[c]);
            }
            t += dt;
        }
        double fd[D];
        if (!f(t, y, fd)) return BG_USER_ERROR;
        push_d(fd);
        push_v();
        ++vlen;
        return BG_OK;
    }

    __device__ __forceinline__ double q_of(double error) {
        return rootn<O>(tol() / (2.0 * error));
    }

    // One AdamsSolver::step (adams.rs:411-561)
    __device__ __forceinline__ int step() {
        yitem = -1;
        if (ym > 0 && ym < O) {  // adams.rs:415-428
            yitem = O - ym - 1;
            ym -= 1;
            if (ym == 0) ym = O + 1;
            return ADAMS_YIELD;
        }
        if (ym == O + 1) {  // adams.rs:434-441
            ym = 0;
            if (!AsBuilt) push_d(impl);
            return ADAMS_YIELD;
        }
        if (t >= end) return ADAMS_DONE;
        if (t + dt >= end) {  // adams.rs:447-451
            dt = end - t;
            const int rc = runge_kutta<1>();
            if (rc) return rc;
            return ADAMS_YIELD;
        }
        // bootstrap(), written out: through the call the compiler keeps the
        // single-instance path of three components in 306 registers, with 474
        // moves to and from the accumulators, instead of 175 (Lorenz-63 to
        // t = 5 at tol 1e-8: 45.7 against 43.7 ms)
        if (vlen == 0) {
#pragma unroll
            for (int c = 0; c < D; ++c) save(c) = y[c];
            if (t + dt * (double)(O - 1) >= end) dt = (end - t) / (double)(O - 1);
            const int rc = runge_kutta<O - 1>();
            if (rc) return rc;
            ym = O;
            return ADAMS_REDO;
        }
        return multistep(impl);
    }

    // adams.rs:453-464
    __device__ __forceinline__ int bootstrap() {
#pragma unroll
        for (int c = 0; c < D; ++c) save(c) = y[c];
        if (t + dt * (double)(O - 1) >= end) dt = (end - t) / (double)(O - 1);
        const int rc = runge_kutta<O - 1>();
        if (rc) return rc;
        ym = O;
        return ADAMS_REDO;
    }

    // Predictor and corrector (adams.rs:466-486) from the derivative history,
    // whose oldest entry is dq[u] (u = 0 outside the ensemble kernel's ordinary
    // steps): corrected value, the predicted point's derivative and the squared
    // distance of the two values.  False if the right-hand side reports an
    // error.
    template <class CF>
    __device__ __forceinline__ bool predict_correct(int u, const CF &cf, double (&co)[D],
                                                    double (&im)[D], double &ss) const {
        double pr[D];
#pragma unroll
        for (int c = 0; c < D; ++c) {
            double sc = dq[u][c] * cf.pred(O - 2);
#pragma unroll
            for (int i = 1; i < O - 1; ++i)
                sc = fma(dq[(u + i) % (O - 1)][c], cf.pred(O - i - 2), sc);
            pr[c] = fma(sc, dt, y[c]);
        }
        if (!f(t + dt, pr, im)) return false;
        ss = 0.0;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            double sc = im[c] * cf.corr(0);
#pragma unroll
            for (int i = 0; i < O - 1; ++i)
                sc = fma(dq[(u + i) % (O - 1)][c], cf.corr(O - i - 1), sc);
            co[c] = fma(sc, dt, y[c]);
            const double df = co[c] - pr[c];
            ss = c == 0 ? df * df : fma(df, df, ss);
        }
        return true;
    }

    // The step from a full history (adams.rs:466-561); im: the derivative at
    // the predicted point
    __device__ __forceinline__ int multistep(double (&im)[D]) {
        double co[D], ss;
        if (!predict_correct(0, CoefAtUse<C>{}, co, im, ss)) return BG_USER_ERROR;
        const double error = (kc(19.0 / 270.0) / dt) * sqrt(ss);
        if (error <= tol()) {  // adams.rs:490-525
#pragma unroll
            for (int c = 0; c < D; ++c) y[c] = co[c];
            t += dt;
            if (ym == O) {
                ym -= 1;
                return ADAMS_REDO;
            }
            push_d(im);  // with the value push: lengths stay O - 1
            if (error < 0.1 * tol()) {
                const double q = q_of(error);
                if (q > 4.0)
                    dt *= 4.0;
                else
                    dt *= q;
                if (dt > dt_max()) dt = dt_max();
                vlen = 0;
            }
            return ADAMS_YIELD;
        }
        ++n_rej;
        if (ym == O) {  // adams.rs:531-536
            t -= dt * (double)(O - 1);
#pragma unroll
            for (int c = 0; c < D; ++c) y[c] = save(c);
        }
        const double q = q_of(error);  // adams.rs:538-556
        if (q < 0.1)
            dt *= 0.1;
        else
            dt *= q;
        if (dt < dt_min()) return BG_MINIMUM_TIME_DELTA_EXCEEDED;
        vlen = 0;
        return ADAMS_REDO;
    }

    __device__ __forceinline__ void load(const bg_ensemble_desc &d, uint64_t i) {
        const uint64_t n = d.n;
#pragma unroll
        for (int c = 0; c < D; ++c) y[c] = d.y0[(uint64_t)c * n + i];
#pragma unroll
        for (int k = 0; k < RHS::P; ++k) p[k] = d.params[(uint64_t)k * n + i];
        t = d.t0 ? d.t0[i] : d.t0_s;
        end = d.t_end ? d.t_end[i] : d.t_end_s;
        const double lo = d.dt_min ? d.dt_min[i] : d.dt_min_s;
        const double hi = d.dt_max ? d.dt_max[i] : d.dt_max_s;
        tol() = d.tol ? d.tol[i] : d.tol_s;
        dt_min() = lo;
        dt_max() = hi;
        dt = (hi + lo) * 0.5;  // adams.rs:288
        vlen = 0;
        ym = 0;
        n_rej = 0;
#pragma unroll
        for (int c = 0; c < D; ++c) impl[c] = 0.0;
#pragma unroll
        for (int k = 0; k < O - 1; ++k)
#pragma unroll
            for (int c = 0; c < D; ++c) dq[k][c] = 0.0;
    }
};

// ---------------------------------------------------------------------------
// Persistent ensemble kernel.
//
// A lane's calls of step() are of two kinds: the ordinary predictor-corrector
// step at an unchanged step size (98 % of them on Lorenz-63 at tol 1e-6), and
// everything around a change of the step size: the exact error and the new
// size, the RK4 bootstrap (four steps, 20 right-hand sides), its first
// multistep, the yields of the bootstrap's values.  In a wave some lane is
// nearly always at the second kind, so running both in each pass costs every
// lane the bootstrap on most of its steps.  Here they are two phases:
//   * the ordinary steps of all lanes, until half of the wave's lanes have
//     met something else.  A lane commits its step if the squared error lies
//     clearly between the two thresholds (error <= tol and not below
//     0.1 tol, each with a margin of 1e-10, far above the rounding of the
//     exact test), which needs neither the square root nor the divisions;
//     any other lane leaves its state as it was and waits;
//   * the calls of the waiting lanes, with the exact test, until most of
//     them are back at ordinary steps.  A bootstrap's yields change nothing
//     but the counters and are settled at once.
// 262,144 Lorenz-63 instances, t in [0, 10], tol 1e-6: 41.4 -> 7.9 ms; 20,000 of
// them 14.8 -> 2.6; 20,000 Lotka-Volterra at tol 1e-5 0.91 -> 0.33 ms.  Waiting
// until a quarter (5/8) of the lanes are left at ordinary steps instead of half:
// 9.6 (7.9), 3.0 (2.8) and 0.29 (0.36) ms.
// ---------------------------------------------------------------------------
template <class RHS, int O, bool AsBuilt>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
    adams_ensemble_kernel(const bg_ensemble_desc, uint32_t *__restrict__ counter) {
    constexpr int D = RHS::D;
    constexpr uint32_t kRoundCalls = 2 * (O + 2);  // at most this many calls per slow round
    const karg_desc dv = kernarg_desc();
    AdamsLane<RHS, O, AsBuilt, false, true> L;
    __shared__ double cold[L.kCold * kColdStride];
    L.cold_lds = cold + threadIdx.x;
    const CoefOnce<AdamsCoef<O>, O> cf;
    const uint64_t max_att = dv->max_attempts;
    const uint32_t cap =
        (uint32_t)((max_att && max_att < kAdamsDefaultMaxSteps) ? max_att : kAdamsDefaultMaxSteps);
    WaveQueue queue(counter);
    int64_t inst = queue.start(dv->n, dv->order);
    bool take = inst >= 0;
    // calls so far: those that yielded (nacc) and those that did not
    uint32_t nacc = 0, other = 0;
    bool slow = false;          // waits for the second phase
    double ss_lo = 0.0, ss_hi = 0.0;  // ordinary steps: ss_lo < ss < ss_hi
    int32_t left = (int32_t)cap;      // passes before a lane could reach the cap
    for (;;) {
        int st = -1;
        if (take) {
            L.load(desc_inputs(dv), (uint64_t)inst);
            nacc = other = 0;
            slow = true;
        }
        const int active = __popcll(ballot(inst >= 0));
        if (active == 0) break;
        const bool drained = queue.drained();
        const int want = drained ? active : 1;
        for (;;) {
            const int running = __popcll(ballot(inst >= 0 && st < 0));
            if (active - running >= want) break;
            // ---- ordinary steps: O - 1 of them a pass, so that every one
            // finds its history in place (a commit overwrites the oldest entry
            // instead of moving the others up)
            bool fast = inst >= 0 && st < 0 && !slow;
            const int stop_at = running / 2;
            int32_t made = 0;
            if (__popcll(ballot(fast)) > stop_at && left >= O - 1) {
                const uint32_t before = nacc;
                do {
#pragma unroll
                    for (int u = 0; u < O - 1; ++u) {
                        // the lanes that wait compute along and keep nothing
                        double co[D], im[D], ss;
                        const double tn = L.t + L.dt;
                        const bool ok = L.predict_correct(u, cf, co, im, ss);
                        fast = fast & ok & (ss > ss_lo) & (ss < ss_hi) & !(tn >= L.end);
                        if (fast) {
                            L.t = tn;
#pragma unroll
                            for (int c = 0; c < D; ++c) {
                                L.y[c] = co[c];
                                L.dq[u][c] = im[c];
                            }
                            ++nacc;
                        }
                    }
                    made += O - 1;
                } while (__popcll(ballot(fast)) > stop_at && made + (O - 1) <= left);
                L.rotate_history((nacc - before) % (uint32_t)(O - 1));
            }
            left -= made;
            queue.ticks += (uint32_t)made + 4u;
            slow = inst >= 0 && st < 0 && !fast;
            if (left <= 0) {
                left = (int32_t)(cap - wave_max_u32(inst >= 0 && st < 0 ? nacc + other : 0u));
                // a lane near the cap: every lane's next call is an exact one
                if (left <= 8 * (int32_t)kRoundCalls) slow = inst >= 0 && st < 0;
            }
            // ---- calls of the lanes that wait
            const int waiting = __popcll(ballot(slow));
            for (int round = 0; round < 8; ++round) {
                left -= (int32_t)kRoundCalls;
                if (slow) {
                    int r = ADAMS_REDO;
                    bool called = true;
                    if (nacc + other >= cap) {
                        st = BG_MAXIMUM_ITERATIONS_EXCEEDED;
                        called = false;
                    } else if (L.t >= L.end) {
                        r = ADAMS_DONE;
                    } else if (L.t + L.dt >= L.end) {  // adams.rs:447-451
                        L.dt = L.end - L.t;
                        r = L.template runge_kutta<1>();
                        if (r == BG_OK) r = ADAMS_YIELD;
                    } else if (L.vlen != 0) {
                        double im[D];
                        r = L.multistep(im);
                        // the first one after a bootstrap: the bootstrap's
                        // yields follow (adams.rs:415-441), one call each
                        if (r == ADAMS_REDO && L.ym == O - 1) {
                            const uint32_t room = cap - 1u - (nacc + other);
                            nacc += (uint32_t)O < room ? (uint32_t)O : room;
                            L.ym = 0;
                            if (!AsBuilt) L.push_d(im);
                        }
                    } else {
                        called = false;
                    }
                    if (called) {
                        if (r == ADAMS_YIELD)
                            ++nacc;
                        else
                            ++other;
                        if (r == ADAMS_DONE)
                            st = BG_OK;
                        else if (r != ADAMS_YIELD && r != ADAMS_REDO)
                            st = r;
                    }
                }
                const bool boot = slow && st < 0 && L.vlen == 0 && nacc + other < cap &&
                                  !(L.t >= L.end) && !(L.t + L.dt >= L.end);
                if (boot) {  // adams.rs:453-464
                    const int r = L.bootstrap();
                    ++other;
                    if (r != ADAMS_REDO) st = r;
                }
                if (slow && (st >= 0 || (L.vlen != 0 && L.ym == 0 && L.t + L.dt < L.end))) {
                    slow = false;
                    // (tol / c)^2 and (0.1 tol / c)^2, c = (19/270) / dt
                    const double c = kc(19.0 / 270.0) / L.dt;
                    const double hi = L.tol() / c, lo = 0.1 * hi;
                    ss_hi = hi * hi * (1.0 - 1e-10);
                    ss_lo = lo * lo * (1.0 + 1e-10);
                    // out of the range in which the margins hold, or a sign
                    // that the squares would lose: every step by the exact
                    // test
                    if (!(ss_lo > 1e-280 && ss_hi < 1e280 && c > 0.0 && hi > 0.0))
                        ss_lo = __builtin_inf();
                }
                if (4 * __popcll(ballot(slow)) <= waiting) break;
            }
        }
        take = inst >= 0 && st >= 0;
        if (take) {
            const bg_ensemble_desc d = desc_outputs(dv);
            const uint64_t n = d.n, i = (uint64_t)inst;
            if (d.t_out) d.t_out[i] = L.t;
            if (d.y_out) {
#pragma unroll
                for (int c = 0; c < D; ++c) d.y_out[(uint64_t)c * n + i] = L.y[c];
            }
            if (d.status) d.status[i] = st;
            if (d.counts) {
                bg_counts cn;
                cn.n_accepted = nacc;
                cn.n_rejected = L.n_rej;
                d.counts[i] = cn;
            }
        }
        if (drained) break;
        const karg_desc du = desc_at_use(dv);
        uint32_t pos;
        const int64_t got = queue.next(counter, (uint32_t)du->n, du->order, take, pos);
        if (take) inst = got;
        take = take && inst >= 0;
    }
}

// Single-instance path production: every yield of the iterator (adams.rs:
// 398-565 through ivp.rs:205-239) into the path buffer; stops when the
// buffer is full (resumable: the lane state goes back to *st) or the solve
// ends.  Steps are counted like the ensemble kernel's, as step() calls.
template <class RHS, int O, bool AsBuilt>
__global__ void __launch_bounds__(64)
    adams_path_kernel(AdamsPathState *__restrict__ st, double *__restrict__ path_t,
                      double *__restrict__ path_y, uint32_t cap) {
    constexpr int D = RHS::D;
    static_assert(D <= 4 && O - 1 <= 4 && RHS::P <= 8, "AdamsPathState sizes");
    if (threadIdx.x != 0) return;
    AdamsLane<RHS, O, AsBuilt, true> L;
    L.t = st->t;
    L.dt = st->dt;
    L.end = st->end;
    L.tol() = st->tol;
    L.dt_min() = st->dt_min;
    L.dt_max() = st->dt_max;
    L.vlen = st->vlen;
    L.ym = st->ym;
    L.yitem = -1;
    L.n_rej = st->n_rejected;
#pragma unroll
    for (int c = 0; c < D; ++c) {
        L.y[c] = st->y[c];
        L.save(c) = st->save[c];
        L.impl[c] = st->impl[c];
    }
#pragma unroll
    for (int k = 0; k < O - 1; ++k) {
        L.vt[k] = st->vt[k];
#pragma unroll
        for (int c = 0; c < D; ++c) {
            L.dq[k][c] = st->dq[k][c];
            L.vy[k][c] = st->vy[k][c];
        }
    }
#pragma unroll
    for (int k = 0; k < RHS::P; ++k) L.p[k] = st->p[k];
    uint64_t steps = st->steps;
    const uint64_t max_steps = st->max_steps;
    uint32_t nacc = st->n_accepted, count = 0;
    int status = st->status, finished = st->finished;
    while (!finished && count < cap) {
        if (steps >= max_steps) {
            status = BG_MAXIMUM_ITERATIONS_EXCEEDED;
            finished = 1;
            break;
        }
        ++steps;
        const int r = L.step();
        if (r == ADAMS_YIELD) {
            ++nacc;
            double yt = L.t, yv[D];
#pragma unroll
            for (int c = 0; c < D; ++c) yv[c] = L.y[c];
#pragma unroll
            for (int k = 0; k < O - 1; ++k) {
                if (L.yitem == k) {
                    yt = L.vt[k];
#pragma unroll
                    for (int c = 0; c < D; ++c) yv[c] = L.vy[k][c];
                }
            }
            path_t[count] = yt;
#pragma unroll
            for (int c = 0; c < D; ++c) path_y[(uint64_t)count * D + c] = yv[c];
            ++count;
        } else if (r == ADAMS_DONE) {
            finished = 1;
        } else if (r != ADAMS_REDO) {
            status = r;
            finished = 1;
        }
    }
    st->t = L.t;
    st->dt = L.dt;
    st->vlen = L.vlen;
    st->ym = L.ym;
    st->n_rejected = L.n_rej;
#pragma unroll
    for (int c = 0; c < D; ++c) {
        st->y[c] = L.y[c];
        st->save[c] = L.save(c);
        st->impl[c] = L.impl[c];
    }
#pragma unroll
    for (int k = 0; k < O - 1; ++k) {
        st->vt[k] = L.vt[k];
#pragma unroll
        for (int c = 0; c < D; ++c) {
            st->dq[k][c] = L.dq[k][c];
            st->vy[k][c] = L.vy[k][c];
        }
    }
    st->steps = steps;
    st->n_accepted = nacc;
    st->status = status;
    st->finished = finished;
    st->count = count;
}

__global__ void adams_counter_kernel(uint32_t *counter, uint32_t lanes) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *counter = lanes;
}

template <class T>
struct AdTag {
    using type = T;
};

template <class V>
static int visit_adams(int method, int rhs, int semantics, uint32_t dim, V &&v) {
    if (method != BG_ADAMS5 && method != BG_ADAMS3) return BG_ERR_INVALID_ARGUMENT;
    if (semantics != BG_AS_BUILT && semantics != BG_INTENDED) return BG_ERR_INVALID_ARGUMENT;
    auto with = [&](auto rtag) -> int {
        using R = typename decltype(rtag)::type;
        if (dim != (uint32_t)R::D) return BG_ERR_INVALID_ARGUMENT;
        const bool ab = semantics == BG_AS_BUILT;
        if (method == BG_ADAMS5)
            return ab ? v(rtag, std::integral_constant<int, 5>{}, std::true_type{})
                      : v(rtag, std::integral_constant<int, 5>{}, std::false_type{});
        return ab ? v(rtag, std::integral_constant<int, 3>{}, std::true_type{})
                  : v(rtag, std::integral_constant<int, 3>{}, std::false_type{});
    };
    switch (rhs) {
    case BG_RHS_EXP: return with(AdTag<RhsExp<1>>{});
    case BG_RHS_NEG: return with(AdTag<RhsNeg<1>>{});
    case BG_RHS_QUADRATIC: return with(AdTag<RhsQuadratic<1>>{});
    case BG_RHS_COS: return with(AdTag<RhsCos<1>>{});
    case BG_RHS_LORENZ: return with(AdTag<RhsLorenz>{});
    case BG_RHS_LOTKA_VOLTERRA: return with(AdTag<RhsLotkaVolterra>{});
    case BG_RHS_OSCILLATOR: return with(AdTag<RhsOscillator>{});
    case BG_RHS_ROBERTSON: return with(AdTag<RhsRobertson>{});
    case BG_RHS_TWO_LEVEL: return with(AdTag<RhsTwoLevel>{});
    default: return BG_ERR_UNSUPPORTED;
    }
}

bool adams_supported(int method, int rhs, uint32_t dim) {
    return visit_adams(method, rhs, BG_INTENDED, dim, [](auto, auto, auto) { return BG_OK; }) ==
           BG_OK;
}

int adams_launch_ensemble(int method, int rhs, int semantics, const bg_ensemble_desc &d,
                          hipStream_t stream, void *ws_in) {
    return visit_adams(method, rhs, semantics, d.dim, [&](auto rtag, auto otag, auto atag) -> int {
        using R = typename decltype(rtag)::type;
        constexpr int O = decltype(otag)::value;
        constexpr bool AB = decltype(atag)::value;
        if (d.n == 0) return BG_OK;
        if (d.n > 0x7fffffffull || !d.y0) return BG_ERR_INVALID_ARGUMENT;
        if (R::P > 0 && (!d.params || d.n_params < (uint32_t)R::P))
            return BG_ERR_INVALID_ARGUMENT;
        int dev = 0;
        BG_HIP_CHECK(hipGetDevice(&dev));
        int per_cu = 0;
        BG_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, adams_ensemble_kernel<R, O, AB>, 256, 0));
        if (per_cu < 1) per_cu = 1;
        uint64_t grid = (uint64_t)per_cu * (uint64_t)device_cu_count(dev);
        const uint64_t need = (d.n + 255) / 256;
        if (grid > need) grid = need;
        // a lane for every instance: no queue, no workspace
        const bool queue = d.n > grid * 256;
        char *ws = (char *)ws_in;
        if (queue) {
            if (!ws_in) BG_HIP_CHECK(hipMallocAsync((void **)&ws, kLaunchWorkspaceBytes, stream));
            adams_counter_kernel<<<1, 64, 0, stream>>>((uint32_t *)ws, (uint32_t)(grid * 256));
        }
        adams_ensemble_kernel<R, O, AB><<<(uint32_t)grid, 256, 0, stream>>>(
            d, queue ? (uint32_t *)ws : nullptr);
        const hipError_t launched = hipGetLastError();
        if (queue && !ws_in) BG_HIP_CHECK(hipFreeAsync(ws, stream));
        BG_HIP_CHECK(launched);
        return BG_OK;
    });
}

int adams_launch_path(int method, int rhs, int semantics, uint32_t dim, AdamsPathState *state,
                      double *path_t, double *path_y, uint32_t cap, hipStream_t stream) {
    return visit_adams(method, rhs, semantics, dim, [&](auto rtag, auto otag, auto atag) -> int {
        using R = typename decltype(rtag)::type;
        constexpr int O = decltype(otag)::value;
        constexpr bool AB = decltype(atag)::value;
        adams_path_kernel<R, O, AB><<<1, 64, 0, stream>>>(state, path_t, path_y, cap);
        BG_HIP_CHECK(hipGetLastError());
        return BG_OK;
    });
}

}  // namespace bg
