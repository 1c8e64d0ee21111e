// rk_kernels.hip — batched embedded Runge-Kutta (RK45 Fehlberg / RK23
// Bogacki-Shampine) for gfx950.
//
// Hot path: bacon-sci's RungeKuttaSolver::step (src/ivp/rk.rs:361-423) driven
// by IVPIterator::next (src/ivp.rs:220-238), recast as an ensemble of
// independent instances.
//
// Layout and schedule:
//  * one lane owns one instance; its state (t, dt, y[D], K[S][D], params)
//    lives in VGPRs for the whole solve;
//  * inputs and outputs are structure-of-arrays in HBM ([component][n]);
//  * the launch is persistent (grid = resident blocks); a wave refills its
//    idle lanes from runs of positions that it claims from a global counter
//    (WaveQueue in bg_device.h), so finished instances retire without
//    stalling the other lanes; an ensemble that fits the resident lanes needs
//    no counter;
//  * an optional schedule permutation hands out instances longest-first.
#include <string.h>

#include <mutex>

#include "bg_device.h"
#include "bg_internal.h"

namespace bg {

static constexpr uint64_t kDefaultMaxAttempts = 10000000ull;

template <class T>
struct Tag {
    using type = T;
};

__device__ __forceinline__ uint32_t attempt_cap(uint64_t max_attempts) {
    return (uint32_t)((max_attempts && max_attempts < kDefaultMaxAttempts) ? max_attempts
                                                                           : kDefaultMaxAttempts);
}

template <class RHS, class Tab, bool H>
__device__ __forceinline__ void rk_load(RkLane<RHS, Tab, H> &L, const bg_ensemble_desc &d,
                                        uint64_t i) {
    constexpr int D = RHS::D, S = Tab::S;
    const uint64_t n = d.n;
#pragma unroll
    for (int k = 0; k < D; ++k) L.y[k] = d.y0[k * n + i];
#pragma unroll
    for (int k = 0; k < RHS::P; ++k) L.p[k] = d.params[k * n + i];
    L.t = d.t0 ? d.t0[i] : d.t0_s;
    L.end = d.t_end ? d.t_end[i] : d.t_end_s;
    L.tol = d.tol ? d.tol[i] : d.tol_s;
    L.dt_min = d.dt_min ? d.dt_min[i] : d.dt_min_s;
    L.dt_max = d.dt_max ? d.dt_max[i] : d.dt_max_s;
    L.dt = (L.dt_max + L.dt_min) * 0.5;  // rk.rs:315
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int k = 0; k < D; ++k) L.K[s][k] = 0.0;  // rk.rs:323-327
    L.set_range();
}

template <class RHS, class Tab, bool H>
__device__ __forceinline__ void rk_store(const RkLane<RHS, Tab, H> &L, const bg_ensemble_desc &d,
                                         uint64_t i, int status, uint32_t nacc, uint32_t nrej) {
    constexpr int D = RHS::D;
    const uint64_t n = d.n;
    if (d.t_out) d.t_out[i] = L.t;
    if (d.y_out) {
#pragma unroll
        for (int k = 0; k < D; ++k) d.y_out[k * n + i] = L.y[k];
    }
    if (d.status) d.status[i] = status;
    if (d.counts) {
        bg_counts c;
        c.n_accepted = nacc;
        c.n_rejected = nrej;
        d.counts[i] = c;
    }
}

// One attempt plus the iterator's bookkeeping.  Returns -1 to continue, or
// the final status (BG_OK at Done).  For the single-lane kernels.
template <class RHS, class Tab, bool H>
__device__ __forceinline__ int rk_advance(RkLane<RHS, Tab, H> &L, uint32_t &attempts, uint32_t cap,
                                          uint32_t &nacc, uint32_t &nrej) {
    if (attempts >= cap) return BG_MAXIMUM_ITERATIONS_EXCEEDED;
    bool failed;
    L.head(L.end);
    uint32_t step = 0;
    const bool accepted = L.attempt(failed, step);
    ++attempts;
    if (failed) return BG_USER_ERROR;
    // rk.rs:414-416
    if (L.dt < L.dt_min && L.t < L.end) return BG_MINIMUM_TIME_DELTA_EXCEEDED;
    if (accepted) {
        ++nacc;
        // the iterator's next step() call would return Done (rk.rs:362-364)
        return L.t >= L.end ? BG_OK : -1;
    }
    ++nrej;
    return -1;
}

// Persistent ensemble kernel.  Outer loop: refill idle lanes, store
// finished instances.  Inner loop: step attempts until at
// least `refill_min` lanes of the wave have finished, or, once the queue is
// used up, all have.  Waves holding an instance among the first `prio_cutoff`
// schedule positions run at raised wave priority so the longest solves are
// not starved.
//
// The attempt loop holds no more bookkeeping than the accepted count and one
// wave-uniform exit test (a lane at its end or below dt_min, or the attempt
// budget that the wave's lanes share until the first could reach its cap);
// statuses and attempt counts are settled outside it.  Lorenz-63 RK45: 193 ->
// 170 vector instructions per attempt.
template <class RHS, class Tab>
__global__ void __launch_bounds__(256)
    rk_ensemble_kernel(const bg_ensemble_desc, uint32_t *__restrict__ counter,
                       uint32_t refill_min, uint32_t prio_cutoff) {
    // the counter kernel may have set fewer blocks to work than were launched
    const uint32_t blocks = counter ? counter[1] : gridDim.x;
    if (blockIdx.x >= blocks) return;
    r8_init();
    const karg_desc dv = kernarg_desc();
    RkLane<RHS, Tab, true> L;
    const uint32_t cap = attempt_cap(dv->max_attempts);
    uint32_t budget = cap;  // attempts until a lane could reach the cap
    WaveQueue queue(counter, blocks);
    uint32_t pos = blockIdx.x * blockDim.x + threadIdx.x;
    int64_t inst = queue.start(dv->n, dv->order);
    bool take = inst >= 0;
    uint32_t attempts = 0, nacc = 0;
    for (;;) {
        // ---- refill --------------------------------------------------------
        int st = -1;  // running; >= 0: the instance's status
        if (take) {
            rk_load(L, desc_inputs(dv), (uint64_t)inst);  // one batch of loads
            attempts = nacc = 0;
            if (L.t >= L.end) st = BG_OK;  // Done before any step
            L.head(L.end);
        }
        if (prio_cutoff) {
            if (ballot(inst >= 0 && pos < prio_cutoff) != 0)
                __builtin_amdgcn_s_setprio(2);
            else
                __builtin_amdgcn_s_setprio(0);
        }
        const int active = __popcll(ballot(inst >= 0));
        if (active == 0) break;
        // ---- attempts ------------------------------------------------------
        const bool drained = queue.drained();
        const int want = drained ? active : min((int)refill_min, active);
        for (;;) {
            const uint64_t running = ballot(inst >= 0 && st < 0);
            if (active - __popcll(running) >= want) break;
            uint32_t made = 0;
            if (inst >= 0 && st < 0) {
                bool accepted, failed;
                uint64_t at_end, low, out;
                do {
                    accepted = L.attempt(failed, nacc);
                    L.head(L.end);
                    ++made;
                    at_end = ballot(L.t >= L.end);
                    low = ballot(L.dt < L.dt_min);
                    out = at_end | low;
                    if constexpr (kRhsFails<RHS>) out |= ballot(failed);
                } while (out == 0 && made < budget);
                attempts += made;
                if (failed) {
                    st = BG_USER_ERROR;
                } else if (lane_bit(low) && L.t < L.end) {  // rk.rs:414-416
                    st = BG_MINIMUM_TIME_DELTA_EXCEEDED;
                    if (accepted) --nacc;
                } else if (lane_bit(at_end)) {
                    // the iterator's next step() would return Done (rk.rs:362-364)
                    st = BG_OK;
                } else if (attempts >= cap) {
                    st = BG_MAXIMUM_ITERATIONS_EXCEEDED;
                }
            }
            const uint32_t rounds = first_of(made, running);
            queue.ticks += rounds;
            budget -= rounds;
            if (budget == 0) budget = cap - wave_max_u32(inst >= 0 && st < 0 ? attempts : 0u);
        }
        take = inst >= 0 && st >= 0;
        if (take) {
            // an attempt that ended in a failure counts as neither
            const uint32_t lost =
                st == BG_USER_ERROR || st == BG_MINIMUM_TIME_DELTA_EXCEEDED ? 1u : 0u;
            rk_store(L, desc_outputs(dv), (uint64_t)inst, st, nacc, attempts - nacc - lost);
        }
        if (drained) break;
        const karg_desc du = desc_at_use(dv);
        const int64_t got = queue.next(counter, (uint32_t)du->n, du->order, take, pos);
        if (take) inst = got;
        take = take && inst >= 0;
    }
}

// Path output for an ensemble: the same persistent scheme as
// rk_ensemble_kernel, and each accepted (t, y) the reference's IVPIterator
// would yield (rk.rs:419, ivp.rs:220-238) is written to a per-instance ring
// buffer: every `every`-th accepted step, or only landings on the shared stop
// times and the end.  Stops: the end clamp of rk.rs:366-368 aims at the next
// stop time and an accepted clamped step lands exactly on it.
//
// PACKED: records go to a workspace, [n][capacity][kRecord] doubles, and
// path_unpack_kernel moves the ring's final content to the caller's arrays.
// Instances drift apart by many steps, so in the caller's layouts an 8-byte
// store is mostly alone in its cache line when the line leaves L2, and every
// record costs 1 + D lines of traffic (262,144 Lorenz-63 instances, 524 M
// records of 32 bytes: 134 GB of lines, 25-40 ms).  Packed, an instance fills
// one line in four steps, and the lines that are open at a time (one per
// resident lane, 3 MB per XCD) fit L2: 41 -> 8.5 ms, of which recording every
// step takes 1.7 and the move 0.2; instance-major 17 -> 8.6.
template <int D>
constexpr int kRecord = (D + 2) / 2 * 2;  // t, y[D], padded to 16 bytes

// Three loops, so that none carries the others' bookkeeping:
//   kRing       no stops, records by count;
//   kRingStops  stops between the records, or too many of them for LDS;
//   kStopsOnly  records at stops and the end only, the stops in LDS.  In a wave
//               of 64 lanes some lane lands on most attempts, so a landing is
//               one branch: the stop after the one aimed at is read ahead.
// The records' addresses advance with them, one per lane, the distances in
// vector registers (the coefficients take the scalar ones).
enum PathLoop { kRing, kRingStops, kStopsOnly };
template <class RHS, class Tab, bool PACKED, PathLoop LOOP>
__global__ void __launch_bounds__(256)
    rk_path_ensemble_kernel(const bg_ensemble_desc, const bg_path_desc pd,
                            uint32_t *__restrict__ counter, double *records,
                            uint32_t *__restrict__ n_records) {
    constexpr int D = RHS::D;
    constexpr bool STOPS = LOOP != kRing;
    r8_init();
    const karg_desc dv = kernarg_desc();
    RkLane<RHS, Tab, true> L;
    const uint32_t cap = attempt_cap(dv->max_attempts);
    const uint64_t n = dv->n;
    const uint32_t every = pd.every ? pd.every : 1u;
    const uint32_t capacity = pd.capacity;
    const bool stops_only = (pd.flags & BG_PATH_STOPS_ONLY) != 0;
    const bool inst_major = (pd.flags & BG_PATH_INSTANCE_MAJOR) != 0;
    uint64_t stride = inst_major ? 1u : n;  // between an entry's components
    asm("" : "+v"(stride));
    const uint32_t n_stops_all = STOPS ? pd.n_stops : 0u;
    __shared__ double stops_lds[STOPS ? kObsLds : 1];
    const bool in_lds = LOOP == kStopsOnly || n_stops_all <= kObsLds;
    bool stops_mid = true;
    if constexpr (STOPS) {
        if (in_lds) stage_obs<true>(stops_lds, pd.stops, n_stops_all);
        stops_mid = in_lds ? times_mid(stops_lds, n_stops_all) : times_mid(pd.stops, n_stops_all);
    }
    // the k-th time to aim at: a stop, else the end
    auto aim = [&](uint32_t k, uint32_t count, double end) -> double {
        if (!STOPS || k >= count) return end;
        return in_lds ? stops_lds[k] : gptr(pd.stops)[k];
    };
    uint32_t budget = cap;
    WaveQueue queue(counter);
    int64_t inst = queue.start(n, dv->order);
    bool take = inst >= 0;
    uint32_t attempts = 0, nacc = 0, next_stop = 0, n_stops = 0, nrec = 0;
    uint32_t every_left = every;  // accepted steps until the next record
    uint32_t room = 0;            // entries until the ring wraps
    double *at_t = nullptr, *at_y = nullptr;  // the next record's place
    double target = 0.0;          // the next stop, else the end
    double after = 0.0;           // the one after it
    auto ring_start = [&]() {
        const uint64_t i = (uint64_t)inst;
        room = capacity;
        if constexpr (PACKED) {
            at_t = records + i * capacity * kRecord<D>;
        } else {
            at_t = pd.path_t + i * (inst_major ? capacity : 1u);
            at_y = pd.path_y + i * (inst_major ? (uint64_t)capacity * D : 1u);
        }
    };
    auto record = [&]() {
        if (capacity) {
            if constexpr (PACKED) {
                typedef double pair_t __attribute__((ext_vector_type(2)));
                auto *p = gptr((pair_t *)at_t);
                p[0] = pair_t{L.t, L.y[0]};
#pragma unroll
                for (int c = 1; c < D; c += 2)
                    p[(c + 1) / 2] = pair_t{L.y[c], L.y[c + 1 < D ? c + 1 : c]};
                at_t += kRecord<D>;
            } else {
                *gptr(at_t) = L.t;
                at_t += stride;
#pragma unroll
                for (int c = 0; c < D; ++c) {
                    *gptr(at_y) = L.y[c];
                    at_y += stride;
                }
            }
            if (--room == 0) ring_start();
        }
        ++nrec;
    };
    for (;;) {
        int st = -1;
        if (take) {
            rk_load(L, desc_inputs(dv), (uint64_t)inst);
            attempts = nacc = nrec = 0;
            every_left = every;
            ring_start();
            if constexpr (STOPS) {
                n_stops = in_lds ? count_stops(stops_lds, n_stops_all, L.end)
                                 : count_stops(pd.stops, n_stops_all, L.end);
                next_stop = in_lds ? count_stops(stops_lds, n_stops, L.t)
                                   : count_stops(pd.stops, n_stops, L.t);
                while (next_stop < n_stops && aim(next_stop, n_stops, 0.0) <= L.t) ++next_stop;
                after = aim(next_stop + 1, n_stops, L.end);
            }
            target = aim(next_stop, n_stops, L.end);
            if (L.t >= L.end) st = BG_OK;
            L.set_range(stops_mid);
            L.head(target);
        }
        const int active = __popcll(ballot(inst >= 0));
        if (active == 0) break;
        const bool drained = queue.drained();
        const int want = drained ? active : 1;
        for (;;) {
            const uint64_t running = ballot(inst >= 0 && st < 0);
            if (active - __popcll(running) >= want) break;
            uint32_t made = 0;
            if (inst >= 0 && st < 0) {
                bool failed, accepted;
                uint64_t at_end, fail, out;
                do {
                    const double dt_proposed = L.dt;
                    accepted = L.attempt(failed, nacc);
                    const bool at_stop =
                        STOPS && accepted && L.clamped && next_stop < n_stops;
                    // an accepted step cut short to land on a stop hands the
                    // next attempt at least the step size proposed before the
                    // cut: a stop just past an accepted time must not shrink
                    // dt below dt_min and fail a solve that succeeds without
                    // the stop
                    if constexpr (STOPS) {
                        const double longer = qmax(L.dt, dt_proposed);
                        L.dt = at_stop ? longer : L.dt;
                    }
                    const bool low = L.dt < L.dt_min && L.t < L.end;
                    if constexpr (LOOP == kStopsOnly) {
                        if (accepted && !low && (at_stop || L.t >= L.end)) {
                            const double read =
                                stops_lds[next_stop + 2 < kObsLds ? next_stop + 2 : kObsLds - 1];
                            const double later = next_stop + 2 < n_stops ? read : L.end;
                            L.t = at_stop ? target : L.t;
                            target = at_stop ? after : target;
                            after = at_stop ? later : after;
                            next_stop += at_stop ? 1u : 0u;
                            record();
                        }
                    } else if (accepted && !low) {
                        if (STOPS && at_stop) {
                            L.t = target;
                            ++next_stop;
                            target = after;
                            after = aim(next_stop + 1, n_stops, L.end);
                        }
                        --every_left;
                        const bool rec = STOPS && stops_only ? (at_stop || L.t >= L.end)
                                                             : (every_left == 0);
                        if (every_left == 0) every_left = every;
                        if (rec) record();
                    }
                    L.head(target);
                    ++made;
                    at_end = ballot(L.t >= L.end);
                    fail = ballot(low);
                    out = at_end | fail;
                    if constexpr (kRhsFails<RHS>) out |= ballot(failed);
                } while (out == 0 && made < budget);
                attempts += made;
                if (failed) {
                    st = BG_USER_ERROR;
                } else if (lane_bit(fail)) {
                    st = BG_MINIMUM_TIME_DELTA_EXCEEDED;
                    if (accepted) --nacc;
                } else if (lane_bit(at_end)) {
                    st = BG_OK;
                } else if (attempts >= cap) {
                    st = BG_MAXIMUM_ITERATIONS_EXCEEDED;
                }
            }
            const uint32_t rounds = first_of(made, running);
            queue.ticks += rounds;
            budget -= rounds;
            if (budget == 0) budget = cap - wave_max_u32(inst >= 0 && st < 0 ? attempts : 0u);
        }
        take = inst >= 0 && st >= 0;
        if (take) {
            const uint32_t lost =
                st == BG_USER_ERROR || st == BG_MINIMUM_TIME_DELTA_EXCEEDED ? 1u : 0u;
            rk_store(L, desc_outputs(dv), (uint64_t)inst, st, nacc, attempts - nacc - lost);
            if (pd.path_len) gptr(pd.path_len)[inst] = nrec;
            if constexpr (PACKED) n_records[inst] = nrec;
        }
        if (drained) break;
        uint32_t pos;
        const int64_t got = queue.next(counter, (uint32_t)n, desc_at_use(dv)->order, take, pos);
        if (take) inst = got;
        take = take && inst >= 0;
    }
}

// The packed records to the caller's arrays: only entries that were written
// (the first min(records, capacity) of an instance) are read and moved.  A
// block moves kUnpackSlots entries of 64 instances at a time through LDS, so
// that it reads runs of kUnpackSlots records and, in the default layout, writes
// 64 neighbours, and stops at the most that any of the 64 has.
// Bound by HBM: 537 MB in, 537 MB out in 0.21 ms (5.1 TB/s).
constexpr int kUnpackSlots = 8;
template <int D>
__global__ void __launch_bounds__(256)
    path_unpack_kernel(const double *__restrict__ records, const uint32_t *__restrict__ n_records,
                       uint64_t n, const bg_path_desc pd) {
    constexpr int W = kRecord<D>, RUN = kUnpackSlots * W;
    __shared__ double tile[64][RUN + 1];
    __shared__ uint32_t have_of[64];
    const uint32_t capacity = pd.capacity;
    const uint64_t i0 = (uint64_t)blockIdx.x * 64;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t have = i0 + lane < n ? n_records[i0 + lane] : 0u;
    have = have < capacity ? have : capacity;
    if (wave == 0) have_of[lane] = have;
    const uint32_t most = wave_max_u32(have);
    __syncthreads();
    for (uint32_t e0 = blockIdx.y * kUnpackSlots; e0 < most; e0 += gridDim.y * kUnpackSlots) {
        for (uint32_t k = threadIdx.x; k < 64 * RUN; k += 256) {
            const uint32_t i = k / RUN, f = k % RUN;
            if (e0 + f / W < have_of[i]) tile[i][f] = records[((i0 + i) * capacity + e0) * W + f];
        }
        __syncthreads();
        if ((pd.flags & BG_PATH_INSTANCE_MAJOR) != 0) {
            // consecutive threads: consecutive values of one instance
            for (uint32_t k = threadIdx.x; k < 64u * kUnpackSlots * (1 + D); k += 256) {
                const uint32_t i = k / (kUnpackSlots * (1 + D)), r = k % (kUnpackSlots * (1 + D));
                const uint32_t e = r < kUnpackSlots ? r : (r - kUnpackSlots) / D;
                if (e0 + e >= have_of[i]) continue;
                const uint64_t at = (i0 + i) * capacity + e0 + e;
                if (r < kUnpackSlots) {
                    pd.path_t[at] = tile[i][e * W];
                } else {
                    const uint32_t c = (r - kUnpackSlots) % D;
                    pd.path_y[at * D + c] = tile[i][e * W + 1 + c];
                }
            }
        } else {
            for (uint32_t r = wave; r < kUnpackSlots * (1 + D); r += 4) {
                const uint32_t e = r / (1 + D), c = r % (1 + D);
                if (e0 + e >= have) break;
                const uint64_t at = e0 + e;
                const double v = tile[lane][e * W + c];
                if (c == 0) pd.path_t[at * n + i0 + lane] = v;
                else pd.path_y[(at * D + c - 1) * n + i0 + lane] = v;
            }
        }
        __syncthreads();  // before the next entries overwrite the tile
    }
}

// Plain path: one instance per launch, one lane.
template <class RHS, class Tab>
__global__ void __launch_bounds__(64) rk_plain_kernel(const bg_ensemble_desc d, uint64_t k) {
    r8_init();
    if (threadIdx.x != 0) return;
    RkLane<RHS, Tab> L;
    const uint64_t i = d.order ? (uint64_t)d.order[k] : k;
    const uint32_t cap = attempt_cap(d.max_attempts);
    rk_load(L, d, i);
    uint32_t attempts = 0;
    uint32_t nacc = 0, nrej = 0;
    int st = L.t >= L.end ? BG_OK : -1;
    while (st < 0) st = rk_advance(L, attempts, cap, nacc, nrej);
    rk_store(L, d, i, st, nacc, nrej);
}

// Single-instance path production: yields every accepted (t, y) into the
// path buffer; stops when the buffer is full (resumable) or the solve ends.
template <class RHS, class Tab>
__global__ void __launch_bounds__(64)
    rk_path_kernel(PathState *__restrict__ st, double *__restrict__ path_t,
                   double *__restrict__ path_y, uint32_t cap) {
    constexpr int D = RHS::D, S = Tab::S;
    r8_init();
    if (threadIdx.x != 0) return;
    RkLane<RHS, Tab> L;
    L.t = st->t;
    L.dt = st->dt;
    L.end = st->end;
    L.tol = st->tol;
    L.dt_min = st->dt_min;
    L.dt_max = st->dt_max;
#pragma unroll
    for (int k = 0; k < D; ++k) L.y[k] = st->y[k];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int k = 0; k < D; ++k) L.K[s][k] = st->K[s][k];
#pragma unroll
    for (int k = 0; k < RHS::P; ++k) L.p[k] = st->p[k];
    L.set_range();
    uint32_t attempts = (uint32_t)st->attempts;
    const uint32_t max_att = (uint32_t)st->max_attempts;
    uint32_t nacc = st->n_accepted, nrej = st->n_rejected, count = 0;
    int status = BG_OK, finished = st->finished;
    while (!finished && count < cap) {
        if (L.t >= L.end) {
            finished = 1;
            break;
        }
        const uint32_t before = nacc;
        const int r = rk_advance(L, attempts, max_att, nacc, nrej);
        if (nacc != before) {
            path_t[count] = L.t;
#pragma unroll
            for (int k = 0; k < D; ++k) path_y[(uint64_t)count * D + k] = L.y[k];
            ++count;
        }
        if (r > 0) {
            status = r;
            finished = 1;
        } else if (r == BG_OK) {
            finished = 1;
        }
    }
    st->t = L.t;
    st->dt = L.dt;
#pragma unroll
    for (int k = 0; k < D; ++k) st->y[k] = L.y[k];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int k = 0; k < D; ++k) st->K[s][k] = L.K[s][k];
    st->attempts = attempts;
    st->n_accepted = nacc;
    st->n_rejected = nrej;
    st->status = status;
    st->finished = finished;
    st->count = count;
}

// Work-queue start: the lanes' own positions are taken (a kernel rather than
// a memset so the launch sequence stays capturable).  counter[1]: the blocks at
// work.
__global__ void rk_counter_kernel(uint32_t *counter, uint32_t blocks, uint32_t block) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        counter[0] = blocks * block;
        counter[1] = blocks;
    }
}

// The same with the choice of rk_default_waves: `many` blocks if the instances
// are alike, by the predicted cost (t_end - t0) tol^(-1/4) of 1,024 of them (its
// fourth power: no root), else `few`.
__global__ void __launch_bounds__(1024)
    rk_look_kernel(uint32_t *counter, uint32_t few, uint32_t many, uint32_t block,
                   const bg_ensemble_desc d) {
    const uint64_t i = (uint64_t)threadIdx.x * d.n / 1024;
    const double t0 = d.t0 ? d.t0[i] : d.t0_s, end = d.t_end ? d.t_end[i] : d.t_end_s;
    const double tol = d.tol ? d.tol[i] : d.tol_s;
    const double span2 = (end - t0) * (end - t0);
    double lo = span2 * span2 / tol, hi = lo;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, m));
        hi = fmax(hi, __shfl_xor(hi, m));
    }
    __shared__ double lows[16], highs[16];
    if (__lane_id() == 0) {
        lows[threadIdx.x >> 6] = lo;
        highs[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) {
            lo = fmin(lo, lows[w]);
            hi = fmax(hi, highs[w]);
        }
        const uint32_t blocks = hi <= 81.0 * lo ? many : few;
        counter[0] = blocks * block;
        counter[1] = blocks;
    }
}

// ---------------------------------------------------------------------------
// Dispatch (method, rhs, dim, semantics) -> template instance.
// ---------------------------------------------------------------------------
template <class V>
static int visit_rk(int method, int rhs, int semantics, uint32_t dim, V &&v) {
    if (semantics != BG_AS_BUILT && semantics != BG_INTENDED) return BG_ERR_INVALID_ARGUMENT;
    auto with_tab = [&](auto rtag) -> int {
        if (method == BG_RK45)
            return semantics == BG_AS_BUILT ? v(rtag, Tag<Tableau<Fehlberg45, true>>{})
                                            : v(rtag, Tag<Tableau<Fehlberg45, false>>{});
        if (method == BG_RK23)
            return semantics == BG_AS_BUILT ? v(rtag, Tag<Tableau<BogackiShampine23, true>>{})
                                            : v(rtag, Tag<Tableau<BogackiShampine23, false>>{});
        return BG_ERR_UNSUPPORTED;
    };
#define BG_SCALAR_FAMILY(ID, TPL)                          \
    case ID:                                               \
        if (dim == 1) return with_tab(Tag<TPL<1>>{});      \
        if (dim == 2) return with_tab(Tag<TPL<2>>{});      \
        return BG_ERR_UNSUPPORTED;
    switch (rhs) {
        BG_SCALAR_FAMILY(BG_RHS_EXP, RhsExp)
        BG_SCALAR_FAMILY(BG_RHS_NEG, RhsNeg)
        BG_SCALAR_FAMILY(BG_RHS_QUADRATIC, RhsQuadratic)
        BG_SCALAR_FAMILY(BG_RHS_COS, RhsCos)
        BG_SCALAR_FAMILY(BG_RHS_FAIL_AFTER, RhsFailAfter)
    case BG_RHS_LORENZ:
        return dim == 3 ? with_tab(Tag<RhsLorenz>{}) : BG_ERR_INVALID_ARGUMENT;
    case BG_RHS_LOTKA_VOLTERRA:
        return dim == 2 ? with_tab(Tag<RhsLotkaVolterra>{}) : BG_ERR_INVALID_ARGUMENT;
    case BG_RHS_OSCILLATOR:
        return dim == 2 ? with_tab(Tag<RhsOscillator>{}) : BG_ERR_INVALID_ARGUMENT;
    case BG_RHS_ROBERTSON:
        return dim == 3 ? with_tab(Tag<RhsRobertson>{}) : BG_ERR_INVALID_ARGUMENT;
    case BG_RHS_TWO_LEVEL:
        return dim == 4 ? with_tab(Tag<RhsTwoLevel>{}) : BG_ERR_INVALID_ARGUMENT;
    default:
        return BG_ERR_UNSUPPORTED;
    }
#undef BG_SCALAR_FAMILY
}

bool rk_supported(int method, int rhs, uint32_t dim) {
    return visit_rk(method, rhs, BG_INTENDED, dim, [](auto, auto) { return BG_OK; }) == BG_OK;
}

static int check_desc(const bg_ensemble_desc &d, int P) {
    if (d.n == 0) return BG_OK;
    if (d.n > 0x7fffffffull) return BG_ERR_INVALID_ARGUMENT;
    if (!d.y0) return BG_ERR_INVALID_ARGUMENT;
    if (P > 0 && (!d.params || d.n_params < (uint32_t)P)) return BG_ERR_INVALID_ARGUMENT;
    return BG_OK;
}

int rk_launch_ensemble(int method, int rhs, int semantics, const bg_ensemble_desc &d,
                       const bg_launch &lc, hipStream_t stream, void *ws_in) {
    // the shared-matrix linear right-hand side runs as a tiled MFMA GEMM kernel
    if (rhs == BG_RHS_LINEAR) return linear_launch_ensemble(method, semantics, d, stream, ws_in);
    return visit_rk(method, rhs, semantics, d.dim, [&](auto rtag, auto ttag) -> int {
        using R = typename decltype(rtag)::type;
        using T = typename decltype(ttag)::type;
        int rc = check_desc(d, R::P);
        if (rc != BG_OK || d.n == 0) return rc;
        const uint32_t block = lc.block ? lc.block : 256;
        if (block % 64 || block > 256) return BG_ERR_INVALID_ARGUMENT;
        int dev = 0;
        BG_HIP_CHECK(hipGetDevice(&dev));
        int per_cu = 0;
        BG_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, rk_ensemble_kernel<R, T>, (int)block, 0));
        const int n_cu = device_cu_count(dev);
        bool look = false;
        const uint32_t waves = rk_default_waves(d.t0 || d.t_end || d.tol, d.n, n_cu, look);
        const uint32_t want = lc.blocks_per_cu ? lc.blocks_per_cu : blocks_of_waves(waves, block);
        if (per_cu < 1) per_cu = 1;
        const uint64_t need = (d.n + block - 1) / block;
        auto grid_of = [&](uint32_t blocks) -> uint64_t {
            const uint64_t g = (blocks < (uint32_t)per_cu ? blocks : (uint64_t)per_cu) * (uint64_t)n_cu;
            return g < need ? g : need;
        };
        const uint64_t grid = grid_of(want);
        const uint64_t few =
            look && !lc.blocks_per_cu ? grid_of(blocks_of_waves(kRkWavesFew, block)) : grid;
        const uint32_t refill_min = lc.refill_min ? lc.refill_min : 1u;
        // a lane for every instance: no queue, no workspace
        const bool queue = d.n > few * block;
        char *ws = (char *)ws_in;
        if (queue) {
            if (!ws_in) BG_HIP_CHECK(hipMallocAsync((void **)&ws, kLaunchWorkspaceBytes, stream));
            if (few < grid)
                rk_look_kernel<<<1, 1024, 0, stream>>>((uint32_t *)ws, (uint32_t)few,
                                                       (uint32_t)grid, block, d);
            else
                rk_counter_kernel<<<1, 64, 0, stream>>>((uint32_t *)ws, (uint32_t)grid, block);
        }
        // With a schedule the longest instances are the first ones: the waves
        // that still hold one of those that they started with go first (the
        // older waves do anyway; once they have finished theirs they give way to
        // the younger ones that have not): 2^20 Lorenz-63 of bounds of their own
        // 54.9 -> 49.5 ms, 50.4 with the first three quarters of the positions.
        const uint32_t prio = lc.prio_cutoff ? lc.prio_cutoff
                              : d.order && queue ? (uint32_t)(few * block) : 0u;
        rk_ensemble_kernel<R, T><<<(uint32_t)grid, block, 0, stream>>>(
            d, queue ? (uint32_t *)ws : nullptr, refill_min, prio);
        const hipError_t launched = hipGetLastError();
        if (queue && !ws_in) BG_HIP_CHECK(hipFreeAsync(ws, stream));
        BG_HIP_CHECK(launched);
        return BG_OK;
    });
}

int rk_launch_plain(int method, int rhs, int semantics, const bg_ensemble_desc &d,
                    hipStream_t stream) {
    return visit_rk(method, rhs, semantics, d.dim, [&](auto rtag, auto ttag) -> int {
        using R = typename decltype(rtag)::type;
        using T = typename decltype(ttag)::type;
        int rc = check_desc(d, R::P);
        if (rc != BG_OK) return rc;
        for (uint64_t k = 0; k < d.n; ++k) {
            rk_plain_kernel<R, T><<<1, 64, 0, stream>>>(d, k);
            BG_HIP_CHECK(hipGetLastError());
            BG_HIP_CHECK(hipStreamSynchronize(stream));
        }
        return BG_OK;
    });
}

int rk_launch_path(int method, int rhs, int semantics, uint32_t dim, PathState *state,
                   double *path_t, double *path_y, uint32_t cap, hipStream_t stream) {
    return visit_rk(method, rhs, semantics, dim, [&](auto rtag, auto ttag) -> int {
        using R = typename decltype(rtag)::type;
        using T = typename decltype(ttag)::type;
        rk_path_kernel<R, T><<<1, 64, 0, stream>>>(state, path_t, path_y, cap);
        BG_HIP_CHECK(hipGetLastError());
        return BG_OK;
    });
}

// Sizes between which the path kernel packs its records (see there).
constexpr size_t kPackedMin = (size_t)32 << 20, kPackedMax = (size_t)1 << 30;

// Workspace of the packed records: a pool of its own on each device that keeps
// up to kPackedMax bytes from one call to the next.  From the default pool,
// which gives everything back at each synchronisation, a call paid for fresh
// memory whenever the driver had to clear it first (28 ms per GB once a program
// has used as much as the card holds: 15 ms for a ring of 537 MB that is
// recorded in 1 ms).  The memory goes back when kPoolSpared calls in a row have
// done without it, or when the pool cannot serve a call.  One lock: the pools
// are shared by all threads and streams, each allocation is ordered on its
// caller's stream.
constexpr uint32_t kPoolSpared = 16;
struct RecordPool {
    hipMemPool_t pool;
    uint32_t spared;
};
static std::mutex g_record_mutex;
static RecordPool g_record_pool[64];

static char *take_records(int dev, size_t bytes, hipStream_t stream) {
    if (dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lk(g_record_mutex);
    RecordPool &rp = g_record_pool[dev];
    if (!rp.pool) {
        hipMemPoolProps props;
        memset(&props, 0, sizeof props);
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        uint64_t keep = kPackedMax;
        if (hipMemPoolCreate(&pool, &props) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) != hipSuccess)
            (void)hipGetLastError();  // then every call allocates
        rp.pool = pool;
    }
    rp.spared = 0;
    for (int attempt = 0; attempt < 2; ++attempt) {
        char *p = nullptr;
        if (hipMallocFromPoolAsync((void **)&p, bytes, rp.pool, stream) == hipSuccess) return p;
        (void)hipGetLastError();
        (void)hipMemPoolTrimTo(rp.pool, 0);
    }
    return nullptr;
}

// A call that needs no records' workspace.
static void spare_records(int dev) {
    if (dev < 0 || dev >= 64) return;
    std::lock_guard<std::mutex> lk(g_record_mutex);
    RecordPool &rp = g_record_pool[dev];
    if (rp.pool && rp.spared < kPoolSpared && ++rp.spared == kPoolSpared)
        (void)hipMemPoolTrimTo(rp.pool, 0);
}

int rk_launch_path_ensemble(int method, int rhs, int semantics, const bg_ensemble_desc &d,
                            const bg_path_desc &p, hipStream_t stream) {
    return visit_rk(method, rhs, semantics, d.dim, [&](auto rtag, auto ttag) -> int {
        using R = typename decltype(rtag)::type;
        using T = typename decltype(ttag)::type;
        int rc = check_desc(d, R::P);
        if (rc != BG_OK || d.n == 0) return rc;
        if (p.capacity && (!p.path_t || !p.path_y)) return BG_ERR_INVALID_ARGUMENT;
        if (p.n_stops && !p.stops) return BG_ERR_INVALID_ARGUMENT;
        int dev = 0;
        BG_HIP_CHECK(hipGetDevice(&dev));
        // Packed records when the caller's arrays are larger than the chip's
        // L2 (below that the lines stay until they are full), unless only
        // stops are recorded (there the lanes of a wave write the same entry
        // within a short time), the array is instance-major and small (its
        // instances' lines, two per lane, fit L2 up to some 10^5 of them; at
        // 131,072 and 128 entries short paths take 0.32 ms direct and 0.41
        // packed, rings that wrap 20 times 7.3 and 5.1, which the host cannot
        // tell apart; at 20,000 0.17 and 0.23, 2.3 and 2.2; at 262,144 and 64
        // entries 17 and 8.7), the workspace, which is sized by the capacity and not by the records,
        // exceeds what its pool keeps (200,000 Lotka-Volterra instances, 50
        // steps each, capacity 1000: see kPackedMax) or the stream is being
        // captured.
        constexpr int W = kRecord<R::D>;
        const size_t record_bytes = (size_t)d.n * p.capacity * W * sizeof(double);
        const size_t bytes = record_bytes + d.n * sizeof(uint32_t);
        double *records = nullptr;
        uint32_t *n_records = nullptr;
        const bool pack = !(p.flags & BG_PATH_STOPS_ONLY) && record_bytes >= kPackedMin &&
                          bytes <= kPackedMax &&
                          !((p.flags & BG_PATH_INSTANCE_MAJOR) && d.n <= 131072);
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {
            (void)hipGetLastError();
            capturing = hipStreamCaptureStatusActive;
        }
        if (capturing == hipStreamCaptureStatusNone) {
            if (pack) {
                // no room: straight to the caller's arrays
                char *ws = take_records(dev, bytes, stream);
                records = (double *)ws;
                if (ws) n_records = (uint32_t *)(ws + record_bytes);
            } else {
                spare_records(dev);
            }
        }
        const bool stops_only = (p.flags & BG_PATH_STOPS_ONLY) != 0;
        const auto kern =
            stops_only && p.n_stops <= kObsLds ? rk_path_ensemble_kernel<R, T, false, kStopsOnly>
            : stops_only || p.n_stops > 0
                ? (records ? rk_path_ensemble_kernel<R, T, true, kRingStops>
                           : rk_path_ensemble_kernel<R, T, false, kRingStops>)
                : (records ? rk_path_ensemble_kernel<R, T, true, kRing>
                           : rk_path_ensemble_kernel<R, T, false, kRing>);
        int per_cu = 0;
        uint32_t *counter = nullptr;
        auto run = [&]() -> hipError_t {
            hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 256, 0);
            if (e != hipSuccess) return e;
            if (per_cu < 1) per_cu = 1;
            uint64_t grid = (uint64_t)per_cu * (uint64_t)device_cu_count(dev);
            const uint64_t need = (d.n + 255) / 256;
            if (grid > need) grid = need;
            if (d.n > grid * 256) {
                e = hipMallocAsync((void **)&counter, kLaunchWorkspaceBytes, stream);
                if (e != hipSuccess) return e;
                rk_counter_kernel<<<1, 64, 0, stream>>>(counter, (uint32_t)grid, 256u);
            }
            kern<<<(uint32_t)grid, 256, 0, stream>>>(d, p, counter, records, n_records);
            if (records) {
                // at most 65,536 blocks, each over as many entries as that takes
                const uint32_t columns = (uint32_t)((d.n + 63) / 64);
                uint32_t rows = (p.capacity + kUnpackSlots - 1) / kUnpackSlots;
                const uint32_t most = columns < 32768u ? 65536u / columns : 2u;
                // (the y dimension of a grid ends at 65,536)
                const dim3 tiles(columns, rows < most ? rows : most < 65535u ? most : 65535u);
                path_unpack_kernel<R::D><<<tiles, 256, 0, stream>>>(records, n_records, d.n, p);
            }
            return hipGetLastError();
        };
        const hipError_t launched = run();
        // the workspaces go back on every path
        const hipError_t f1 = counter ? hipFreeAsync(counter, stream) : hipSuccess;
        const hipError_t f2 = records ? hipFreeAsync(records, stream) : hipSuccess;
        BG_HIP_CHECK(launched);
        BG_HIP_CHECK(f1);
        BG_HIP_CHECK(f2);
        return BG_OK;
    });
}

}  // namespace bg
