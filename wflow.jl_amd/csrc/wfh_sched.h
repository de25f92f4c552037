// The exchange of the routing kernels: outflow slots between waves, the passes of one routing family
// over the 64 cells of a wave (run_sched), and the ranks that order them (chunk_ranks).
//
// The file needs of its includer the wave's operations only (__any, __ballot, the wave barrier, the
// atomics), so that a host build can run the same source, a lane at a time, under any interleaving
// of the waves (tests/sched_host.cpp).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "wfh_math.h"

namespace wfh {

constexpr uint64_t SLOT_EMPTY = 0xFFF40000DEADBEEFULL;  // signalling NaN, never produced by arithmetic
constexpr int WAVE = 64;

__device__ __forceinline__ void slot_put(uint64_t* s, double v) {
    __hip_atomic_store(s, wfh_bits(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool slot_take(uint64_t* s, double& v) {
    const uint64_t b = __hip_atomic_load(s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (b == SLOT_EMPTY) return false;
    __hip_atomic_store(s, SLOT_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = wfh_from_bits(b);
    return true;
}

// Folds of the upstream discharge in the reference's left-fold order (sum_at, utils.jl:472-477).
//   FOLD_SSF: acc1 = sum q (1 - f)  (q_in),   acc2 = sum q f  (to_river)   lateral_subsurface_flow.jl:228-240
//   FOLD_OL:  acc1 = sum q f (to_river),      acc2 = sum q (1 - f) (qin)    surface_kinwave.jl:317-326
//   FOLD_RIV: acc1 = sum q                                                  surface_kinwave.jl:520
//   FOLD_SNOW: acc1 = own material + material passed on by each upstream cell, in the reference's
//              topological order of the upstream cells (accucapacityflux!  routing/utils.jl:82-108)
//   FOLD_RIV_RES (a model with reservoirs): acc1 = sum q over the non-reservoir upstream cells,
//             acc2 = outflow of an upstream reservoir (f = 1 on that edge)  surface_kinwave.jl:478,520
enum { FOLD_SSF = 0, FOLD_OL = 1, FOLD_RIV = 2, FOLD_RIV_RES = 3, FOLD_SNOW = 4 };

template <int FOLD>
__device__ __forceinline__ void fold_in(double& acc1, double& acc2, double q, double f) {
    if (FOLD == FOLD_SSF) {
        acc1 = acc1 + q * (1.0 - f);
        acc2 = acc2 + q * f;
    } else if (FOLD == FOLD_OL) {
        acc1 = acc1 + q * f;
        acc2 = acc2 + q * (1.0 - f);
    } else if (FOLD == FOLD_RIV_RES && f != 0.0) {
        acc2 = q;  // a reservoir's outflow is assigned to the downstream inflow (surface_kinwave.jl:478)
    } else {
        acc1 = acc1 + q;
    }
}

// One family of routing sub-steps (all subsurface, all overland or all river sub-steps of the
// model step) for the 64 cells of a wave, as a sequence of passes in which the lanes of the pass
// compute one sub-step each.
//
// Bound: the latency of one pass times the cells of the longest path, and in a pass the number of
// instructions (4.5 cycles each, dependent or not) and of branches on votes (about 60 cycles). A
// pass therefore holds little but what the next cell waits for: the inflow of the lane's sub-step
// is read from LDS in one round trip (an in-wave upstream cell's outflow from the wave's table, an
// outflow from another wave from this lane's inbox, a zero for an edge that is not there, at
// addresses fixed beforehand), folded in ascending edge order (the reference's sum_at order), solved
// (`compute`), published and written to the table; lanes whose solve turns out long follow
// (`finish`), then the sums and the preparation of the next sub-step (`after`).
//   One sub-step: a lane computes as soon as its inflow is there. Which in-wave cells are left is
// one wave-uniform bit mask, held against each lane's mask of in-wave upstream cells, so a lane
// that waits for a late inflow holds up nobody else.
//   Several sub-steps: a fixed schedule. `rank` is the cell's place in its chunk (chunk_ranks), an
// in-wave upstream cell having the next lower rank, and in pass t a lane computes sub-step
// t - rank: the sub-steps of a chain run as a diagonal, and the lanes of a wave stay in step.
//   Once the inflow from other waves is complete, either kind runs its remaining passes in the
// order of the ranks, without a vote: 260 cycles a pass (trivial solve) instead of 950.
//   A chunk in which some cell has more than SCHED_PF upstream cells keeps the votes to its last pass, and
// such a cell reads its further edges inside its pass (from the table, from memory, or waiting for a
// slot while the pass's other lanes wait with it). No river cell of the timed basins has that many, but
// 0.5 to 1.5 % of the cells have five, in 24 to 33 % of the land chunks, and they gather on main stems: of
// the longest path's cells 98 % lie in such chunks at 61 x 67, 97 % at 256 x 256, 60 % at 509 x 487 and
// 35 % at 4096 x 4096.
//
// Outflow to a consumer in another wave goes through that consumer's global slot (one per edge
// and sub-step, cleared by the consumer). Slots are polled for all lanes of the wave together, at
// most RING sub-steps ahead, when a pass lacks one (or, overlapped with the pass, when a lane of
// the next passes does), and taken into the inbox; so a wave that waits for its main stem has the
// inflow of its tributaries before the main stem arrives. A wave waits only for chunks of smaller
// index, so the ticket order keeps the launch free of deadlock. Returns false when the wave has to
// stop (a wait exceeded its limit, or another wave raised the abort flag).
//
// The exchange before this one compared (sub-step, outflow) pairs of the upstream cells in every
// pass and let each lane compute whenever it was ready; the lanes of a wave drifted apart until each
// sub-step of each cell took a pass of its own. With it and the solves of that time an hourly step
// took 0.56 ms on 61 x 67 cells, 2.43 ms on 509 x 487 and 18.1 ms on 4096 x 4096, a daily one (24
// land and 96 river sub-steps) 14.6 ms on 256 x 256; now 0.30, 1.68, 15.7 and 2.0 ms.
constexpr int SCHED_PF = 4;                             // upstream edges with a place in the inbox
constexpr int SCHED_ZERO = (SCHED_PF + 1) * WAVE;       // a zero after the table row and the inbox rows
constexpr int SCHED_ROWS = SCHED_ZERO + 8;              // doubles of one sub-step
constexpr int SCHED_RING = 4;                           // sub-steps the inbox holds

// The abort flag as a wave-uniform value (a branch on the value a lane loaded is a per-lane one)
template <class Args>
__device__ __forceinline__ bool aborted(const Args& a) {
    return __builtin_amdgcn_readfirstlane(
               __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}
// The next ticket, the same for all lanes and known to be so (a shuffle's result is not)
__device__ __forceinline__ unsigned long long next_ticket(unsigned long long* counter, const int lane) {
    unsigned long long t = 0;
    if (lane == 0) t = atomicAdd(counter, 1ull);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)t);
    const unsigned hi = __builtin_amdgcn_readfirstlane((int)(unsigned)(t >> 32));
    return (unsigned long long)hi << 32 | lo;
}

// for the families' lambdas, which run_sched calls at two places
#define ROUTE_INLINE __attribute__((always_inline))

template <int RING>
__device__ __forceinline__ void sched_init(double* lds, const int lane) {
    if (lane < RING) lds[lane * SCHED_ROWS + SCHED_ZERO] = 0.0;
}

template <int FOLD, int RING, class Args, class Compute, class Finish, class After>
__device__ __forceinline__ bool run_sched(const Args& a, const int lane, const int c, const bool part,
                                          const int S, const int rank, const int nrank,
                                          const int* __restrict__ up_node, const int* __restrict__ up_slot,
                                          const double* __restrict__ up_f, const int e0, const int e1, uint64_t* slots,
                                          const size_t stride, const int my_slot, const bool pub_cross, double* lds,
                                          Compute& compute, const Finish& finish, const After& after,
                                          const double acc0 = 0.0) {
    constexpr int PF = SCHED_PF;
    static_assert((RING & (RING - 1)) == 0, "sub-step k uses row k mod RING");
    constexpr bool FRAC = FOLD != FOLD_RIV && FOLD != FOLD_SNOW;
    const int ne = part ? e1 - e0 : 0;
    int at[PF], es[PF];
    double ef[PF];
    unsigned ext = 0;   // bit j: edge e0 + j comes from another wave
    uint64_t need = 0;  // in-wave upstream lanes (used with one sub-step)
    {
        // Every lane loads PF entries (unused ones at a valid index); the empty asm takes them all
        // as operands, so the compiler issues the loads together and waits once, instead of moving
        // each into the per-lane branch that uses it and waiting for them one by one.
        int un[PF], us[PF];
        double uf[PF];
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            const int ej = j < ne ? e0 + j : (ne > 0 ? e0 : 0);
            un[j] = up_node[ej];
            us[j] = up_slot[ej];
            uf[j] = FRAC ? up_f[ej] : 0.0;
        }
        static_assert(PF == 4, "the operand list below names four edges");
        asm volatile("" : "+v"(un[0]), "+v"(un[1]), "+v"(un[2]), "+v"(un[3]), "+v"(us[0]), "+v"(us[1]), "+v"(us[2]),
                     "+v"(us[3]), "+v"(uf[0]), "+v"(uf[1]), "+v"(uf[2]), "+v"(uf[3]));
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            const bool use = j < ne, in = (un[j] >> 6) == c;
            at[j] = !use ? SCHED_ZERO : in ? (un[j] & (WAVE - 1)) : (1 + j) * WAVE + lane;
            es[j] = us[j];
            ef[j] = use ? uf[j] : 0.0;
            ext |= (use && !in) ? (1u << j) : 0u;
            need |= (use && in) ? 1ull << (un[j] & (WAVE - 1)) : 0ull;
        }
    }
    const bool many = __any(ne > PF);  // wave-uniform
    if (many)
        for (int e = e0 + PF; e < e0 + ne; ++e) {
            const int u = up_node[e];
            need |= (u >> 6) == c ? 1ull << (u & (WAVE - 1)) : 0ull;
        }
    int kf = ext ? 0 : S;  // sub-steps of this lane whose inflow from other waves is in the inbox
    unsigned got = 0;      // bit j: edge e0 + j of sub-step kf has arrived
    uint64_t v[PF];        // the poll in flight
    const auto fetch = [&](const bool want) {
        const unsigned miss = want ? ext & ~got : 0u;
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            v[j] = SLOT_EMPTY;
            if (miss >> j & 1u)
                v[j] = __hip_atomic_load(slots + (size_t)kf * stride + es[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_wave_barrier();  // (see the loop)
    };
    bool complete = !__any(kf < S);  // all inflow from other waves is in the inbox (wave-uniform)
    const auto collect = [&]() -> bool {  // true when something arrived
        bool in[PF], any = false;
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            in[j] = v[j] != SLOT_EMPTY;
            any = any || in[j];
        }
        if (!__any(any)) return false;
#pragma unroll
        for (int j = 0; j < PF; ++j)
            if (in[j]) {
                __hip_atomic_store(slots + (size_t)kf * stride + es[j], SLOT_EMPTY, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                lds[(kf & (RING - 1)) * SCHED_ROWS + (1 + j) * WAVE + lane] = wfh_from_bits(v[j]);
                got |= 1u << j;
            }
        __builtin_amdgcn_wave_barrier();  // (see the loop)
        const bool full = kf < S && got == ext;
        kf = full ? kf + 1 : kf;
        got = full ? 0u : got;
        complete = !__any(kf < S);
        return true;
    };
    // A pass of the lanes that execute: inflow, solve, publish. The lanes whose solve does not end in
    // its straight part publish after the others (`finish`), so that a long solve (an overland one
    // can take 126 updates) does not hold up the cells below the other lanes.
    const auto pass = [&](const int k, double acc1, double acc2) ROUTE_INLINE {
        double* const out = lds + (k & (RING - 1)) * SCHED_ROWS + lane;
        uint64_t* const slot = slots + (size_t)k * stride + my_slot;
        bool open = false;
        const double q1 = compute(k, acc1, acc2, open);
        if (!open) {
            *out = q1;
            if (pub_cross) slot_put(slot, q1);
        }
        if (__any(open)) {
            if (open) {
                const double q2 = finish(k);
                *out = q2;
                if (pub_cross) slot_put(slot, q2);
            }
        }
        after(k);
    };
    const int T = nrank > 0 ? nrank + S - 1 : 0;
    uint64_t left = __ballot(part);  // one sub-step: lanes that have not computed
    int mine = part ? rank : -S;     // this lane's first pass; -S once it has computed its only sub-step
    int t = 0;

    // ---- some inflow from other waves is still to come ----
    // The per-lane branches of a poll, of a look at its values and of a pass are each closed by a wave
    // barrier (no instruction): the compiler would else merge their ends with the ways round them, and
    // take every wave-uniform variable that has two values there for a per-lane one, that is, keep
    // the whole loop's state in vector registers and its branches under execution masks (1250 cycles
    // for a pass with a trivial solve, where the scheduled passes below take 260).
    // A poll issued beside a pass is looked at PASSES_PER_POLL passes later, when its values are
    // there, so that no pass waits for memory.
    constexpr int PASSES_PER_POLL = 2;
    int pending = 0;  // passes until the poll in flight is looked at (0: none)
    long spin = 0;
    while (!complete || many) {
        bool act, go;  // lanes of the pass; whether there is one (else the wave waits)
        int k = 0;
        if (S > 1) {
            if (t >= T) break;
            k = t - mine;
            act = (unsigned)k < (unsigned)S;
            go = !__any(act && kf <= k);
        } else {
            if (left == 0) break;
            act = mine >= 0 && kf > 0 && !(need & left);
            go = __any(act);
            left &= ~__ballot(act);
            mine = act ? -1 : mine;
        }
        // polls: inflow that this pass lacks, or that the next passes do
        const int kring = (k > 0 ? k : 0) + RING;  // inbox rows before this one are free or filled
        const bool want = kf < S && kf < kring;
        const bool soon = S > 1 ? kf <= k + PASSES_PER_POLL : mine >= 0 && !(need & left);
        if (pending == 0 && (!go || __any(want && soon))) {
            fetch(want);
            pending = PASSES_PER_POLL + 1;
        }
        bool stop = false;
        __builtin_amdgcn_wave_barrier();
        if (act && go) {
            const double* const row = lds + (k & (RING - 1)) * SCHED_ROWS;
            double acc1 = acc0, acc2 = 0.0;
#pragma unroll
            for (int j = 0; j < PF; ++j) fold_in<FOLD>(acc1, acc2, row[at[j]], ef[j]);
            for (int e = e0 + PF; e < e0 + ne; ++e) {
                const int u = up_node[e];
                const double f = FRAC ? up_f[e] : 0.0;
                double qe = row[u & (WAVE - 1)];
                if ((u >> 6) != c) {
                    uint64_t* const sl = slots + (size_t)k * stride + up_slot[e];
                    for (long w = 0; !stop && !slot_take(sl, qe); ++w) {
                        __builtin_amdgcn_s_sleep(1);
                        stop = w > a.spin_limit ||
                               ((w & 255) == 255 &&
                                __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    }
                }
                fold_in<FOLD>(acc1, acc2, qe, f);
            }
            if (!stop) pass(k, acc1, acc2);  // (a lane that has given up has no inflow to publish from)
        }
        __builtin_amdgcn_wave_barrier();
        if (many && __any(stop)) {  // (wave-uniform)
            __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        t += go && S > 1 ? 1 : 0;
        pending -= pending > 0 ? 1 : 0;
        if (!complete && (!go || pending == 1)) {
            pending = 0;
            if (collect()) spin = -1;
        }
        if (!go) {
            ++spin;
            if ((spin & 255) == 255 && aborted(a)) return false;
            if (spin > a.spin_limit) {
                __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
        } else {
            spin = 0;
        }
    }
    if (many) return true;

    // ---- all inflow from other waves is in the inbox: the passes left, in the order of the ranks ----
    for (; t < T; ++t) {
        const int k = t - mine;
        if ((unsigned)k < (unsigned)S) {
            const double* const row = lds + (k & (RING - 1)) * SCHED_ROWS;
            double acc1 = acc0, acc2 = 0.0;
            // an edge that is not there adds 0 (sums that start from 0 are never -0, so that is exact)
#pragma unroll
            for (int j = 0; j < PF; ++j) fold_in<FOLD>(acc1, acc2, row[at[j]], ef[j]);
            pass(k, acc1, acc2);
        }
        __builtin_amdgcn_wave_barrier();
    }
    return true;
}

// The pass schedule of every chunk of 64 positions (run_sched). A cell of the chunk that drains
// inside it gets the rank just below its consumer's, so its outflow is used in the next pass; the
// last cell of such a tree is placed by its network level, so that trees whose inflow comes early
// (small levels) run before, not after, a main stem whose inflow comes late. Ranks are the chunk's
// distinct places in order, 0 first, with up to `gap` ranks from one place to the next where the
// levels are that far apart: with several sub-steps, an early tree then has its first sub-steps done
// before the pass that waits for a late one. nrank is the number of ranks, at most 253.
constexpr int SCHED_GAP = 4;
static_assert((WAVE - 1) * SCHED_GAP + 1 <= 255, "ranks are stored in 8 bits");
template <class Part>
static void chunk_ranks(const int64_t n, const Part& part, const std::vector<int>& down, const std::vector<int>& level,
                        const int gap, std::vector<uint8_t>& rank, std::vector<uint8_t>& nrank) {
    const int64_t nch = (n + WAVE - 1) / WAVE;
    rank.assign(n, 0);
    nrank.assign(std::max<int64_t>(nch, 1), 0);
    for (int64_t c = 0; c < nch; ++c) {
        const int64_t q0 = c * WAVE, q1 = std::min<int64_t>(q0 + WAVE, n);
        int key[WAVE], seen[WAVE], place[WAVE] = {0}, m = 0;
        for (int64_t q = q1 - 1; q >= q0; --q) {  // downstream cells first
            if (!part(q)) continue;
            const int dn = down[q];
            key[q - q0] = dn > q && dn < q1 ? key[dn - q0] - 1 : level[q];
            seen[m++] = key[q - q0];
        }
        std::sort(seen, seen + m);
        m = (int)(std::unique(seen, seen + m) - seen);
        for (int j = 1; j < m; ++j) place[j] = place[j - 1] + std::min(seen[j] - seen[j - 1], gap);
        for (int64_t q = q0; q < q1; ++q)
            if (part(q)) rank[q] = (uint8_t)place[std::lower_bound(seen, seen + m, key[q - q0]) - seen];
        nrank[c] = (uint8_t)(m > 0 ? place[m - 1] + 1 : 0);
    }
}

}  // namespace wfh
