// Host run of the routing exchange (run_sched and chunk_ranks of wfh_sched.h, the source the kernels
// are built from) for CPU tests. A wave is 64 fibers. Every wave operation (__any, __ballot, the wave
// barrier, readfirstlane) is a meeting point: a lane runs alone up to the next one, in a random order
// of the lanes, and lanes that have left a branch early wait at the barrier that follows it. Waves take
// their chunks by ticket, a limited number of them is resident, which of them runs next is random at
// every meeting point, and what a wave publishes becomes visible to the others after a random while.
#include <setjmp.h>
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <random>
#include <vector>

#include "wfh_math.h"

namespace emu {

enum { AT_ANY, AT_BALLOT, AT_BARRIER, AT_FIRST };

struct Lane {
    ucontext_t ctx;  // for the first entry; after it the switches are jumps
    jmp_buf at;
    std::unique_ptr<char[]> stack;
    bool done = true, entered = false;
    int kind = 0, line = 0;  // the meeting point it waits at
    bool waits = false;
    uint64_t value = 0, result = 0;
};

struct Wave {
    Lane lane[64];
    std::function<void(int)> body;
    bool live = false;
};

constexpr size_t STACK = 256 << 10;
jmp_buf main_at;
Wave* cur_wave = nullptr;
int cur_lane = -1;
std::mt19937 rng;
const char* error = nullptr;

// ---- global memory: a wave's stores reach the others late ----
struct Store {
    uint64_t* p;
    uint64_t v;
    int left;
};
std::deque<Store> stores;
int max_delay = 0;

void age_stores() {  // (stores to one address keep their order: a slot is written once by each side)
    for (size_t k = 0; k < stores.size();) {
        if (stores[k].left-- <= 0) {
            *stores[k].p = stores[k].v;
            stores.erase(stores.begin() + k);
        } else {
            ++k;
        }
    }
}

std::function<void(const uint64_t*, uint64_t)> on_put;  // every value published

uint64_t load(const uint64_t* p) { return *p; }
int load(const int* p) { return *p; }
void store(uint64_t* p, uint64_t v, uint64_t empty) {
    if (v == empty) {
        *p = v;
        return;
    }
    on_put(p, v);
    stores.push_back({p, v, max_delay > 0 ? (int)(rng() % (unsigned)max_delay) : 0});
}
void store(int* p, int v, uint64_t) { *p = v; }

// ---- the wave ----
void leave(Lane& l) {  // to run()
    if (!_setjmp(l.at)) _longjmp(main_at, 1);
}

uint64_t meet(const int kind, const int line, const uint64_t value) {
    Lane& l = cur_wave->lane[cur_lane];
    l.kind = kind, l.line = line, l.value = value, l.waits = true;
    leave(l);
    return l.result;
}

void entry() {
    Lane& l = cur_wave->lane[cur_lane];
    cur_wave->body(cur_lane);
    l.done = true;
    leave(l);
}

void start(Wave& w, std::function<void(int)> body) {
    w.body = std::move(body);
    w.live = true;
    for (Lane& l : w.lane) {
        if (!l.stack) l.stack.reset(new char[STACK]);
        getcontext(&l.ctx);
        l.ctx.uc_stack.ss_sp = l.stack.get();
        l.ctx.uc_stack.ss_size = STACK;
        l.ctx.uc_link = nullptr;
        makecontext(&l.ctx, entry, 0);
        l.done = l.entered = l.waits = false;
    }
}

__attribute__((noinline)) void enter(Lane& l) {
    if (_setjmp(main_at)) return;
    if (l.entered) _longjmp(l.at, 1);
    l.entered = true;
    setcontext(&l.ctx);
}

// Runs the wave's lanes up to their meeting points (or a sleep), then resolves one meeting. The lanes
// that wait at a barrier are the ones that went round a branch, so another meeting comes first.
void run(Wave& w) {
    int order[64];
    for (int k = 0; k < 64; ++k) order[k] = k;
    std::shuffle(order, order + 64, rng);
    cur_wave = &w;
    bool blocked = true;
    for (int k : order) {
        Lane& l = w.lane[k];
        if (l.done || l.waits) continue;
        cur_lane = k;
        enter(l);
        blocked = blocked && (l.done || l.waits);
    }
    if (!blocked) return;  // a lane sleeps: the others wait for it
    std::vector<Lane*> at, all;
    for (Lane& l : w.lane)
        if (!l.done) {
            all.push_back(&l);
            if (l.kind != AT_BARRIER) at.push_back(&l);
        }
    if (all.empty()) {
        w.live = false;
        return;
    }
    if (at.empty()) at = all;
    for (Lane* l : at)
        if (l->line != at[0]->line || l->kind != at[0]->kind) {
            error = "the lanes of a wave wait at different points";
            return;
        }
    bool finished = false;
    for (const Lane& l : w.lane) finished = finished || l.done;
    if (finished) {
        error = "some lanes of a wave have returned, some have not";
        return;
    }
    uint64_t any = 0, ballot = 0;
    for (Lane* l : at)
        if (l->value) any = 1, ballot |= 1ull << (l - w.lane);
    const uint64_t first = at[0]->value;
    for (Lane* l : at) {
        l->result = l->kind == AT_ANY ? any : l->kind == AT_BALLOT ? ballot : first;
        l->waits = false;
    }
}

}  // namespace emu

#define __device__
#define __forceinline__ inline
#define __any(x) (emu::meet(emu::AT_ANY, __LINE__, (x) ? 1 : 0) != 0)
#define __ballot(x) (emu::meet(emu::AT_BALLOT, __LINE__, (x) ? 1 : 0))
#define __builtin_amdgcn_wave_barrier() ((void)emu::meet(emu::AT_BARRIER, __LINE__, 0))
#define __builtin_amdgcn_readfirstlane(x) ((int)emu::meet(emu::AT_FIRST, __LINE__, (uint64_t)(unsigned)(x)))
// a sleep: the lane goes on when its wave is run again
#define __builtin_amdgcn_s_sleep(x) (emu::leave(emu::cur_wave->lane[emu::cur_lane]))
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) (emu::load(p))
#define __hip_atomic_store(p, v, order, scope) (emu::store((p), (v), wfh::SLOT_EMPTY))
static unsigned long long atomicAdd(unsigned long long* p, unsigned long long v) {
    const unsigned long long t = *p;
    *p += v;
    return t;
}

#include "wfh_sched.h"

using namespace wfh;

namespace {
struct Args {
    int* abort_flag;
    long spin_limit;
};

// The cell of a test family: its outflow from its previous outflow, its inflow (both folds) and a
// value of its own.
struct Cell {
    double q, lat, acc = 0.0;
    bool opens;  // its solves end in `finish`
    double solve(const double a1, const double a2, const int k) {
        acc = acc + a1;
        return 0.5 * q + 0.25 * a1 + 0.125 * a2 + lat * (1.0 + k);
    }
};
}  // namespace

// chunk_ranks of n positions
extern "C" void host_ranks(long n, const uint8_t* part, const int* down, const int* level, int gap, uint8_t* rank,
                           uint8_t* nrank) {
    std::vector<uint8_t> r, nr;
    chunk_ranks(
        n, [&](int64_t q) { return part[q] != 0; }, std::vector<int>(down, down + n), std::vector<int>(level, level + n),
        gap, r, nr);
    std::memcpy(rank, r.data(), r.size());
    std::memcpy(nrank, nr.data(), nr.size());
}

// A step of `fams` families of S sub-steps over n positions: inflow edges up_ptr / up_node (position) /
// up_slot (outflow slot) / up_f in fold order, down (position or -1), and of each family's cells the first
// outflow q0 and the value lat, [fams][n]. `expect` [fams][S][n]: what each cell has to publish. Results:
// q [fams][n] last outflow, acc [fams][n] sum of the first fold. slots: [fams][S][stride], empty at the
// start; reverse: tickets in the reverse order of the chunks. Returns 0 when the step has drained, 1 when it was given up, and a negative number for an error
// of the protocol: -1 a wave operation met by part of a wave, -2 the run did not end, -3 a slot was left
// full, -4 a published value is not the expected one, -5 a value published twice.
template <int FOLD, int RING>
static int run_step(const long n, const int S, const int fams, const uint8_t* part, const int* up_ptr,
                    const int* up_node, const int* up_slot, const double* up_f, const int* down, const uint8_t* rank,
                    const uint8_t* nrank, const double* q0, const double* lat, const uint8_t* opens, const double* expect,
                    const double* acc0, const long stride, const int resident, const unsigned seed, const int max_delay,
                    const long spin_limit, const bool reverse, double* q_out, double* acc_out) {
    emu::rng.seed(seed);
    emu::error = nullptr;
    emu::stores.clear();
    emu::max_delay = max_delay;
    std::vector<uint64_t> slots((size_t)fams * S * stride, SLOT_EMPTY);
    std::vector<uint8_t> put(slots.size(), 0);
    int wrong = 0;
    emu::on_put = [&](const uint64_t* p, const uint64_t v) {
        const size_t i = p - slots.data();
        const size_t row = i / stride, q = i % stride;
        if (put[i]++) wrong = -5;
        if ((long)q >= n || v != wfh_bits(expect[row * n + q])) wrong = wrong ? wrong : -4;
    };
    int abort_flag = 0;
    const Args a{&abort_flag, spin_limit};
    const int nchunks = (int)((n + WAVE - 1) / WAVE);
    unsigned long long ticket = 0;
    std::vector<std::unique_ptr<emu::Wave>> waves;
    std::vector<std::vector<double>> lds(resident);
    for (int w = 0; w < resident; ++w) {
        waves.emplace_back(new emu::Wave);
        lds[w].assign(RING * SCHED_ROWS, 0.0 / 0.0);
        double* const table = lds[w].data();
        emu::start(*waves[w], [&, table](const int lane) {
            sched_init<RING>(table, lane);
            for (;;) {
                const unsigned long long t = next_ticket(&ticket, lane);
                if (t >= (unsigned long long)nchunks) return;
                const int c = reverse ? nchunks - 1 - (int)t : (int)t;
                const long p = (long)c * WAVE + lane;
                const bool valid = p < n && part[p];
                const long q = valid ? p : 0;
                const int e0 = up_ptr[q], e1 = valid ? up_ptr[q + 1] : e0;
                const bool cross = valid && down[q] >= 0 && down[q] / WAVE != c;
                for (int fam = 0; fam < fams; ++fam) {
                    Cell cell{q0[fam * n + q], lat[fam * n + q], 0.0, opens[q] != 0};
                    double a1 = 0.0, a2 = 0.0, qn = 0.0;
                    auto compute = [&](int k, double acc1, double acc2, bool& open) -> double {
                        a1 = acc1, a2 = acc2;
                        open = cell.opens && ((q + k) & 1);
                        qn = open ? -1.0 : cell.solve(a1, a2, k);
                        return qn;
                    };
                    const auto finish = [&](int k) -> double { return qn = cell.solve(a1, a2, k); };
                    const auto after = [&](int) { cell.q = qn; };
                    if (!run_sched<FOLD, RING>(a, lane, c, valid, S, valid ? rank[p] : 0, nrank[c], up_node, up_slot,
                                               up_f, e0, e1, slots.data() + (size_t)fam * S * stride, (size_t)stride,
                                               (int)q, cross, table, compute, finish, after,
                                               acc0 ? acc0[fam * n + q] : 0.0))
                        return;
                    if (valid) {
                        q_out[fam * n + p] = cell.q;
                        acc_out[fam * n + p] = cell.acc;
                    }
                }
            }
        });
    }
    for (long turns = 0;; ++turns) {
        std::vector<emu::Wave*> live;
        for (auto& w : waves)
            if (w->live) live.push_back(w.get());
        if (live.empty()) break;
        if (turns > 40000000) return -2;
        emu::age_stores();
        // several turns in a row, so that a wave can fall far behind another
        emu::Wave* const w = live[emu::rng() % live.size()];
        for (int k = 1 + (int)(emu::rng() % 40u); k > 0 && w->live; --k) {
            emu::run(*w);
            if (emu::error) {
                std::fprintf(stderr, "%s\n", emu::error);
                return -1;
            }
        }
    }
    while (!emu::stores.empty()) emu::age_stores();
    if (wrong) return wrong;
    if (abort_flag) return 1;
    for (uint64_t s : slots)
        if (s != SLOT_EMPTY) return -3;
    return 0;
}

extern "C" int host_step(int fold, int ring, long n, int S, int fams, const uint8_t* part, const int* up_ptr,
                         const int* up_node, const int* up_slot, const double* up_f, const int* down, const uint8_t* rank,
                         const uint8_t* nrank, const double* q0, const double* lat, const uint8_t* opens,
                         const double* expect, const double* acc0, long stride, int resident, unsigned seed,
                         int max_delay, long spin_limit, int reverse, double* q_out, double* acc_out) {
#define RUN(F, R)                                                                                                    \
    if (fold == F && ring == R)                                                                                      \
        return run_step<F, R>(n, S, fams, part, up_ptr, up_node, up_slot, up_f, down, rank, nrank, q0, lat, opens,   \
                              expect, acc0, stride, resident, seed, max_delay, spin_limit, reverse != 0, q_out, acc_out);
    RUN(FOLD_SSF, SCHED_RING)
    RUN(FOLD_OL, SCHED_RING)
    RUN(FOLD_RIV_RES, SCHED_RING)
    RUN(FOLD_SSF, 1)
    RUN(FOLD_SNOW, 1)
    return -100;
}

extern "C" void host_constants(int* pf, int* ring, int* gap) { *pf = SCHED_PF, *ring = SCHED_RING, *gap = SCHED_GAP; }
