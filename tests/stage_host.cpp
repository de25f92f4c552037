// Host run of the staged upload (stage_ready, stage_pieces of wfh_stage.h) for CPU tests: the transfers
// are copies, and their events, waits and failures are the test's.
#include <dirent.h>
#include <sys/resource.h>

#include <chrono>
#include <cstdlib>
#include <vector>

#include "wfh_stage.h"

using namespace wfh;

static int process_threads() {
    int n = 0;
    if (DIR* d = opendir("/proc/self/task")) {
        while (const dirent* e = readdir(d)) n += e->d_name[0] != '.';
        closedir(d);
    }
    return n;
}

// Three arrays of n doubles in `in` to `out` [3 n]. Fails the wait or the send of piece fail_wait /
// fail_send (counted from 0, -1: none); each wait takes wait_us of sleep. info: seconds of CPU time,
// seconds, pieces sent, a slot sent again before it was waited for (0 / 1), threads of the call. Returns
// stage_pieces's result.
extern "C" int host_stage(const double* in, double* out, long n, int fail_wait, int fail_send, int wait_us,
                          double* info) {
    const double* const src[3] = {in, in + n, in + 2 * n};
    std::vector<double> pin(HF_SLOTS * HF_SLOT);
    bool pending[HF_SLOTS] = {};
    int waits = 0, sends = 0;
    bool reused = false;
    const int before = process_threads();
    int threads = 0;
    const auto cpu = [] {
        rusage u;
        getrusage(RUSAGE_SELF, &u);
        return (double)(u.ru_utime.tv_sec + u.ru_stime.tv_sec) + 1e-6 * (double)(u.ru_utime.tv_usec + u.ru_stime.tv_usec);
    };
    const double c0 = cpu();
    const auto t0 = std::chrono::steady_clock::now();
    const bool ok = stage_pieces(
        src, (size_t)n, pin.data(),
        [&](const int slot) {
            threads = std::max(threads, process_threads() - before + 1);
            if (waits++ == fail_wait) return false;
            if (wait_us > 0) std::this_thread::sleep_for(std::chrono::microseconds(wait_us));
            pending[slot] = false;
            return true;
        },
        [&](const size_t off, const int slot, const size_t len) {
            if (sends++ == fail_send) return false;
            reused = reused || pending[slot];
            pending[slot] = true;
            std::memcpy(out + off, pin.data() + (size_t)slot * HF_SLOT, len * sizeof(double));
            return true;
        });
    info[0] = cpu() - c0;
    info[1] = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    info[2] = sends;
    info[3] = reused;
    info[4] = threads;
    return ok;
}

// stage_ready with an allocation or event (counted together from 0) that fails at `fail`, then again with
// none: results of both calls in rc, whether every event is there after each in made, events and
// allocations made in all in count.
extern "C" void host_ready(int fail, int* rc, int* made, int* count) {
    double* pin = nullptr;
    int* slot[HF_SLOTS] = {};
    int calls = 0;
    static int object;
    count[0] = count[1] = 0;
    for (int k = 0; k < 2; ++k) {
        rc[k] = stage_ready(
            pin, slot,
            [&](double*& p) {
                p = (double*)&object;  // (a failing call may leave anything)
                if (calls++ == fail) return false;
                ++count[0];
                return true;
            },
            [&](int*& e) {
                e = &object;
                if (calls++ == fail) return false;
                ++count[1];
                return true;
            });
        made[k] = pin != nullptr;
        for (int* e : slot) made[k] = made[k] && e != nullptr;
    }
}

extern "C" long host_slot() { return (long)HF_SLOT; }
