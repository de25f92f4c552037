// Host arrays to the device through a ring of pinned slots: the copies by several threads, and the
// slots' memory and events. The runtime's calls come from the caller, so that a host build can run it.
#pragma once

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace wfh {

constexpr size_t HF_SLOT = 1u << 18;  // doubles of a slot (2 MiB)
constexpr int HF_SLOTS = 4, HF_THREADS = 8;
constexpr int HF_LOOKS = 256;  // (a yield each)

// The slots' memory and the event of each, as far as they are not there yet: alloc(pin) and make(event)
// return whether they could. What has been made stays for the next call.
template <class Event, class Alloc, class Make>
bool stage_ready(double*& pin, Event (&slot)[HF_SLOTS], const Alloc& alloc, const Make& make) {
    if (!pin && !alloc(pin)) {
        pin = nullptr;
        return false;
    }
    for (Event& e : slot)
        if (!e && !make(e)) {
            e = Event{};
            return false;
        }
    return true;
}

// CPUs that the process may run on
inline int usable_cpus() {
    cpu_set_t set;
    CPU_ZERO(&set);
    return sched_getaffinity(0, sizeof set, &set) == 0 ? std::max(CPU_COUNT(&set), 1) : 1;
}

// Sends three arrays of n doubles, piece by piece: wait(slot) until the slot's last transfer is over,
// the piece is copied into it by all threads, a stripe each, then send(offset, slot, length) on its way,
// offset counted over the three arrays one after another. Returns when all has been read, or at the
// first wait or send that returns false, with that.
// At most HF_THREADS threads and one for each CPU that the process may use, the caller among them. A
// helper looks HF_LOOKS times for the next piece and then sleeps until it is there. While the transfers
// run at the link's rate it finds the piece by looking: with transfers of 45 GB/s played on an eight-CPU
// host, three arrays of 1,017,937 doubles take 0.81 ms (0.75 with endless looking, 1.0 with 64 looks and
// 1.35 with none). While they do not, no core is kept busy for them.
template <class Wait, class Send>
bool stage_pieces(const double* const src[3], const size_t n, double* const pin, const Wait& wait, const Send& send) {
    const size_t per = (n + HF_SLOT - 1) / HF_SLOT;  // pieces of an array
    const int pieces = (int)(3 * per);
    // A piece is published by its number and copied by all threads, a stripe each.
    std::atomic<int> go{-1}, done{0};
    std::mutex mutex;
    std::condition_variable next;
    int threads = 1;  // set before the first piece is published
    const auto publish = [&](const int i) {
        {
            std::lock_guard<std::mutex> lock(mutex);
            go.store(i, std::memory_order_release);
        }
        next.notify_all();
    };
    const auto copy = [&](const int i, const int t) {
        const size_t off = (size_t)i % per * HF_SLOT, len = std::min(HF_SLOT, n - off);
        const size_t a = len * t / threads, b = len * (t + 1) / threads;
        std::memcpy(pin + (size_t)(i % HF_SLOTS) * HF_SLOT + a, src[(size_t)i / per] + off + a, (b - a) * sizeof(double));
    };
    const auto work = [&](const int t) {
        for (int i = 0; i < pieces; ++i) {
            for (int k = 0; k < HF_LOOKS && go.load(std::memory_order_acquire) < i; ++k) std::this_thread::yield();
            if (go.load(std::memory_order_acquire) < i) {
                std::unique_lock<std::mutex> lock(mutex);
                next.wait(lock, [&] { return go.load(std::memory_order_acquire) >= i; });
            }
            if (go.load(std::memory_order_acquire) >= pieces) return;  // given up
            copy(i, t);
            done.fetch_add(1, std::memory_order_release);
        }
    };
    std::thread helpers[HF_THREADS - 1];
    const int want = std::min(HF_THREADS, usable_cpus()) - 1;
    int started = 0;
    try {
        for (; started < want; ++started) helpers[started] = std::thread(work, started + 1);
    } catch (const std::exception&) {  // fewer threads than wanted
    }
    threads = started + 1;
    bool ok = true;
    for (int i = 0; i < pieces; ++i) {
        const int slot = i % HF_SLOTS;
        if (!(ok = wait(slot))) break;
        publish(i);
        copy(i, 0);
        while (done.load(std::memory_order_acquire) < (i + 1) * started) std::this_thread::yield();
        const size_t off = (size_t)i % per * HF_SLOT, len = std::min(HF_SLOT, n - off);
        if (!(ok = send((size_t)i / per * n + off, slot, len))) break;
    }
    if (!ok) publish(pieces);
    for (int t = 0; t < started; ++t) helpers[t].join();
    return ok;
}

}  // namespace wfh
