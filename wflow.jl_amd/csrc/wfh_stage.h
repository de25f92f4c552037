// Host arrays to the device through a ring of pinned slots: the copies by several threads, and the
// slots' memory and events. The runtime's calls come from the caller, so that a host build can run it.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <thread>

namespace wfh {

constexpr size_t HF_SLOT = 1u << 18;  // doubles of a slot (2 MiB)
constexpr int HF_SLOTS = 4, HF_THREADS = 8;

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

// Sends three arrays of n doubles, piece by piece: wait(slot) until the slot's last transfer is over,
// the piece is copied into it by all threads, a stripe each, then send(offset, slot, length) on its way,
// offset counted over the three arrays one after another. Returns when all has been read, or at the
// first wait or send that returns false, with that.
template <class Wait, class Send>
bool stage_pieces(const double* const src[3], const size_t n, double* const pin, const Wait& wait, const Send& send) {
    const size_t per = (n + HF_SLOT - 1) / HF_SLOT;  // pieces of an array
    const int pieces = (int)(3 * per);
    // A piece is published by its number and copied by all threads, a stripe each.
    std::atomic<int> go{-1}, done{0};
    const auto copy = [&](const int i, const int t, const int threads) {
        const size_t off = (size_t)i % per * HF_SLOT, len = std::min(HF_SLOT, n - off);
        const size_t a = len * t / threads, b = len * (t + 1) / threads;
        std::memcpy(pin + (size_t)(i % HF_SLOTS) * HF_SLOT + a, src[(size_t)i / per] + off + a, (b - a) * sizeof(double));
    };
    std::thread helpers[HF_THREADS - 1];
    std::atomic<int> threads{0};  // set once the number of helpers is known
    int started = 0;
    const auto work = [&](const int t) {
        int nt;
        while ((nt = threads.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
        for (int i = 0; i < pieces; ++i) {
            int g;
            while ((g = go.load(std::memory_order_acquire)) < i) std::this_thread::yield();
            if (g >= pieces) return;  // given up
            copy(i, t, nt);
            done.fetch_add(1, std::memory_order_release);
        }
    };
    try {
        for (; started < HF_THREADS - 1; ++started) helpers[started] = std::thread(work, started + 1);
    } catch (const std::exception&) {  // fewer threads than wanted
    }
    const int nt = started + 1;
    threads.store(nt, std::memory_order_release);
    bool ok = true;
    for (int i = 0; i < pieces; ++i) {
        const int slot = i % HF_SLOTS;
        if (!(ok = wait(slot))) break;
        go.store(i, std::memory_order_release);
        copy(i, 0, nt);
        while (done.load(std::memory_order_acquire) < (i + 1) * started) std::this_thread::yield();
        const size_t off = (size_t)i % per * HF_SLOT, len = std::min(HF_SLOT, n - off);
        if (!(ok = send((size_t)i / per * n + off, slot, len))) break;
    }
    if (!ok) go.store(pieces, std::memory_order_release);
    for (int t = 0; t < started; ++t) helpers[t].join();
    return ok;
}

}  // namespace wfh
