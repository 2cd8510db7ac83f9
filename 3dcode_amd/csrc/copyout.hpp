// Device results to the caller's memory (copy_out).  A names the few runtime
// calls it makes: HIP's in cav3d.hip, and ones that fail on demand in the
// host tests.
//
// The copy of pageable memory inside the runtime is a serial chain of a
// transfer to its staging buffer and one thread's memcpy from it (20 and 70 us
// per chunk), the memcpy paying the page faults of a fresh array as well.
// Here THREADS threads each own BUFS / THREADS pinned chunks of the context: a
// thread copies one out while its next is being filled.  128x64x64: the state
// (47 MB) 2.75 -> 1.59 ms, the residual and its Jacobians (75 MB into fresh
// arrays, with the 0.9 ms of the kernels) 8.6 -> 4.3 ms.
// Below MIN the plain copy is the faster one (the threads cost some 50 us), and
// so it is into memory the runtime knows: a transfer into pinned memory goes
// straight there (the same state 0.92 ms, 1.59 through the chunks), and device
// memory is not a thread's to write.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>

namespace cav {

template <class A> struct CopyRing {
    using Error = typename A::Error;
    static constexpr int BUFS = 8, THREADS = 4;
    static constexpr size_t CHUNK = 1u << 20, MIN = 4 * CHUNK;
    char *pin = nullptr;
    typename A::Event ev[BUFS] = {};

    // buffers and events on device dev (an event is recorded on its own
    // device's streams only); the caller's device stays
    bool open(int dev)
    {
        const int cur = A::device();
        if (cur != dev) A::set_device(dev);
        bool ok = A::alloc(&pin, BUFS * CHUNK) == A::OK;
        for (int q = 0; ok && q < BUFS; q++) ok = A::event_create(&ev[q]) == A::OK;
        if (!ok) {
            A::clear_error();
            close();
        }
        if (cur != dev) A::set_device(cur);
        return ok;
    }

    void close()
    {
        if (pin) A::release(pin);
        pin = nullptr;
        for (auto &e : ev) {
            if (e) A::event_destroy(e);
            e = {};
        }
    }

    // src (device dev, ordered behind what is on st) into dst, complete on
    // return unless wait is false: then a later copy's wait may be the one that completes it
    Error copy(typename A::Stream st, int dev, void *dst, const void *src, size_t bytes, bool wait = true)
    {
        if (bytes < MIN || !A::pageable(dst) || (!pin && !open(dev))) {
            const Error e = A::to_host(dst, src, bytes, st);
            return e == A::OK && wait ? A::stream_wait(st) : e;
        }
        const long n = (long)((bytes + CHUNK - 1) / CHUNK);
        std::atomic<Error> err{A::OK};
        auto size = [&](long q) { return std::min(CHUNK, bytes - (size_t)q * CHUNK); };
        auto fill = [&](long q) {        // chunk q into its buffer
            const int b = (int)(q % BUFS);
            Error e = A::to_host(pin + b * CHUNK, (const char *)src + q * CHUNK, size(q), st);
            if (e == A::OK) e = A::event_record(ev[b], st);
            if (e != A::OK) err = e;
        };
        for (long q = 0; q < std::min<long>(n, BUFS); q++) fill(q);
        auto work = [&](int t) {         // chunks t, t + THREADS, ...
            for (long q = t; q < n && err == A::OK; q += THREADS) {
                const int b = (int)(q % BUFS);
                const Error e = A::event_wait(ev[b]);
                if (e != A::OK) { err = e; break; }
                memcpy((char *)dst + q * CHUNK, pin + b * CHUNK, size(q));
                if (q + BUFS < n) fill(q + BUFS);
            }
        };
        auto other = [&](int t) {        // (the caller's own thread keeps its device)
            A::set_device(dev);
            work(t);
        };
        typename A::Thread th[THREADS - 1];
        int started = 0;
        try {
            for (; started < THREADS - 1; started++) th[started] = typename A::Thread(other, started + 1);
        } catch (...) {                  // (no thread: std::system_error; no memory for its state: std::bad_alloc)
        }
        work(0);
        for (int t = started + 1; t < THREADS; t++) work(t);      // the threads that could not be started
        for (int t = 0; t < started; t++) th[t].join();
        if (err != A::OK) (void)A::stream_wait(st);
        return err;
    }
};

}  // namespace cav
