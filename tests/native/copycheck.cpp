// CopyRing of 3dcode_amd/csrc/copyout.hpp over runtime calls that live on the
// host and fail on demand.  Test infrastructure only.
#include "../../3dcode_amd/csrc/copyout.hpp"
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace {

std::mutex lock;
thread_local int current = 0;                 // the thread's device
int events, pinned, waits, copies, fail_event, fail_thread, thread_error;
const char *known = nullptr;                  // memory the runtime knows

struct Host {
    using Error = int;
    struct Ev { int dev; };
    using Event = Ev *;
    using Stream = int;                       // the device it is on
    static constexpr Error OK = 0;
    struct Thread : std::thread {
        Thread() {}
        template <class F> Thread(F f, int t) : std::thread((check(), f), t) {}
        static void check()
        {
            if (fail_thread-- != 0) return;
            if (thread_error == 1) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
            throw std::bad_alloc();
        }
    };
    static Error alloc(char **p, size_t n) { pinned++; *p = new char[n]; return OK; }
    static void release(char *p) { pinned--; delete[] p; }
    static Error event_create(Event *e)
    {
        if (fail_event-- == 0) return 2;
        std::lock_guard<std::mutex> g(lock);
        events++;
        *e = new Ev{current};
        return OK;
    }
    static void event_destroy(Event e) { events--; delete e; }
    static Error event_record(Event e, Stream st) { return e->dev == st ? OK : 400; }
    static Error event_wait(Event) { return OK; }
    static bool pageable(const void *p) { return p != known; }
    static Error to_host(void *d, const void *s, size_t n, Stream) { copies++; memcpy(d, s, n); return OK; }
    static Error stream_wait(Stream) { waits++; return OK; }
    static int device() { return current; }
    static void set_device(int d) { current = d; }
    static void clear_error() {}
};

}  // namespace

extern "C" {

// one copy of the given size; out = {error, copied, the caller's device afterwards,
// events and pinned buffers alive after close, stream waits, transfers}; registered:
// into memory the runtime knows; again: further copies, or -1 for one more in two parts
void cc_copy(long bytes, int dev, int caller, int bad_event, int bad_thread, int bad_kind, int again, int registered, int *out)
{
    events = pinned = waits = copies = 0;
    fail_event = bad_event;
    fail_thread = bad_thread;
    thread_error = bad_kind;
    std::vector<unsigned char> a(bytes), b(bytes, 0);
    for (long q = 0; q < bytes; q++) a[q] = (unsigned char)(q * 131 + (q >> 12));
    known = registered ? (const char *)b.data() : nullptr;
    const int before = current;
    current = caller;
    cav::CopyRing<Host> r;
    out[0] = r.copy(dev, dev, b.data(), a.data(), (size_t)bytes);
    out[1] = a == b;
    for (int q = 0; q < again && !out[0]; q++) {
        std::fill(b.begin(), b.end(), 0);
        out[0] = r.copy(dev, dev, b.data(), a.data(), (size_t)bytes);
        out[1] = out[1] && a == b;
    }
    out[2] = current;
    if (again < 0) {                          // two results of one call, the first not waited for by itself
        std::fill(b.begin(), b.end(), 0);
        waits = 0;
        const long n1 = bytes / 2;
        out[0] = r.copy(dev, dev, b.data(), a.data(), (size_t)n1, false) || r.copy(dev, dev, b.data() + n1, a.data() + n1, (size_t)(bytes - n1));
        out[1] = out[1] && a == b;
    }
    r.close();
    out[3] = events; out[4] = pinned; out[5] = waits; out[6] = copies;
    current = before;
}

}
