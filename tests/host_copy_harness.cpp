// Drives the library's host transfers (host_copy in mpcf_capi.cpp) on the CPU:
// linked with that file and the few HIP runtime calls it makes, played here by
// host memory, with two devices, streams that can be held busy, and refusals.
//   host_copy_harness MODE   -> exit code 0 if the transfers do what they should
#include <hip/hip_runtime.h>
#include <cerrno>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <string>
#include <thread>
#include <vector>
#include "mpcf_internal.h"

namespace {

struct Stream
{
    int device = 0;
    bool held = false;                        // work queued on it waits
    std::deque<std::function<void()>> work;
};
struct Event { int device; Stream* s = nullptr; };

std::mutex mu;
std::condition_variable cv;
int waiting = 0;                              // callers inside a wait for a held stream
thread_local int device = 0;
bool refuse_pinned = false;
int pinned = 0;
int threads_left = 1 << 20;                   // threads that the host still gives
Stream null_stream;

Stream* stream(hipStream_t s) { return s ? (Stream*)s : &null_stream; }

void wait(Stream* s)
{
    std::unique_lock<std::mutex> lk(mu);
    ++waiting;
    cv.notify_all();
    cv.wait(lk, [&] { return !s->held; });
    --waiting;
}

void release(Stream& s)
{
    std::lock_guard<std::mutex> lk(mu);
    for (auto& w : s.work) w();
    s.work.clear();
    s.held = false;
    cv.notify_all();
}

}  // namespace

extern "C" {
// every thread of the program starts here (the linker wraps the calls)
int __real_pthread_create(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
int __wrap_pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x)
{
    return threads_left-- > 0 ? __real_pthread_create(t, a, f, x) : EAGAIN;
}
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s ? stream(s)->device : device; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (refuse_pinned) return hipErrorOutOfMemory;
    ++pinned;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Event{device}; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (((Event*)e)->device != stream(s)->device) return hipErrorInvalidHandle;
    ((Event*)e)->s = stream(s);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (((Event*)e)->s) wait(((Event*)e)->s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { wait(stream(s)); return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s)
{
    std::lock_guard<std::mutex> lk(mu);
    if (stream(s)->held) stream(s)->work.push_back([=] { std::memcpy(dst, src, n); });
    else std::memcpy(dst, src, n);
    return hipSuccess;
}
}

namespace {

// nh arrays of `per` bytes to a "device" buffer and back, on s
bool round_trip(Stream& s, const int nh, const size_t per, const unsigned seed)
{
    std::vector<std::vector<unsigned char>> a(nh), b(nh);
    std::vector<void*> pa(nh), pb(nh);
    for (int q = 0; q < nh; ++q) {
        a[q].resize(per); b[q].resize(per);
        for (size_t i = 0; i < per; ++i) a[q][i] = (unsigned char)((i * 2654435761u + q * 40503u + seed) >> 11);
        pa[q] = a[q].data(); pb[q] = b[q].data();
    }
    std::vector<unsigned char> dev(nh * per);
    if (mpcf::detail::host_copy((hipStream_t)&s, dev.data(), pa.data(), nh, per, true) != MPCF_OK) return false;
    if (mpcf::detail::host_copy((hipStream_t)&s, dev.data(), pb.data(), nh, per, false) != MPCF_OK) return false;
    for (int q = 0; q < nh; ++q)
        if (a[q] != b[q] || std::memcmp(dev.data() + q * per, a[q].data(), per)) return false;
    return true;
}

// a transfer behind a busy stream does not keep another stream's waiting
bool busy()
{
    Stream s0, s1;
    if (!round_trip(s1, 7, 200000, 1)) return false;
    s0.held = true;
    std::vector<char> dev(3 << 20, 'd'), host(3 << 20);
    void* h = host.data();
    int rc0 = -1;
    std::thread A([&] { rc0 = mpcf::detail::host_copy((hipStream_t)&s0, dev.data(), &h, 1, dev.size(), false); });
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [] { return waiting > 0; });
    }
    bool done = false, same = false;
    std::thread B([&] {
        const bool r = round_trip(s1, 7, 200000, 2);
        std::lock_guard<std::mutex> lk(mu);
        done = true; same = r;
        cv.notify_all();
    });
    bool first;
    {
        std::unique_lock<std::mutex> lk(mu);
        first = cv.wait_for(lk, std::chrono::seconds(3), [&] { return done; });
    }
    release(s0);
    A.join();
    B.join();
    return first && same && rc0 == MPCF_OK && host == dev;
}

// contexts on two devices, the current device not always the stream's
bool devices()
{
    Stream s[2];
    s[1].device = 1;
    for (int k = 0; k < 6; ++k) {
        device = k & 1;
        if (!round_trip(s[(k >> 1) & 1], 7, 100000 + 900000 * k, k) || device != (k & 1)) return false;
    }
    return pinned > 0;
}

// sizes on both sides of the line to plain copies, chunk edges inside arrays,
// the small chunks growing into the large ones, more than two full chunks
bool sizes()
{
    Stream s;
    bool ok = true;
    for (const size_t per : {size_t(37449), size_t(37450), size_t(600001), size_t(3000017), size_t(24000031)})
        ok = ok && round_trip(s, 7, per, 7);
    for (const size_t n : {(size_t(1) << 20), (size_t(1) << 20) + 1, (size_t(4) << 20), (size_t(4) << 20) + 5})
        ok = ok && round_trip(s, 1, n, 8);
    return ok;
}

// one array of up to 4 MB, or 1 MB downloaded, goes to the runtime as it is
bool single()
{
    Stream s;
    std::vector<char> host(4 << 20, 'h'), dev(4 << 20, 'd');
    void* h = host.data();
    bool ok = mpcf::detail::host_copy((hipStream_t)&s, dev.data(), &h, 1, dev.size(), true) == MPCF_OK && host == dev;
    host.assign(1 << 20, 'x');
    h = host.data();
    ok = ok && mpcf::detail::host_copy((hipStream_t)&s, dev.data(), &h, 1, host.size(), false) == MPCF_OK &&
         std::memcmp(host.data(), dev.data(), host.size()) == 0;
    return ok && pinned == 0;
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string mode = argc > 1 ? argv[1] : "";
    bool ok = false;
    if (mode == "busy") ok = busy();
    if (mode == "devices") ok = devices();
    if (mode == "sizes") ok = sizes();
    if (mode == "single") ok = single();
    if (mode == "refused") { refuse_pinned = true; ok = sizes() && pinned == 0; }
    if (mode == "threads") { threads_left = std::atoi(argv[2]); ok = sizes(); }
    std::printf("%s %s\n", mode.c_str(), ok ? "ok" : "failed");
    std::fflush(stdout);
    std::_Exit(ok ? 0 : 1);   // the library's copy threads live as long as the process
}
