// Copies of device buffers into the caller's pageable arrays.
//
// A plain hipMemcpy to pageable memory stages through the runtime's buffers on
// one thread, and a fresh array's page faults are taken there too.  Here chunks
// of 1 MiB go through pinned buffers of the solver, and from kParallel bytes on
// several threads move them (two chunks in flight each).  Measured, plain -> four
// threads, into an array used before (a fresh one): 2.1 MB 118 -> 118 us, 3.2 MB
// 185 -> 193, 4.2 MB 237 -> 225, 6.3 MB 360 -> 290, 17 MB 0.97 -> 0.63 ms, 105 MB
// 5.9 (24) -> 3.4 (8.2) ms: below kParallel the plain copy is used unless rows
// have to be placed.  Results of 384x256x256 cells (2 x 101 MB): 26 -> 8 ms.
// Uploads are plain copies: 3.2 / 26 / 105 MB take 0.11 / 0.71 / 3.5 ms so, and
// took 0.19 / 0.92 / 3.45 through such buffers.  A solver's first copy pays for
// the buffers: 0.35 ms for 8 MiB.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <thread>

namespace dn {

// One device range [0, bytes) and where its rows of `row` bytes lie on the host:
// row r at host + (r % n1) p1 + (r / n1 % n2) p2 + (r / (n1 n2)) p3.
struct HostRows {
    char* dev;
    char* host;
    size_t bytes, row;
    long long n1, n2;
    ptrdiff_t p1, p2, p3;
};
inline HostRows host_block(const void* dev, const void* host, size_t bytes)
{
    return HostRows{(char*)dev, (char*)host, bytes, bytes, 1, 1, 0, 0, 0};
}

class HostPipe {
public:
    static constexpr size_t kChunk = 1u << 20, kParallel = 4u << 20;
    static constexpr int kWorkers = 4;

    ~HostPipe() { release(); }

    // Memory that HIP knows (device, managed, pinned) is left to hipMemcpy.
    static bool pageable(const void* p)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }

    // Moves the jobs' ranges in stream order; the host side is done on return.
    hipError_t run(int device, hipStream_t st, const HostRows* jobs, int njobs)
    {
        Chunks ch{jobs, njobs, 0};
        size_t total = 0;
        for (int j = 0; j < njobs; ++j) {
            total += jobs[j].bytes;
            ch.n += Chunks::of(jobs[j]);
        }
        if (ch.n == 0) return hipSuccess;
        const int T = total < kParallel ? 1 : kWorkers;
        hipError_t e = ensure(T == 1 && ch.n == 1 ? 1 : 2 * T);
        if (e != hipSuccess) return e;
        hipError_t err[kWorkers] = {hipSuccess, hipSuccess, hipSuccess, hipSuccess};
        std::thread th[kWorkers];
        int made = 1;
        try {
            for (; made < T; ++made)
                th[made] = std::thread([&, made] {
                    err[made] = hipSetDevice(device);
                    if (err[made] == hipSuccess) err[made] = work(st, ch, made, T);
                });
        } catch (...) {   // no thread to be had, or no memory for one: this one does the rest
        }
        err[0] = work(st, ch, 0, T);
        for (int t = made; t < T; ++t) err[t] = work(st, ch, t, T);
        for (int t = 1; t < made; ++t) th[t].join();
        for (int t = 0; t < T; ++t)
            if (err[t] != hipSuccess) return err[t];
        return hipSuccess;
    }

private:
    struct Chunk {
        const HostRows* j;
        size_t off, len;
    };
    struct Chunks {   // the jobs' ranges in pieces of kChunk (nothing allocated)
        const HostRows* jobs;
        int njobs;
        size_t n;
        static size_t of(const HostRows& j) { return (j.bytes + kChunk - 1) / kChunk; }
        Chunk operator[](size_t c) const
        {
            const HostRows* j = jobs;
            for (; c >= of(*j); ++j) c -= of(*j);
            return Chunk{j, c * kChunk, std::min(kChunk, j->bytes - c * kChunk)};
        }
    };
    char* pin_ = nullptr;
    int slots_ = 0;
    hipEvent_t ev_[2 * kWorkers] = {};

    void release()
    {
        for (int i = 0; i < slots_; ++i) (void)hipEventDestroy(ev_[i]);
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
        slots_ = 0;
    }
    hipError_t ensure(int slots)
    {
        if (slots <= slots_) return hipSuccess;
        release();
        hipError_t e = hipHostMalloc((void**)&pin_, (size_t)slots * kChunk, hipHostMallocDefault);
        if (e != hipSuccess) {
            pin_ = nullptr;
            return e;
        }
        for (; slots_ < slots; ++slots_)
            if ((e = hipEventCreateWithFlags(&ev_[slots_], hipEventDisableTiming)) != hipSuccess) {
                release();
                return e;
            }
        return hipSuccess;
    }
    static void rows(const Chunk& c, const char* pin)
    {
        const HostRows& j = *c.j;
        for (size_t o = c.off; o < c.off + c.len;) {
            const long long r = (long long)(o / j.row);
            const size_t in = o - (size_t)r * j.row, n = std::min(j.row - in, c.off + c.len - o);
            memcpy(j.host + (r % j.n1) * j.p1 + (r / j.n1 % j.n2) * j.p2 + (r / (j.n1 * j.n2)) * j.p3 + in, pin + (o - c.off), n);
            o += n;
        }
    }
    // worker t of T: chunks t, t + T, ..., alternating between its two slots
    hipError_t work(hipStream_t st, const Chunks& ch, int t, int T)
    {
        hipError_t e = hipSuccess;
        const size_t n = ch.n;
        auto slot = [&](size_t c) { return 2 * t + (int)((c / T) & 1); };
        auto pin = [&](size_t c) { return pin_ + (size_t)slot(c) * kChunk; };
        auto issue = [&](size_t c) -> hipError_t {
            const Chunk k = ch[c];
            const hipError_t r = hipMemcpyAsync(pin(c), k.j->dev + k.off, k.len, hipMemcpyDeviceToHost, st);
            return r != hipSuccess ? r : hipEventRecord(ev_[slot(c)], st);
        };
        if ((size_t)t < n) e = issue(t);
        for (size_t c = t; c < n && e == hipSuccess; c += T) {
            if (c + T < n && (e = issue(c + T)) != hipSuccess) break;
            if ((e = hipEventSynchronize(ev_[slot(c)])) != hipSuccess) break;
            rows(ch[c], pin(c));
        }
        // after an error the slots are free again when the call returns (an event
        // never recorded counts as complete)
        if (e != hipSuccess)
            for (int i = 2 * t; i < std::min(2 * t + 2, slots_); ++i) (void)hipEventSynchronize(ev_[i]);
        return e;
    }
};

}  // namespace dn
