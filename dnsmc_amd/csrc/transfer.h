// Copies between device buffers and the caller's pageable arrays.
//
// A plain hipMemcpy of pageable memory stages through the runtime's buffers on
// one thread, and a fresh array's page faults are taken there too: 7 to 15 GB/s.
// Here chunks of 1 MiB go through pinned buffers of the solver, and from
// kParallel bytes on several threads move them (two chunks in flight each).
// Results of 384x256x256 cells (2 x 101 MB): 26 -> 8 ms, a field of them in 3 ms;
// four FP64 results of 256x128x128 cells (134 MB): 20 -> 6 ms.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <system_error>
#include <thread>
#include <vector>

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
    static constexpr size_t kChunk = 1u << 20, kParallel = 2u << 20;
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
    hipError_t run(int device, hipStream_t st, bool up, const HostRows* jobs, int njobs)
    {
        std::vector<Chunk> ch;
        size_t total = 0;
        for (int j = 0; j < njobs; ++j) {
            total += jobs[j].bytes;
            for (size_t o = 0; o < jobs[j].bytes; o += kChunk) ch.push_back(Chunk{jobs + j, o, std::min(kChunk, jobs[j].bytes - o)});
        }
        if (ch.empty()) return hipSuccess;
        const int T = total < kParallel ? 1 : kWorkers;
        hipError_t e = ensure(T == 1 && ch.size() == 1 ? 1 : 2 * T);
        if (e != hipSuccess) return e;
        hipError_t err[kWorkers] = {hipSuccess, hipSuccess, hipSuccess, hipSuccess};
        std::thread th[kWorkers];
        int made = 1;
        try {
            for (; made < T; ++made)
                th[made] = std::thread([&, made] {
                    err[made] = hipSetDevice(device);
                    if (err[made] == hipSuccess) err[made] = work(st, up, ch, made, T);
                });
        } catch (const std::system_error&) {   // no thread to be had: this one does the rest
        }
        err[0] = work(st, up, ch, 0, T);
        for (int t = made; t < T; ++t) err[t] = work(st, up, ch, t, T);
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
    static void rows(const Chunk& c, char* pin, bool up)
    {
        const HostRows& j = *c.j;
        for (size_t o = c.off; o < c.off + c.len;) {
            const long long r = (long long)(o / j.row);
            const size_t in = o - (size_t)r * j.row, n = std::min(j.row - in, c.off + c.len - o);
            char* h = j.host + (r % j.n1) * j.p1 + (r / j.n1 % j.n2) * j.p2 + (r / (j.n1 * j.n2)) * j.p3 + in;
            if (up) memcpy(pin + (o - c.off), h, n);
            else memcpy(h, pin + (o - c.off), n);
            o += n;
        }
    }
    // worker t of T: chunks t, t + T, ..., alternating between its two slots
    hipError_t work(hipStream_t st, bool up, const std::vector<Chunk>& ch, int t, int T)
    {
        hipError_t e = hipSuccess;
        const size_t n = ch.size();
        auto slot = [&](size_t c) { return 2 * t + (int)((c / T) & 1); };
        auto pin = [&](size_t c) { return pin_ + (size_t)slot(c) * kChunk; };
        auto issue = [&](size_t c) -> hipError_t {
            char* d = ch[c].j->dev + ch[c].off;
            hipError_t r = up ? hipMemcpyAsync(d, pin(c), ch[c].len, hipMemcpyHostToDevice, st)
                              : hipMemcpyAsync(pin(c), d, ch[c].len, hipMemcpyDeviceToHost, st);
            return r != hipSuccess ? r : hipEventRecord(ev_[slot(c)], st);
        };
        if (!up && (size_t)t < n) e = issue(t);
        size_t c = t;
        for (; c < n && e == hipSuccess; c += T) {
            if (up) {
                if (c >= 2 * (size_t)T && (e = hipEventSynchronize(ev_[slot(c)])) != hipSuccess) break;
                rows(ch[c], pin(c), true);
                e = issue(c);
            } else {
                if (c + T < n && (e = issue(c + T)) != hipSuccess) break;
                if ((e = hipEventSynchronize(ev_[slot(c)])) != hipSuccess) break;
                rows(ch[c], pin(c), false);
            }
        }
        // the slots are free again when the call returns (an event never recorded
        // counts as complete)
        if (up || e != hipSuccess)
            for (int i = 2 * t; i < std::min(2 * t + 2, slots_); ++i) {
                const hipError_t r = hipEventSynchronize(ev_[i]);
                if (e == hipSuccess) e = r;
            }
        return e;
    }
};

}  // namespace dn
