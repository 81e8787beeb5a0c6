// Host side of the per-iteration entry points' transfers.
//
// Inputs are packed into a pinned buffer and outputs go through a ring of pinned chunks, pieces
// that are neighbours in device memory as one copy.  The runtime's own path for pageable memory
// takes 10-20 us a call and 10 GB/s into pages not touched before; a pinned copy takes 5 us to issue
// and 56 GB/s, and several threads fill the caller's arrays from the ring as its chunks arrive.
// They are started once the call's kernels are queued and first have the kernel map the arrays'
// pages, so that both hide behind the kernels.  They end with the call.
// Measured, before (pageable copies, workspaces allocated per call) and so: the c2 build with gas_cap
// (16 MB) on the host 1.94 -> 1.05 ms, its precision form 1.66 -> 0.84 ms, the NLTE build (80 MB)
// 8.6 -> 3.3 ms, a build of 64 x 250 with every output 243 -> 151 us.
#pragma once

#include <hip/hip_runtime.h>
#include <sched.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>

namespace slgpu {

// The pinned memory of one context, 16 MiB at most: a ring of 12 MiB for outputs, less where its largest
// output is smaller, and up to 4 MiB of inputs.
struct HostIO {
    static constexpr int SLOTS = 6;
    static constexpr size_t CHUNK = (size_t)2 << 20;
    char *in = nullptr, *ring = nullptr;
    size_t in_cap = 0, in_used = 0, chunk = 0;
    int slots = 0;
    hipEvent_t ev[SLOTS] = {};
    bool busy = false;          // a call that failed may have left copies from `in` under way

    // in_bytes: the largest call's inputs; out_bytes: its outputs
    hipError_t create(size_t in_bytes, size_t out_bytes)
    {
        in_cap = in_bytes;
        chunk = std::min(CHUNK, (out_bytes + 4095) / 4096 * 4096);
        slots = (int)std::min<size_t>(SLOTS, (out_bytes + chunk - 1) / chunk);
        hipError_t e = hipHostMalloc((void **)&in, in_cap, hipHostMallocDefault);
        if (e == hipSuccess) e = hipHostMalloc((void **)&ring, chunk * slots, hipHostMallocDefault);
        for (int k = 0; k < slots && e == hipSuccess; ++k)
            e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        return e;
    }
    void destroy()
    {
        if (in) (void)hipHostFree(in);
        if (ring) (void)hipHostFree(ring);
        for (hipEvent_t &x : ev)
            if (x) (void)hipEventDestroy(x);
    }
};

// Ordinary host memory, which the CPU may copy; anything HIP knows (pinned, managed, device) keeps
// its own copy.
inline bool plain_host(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// The inputs of one call, which ends with the stream drained: construct, add in the order of the
// device memory, send before the first kernel.
class Inputs {
public:
    Inputs(HostIO &io, hipStream_t stream) : io_(io), s_(stream)
    {
        if (io_.busy) (void)hipStreamSynchronize(s_);
        io_.busy = true;
        io_.in_used = 0;
    }
    // joins: dst is in the allocation of the piece added before it (only such pieces share a copy:
    // separate allocations can lie side by side too)
    void add(void *dst, const void *src, size_t n, bool joins = false)
    {
        if (e_ != hipSuccess || n == 0) return;
        if (io_.in_used + n > io_.in_cap || !plain_host(src)) {
            send();
            if (e_ == hipSuccess) e_ = hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s_);
            return;
        }
        if (n_ && !(joins && dst_ + n_ == (char *)dst)) send();
        if (!n_) {
            io_.in_used = std::min(io_.in_cap, (io_.in_used + 15) / 16 * 16);
            if (io_.in_used + n > io_.in_cap) {
                if (e_ == hipSuccess) e_ = hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s_);
                return;
            }
            dst_ = (char *)dst;
            off_ = io_.in_used;
        }
        std::memcpy(io_.in + io_.in_used, src, n);
        io_.in_used += n;
        n_ += n;
    }
    hipError_t send()
    {
        if (n_ && e_ == hipSuccess)
            e_ = hipMemcpyAsync(dst_, io_.in + off_, n_, hipMemcpyHostToDevice, s_);
        n_ = 0;
        return e_;
    }

private:
    HostIO &io_;
    hipStream_t s_;
    char *dst_ = nullptr;
    size_t off_ = 0, n_ = 0;
    hipError_t e_ = hipSuccess;
};

// The outputs of one call: add them, start() once the kernels are queued, finish() to have them.
class Outputs {
public:
    Outputs(HostIO &io, hipStream_t stream) : io_(io), s_(stream) {}
    ~Outputs() { end(); }
    // joins: as for Inputs, of src
    void add(void *dst, const void *src, size_t n, bool joins = false)
    {
        if (dst && n) items_.push_back({(char *)dst, (const char *)src, n, joins});
    }

    void start()
    {
        size_t total = 0;
        for (Item &t : items_) {
            t.direct = !plain_host(t.dst);
            if (t.direct) continue;
            for (size_t o = 0; o < t.n;) {
                const bool next = t.joins && o == 0 && !segs_.empty() && segs_.back().src + segs_.back().n == t.src;
                size_t at = chunks_.empty() ? io_.chunk : chunks_.back().n;
                if (!next) at = (at + 63) / 64 * 64;
                if (at >= io_.chunk) {
                    chunks_.push_back({(int)segs_.size(), 0, 0});
                    at = 0;
                }
                const size_t n = std::min(t.n - o, io_.chunk - at);
                segs_.push_back({t.dst + o, t.src + o, at, n, next && at > 0});
                chunks_.back().nseg++;
                chunks_.back().n = at + n;
                o += n;
            }
            total += t.n;
        }
        // a thread per MiB, up to 8 (one copies 8-10 GB/s), on cores beside the caller's: a rank bound to
        // one core copies by itself
        workers_ = (int)std::min<size_t>(std::min(8, spare_cores()), total >> 20);
        if (!workers_) return;
        done_.reset(new std::atomic<int>[chunks_.size()]);
        for (size_t k = 0; k < chunks_.size(); ++k) done_[k].store(0, std::memory_order_relaxed);
        int made = 0;
        try {
            threads_.reserve(workers_);
            gate_.store(0, std::memory_order_relaxed);
            for (; made < workers_; ++made) threads_.emplace_back([this, made] { work(made); });
        } catch (...) {                                    // fewer threads than asked for, or none
        }
        workers_ = made;
        gate_.store(made ? made : -1, std::memory_order_release);
    }

    // `last` follows the last copy on the stream, which is drained on return
    hipError_t finish(hipEvent_t last)
    {
        hipError_t e = hipSuccess;
        for (const Item &t : items_)
            if (t.direct && e == hipSuccess) e = hipMemcpyAsync(t.dst, t.src, t.n, hipMemcpyDeviceToHost, s_);
        const int n = (int)chunks_.size();
        if (n == 0) {
            if (e == hipSuccess) e = hipEventRecord(last, s_);
            if (e == hipSuccess) e = hipEventSynchronize(last);
            if (e == hipSuccess) io_.busy = false;
            return e;
        }
        int issued = 0;
        auto t_last = std::chrono::steady_clock::now();
        for (int k = 0; k < n && e == hipSuccess; ++k) {
            while (issued < n && issued < k + io_.slots && e == hipSuccess) {
                if (issued >= io_.slots && workers_ > 0) {
                    std::atomic<int> &d = done_[issued - io_.slots];
                    if (d.load(std::memory_order_acquire) < workers_) {
                        if (issued > k) break;             // chunk k can be waited for meanwhile
                        while (d.load(std::memory_order_acquire) < workers_) std::this_thread::yield();
                    }
                }
                e = issue(issued, issued == n - 1 ? last : io_.ev[issued % io_.slots]);
                ++issued;
            }
            if (e == hipSuccess) e = hipEventSynchronize(k == n - 1 ? last : io_.ev[k % io_.slots]);
            if (e != hipSuccess) break;
            t_last = std::chrono::steady_clock::now();
            if (workers_ > 0) ready_.store(k + 1, std::memory_order_release);
            else copy(k, 0, chunks_[k].n);
        }
        if (e != hipSuccess) stop_.store(true, std::memory_order_release);
        else io_.busy = false;
        end();
        tail_ms_ = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_last).count();
        return e;
    }

    // from `last` until the caller's arrays held everything, which the event does not cover
    double tail_ms() const { return tail_ms_; }

private:
    struct Item {
        char *dst;
        const char *src;
        size_t n;
        bool joins, direct = false;
    };
    struct Seg {
        char *dst;
        const char *src;
        size_t at, n;                  // place in the chunk
        bool joins;                    // one copy with the segment before it
    };
    struct Chunk {
        int seg, nseg;
        size_t n;
    };

    // cores that threads of the caller may run on, less its own
    static int spare_cores()
    {
        cpu_set_t s;
        return sched_getaffinity(0, sizeof(s), &s) == 0 ? CPU_COUNT(&s) - 1 : 8;
    }

    hipError_t issue(int k, hipEvent_t done)
    {
        char *slot = io_.ring + (size_t)(k % io_.slots) * io_.chunk;
        const Chunk &c = chunks_[k];
        hipError_t e = hipSuccess;
        for (int s = c.seg; s < c.seg + c.nseg && e == hipSuccess;) {
            const Seg &a = segs_[s];
            size_t n = a.n;
            int t = s + 1;
            while (t < c.seg + c.nseg && segs_[t].joins) n += segs_[t++].n;
            e = hipMemcpyAsync(slot + a.at, a.src, n, hipMemcpyDeviceToHost, s_);
            s = t;
        }
        return e == hipSuccess ? hipEventRecord(done, s_) : e;
    }

    // bytes [lo, hi) of chunk k to their places
    void copy(int k, size_t lo, size_t hi) const
    {
        const char *slot = io_.ring + (size_t)(k % io_.slots) * io_.chunk;
        const Chunk &c = chunks_[k];
        for (int s = c.seg; s < c.seg + c.nseg; ++s) {
            const Seg &a = segs_[s];
            const size_t x = std::max(lo, a.at), y = std::min(hi, a.at + a.n);
            if (x < y) std::memcpy(a.dst + (x - a.at), slot + x, y - x);
        }
    }

    void work(int w)
    {
        int nw;
        while ((nw = gate_.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
        // the pages of the w-th part of every large array, without changing what they hold
        const size_t page = (size_t)sysconf(_SC_PAGESIZE);
#ifdef MADV_POPULATE_WRITE
        for (const Item &t : items_) {
            if (t.direct || t.n < ((size_t)1 << 20)) continue;
            const uintptr_t b = (uintptr_t)t.dst, lo = (b + t.n * w / nw) / page * page;
            const uintptr_t hi = (b + t.n * (w + 1) / nw + page - 1) / page * page;
            (void)madvise((void *)lo, hi - lo, MADV_POPULATE_WRITE);
        }
#endif
        const auto t0 = std::chrono::steady_clock::now();
        for (int k = 0; k < (int)chunks_.size(); ++k) {
            while (ready_.load(std::memory_order_acquire) <= k) {
                if (stop_.load(std::memory_order_acquire)) return;
                // long kernels: off the core after the first millisecond
                if (std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(1)) std::this_thread::yield();
                else std::this_thread::sleep_for(std::chrono::microseconds(20));
            }
            const size_t n = chunks_[k].n;
            copy(k, n * w / nw, n * (w + 1) / nw);
            done_[k].fetch_add(1, std::memory_order_acq_rel);
        }
    }

    void end()
    {
        if (threads_.empty()) return;
        if (ready_.load() < (int)chunks_.size()) stop_.store(true, std::memory_order_release);
        for (std::thread &t : threads_) t.join();
        threads_.clear();
    }

    HostIO &io_;
    hipStream_t s_;
    std::vector<Item> items_;
    std::vector<Seg> segs_;
    std::vector<Chunk> chunks_;
    std::vector<std::thread> threads_;
    std::unique_ptr<std::atomic<int>[]> done_;
    std::atomic<int> ready_{0}, gate_{0};
    std::atomic<bool> stop_{false};
    int workers_ = 0;
    double tail_ms_ = 0.0;
};

}  // namespace slgpu
