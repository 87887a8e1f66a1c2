// Records from the device into the caller's memory (host side).
//
// A batch's records are its largest result (168 MB for 128 windows of 820
// receivers x 200 samples), and the caller's buffer is usually fresh: its
// pages do not exist yet and it is not pinned.  A plain copy of those 168 MB
// took 16-18 ms, 6 of them page faults; from pinned memory it takes 3.  So the
// pages are made while the device still computes (prepare), and the copy goes
// through two pinned pieces, each emptied by several threads while the next
// one arrives: 3.8 ms.  Below 8 MB the plain copy (17 GB/s, 0.5 ms) is kept: the
// threads' start would cost as much, and for destinations that HIP knows.
#pragma once
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace ds2d {

class RecordCopy {
  public:
    static constexpr size_t kStaged = 8u << 20;

    RecordCopy() = default;
    RecordCopy(const RecordCopy&) = delete;
    RecordCopy& operator=(const RecordCopy&) = delete;
    ~RecordCopy() {
        if (pin_) (void)hipHostFree(pin_);
        for (hipEvent_t e : ev_)
            if (e) (void)hipEventDestroy(e);
    }

    // Makes the whole pages of [p, p + bytes) without touching what they hold
    // (a hint: kernels that do not know it leave the copy to do it).
    static void prepare(void* p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
        const int how = MADV_POPULATE_WRITE;
#else
        const int how = 23;
#endif
        const uintptr_t page = 4096, a = ((uintptr_t)p + page - 1) / page * page, b = ((uintptr_t)p + bytes) / page * page;
        if (p && b > a) (void)madvise((void*)a, b - a, how);
    }

    // n floats to each destination that is not null, complete on return.
    hipError_t fetch(hipStream_t st, size_t n, float* z, const float* dz, float* x, const float* dx) {
        const Piece whole[2] = {{(char*)z, (const char*)dz, z ? n * 4 : 0}, {(char*)x, (const char*)dx, x ? n * 4 : 0}};
        if (whole[0].bytes + whole[1].bytes < kStaged || known(z) || known(x) || !staging()) {
            for (const Piece& q : whole) {
                const hipError_t e = q.bytes ? hipMemcpyAsync(q.dst, q.src, q.bytes, hipMemcpyDeviceToHost, st) : hipSuccess;
                if (e != hipSuccess) return e;
            }
            return hipStreamSynchronize(st);
        }
        std::vector<Piece> todo;
        for (const Piece& q : whole)
            for (size_t o = 0; o < q.bytes; o += kPiece)
                todo.push_back({q.dst + o, q.src + o, std::min(kPiece, q.bytes - o)});
        return staged(st, todo);
    }

  private:
    struct Piece {
        char* dst;
        const char* src;
        size_t bytes;
    };
    static constexpr size_t kPiece = 4u << 20;
    char* pin_ = nullptr;
    hipEvent_t ev_[2] = {nullptr, nullptr};

    // Memory that HIP knows, which the runtime copies to at full rate by itself
    // (pinned) and a host thread may not be able to write (device).
    static bool known(const void* p) {
        hipPointerAttribute_t a;
        if (p && hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return false;
    }

    bool staging() {
        for (hipEvent_t& e : ev_)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                (void)hipGetLastError();
                return false;
            }
        if (!pin_ && hipHostMalloc((void**)&pin_, 2 * kPiece, hipHostMallocDefault) != hipSuccess) {
            pin_ = nullptr;
            (void)hipGetLastError();
        }
        return pin_ != nullptr;
    }

    // Piece i passes through half i % 2.  Thread t copies the t-th share of
    // every piece as it arrives; a half is filled again once all have left it.
    hipError_t staged(hipStream_t st, const std::vector<Piece>& todo) {
        const int n = (int)todo.size();
        std::atomic<int> arrived{0};
        std::atomic<bool> stop{false};
        std::vector<std::atomic<int>> left(n);
        for (auto& l : left) l.store(0);
        int helpers = (int)std::min(3u, std::max(1u, std::thread::hardware_concurrency()) - 1), started = 0;
        const auto share = [&](int i, int t, int of) {
            const Piece& q = todo[i];
            const size_t a = q.bytes * t / of, b = q.bytes * (t + 1) / of;
            memcpy(q.dst + a, pin_ + (i & 1) * kPiece + a, b - a);
            left[i].fetch_add(1, std::memory_order_release);
        };
        std::atomic<int> of{0};  // threads that share a piece, known once all have started
        const auto help = [&](int t) {
            while (!of.load(std::memory_order_acquire)) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            for (int i = 0; i < n; ++i) {
                while (arrived.load(std::memory_order_acquire) <= i) {
                    if (stop.load(std::memory_order_relaxed)) return;
                    std::this_thread::yield();
                }
                share(i, t, of.load(std::memory_order_relaxed));
            }
        };
        const auto start = [&](int i) {
            const hipError_t e = hipMemcpyAsync(pin_ + (i & 1) * kPiece, todo[i].src, todo[i].bytes, hipMemcpyDeviceToHost, st);
            return e != hipSuccess ? e : hipEventRecord(ev_[i & 1], st);
        };
        hipError_t e = start(0);
        if (e == hipSuccess && n > 1) e = start(1);
        // threads start once the first piece is there: until then the stream may have seconds of work before it
        if (e == hipSuccess) e = hipEventSynchronize(ev_[0]);
        std::vector<std::thread> pool;
        if (e != hipSuccess) helpers = 0;
        try {
            pool.reserve(helpers);
            for (; started < helpers; ++started) pool.emplace_back(help, started + 1);
        } catch (const std::exception&) {  // fewer threads, then
        }
        const int all = started + 1;
        of.store(all, std::memory_order_release);
        for (int i = 0; i < n && e == hipSuccess; ++i) {
            if (i > 0 && i + 1 < n) {  // the other half still holds piece i - 1
                while (left[i - 1].load(std::memory_order_acquire) < all) std::this_thread::yield();
                e = start(i + 1);
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev_[i & 1]);
            if (e != hipSuccess) break;
            arrived.store(i + 1, std::memory_order_release);
            share(i, 0, all);
        }
        if (e != hipSuccess) {
            stop.store(true);
            (void)hipStreamSynchronize(st);
        }
        for (std::thread& t : pool) t.join();
        return e;
    }
};

}  // namespace ds2d
