// Transfers between the caller's (pageable) arrays and the device.
//
// hipMemcpy on pageable memory runs on one host thread at 18 GB/s, 10 where the
// pages are new to the process, while the bus carries 56 GB/s; what a lane holds
// (pinned memory, a stream, the stack backing store of ray queries) takes tens of
// microseconds and more to allocate. So lanes are made once per process and
// device, lent to a call, and several at a time work on the parts of a large
// transfer, each on a thread of its own. A call takes idle lanes or new ones, at
// most LANES_PER_CALL; at most POOL_LANES idle ones are kept, and the last
// renderer that is destroyed gives them all back. Every function here may be
// called from several threads.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace ptx {

constexpr size_t LANE_PINNED = size_t{4} << 20;  // pinned bytes of a lane,
constexpr size_t LANE_SMALL = size_t{64} << 10;  // or these (4 MB take 0.1 ms to pin, 0.1 to give back)
constexpr int LANES_PER_CALL = 8;
constexpr int POOL_LANES = 16;

struct Lane {
    int device = 0;
    hipStream_t stream = nullptr;
    char* pinned = nullptr;
    size_t pinned_n = 0;
    int* spill = nullptr;    // device: the query's traversal-stack backing store
    size_t spill_n = 0;

    Lane() = default;
    Lane(const Lane&) = delete;
    Lane& operator=(const Lane&) = delete;
    ~Lane() {
        if (stream) (void)hipStreamDestroy(stream);
        if (pinned) (void)hipHostFree(pinned);
        if (spill) (void)hipFree(spill);
    }
    hipError_t open(int dev) {
        device = dev;
        return hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
    }
    hipError_t ensure_pinned(size_t bytes) {  // bytes <= LANE_PINNED
        if (pinned_n >= bytes) return hipSuccess;
        if (pinned) (void)hipHostFree(pinned);
        pinned = nullptr;
        pinned_n = 0;
        const size_t n = bytes <= LANE_SMALL ? LANE_SMALL : LANE_PINNED;
        const hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&pinned), n, hipHostMallocDefault);
        if (e == hipSuccess) pinned_n = n;
        return e;
    }
    hipError_t ensure_spill(size_t ints) {
        if (spill_n >= ints) return hipSuccess;
        if (spill) (void)hipFree(spill);
        spill = nullptr;
        spill_n = 0;
        const hipError_t e = hipMalloc(reinterpret_cast<void**>(&spill), ints * sizeof(int));
        if (e == hipSuccess) spill_n = ints;
        return e;
    }
};

class Pool {
public:
    static Pool& get() {
        static Pool* p = new Pool;  // never destroyed: no device calls at process exit
        return *p;
    }
    void add_user() {
        std::lock_guard<std::mutex> g(m_);
        ++users_;
    }
    void drop_user() {
        Lane* gone[POOL_LANES];
        int n = 0;
        {
            std::lock_guard<std::mutex> g(m_);
            if (--users_ == 0)
                while (idle_n_ > 0) gone[n++] = idle_[--idle_n_];
        }
        for (int i = 0; i < n; ++i) discard(gone[i]);
    }
    // An idle lane of the device or a new one, with `bytes` of pinned memory; null
    // where that cannot be had.
    Lane* take(int device, size_t bytes) {
        Lane* l = nullptr;
        {
            std::lock_guard<std::mutex> g(m_);
            for (int i = idle_n_; i-- > 0 && !l;)
                if (idle_[i]->device == device) {
                    l = idle_[i];
                    std::copy(idle_ + i + 1, idle_ + idle_n_, idle_ + i);
                    --idle_n_;
                }
        }
        const bool made = !l;
        if (made) l = new (std::nothrow) Lane;
        if (l && ((made && l->open(device) != hipSuccess) || l->ensure_pinned(bytes) != hipSuccess)) {
            (void)hipGetLastError();
            delete l;
            l = nullptr;
        }
        return l;
    }
    void give(Lane* l) {
        {
            std::lock_guard<std::mutex> g(m_);
            if (users_ > 0 && idle_n_ < POOL_LANES) {
                idle_[idle_n_++] = l;
                return;
            }
        }
        discard(l);
    }

private:
    static void discard(Lane* l) {
        int current = l->device;
        (void)hipGetDevice(&current);
        (void)hipSetDevice(l->device);
        delete l;
        (void)hipSetDevice(current);
    }
    std::mutex m_;
    Lane* idle_[POOL_LANES];  // no container: a lane is given back where nothing may throw
    int idle_n_ = 0;
    int users_ = 0;
};

// Lanes lent to one call, each with `bytes` of pinned memory.
class Lanes {
public:
    Lanes(int device, int want, size_t bytes) {
        for (int i = 0; i < std::min(want, LANES_PER_CALL); ++i) {
            Lane* l = Pool::get().take(device, bytes);
            if (!l) break;
            l_[n_++] = l;
        }
    }
    Lanes(const Lanes&) = delete;
    Lanes& operator=(const Lanes&) = delete;
    ~Lanes() {
        for (int i = 0; i < n_; ++i) {
            (void)hipStreamSynchronize(l_[i]->stream);  // nothing in flight on a lane that is given back
            Pool::get().give(l_[i]);
        }
    }
    int size() const { return n_; }
    Lane& operator[](int i) { return *l_[i]; }

    // part(lane, k) for k = 0..n-1, the lanes on threads of their own taking
    // the next part each; the first error ends it and is thrown here.
    template <class F>
    void each(int n, F&& part) {
        std::atomic<int> next{0};
        std::exception_ptr err;
        std::mutex em;
        auto work = [&](Lane& lane) {
            try {
                for (int k = next.fetch_add(1); k < n; k = next.fetch_add(1)) part(lane, k);
            } catch (...) {
                std::lock_guard<std::mutex> g(em);
                if (!err) err = std::current_exception();
                next.store(n);
            }
        };
        std::vector<std::thread> threads;
        const int t = std::min(size(), n);
        try {
            for (int i = 1; i < t; ++i)
                threads.emplace_back([&, i] {
                    (void)hipSetDevice((*this)[i].device);
                    work((*this)[i]);
                });
        } catch (...) {  // no thread to be had: the others do its parts
        }
        work((*this)[0]);
        for (std::thread& th : threads) th.join();
        if (err) std::rethrow_exception(err);
    }

private:
    Lane* l_[LANES_PER_CALL];
    int n_ = 0;
};

// Touches the pages of [p, p + n) (values kept) while `busy` says the device is
// still at work, so that a later copy does not wait for the system to supply
// them: 10 -> 18 GB/s and more.
template <class Busy>
inline void supply_pages(void* p, size_t n, Busy&& busy) {
    constexpr size_t page = 4096, step = 256 * page;
    volatile char* c = static_cast<volatile char*>(p);
    for (size_t a = 0; a < n; a += step) {
        if (!busy()) return;
        for (size_t i = a; i < std::min(n, a + step); i += page) c[i] = c[i];
    }
    if (n > 0) c[n - 1] = c[n - 1];
}

}  // namespace ptx
