// staging.h -- copies between device memory and the caller's (pageable) arrays
// through a ring of pinned chunks held by the handle.
//
// A hipMemcpy to or from pageable memory takes 35 us for 64 KiB, 0.45 ms for 1
// MiB and, into fresh memory, 15.6 ms for 64 MiB (most of it first-touch page
// faults); through pinned memory the bus takes 9 us, 27 us and 1.2 ms, and a
// host copy in several threads 2 us, 42 us and 2.9 ms.  So small transfers are
// one pinned copy and a memcpy, and large ones run chunk by chunk, the bus
// filling (or draining) one chunk while threads copy the others.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace nbh {

class Staging {
public:
    struct Part {
        void* host;   // caller's array
        size_t bytes;
    };

    ~Staging() { release(); }
    void release() {
        if (pin_) (void)hipHostFree(pin_);
        for (hipEvent_t& e : ev_)
            if (e) (void)hipEventDestroy(e), e = nullptr;
        pin_ = nullptr;
        cap_ = 0;
    }

    // the parts, which lie one after the other at dev, to the host; returns
    // when the caller's arrays are written
    hipError_t to_host(const Part* parts, int n, const void* dev, hipStream_t st) { return move(parts, n, (char*)dev, true, st); }
    // the caller's arrays to dev, one after the other, in stream order (the
    // caller's arrays are free on return, the stream may still be copying)
    hipError_t to_device(const Part* parts, int n, void* dev, hipStream_t st) { return move(parts, n, (char*)dev, false, st); }

private:
    static constexpr size_t CHUNK = 2u << 20;
    static constexpr int SLOTS = 8;          // at most 16 MiB pinned
    static constexpr int THREADS = 8;
    static constexpr size_t SMALL = 2 * CHUNK;  // one copy, on this thread
    struct Piece {
        char* host;
        char* dev;
        size_t bytes;
    };

    char* pin_ = nullptr;
    size_t cap_ = 0;
    hipEvent_t ev_[SLOTS] = {};

    hipError_t ensure(size_t bytes) {
        if (bytes <= cap_) return hipSuccess;
        // (the last upload may still be in flight; a device-wide wait would also
        // wait for other handles, and meet a stream that another thread captures)
        hipError_t e = drain();
        if (e != hipSuccess) return e;
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
        cap_ = 0;
        size_t want = 64u << 10;
        while (want < bytes) want *= 2;
        e = hipHostMalloc((void**)&pin_, want, hipHostMallocDefault);
        if (e != hipSuccess) { pin_ = nullptr; return e; }
        cap_ = want;
        return hipSuccess;
    }

    // the ring's last upload has left it
    hipError_t drain() {
        for (hipEvent_t ev : ev_) {
            const hipError_t e = hipEventSynchronize(ev);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

    hipError_t move(const Part* parts, int n, char* dev, bool down, hipStream_t st) {
        size_t total = 0;
        for (int k = 0; k < n; ++k) total += parts[k].bytes;
        if (!total) return hipSuccess;
        for (hipEvent_t& e : ev_)
            if (!e) {
                const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
                if (r != hipSuccess) { e = nullptr; return r; }
            }
        if (total <= SMALL) {
            hipError_t e = ensure(total);
            if (e != hipSuccess) return e;
            if (down) {
                e = hipMemcpyAsync(pin_, dev, total, hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipStreamSynchronize(st);
                if (e != hipSuccess) return e;
            } else if ((e = drain()) != hipSuccess) {
                return e;
            }
            size_t o = 0;
            for (int k = 0; k < n; ++k) {
                if (down) std::memcpy(parts[k].host, pin_ + o, parts[k].bytes);
                else std::memcpy(pin_ + o, parts[k].host, parts[k].bytes);
                o += parts[k].bytes;
            }
            if (!down) {
                e = hipMemcpyAsync(dev, pin_, total, hipMemcpyHostToDevice, st);
                if (e == hipSuccess) e = hipEventRecord(ev_[0], st);
            }
            return e;
        }
        hipError_t e = ensure(SLOTS * CHUNK);
        if (e != hipSuccess) return e;
        std::vector<Piece> pc;
        try {
            for (int k = 0; k < n; ++k)
                for (size_t o = 0; o < parts[k].bytes; o += CHUNK) {
                    const size_t b = std::min(CHUNK, parts[k].bytes - o);
                    pc.push_back({(char*)parts[k].host + o, dev, b});
                    dev += b;
                }
        } catch (...) {
            return hipErrorOutOfMemory;
        }
        return down ? large_down(pc, st) : large_up(pc, st);
    }

    // piece c goes through slot c % SLOTS.  This thread drives the bus; the
    // helpers (and this thread, where it would wait) copy pieces on the host.
    hipError_t large_down(const std::vector<Piece>& pc, hipStream_t st) {
        const int np = (int)pc.size();
        std::atomic<int> ready{0}, next{0}, failed{0};
        std::atomic<int> done[SLOTS];  // pieces of the slot copied out so far
        for (auto& d : done) d.store(0);
        auto work = [&](bool wait) {  // true: a piece was copied
            int c = next.load();
            do {
                if (c >= np || (!wait && c >= ready.load(std::memory_order_acquire))) return false;
            } while (!next.compare_exchange_weak(c, c + 1));
            while (ready.load(std::memory_order_acquire) <= c) {
                if (failed.load()) return false;
                std::this_thread::yield();
            }
            std::memcpy(pc[c].host, pin_ + (size_t)(c % SLOTS) * CHUNK, pc[c].bytes);
            done[c % SLOTS].fetch_add(1, std::memory_order_release);
            return true;
        };
        std::thread th[THREADS - 1];
        const int nt = helpers();
        for (int k = 0; k < nt; ++k) {
            try {
                th[k] = std::thread([&] { while (work(true)) {} });
            } catch (const std::system_error&) {
                break;  // fewer threads
            }
        }
        hipError_t e = hipSuccess;
        int issued = 0;
        while (ready.load() < np && e == hipSuccess) {
            while (issued < np && issued < ready.load() + SLOTS && e == hipSuccess) {
                const int s = issued % SLOTS;
                if (done[s].load(std::memory_order_acquire) < issued / SLOTS) {  // its last piece is not out yet
                    if (issued > ready.load()) break;
                    if (!work(false)) std::this_thread::yield();
                    continue;
                }
                e = hipMemcpyAsync(pin_ + (size_t)s * CHUNK, pc[issued].dev, pc[issued].bytes, hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(ev_[s], st);
                ++issued;
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev_[ready.load() % SLOTS]);
            if (e == hipSuccess) ready.fetch_add(1, std::memory_order_release);
        }
        if (e != hipSuccess) failed.store(1);
        else while (work(true)) {}
        for (std::thread& t : th)
            if (t.joinable()) t.join();
        return e;
    }

    hipError_t large_up(const std::vector<Piece>& pc, hipStream_t st) {
        const int np = (int)pc.size();
        hipError_t e = drain();
        if (e != hipSuccess) return e;
        std::atomic<int> free_until{std::min(np, (int)SLOTS)}, next{0}, failed{0};
        std::atomic<int> filled[SLOTS];  // pieces put into the slot so far
        for (auto& d : filled) d.store(0);
        auto work = [&](bool wait) {
            int c = next.load();
            do {
                if (c >= np || (!wait && c >= free_until.load(std::memory_order_acquire))) return false;
            } while (!next.compare_exchange_weak(c, c + 1));
            while (free_until.load(std::memory_order_acquire) <= c) {
                if (failed.load()) return false;
                std::this_thread::yield();
            }
            std::memcpy(pin_ + (size_t)(c % SLOTS) * CHUNK, pc[c].host, pc[c].bytes);
            filled[c % SLOTS].fetch_add(1, std::memory_order_release);
            return true;
        };
        std::thread th[THREADS - 1];
        const int nt = helpers();
        for (int k = 0; k < nt; ++k) {
            try {
                th[k] = std::thread([&] { while (work(true)) {} });
            } catch (const std::system_error&) {
                break;
            }
        }
        for (int c = 0; c < np && e == hipSuccess; ++c) {
            const int s = c % SLOTS;
            while (filled[s].load(std::memory_order_acquire) <= c / SLOTS)
                if (!work(false)) std::this_thread::yield();
            e = hipMemcpyAsync(pc[c].dev, pin_ + (size_t)s * CHUNK, pc[c].bytes, hipMemcpyHostToDevice, st);
            if (e == hipSuccess) e = hipEventRecord(ev_[s], st);
            // the piece SLOTS ahead of the oldest one in flight may be filled
            const int old = c + 1 - SLOTS / 2;
            if (e == hipSuccess && old >= 0 && old + SLOTS < np) {
                e = hipEventSynchronize(ev_[old % SLOTS]);
                if (e == hipSuccess) free_until.store(old + SLOTS + 1, std::memory_order_release);
            }
        }
        if (e != hipSuccess) failed.store(1);
        for (std::thread& t : th)
            if (t.joinable()) t.join();
        return e;
    }

    static int helpers() {
        const unsigned hw = std::thread::hardware_concurrency();
        return (int)std::min<unsigned>(THREADS - 1, hw > 1 ? hw - 1 : 0);
    }
};

}  // namespace nbh
