// Reading a field back into the caller's array of doubles.
//
// A plain copy into pageable memory is staged by the runtime on the calling
// thread, the float fields of a mixed case were then widened by the same
// thread, and a fresh destination's pages are faulted in on it too: 256 x 256
// x 192 points took 19 ms (mixed) and 15.5 ms (FP64), against 1 and 2 ms on
// the link (56 GB/s).  Fields of HC_MIN values and more are moved in chunks through a ring
// of pinned buffers instead: the calling thread keeps HC_AHEAD copies in
// flight, and up to HC_THREADS threads, started for the call and joined before
// it returns, widen or copy finished chunks into the destination.  Below
// HC_MIN the threads cost what they save, and the plain copy stays; it also
// stays where no pinned memory or no thread can be had, and for a call that
// finds the ring in use by another thread.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

#include "common.hpp"

namespace lg {

// values a chunk: 2 MiB of the destination, whose chunks also end on 2 MiB
// addresses, so that no two threads fault in one huge page (with chunks of
// 1 MiB two did, each clearing it whole: FP64 14.3 ms)
constexpr long HC_CHUNK = 1L << 18;
constexpr int HC_BUFS = 12;             // chunks in the ring, at most
constexpr int HC_AHEAD = 3;             // copies in flight
constexpr int HC_THREADS = 8;
// Smallest field that takes the ring, in values: 32 MiB of doubles.  Reads of
// four fields in turn, ring and plain copy, ms a field: 256 x 256 x 192 (12.8 M
// values) mixed 2.1 and 18.9, FP64 3.0 and 10.0; 192^3 (7.2 M) 1.4 and 6.0, 5.3
// and 6.1; 192 x 144 x 160 (4.5 M) 1.05 and 3.75, 3.3 and 3.8; just below the
// line, 144 x 144 x 190 (4.0 M), 0.9 and 2.8, 2.2 and 2.6; 128^3 1.5 and 1.9, 0.7
// and 1.0; 64^3 0.43 and 0.29, 0.6 and 0.4.  The line is not where the reads by
// themselves cross (near 10^6 values) but above 128^3, where what the program
// did next cost more than the ring saved: the plain copy leaves a field in
// the cache of the caller's core, the ring in eight others', and a pass of 128^3
// steps that reads and converts four fields took 6 ms longer (54 and 60).
constexpr long HC_MIN = 1L << 22;

class HostCopy {
    std::mutex use;                     // one call at a time in the ring
    char* pin = nullptr;
    int nbuf = 0;
    hipEvent_t ev[HC_BUFS] = {};
    int nev = 0;

    template <typename T>
    static void widen(double* dst, const T* src, long n) {
        if constexpr (std::is_same<T, double>::value) {
            std::memcpy(dst, src, (size_t)n * sizeof(double));
        } else {
            for (long i = 0; i < n; ++i) dst[i] = (double)src[i];
        }
    }

    template <typename T>
    static void plain(const T* dev, double* host, long n, hipStream_t s) {
        if constexpr (std::is_same<T, double>::value) {
            LG_HIP(hipMemcpyAsync(host, dev, n * sizeof(T), hipMemcpyDeviceToHost, s));
            LG_HIP(hipStreamSynchronize(s));
        } else {
            std::vector<T> tmp((size_t)n);
            LG_HIP(hipMemcpyAsync(tmp.data(), dev, n * sizeof(T), hipMemcpyDeviceToHost, s));
            LG_HIP(hipStreamSynchronize(s));
            widen(host, tmp.data(), n);
        }
    }

    template <typename T>
    void ring(const T* dev, double* host, long n, hipStream_t s) {
        const long past = (long)((reinterpret_cast<uintptr_t>(host) / sizeof(double)) % HC_CHUNK);
        const int K = (int)((past + n + HC_CHUNK - 1) / HC_CHUNK);
        std::mutex mu;
        std::condition_variable cv_ready, cv_done;
        int ready = 0;                       // chunks 0 .. ready-1 have arrived
        bool stop = false;
        std::vector<char> done((size_t)K, 0);
        std::atomic<int> next{0};
        auto buf = [&](int k) { return reinterpret_cast<T*>(pin) + (k % nbuf) * HC_CHUNK; };
        auto beg = [&](int k) { return std::max(0L, (long)k * HC_CHUNK - past); };
        auto len = [&](int k) { return std::min(n, (long)(k + 1) * HC_CHUNK - past) - beg(k); };
        auto work = [&] {
            for (int k; (k = next.fetch_add(1)) < K;) {
                {
                    std::unique_lock<std::mutex> lk(mu);
                    cv_ready.wait(lk, [&] { return ready > k || stop; });
                    if (ready <= k) return;
                }
                widen(host + beg(k), buf(k), len(k));
                std::lock_guard<std::mutex> lk(mu);
                done[(size_t)k] = 1;
                cv_done.notify_one();
            }
        };
        auto issue = [&](int k) {
            if (k >= nbuf) {                 // the buffer's last chunk has to be out of it
                std::unique_lock<std::mutex> lk(mu);
                cv_done.wait(lk, [&] { return done[(size_t)(k - nbuf)] != 0; });
            }
            LG_HIP(hipMemcpyAsync(buf(k), dev + beg(k), (size_t)len(k) * sizeof(T),
                                  hipMemcpyDeviceToHost, s));
            LG_HIP(hipEventRecord(ev[k % nbuf], s));
        };
        // no throw between the first thread and the last join but through
        // here: `host`, `mu` and the rest live until every thread has ended
        std::vector<std::thread> th;
        auto join = [&] {
            {
                std::lock_guard<std::mutex> lk(mu);
                stop = true;
            }
            cv_ready.notify_all();
            for (auto& t : th) t.join();
        };
        try {
            const int ahead = std::min(HC_AHEAD, nbuf);
            for (int k = 0; k < std::min(ahead, K); ++k) issue(k);
            const int hw = std::max(1, (int)std::thread::hardware_concurrency());
            const int want = std::min({HC_THREADS, hw, K});
            th.reserve((size_t)want);
            try {
                for (int i = 0; i < want; ++i) th.emplace_back(work);
            } catch (const std::system_error&) {
                if (th.empty()) throw;       // fewer threads do as well
            }
            for (int k = 0; k < K; ++k) {
                LG_HIP(hipEventSynchronize(ev[k % nbuf]));
                {
                    std::lock_guard<std::mutex> lk(mu);
                    ready = k + 1;
                }
                cv_ready.notify_all();             // the threads wait for different chunks
                if (k + ahead < K) issue(k + ahead);
            }
            join();
        } catch (...) {
            join();
            (void)hipStreamSynchronize(s);   // copies in flight into the ring
            throw;
        }
    }

public:
    HostCopy() = default;
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;

    // The ring for fields of n values of `size` bytes on the device; without
    // one every read takes the plain copy.
    void prepare(long n, size_t size) {
        if (n < HC_MIN) return;
        const int nb = (int)std::min((long)HC_BUFS, (n + HC_CHUNK - 1) / HC_CHUNK + 1);
        void* p = nullptr;
        if (hipHostMalloc(&p, (size_t)nb * HC_CHUNK * size, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        pin = static_cast<char*>(p);
        while (nev < nb) {
            if (hipEventCreateWithFlags(&ev[nev], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return;                      // nbuf stays 0: plain copies
            }
            ++nev;
        }
        nbuf = nb;
    }

    ~HostCopy() {
        for (int i = 0; i < nev; ++i) (void)hipEventDestroy(ev[i]);
        if (pin) (void)hipHostFree(pin);
    }

    // n values at dev, after the work queued on s, to host; returns when
    // they are there.
    template <typename T>
    void read(const T* dev, double* host, long n, hipStream_t s) {
        std::unique_lock<std::mutex> lk(use, std::defer_lock);
        if (nbuf > 0 && n >= HC_MIN && lk.try_lock()) {
            try {
                ring(dev, host, n, s);
                return;
            } catch (const std::system_error&) {
                // no thread could be started
            }
        }
        plain(dev, host, n, s);
    }
};

}  // namespace lg
