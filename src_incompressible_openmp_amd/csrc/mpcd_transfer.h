/*
 * mpcd_transfer.h -- copies between a caller's pageable host arrays and device
 * memory.
 *
 * The runtime's own staged copies reach 9-10 GB/s into a pageable destination
 * and 28 GB/s out of one here, a fraction of the link's rate: one download of
 * 10.5 million particles (336 MB) took 32 ms, 37 into fresh pages, as long as
 * 20 time steps.  A copy of UP_MIN or DOWN_MIN bytes or more is cut into chunks instead,
 * which a few threads move: each owns two pinned chunks, so its copy on one
 * side runs beside the device's on the other, and the page faults of a fresh
 * destination are shared.  The same download takes 9.7 ms (10.0 fresh), the
 * upload 8.6 instead of 12.0 (39 GB/s).  Two threads leave the download at
 * 15-21 ms and eight gain nothing over four; chunks of 1 MiB cost 20 % (about
 * 9 us a chunk beside the copy), of 512 KiB 65 %.  An array that the runtime
 * knows (pinned, managed or device memory) goes to it in one piece: 2^21
 * particles in pinned arrays take 1.25 ms up and 1.24 down, in chunks 1.93
 * and 1.90.
 */
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "mpcd_hip_util.h"

namespace mpcdk {

/* The pinned chunks, shared by every simulation, ensemble and network of the
 * process: allocated at the first large copy, freed with the last object that
 * holds a lease.  One copy uses them at a time; a copy that finds them taken
 * goes the runtime's way. */
class PinnedChunks {
   public:
    static constexpr size_t BYTES = (size_t)2 << 20;
    static constexpr int THREADS = 4;
    static PinnedChunks& instance() {
        static PinnedChunks p;
        return p;
    }
    void lease() {
        std::lock_guard<std::mutex> lk(mu_);
        ++leases_;
    }
    void release() {
        std::lock_guard<std::mutex> lk(mu_);
        if (--leases_ == 0) {
            /* (no copy runs: a copy's object holds a lease) */
            for (void*& b : buf_) {
                if (b) (void)hipHostFree(b);
                b = nullptr;
            }
        }
    }
    std::mutex& busy() { return busy_; }
    /* chunk k, allocated when first asked for (null if there is no memory to
     * pin); busy() held */
    void* chunk(int k) {
        std::lock_guard<std::mutex> lk(mu_);
        if (!buf_[k] && hipHostMalloc(&buf_[k], BYTES, hipHostMallocPortable) != hipSuccess) {
            buf_[k] = nullptr;
            (void)hipGetLastError();
        }
        return buf_[k];
    }

   private:
    std::mutex mu_, busy_;
    int leases_ = 0;
    void* buf_[2 * THREADS] = {};
};

/* Held by every object that copies; the copies themselves. */
class HostCopy {
   public:
    /* Down, two threads' worth of chunks: 8 MiB take 0.35 ms chunked, 0.51 not
     * (the threads' start costs what is gained below).  The runtime's uploads
     * are three times as fast, so chunks pay later.  Arrays uploaded again and
     * again: 8 MiB take 0.30 ms chunked, 0.25 not, 10 MiB 0.34 and 0.30, 14 MiB
     * 0.46 and 0.42, 16 MiB 0.51 both, 20 MiB 0.62 and 0.69.  New arrays at each
     * call, the program that calls the stages one by one: a step with arrays of
     * 8.2 MiB takes 11.2 ms chunked, 10.8 not, of 10 MiB 12.0 and 12.2, of 14.3
     * MiB 17.1 and 17.3.  The line is the latter's. */
    static constexpr size_t DOWN_MIN = 4 * PinnedChunks::BYTES, UP_MIN = 5 * PinnedChunks::BYTES;

    HostCopy() { PinnedChunks::instance().lease(); }
    ~HostCopy() { PinnedChunks::instance().release(); }
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;

    /* device to host, complete on return */
    void download(void* dst, const void* src, size_t bytes, hipStream_t st) {
        if (!download_later(dst, src, bytes, st)) HIP_OK(hipStreamSynchronize(st));
    }
    /* the same for one of several arrays that share one wait: complete at the
     * latest once the caller has waited for the stream; true if it is on
     * return */
    bool download_later(void* dst, const void* src, size_t bytes, hipStream_t st) {
        if (staged(dst, const_cast<void*>(src), bytes, st, false)) return true;
        HIP_OK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
        return false;
    }
    /* host to device, ordered on the stream: a pageable array may change on
     * return, a pinned one once the stream has got there (every caller waits
     * for it before it returns) */
    void upload(void* dst, const void* src, size_t bytes, hipStream_t st) {
        if (!staged(const_cast<void*>(src), dst, bytes, st, true))
            HIP_OK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    }

   private:
    static bool pageable(const void* host) {
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, host) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError(); /* an unknown pointer, where that is an error */
        return true;
    }

    bool staged(void* host, void* dev, size_t bytes, hipStream_t st, bool up) {
        if (bytes < (up ? UP_MIN : DOWN_MIN) || !pageable(host)) return false;
        PinnedChunks& pc = PinnedChunks::instance();
        std::unique_lock<std::mutex> lk(pc.busy(), std::try_to_lock);
        if (!lk.owns_lock()) return false;
        const size_t B = PinnedChunks::BYTES;
        const long long nch = (long long)((bytes + B - 1) / B);
        const int T = (int)std::min<long long>(PinnedChunks::THREADS, nch / 2);
        void* bufs[2 * PinnedChunks::THREADS];
        for (int k = 0; k < 2 * T; ++k)
            if (!(bufs[k] = pc.chunk(k))) return false;
        int device = 0;
        HIP_OK(hipGetDevice(&device));
        std::exception_ptr failed[PinnedChunks::THREADS];
        auto work = [&](int t) {
            hipEvent_t ev[2] = {nullptr, nullptr};
            try {
                HIP_OK(hipSetDevice(device));
                for (hipEvent_t& e : ev) HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
                auto len = [&](long long c) { return std::min(B, bytes - (size_t)c * B); };
                long long prev = -1;
                int s = 0;
                for (long long c = t; c < nch; c += T, s ^= 1) {
                    char* const h = (char*)host + (size_t)c * B;
                    char* const d = (char*)dev + (size_t)c * B;
                    void* const b = bufs[2 * t + s];
                    if (up) {
                        if (c >= t + 2 * T) HIP_OK(hipEventSynchronize(ev[s])); /* the chunk's last use */
                        std::memcpy(b, h, len(c));
                        HIP_OK(hipMemcpyAsync(d, b, len(c), hipMemcpyHostToDevice, st));
                        HIP_OK(hipEventRecord(ev[s], st));
                    } else {
                        HIP_OK(hipMemcpyAsync(b, d, len(c), hipMemcpyDeviceToHost, st));
                        HIP_OK(hipEventRecord(ev[s], st));
                        if (prev >= 0) {
                            HIP_OK(hipEventSynchronize(ev[s ^ 1]));
                            std::memcpy((char*)host + (size_t)prev * B, bufs[2 * t + (s ^ 1)], len(prev));
                        }
                        prev = c;
                    }
                }
                if (!up && prev >= 0) {
                    HIP_OK(hipEventSynchronize(ev[s ^ 1]));
                    std::memcpy((char*)host + (size_t)prev * B, bufs[2 * t + (s ^ 1)], len(prev));
                }
            } catch (...) {
                failed[t] = std::current_exception();
            }
            for (hipEvent_t e : ev)
                if (e) (void)hipEventDestroy(e);
        };
        std::vector<std::thread> th;
        int started = 1;
        try {
            for (; started < T; ++started) th.emplace_back(work, started);
        } catch (...) {
            /* no thread to be had: this one takes the rest's share below */
        }
        work(0);
        for (std::thread& x : th) x.join();
        for (int t = started; t < T; ++t) work(t);
        /* an upload's chunks are free again, and nothing is in flight on an error */
        const hipError_t e = hipStreamSynchronize(st);
        for (int t = 0; t < T; ++t)
            if (failed[t]) std::rethrow_exception(failed[t]);
        HIP_OK(e);
        return true;
    }
};

}  // namespace mpcdk
