// Device-to-host transfers of a context through one pinned buffer.
//
// A copy to pageable memory costs about 12 us a call for a few kilobytes, and
// a large one runs at the rate of one core that faults the destination's
// pages in (112 MB to fresh memory: 27 ms, 4 GB/s).  Here
//  - a few arrays of at most SMALL bytes in all are written to the buffer by
//    one kernel (launch_pack) and copied out: six arrays of 64 KB in all
//    15 us against 92 us as six copies, of 2 MB in all 110 against 133 us;
//  - larger ones go in pieces of CHUNK bytes, which several threads of the
//    call copy out as they arrive, two pieces in flight for each: 14 MB to
//    fresh pages 0.45 against 0.85 ms, 112 MB 5.8 against 27 ms (eight
//    threads; four: 8.7 ms, pieces of 512 KB: 6.1 ms).
// The buffer grows with the largest request, to at most 2 * THREADS * CHUNK
// bytes, and is freed with its owner.  Calls on one object are serialised.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

#include "bw_common.h"

namespace bw {

void launch_pack(const PackSegs &, int *dst, hipStream_t);

// bytes from src (device) to dst (host), whole 32-bit words; a null dst is skipped
struct StageSeg {
    void *dst;
    const void *src;
    size_t bytes;
};

class Staging {
  public:
    static constexpr size_t SMALL = (size_t)2 << 20, CHUNK = (size_t)2 << 20;
    static constexpr int THREADS = 8;

    Staging() = default;
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;
    ~Staging() {
        for (int i = 0; i < n_ev_; i++) (void)hipEventDestroy(ev_[i]);
        if (buf_) (void)hipHostFree(buf_);
    }

    // copies every segment after the work submitted to st; returns when done
    hipError_t download(const StageSeg *seg, int n, hipStream_t st) {
        StageSeg s[PackSegs::MAX];
        int k = 0;
        size_t total = 0;
        for (int i = 0; i < n; i++)
            if (seg[i].dst && seg[i].bytes) {
                s[k++] = seg[i];
                total += seg[i].bytes;
            }
        std::lock_guard<std::mutex> lock(m_);
        if (!k) return hipStreamSynchronize(st);
        // threads for the pieces; no more than half as many as there are pieces
        const int nt = total <= SMALL ? 0 : (int)std::clamp<size_t>(total / (2 * CHUNK), 1, THREADS);
        if (!reserve(nt ? 2 * (size_t)nt * CHUNK : total, 2 * nt)) return plain(s, k, st);
        return nt ? pieces(s, k, nt, st) : small(s, k, st);
    }

  private:
    std::mutex m_;
    char *buf_ = nullptr;
    size_t cap_ = 0;
    hipEvent_t ev_[2 * THREADS];
    int n_ev_ = 0;

    bool reserve(size_t bytes, int events) {
        if (bytes > cap_) {
            if (buf_) (void)hipHostFree(buf_);
            buf_ = nullptr;
            cap_ = 0;
            void *p = nullptr;
            bytes = std::max(bytes, (size_t)64 << 10);
            if (hipHostMalloc(&p, bytes, 0) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            buf_ = (char *)p;
            cap_ = bytes;
        }
        for (; n_ev_ < events; n_ev_++)
            if (hipEventCreateWithFlags(&ev_[n_ev_], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        return true;
    }
    // no pinned memory to be had
    static hipError_t plain(const StageSeg *s, int k, hipStream_t st) {
        hipError_t e = hipStreamSynchronize(st);
        for (int i = 0; i < k && e == hipSuccess; i++) e = hipMemcpy(s[i].dst, s[i].src, s[i].bytes, hipMemcpyDeviceToHost);
        return e;
    }
    hipError_t small(const StageSeg *s, int k, hipStream_t st) {
        PackSegs p;
        p.n = k;
        p.off[0] = 0;
        for (int i = 0; i < k; i++) {
            p.src[i] = (const int *)s[i].src;
            p.off[i + 1] = p.off[i] + (int)(s[i].bytes / 4);
        }
        launch_pack(p, (int *)buf_, st);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
        for (int i = 0; i < k; i++) std::memcpy(s[i].dst, buf_ + (size_t)p.off[i] * 4, s[i].bytes);
        return hipSuccess;
    }
    // The pieces are handed out in order.  A thread owns two places of the
    // buffer and their events: while one piece is copied out the next is on
    // its way.  (A thread that cannot be started, for want of memory or of
    // threads, leaves its share to the others.)
    hipError_t pieces(const StageSeg *s, int k, int nt, hipStream_t st) {
        size_t first[PackSegs::MAX + 1] = {0};
        for (int i = 0; i < k; i++) first[i + 1] = first[i] + (s[i].bytes + CHUNK - 1) / CHUNK;
        int device = 0;
        hipError_t e0 = hipGetDevice(&device);
        if (e0 != hipSuccess) return e0;
        std::atomic<size_t> next{0};
        std::atomic<int> error{(int)hipSuccess};
        auto work = [&](int w) {
            struct { char *dst; size_t bytes; } piece[2];
            auto issue = [&](int q) {
                piece[q].bytes = 0;
                const size_t c = next.fetch_add(1);
                if (c >= first[k] || error.load() != hipSuccess) return hipSuccess;
                int i = 0;
                while (c >= first[i + 1]) i++;
                const size_t o = (c - first[i]) * CHUNK, b = std::min(CHUNK, s[i].bytes - o);
                hipError_t e = hipMemcpyAsync(place(w, q), (const char *)s[i].src + o, b, hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(ev_[2 * w + q], st);
                if (e != hipSuccess) return e;
                piece[q].dst = (char *)s[i].dst + o;
                piece[q].bytes = b;
                return hipSuccess;
            };
            hipError_t e = hipSetDevice(device);
            piece[0].bytes = piece[1].bytes = 0;
            for (int q = 0; q < 2 && e == hipSuccess; q++) e = issue(q);
            for (int q = 0; e == hipSuccess && piece[q].bytes; q ^= 1) {
                e = hipEventSynchronize(ev_[2 * w + q]);
                if (e != hipSuccess) break;
                std::memcpy(piece[q].dst, place(w, q), piece[q].bytes);
                e = issue(q);
            }
            if (e != hipSuccess) error.store((int)e);
        };
        std::thread threads[THREADS];
        try {
            for (int w = 1; w < nt; w++) threads[w] = std::thread(work, w);
        } catch (const std::exception &) {
        }
        work(0);
        for (auto &t : threads)
            if (t.joinable()) t.join();
        const hipError_t e = hipStreamSynchronize(st);  // also after an error: nothing of the buffer is in flight
        return error.load() != hipSuccess ? (hipError_t)error.load() : e;
    }
    char *place(int w, int q) const { return buf_ + (size_t)(2 * w + q) * CHUNK; }
};

}  // namespace bw
