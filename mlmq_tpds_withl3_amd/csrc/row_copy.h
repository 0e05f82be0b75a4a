// Copies of device rows into ordinary host memory.
//
// Such a copy is bound by the host: new memory of the caller's is not backed
// by pages yet, and to fault them in one by one while copying costs 0.7 us per
// 4 KiB (the card would deliver them in 0.1 us).  Here the rows come over the
// bus into a pinned buffer while the kernel is asked for all of the
// destination's pages at once (0.3 us per page), and are copied from there.
// New rows of 20,011 / 50,021 / 264,346 / 1,070,376 / 6,262,104 vertices:
// hipMemcpy 56 / 45-120 / 256 / 763 / 2796 us, this 11 / 16 / 119 / 364 /
// 1753 us; into memory that has its pages 42 / 17 / 69 / 244 / 1398 us against
// 12 / 17 / 61 / 219 / 1245 us.
#pragma once

#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>

namespace mlmq {

struct RowCopy {
    void *dst = nullptr;          // host
    const void *src = nullptr;    // device
    size_t bytes = 0;
};

class RowStage {
public:
    static constexpr size_t kPiece = 4u << 20;   // bytes on their way at once, twice over

    // A pinned buffer for `bytes` (at most two pieces: one fills while the
    // other is copied out).  Without one, rows are copied directly.
    hipError_t reserve(size_t bytes) {
        const size_t size = bytes > kPiece ? 2 * kPiece : (bytes + 4095) & ~(size_t)4095;
        if (size <= size_) return hipSuccess;
        release();
        hipError_t e = hipHostMalloc((void **)&buf_, size, hipHostMallocDefault);
        for (hipEvent_t &ev : ev_)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) release();
        else size_ = size;
        return e;
    }
    void release() {
        if (buf_) (void)hipHostFree(buf_);
        for (hipEvent_t &ev : ev_) {
            if (ev) (void)hipEventDestroy(ev);
            ev = nullptr;
        }
        buf_ = nullptr;
        size_ = 0;
    }
    // Copies the rows in stream order and waits for them.
    hipError_t copy(const RowCopy *rows, size_t count, hipStream_t s) {
        const size_t piece = std::min(size_, kPiece);
        const int pieces = size_ > kPiece ? 2 : 1;
        hipError_t e = hipSuccess;
        if (count == 1 && rows[0].bytes <= piece && ordinary(rows[0].dst)) {
            // (waiting for an event takes 8 us longer than for the stream)
            e = hipMemcpyAsync(buf_, rows[0].src, rows[0].bytes, hipMemcpyDeviceToHost, s);
            populate((char *)rows[0].dst, rows[0].bytes);
            if (e == hipSuccess) e = hipStreamSynchronize(s);
            if (e == hipSuccess) std::memcpy(rows[0].dst, buf_, rows[0].bytes);
            return e;
        }
        Place in, out;
        int filled = 0, emptied = 0;
        while (e == hipSuccess && out.row < count) {
            const RowCopy &r = rows[out.row];
            if (out.at == 0 && (!buf_ || !ordinary(r.dst))) {
                if (in.row == out.row && in.at == 0) in.next(r.bytes, r.bytes);
                e = hipMemcpyAsync(r.dst, r.src, r.bytes, hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipStreamSynchronize(s);
                out.next(r.bytes, r.bytes);
                continue;
            }
            while (e == hipSuccess && filled - emptied < pieces && in.row < count && (in.at || ordinary(rows[in.row].dst))) {
                const size_t n = std::min(piece, rows[in.row].bytes - in.at);
                e = hipMemcpyAsync(buf_ + filled % pieces * piece, (const char *)rows[in.row].src + in.at, n,
                                   hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(ev_[filled % pieces], s);
                ++filled;
                in.next(n, rows[in.row].bytes);
            }
            const size_t n = std::min(piece, r.bytes - out.at);
            populate((char *)r.dst + out.at, n);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[emptied % pieces]);
            if (e == hipSuccess) std::memcpy((char *)r.dst + out.at, buf_ + emptied % pieces * piece, n);
            ++emptied;
            out.next(n, r.bytes);
        }
        if (e != hipSuccess && filled != emptied) (void)hipStreamSynchronize(s);   // nothing still writes the buffer
        return e;
    }

private:
    struct Place {
        size_t row = 0, at = 0;
        void next(size_t n, size_t of) {
            at += n;
            if (at < of) return;
            ++row;
            at = 0;
        }
    };
    // Memory that the runtime knows (pinned, device) is copied to directly.
    static bool ordinary(const void *p) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return true;
    }
    // Pages of [p, p + n) that are not there yet; where this is not supported
    // the copy faults them in.
    static void populate(char *p, size_t n) {
#ifdef MADV_POPULATE_WRITE
        constexpr int kPopulate = MADV_POPULATE_WRITE;
#else
        constexpr int kPopulate = 23;
#endif
        if (n < kPopulateFrom) return;
        const uintptr_t lo = ((uintptr_t)p + 4095) & ~(uintptr_t)4095, hi = ((uintptr_t)p + n) & ~(uintptr_t)4095;
        if (lo < hi) (void)madvise((void *)lo, hi - lo, kPopulate);
    }
    // (a call costs as much as the faults of a few pages)
    static constexpr size_t kPopulateFrom = 32u << 10;

    char *buf_ = nullptr;
    size_t size_ = 0;
    hipEvent_t ev_[2] = {nullptr, nullptr};
};

}  // namespace mlmq
