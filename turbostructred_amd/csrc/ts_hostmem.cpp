// ts_hostmem.cpp -- host memory of states and their transfers (see ts_hostmem.hpp).
#include "ts_hostmem.hpp"

#include <sys/mman.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>

namespace tsr {

void host_copy(void* dst, const void* src, size_t bytes) {
    if (bytes < kThreadedCopy) {
        std::memcpy(dst, src, bytes);
        return;
    }
    for_chunks(bytes, size_t(1) << 20, copy_threads(),
               [&](int, size_t b, size_t e) { std::memcpy((char*)dst + b, (const char*)src + b, e - b); });
}

bool HostArray::allocate(size_t n) {
    release();
    const size_t bytes = n * sizeof(double), huge = size_t(2) << 20;
    void* q = nullptr;
    if (bytes < 2 * huge) {
        q = std::malloc(bytes ? bytes : 1);
        if (!q) return false;
    } else {
        if (posix_memalign(&q, huge, bytes)) return false;
        (void)madvise(q, bytes / huge * huge, MADV_HUGEPAGE);  // a hint: small pages serve as well
    }
    p_ = (double*)q;
    n_ = n;
    return true;
}

void HostArray::release() {
    std::free(p_);
    p_ = nullptr;
    n_ = 0;
}

hipError_t Staging::ensure() {
    if (buf_) return hipSuccess;
    pinned_ = hipHostMalloc((void**)&buf_, kBytes, hipHostMallocDefault) == hipSuccess;
    if (!pinned_) buf_ = nullptr;
    for (int i = 0; pinned_ && i < kSlots; i++)
        if (hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) != hipSuccess) {
            ev_[i] = nullptr;
            release();
        }
    if (!pinned_) {
        (void)hipGetLastError();  // handled here: not the next launch's
        buf_ = (char*)std::malloc(kBytes);
    }
    return buf_ ? hipSuccess : hipErrorOutOfMemory;
}

void Staging::release() {
    for (hipEvent_t& ev : ev_) {
        if (ev) (void)hipEventDestroy(ev);
        ev = nullptr;
    }
    if (buf_ && pinned_) (void)hipHostFree(buf_);
    else std::free(buf_);
    buf_ = nullptr;
    pinned_ = false;
    used_ = 0;
}

// Every thread has a slot of its own: up, it fills the slot and sends it, and waits before it fills it
// again; down, it fetches a chunk, waits for it and copies it out.
hipError_t Staging::chunked(char* dst, const char* src, size_t bytes, int device, hipStream_t stream, bool up) {
    std::atomic<int> failed{int(hipSuccess)};
    bool pending[kSlots] = {};  // each entry is its thread's own
    size_t chunk = bytes / (4 * kSlots);
    chunk = chunk < (size_t(512) << 10) ? size_t(512) << 10 : chunk > kSlot ? kSlot : chunk;
    chunk &= ~size_t(4095);
    static_assert(kSlots == 4, "copy_threads gives at most one thread per slot");
    for_chunks(bytes, chunk, copy_threads(), [&](int w, size_t b, size_t e) {
        if (failed.load() != hipSuccess) return;
        char* slot = buf_ + w * kSlot;
        hipError_t r = hipSetDevice(device);
        if (up) {
            if (r == hipSuccess && pending[w]) r = hipEventSynchronize(ev_[w]);
            if (r == hipSuccess) {
                std::memcpy(slot, src + b, e - b);
                r = hipMemcpyAsync(dst + b, slot, e - b, hipMemcpyHostToDevice, stream);
            }
            if (r == hipSuccess) r = hipEventRecord(ev_[w], stream);
            pending[w] = true;
        } else {
            if (r == hipSuccess) r = hipMemcpyAsync(slot, src + b, e - b, hipMemcpyDeviceToHost, stream);
            if (r == hipSuccess) r = hipEventRecord(ev_[w], stream);
            if (r == hipSuccess) r = hipEventSynchronize(ev_[w]);
            if (r == hipSuccess) std::memcpy(dst + b, slot, e - b);
        }
        if (r != hipSuccess) failed = int(r);
    });
    const hipError_t last = hipStreamSynchronize(stream);
    return failed.load() != hipSuccess ? hipError_t(failed.load()) : last;
}

hipError_t Staging::to_device(void* dst, const void* src, size_t bytes, int device, hipStream_t stream) {
    if (bytes < kThreadedUpload || copy_threads() == 1 || ensure() != hipSuccess || !pinned_) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
    }
    const hipError_t e = used_ ? hipStreamSynchronize(stream) : hipSuccess;  // what take() handed out
    used_ = 0;
    return e != hipSuccess ? e : chunked((char*)dst, (const char*)src, bytes, device, stream, true);
}

hipError_t Staging::to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t stream) {
    if (bytes < kThreadedCopy || copy_threads() == 1 || ensure() != hipSuccess || !pinned_) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
        return e != hipSuccess ? e : hipStreamSynchronize(stream);
    }
    const hipError_t e = used_ ? hipStreamSynchronize(stream) : hipSuccess;
    used_ = 0;
    return e != hipSuccess ? e : chunked((char*)dst, (const char*)src, bytes, device, stream, false);
}

char* Staging::take(size_t bytes, hipStream_t stream, hipError_t* e) {
    *e = ensure();
    if (*e != hipSuccess) return nullptr;
    bytes = (bytes + 255) & ~size_t(255);
    if (used_ + bytes > kBytes) {
        *e = hipStreamSynchronize(stream);
        if (*e != hipSuccess) return nullptr;
        used_ = 0;
    }
    char* p = buf_ + used_;
    used_ += bytes;
    return p;
}

}  // namespace tsr
