// ts_hostmem.hpp -- host memory of states: transfers between the caller's (pageable) arrays and the
// device, and the batch engine's own copies of states.
//
// What bounds them is not PCIe.  hipMemcpy from and to pageable memory goes through one thread, at
// 28 GB/s up and 17 GB/s down, and a freshly allocated array costs that thread its page faults as
// well (168 MB: 6 to 30 ms, by page size), where pinned memory takes 53 GB/s either way.  So large
// transfers go in chunks through a small pinned buffer, with a few threads that each copy their
// chunks to or from the caller's array (faulting its pages in side by side) while the others' are
// on the bus.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <system_error>
#include <thread>
#include <vector>

namespace tsr {

// Bytes from which a copy is shared between threads, and the same for an upload, whose array is there
// and needs no page faults.  They start well above the cost of starting threads: the caller's own
// threads (an OpenMP pool) often spin on every CPU for a while after their last work, and then the
// helpers wait for a time slice each.  Behind such a pool a 9 MB download by four threads took 1.9 ms
// instead of 1.0 and a 10 MB upload 4 ms instead of 0.4; a 42 MB download still gains, 4.9 to 1.9 ms, and a
// 168 MB upload 6.0 to 4.4 ms.
constexpr size_t kThreadedCopy = size_t(24) << 20;
constexpr size_t kThreadedUpload = size_t(64) << 20;
constexpr size_t kSmallState = size_t(4) << 20;  // bytes below which the batch gathers states in pinned memory

// Calls f(worker, begin, end) for chunks that cover [0, total), on at most `most` threads, the calling one
// among them; chunks go to whichever thread is free.  Needs none of the threads it asks for.
template <typename F>
void for_chunks(size_t total, size_t chunk, int most, F&& f) {
    std::atomic<size_t> next{0};
    auto work = [&](int w) {
        for (;;) {
            const size_t b = next.fetch_add(chunk);
            if (b >= total) return;
            f(w, b, b + chunk < total ? b + chunk : total);
        }
    };
    std::vector<std::thread> helpers;
    const size_t chunks = (total + chunk - 1) / chunk;
    try {
        for (int w = 1; w < most && size_t(w) < chunks; w++) helpers.emplace_back(work, w);
    } catch (const std::exception&) {  // no thread or no memory for one: fewer share the work
    }
    work(0);
    for (std::thread& t : helpers) t.join();
}

// Threads that a copy of at least kThreadedCopy bytes is shared between.  Four reach 100 GB/s between pages
// that are there, and fault fresh ones in faster than eight do (5 against 8 ms for 168 MB).
inline int copy_threads() { return std::thread::hardware_concurrency() >= 8 ? 4 : 1; }

// dst[0, bytes) = src[0, bytes)
void host_copy(void* dst, const void* src, size_t bytes);

// An uninitialised array of doubles.  Large ones are on huge pages where the system has them.
class HostArray {
   public:
    HostArray() = default;
    ~HostArray() { release(); }
    HostArray(const HostArray&) = delete;
    HostArray& operator=(const HostArray&) = delete;
    bool allocate(size_t n);  // false: no memory
    void release();
    double* data() { return p_; }
    const double* data() const { return p_; }
    size_t size() const { return n_; }

   private:
    double* p_ = nullptr;
    size_t n_ = 0;
};

// A pinned buffer for the transfers of one context or batch, allocated at the first transfer that uses it and
// freed with its owner.  Where the system has no pinned memory to give, the buffer is an ordinary one: copies
// through it are slower, and large ones go to the runtime as they are.  One thread uses it at a time.
class Staging {
   public:
    static constexpr int kSlots = 4;  // one to a thread
    static constexpr size_t kSlot = size_t(2) << 20;
    static constexpr size_t kBytes = kSlots * kSlot;
    static_assert(kBytes >= 2 * kSmallState);
    // On `device`, in the stream's order.  to_host waits until the data are there; to_device may return before
    // they are, and the caller keeps `src` until it has waited for the stream.  Small copies, and all
    // in a process with few CPUs, are left to the runtime: one thread would take turns with the bus, where the
    // runtime's own copy of pageable memory overlaps the two.
    hipError_t to_device(void* dst, const void* src, size_t bytes, int device, hipStream_t stream);
    hipError_t to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t stream);
    // `bytes` <= kBytes of the buffer for an asynchronous copy on `stream`: free again after the next wait
    // (null with an error in `e`).  The buffer is handed out in order; a full one waits for the stream.
    char* take(size_t bytes, hipStream_t stream, hipError_t* e);
    void all_free() { used_ = 0; }  // the stream has been waited for
    void release();

   private:
    hipError_t ensure();
    hipError_t chunked(char* dst, const char* src, size_t bytes, int device, hipStream_t stream, bool up);
    char* buf_ = nullptr;
    bool pinned_ = false;
    hipEvent_t ev_[kSlots] = {};
    size_t used_ = 0;
};

}  // namespace tsr
