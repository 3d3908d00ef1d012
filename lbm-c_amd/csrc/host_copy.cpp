// A copy of a large device array into pageable memory by hipMemcpy runs on one
// thread, which also takes the page faults of a fresh destination; widening
// floats to doubles is another pass over both.  Here up to 8 threads each
// take pieces in turn: an asynchronous copy into the thread's own pinned slot,
// then the (widening) copy out of it, so the link, the page faults and the
// conversion overlap.  Reading rho and u of a 256^3 FP32 lattice (268 MB over
// the link, 537 MB of doubles) took 80-127 ms by hipMemcpy and a loop, and takes
// 9-12 ms; of a 131x97x75 FP64 lattice the 15 populations (114 MB) in took 4.8
// ms, out 15.1 ms, rho and u 2.5 ms, and take 3.1, 3.4 and 1.0 ms; 12 bytes of
// one node 33 and 17 us, by one wait instead of three.
#include "host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace lbmc {

namespace {

constexpr int kSlots = 8;
constexpr size_t kSlotBytes = 2u << 20;
// Reads up to this size go through one small buffer with a single wait: 3
// arrays of 192 KB take 170 us this way, as with threads; at 3 x 512 KB
// threads are ahead, 250 against 400
constexpr size_t kSmallBytes = 1u << 20;
// A thread per 512 KB, two pieces each (at least 512 KB, so that the cost of
// an enqueue and a wait stays small against the copy): of ten such settings
// the one that was best or near it at every size from 1 to 200 MB; 2 MB pieces
// throughout cost up to 2.5 times as much at 4 MB, where too few overlap
constexpr size_t kMinPiece = 512u << 10;
// Writes: up to 256 KB through the small buffer (100 KB 48 -> 16 us), from
// 24 MB in pieces (28 MB 999 -> 919 us, 115 MB 4.3 -> 3.1 ms); between them
// hipMemcpy is ahead (3 MB 109 us against 216: a source has no page faults to
// overlap, and threads cost more than they save)
constexpr size_t kSmallWrite = 256u << 10;
constexpr size_t kPieceWrite = 24u << 20;

struct Staging {
    std::mutex mu;  // one transfer at a time; others go through hipMemcpy
    std::mutex hold_mu;
    int holders = 0;
    // each with the first transfer that takes it: a program that makes and
    // closes one lattice after another pins and unpins for those that read
    // only (14 and 20 us for 1 MB; 0.4 ms with the first use of the slots)
    char *small = nullptr;  // kSmallBytes
    char *slots = nullptr;  // kSlots * kSlotBytes
};

Staging g_staging;

// One transfer's pieces: piece k covers elements of one array
struct Piece {
    int array;
    size_t first, n;
};

int thread_count(size_t bytes) { return (int)std::clamp<size_t>(bytes / kMinPiece, 1, kSlots); }

size_t piece_bytes(size_t bytes)
{
    return std::clamp(bytes / (2 * (size_t)thread_count(bytes)) & ~(size_t)4095, kMinPiece, kSlotBytes);
}

char *pinned(size_t bytes)
{
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocPortable) == hipSuccess) return (char *)p;
    (void)hipGetLastError();
    return nullptr;
}

// the staging memory for a transfer of a holder, its mutex held; null: none
char *staging_for(bool small)
{
    char *&p = small ? g_staging.small : g_staging.slots;
    if (!p) p = pinned(small ? kSmallBytes : kSlots * kSlotBytes);
    return p;
}

// work(piece, slot, event) for every piece by up to `threads` threads, the
// calling one included (fewer when the system gives no more), each with its own
// slot and event; ends with stream s idle, also after an error
template <class Work>
hipError_t for_pieces(const std::vector<Piece> &pieces, int threads, char *staging, int device, hipStream_t s,
                      const Work &work)
{
    std::atomic<size_t> next{0};
    std::atomic<int> status{(int)hipSuccess};
    auto body = [&](int w) {
        hipEvent_t ev = nullptr;
        hipError_t e = hipSetDevice(device);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        while (e == hipSuccess && status.load() == (int)hipSuccess) {
            const size_t k = next.fetch_add(1);
            if (k >= pieces.size()) break;
            e = work(pieces[k], staging + (size_t)w * kSlotBytes, ev);
        }
        if (ev) (void)hipEventDestroy(ev);
        if (e != hipSuccess) status.store((int)e);
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(kSlots);
        for (int w = 1; w < std::min<int>(threads, (int)pieces.size()); w++) pool.emplace_back([&body, w] { body(w); });
    } catch (...) {
        // the threads that did start, and this one, take all pieces
    }
    body(0);
    for (std::thread &t : pool) t.join();
    const hipError_t w = hipStreamSynchronize(s);
    return status.load() != (int)hipSuccess ? (hipError_t)status.load() : w;
}

}  // namespace

void staging_hold()
{
    std::lock_guard<std::mutex> lock(g_staging.hold_mu);
    g_staging.holders++;
}

void staging_release()
{
    std::lock_guard<std::mutex> lock(g_staging.hold_mu);
    if (--g_staging.holders == 0) {
        std::lock_guard<std::mutex> busy(g_staging.mu);
        for (char **p : {&g_staging.small, &g_staging.slots}) {
            if (*p) (void)hipHostFree(*p);
            *p = nullptr;
        }
    }
}

hipError_t read_arrays(const HostRead *arrays, int count, int bytes, bool widen, int device, hipStream_t s)
{
    std::unique_lock<std::mutex> lock(g_staging.mu, std::try_to_lock);
    size_t total = 0;
    for (int k = 0; k < count; k++) total += arrays[k].n * (size_t)bytes;
    const bool small = total <= kSmallBytes;
    char *const staging = lock.owns_lock() ? staging_for(small) : nullptr;
    try {
        if (!staging) {
            hipError_t e = hipStreamSynchronize(s);
            std::vector<float> tmp;
            for (int k = 0; k < count && e == hipSuccess; k++) {
                const HostRead &r = arrays[k];
                if (widen) tmp.resize(r.n);
                e = hipMemcpy(widen ? (void *)tmp.data() : r.dst, r.src, r.n * (size_t)bytes, hipMemcpyDeviceToHost);
                if (widen && e == hipSuccess) std::copy(tmp.begin(), tmp.end(), (double *)r.dst);
            }
            return e;
        }
        auto out = [&](const HostRead &r, size_t first, size_t n, const char *slot) {
            if (widen) {
                double *d = (double *)r.dst + first;
                const float *f = (const float *)slot;
                for (size_t i = 0; i < n; i++) d[i] = f[i];
            } else {
                memcpy((char *)r.dst + first * (size_t)bytes, slot, n * (size_t)bytes);
            }
        };
        if (small) {
            // all arrays side by side, one wait
            hipError_t e = hipSuccess;
            size_t at = 0;
            for (int k = 0; k < count && e == hipSuccess; k++) {
                e = hipMemcpyAsync(staging + at, arrays[k].src, arrays[k].n * (size_t)bytes,
                                   hipMemcpyDeviceToHost, s);
                at += arrays[k].n * (size_t)bytes;
            }
            const hipError_t w = hipStreamSynchronize(s);  // the slot is idle again, also after an error
            if (e == hipSuccess) e = w;
            at = 0;
            for (int k = 0; k < count && e == hipSuccess; k++) {
                out(arrays[k], 0, arrays[k].n, staging + at);
                at += arrays[k].n * (size_t)bytes;
            }
            return e;
        }
        std::vector<Piece> pieces;
        const size_t per = piece_bytes(total) / (size_t)bytes;
        for (int k = 0; k < count; k++)
            for (size_t i = 0; i < arrays[k].n; i += per) pieces.push_back({k, i, std::min(per, arrays[k].n - i)});
        return for_pieces(pieces, thread_count(total), staging, device, s,
                          [&](const Piece &p, char *slot, hipEvent_t ev) {
                              const HostRead &r = arrays[p.array];
                              hipError_t e = hipMemcpyAsync(slot, (const char *)r.src + p.first * (size_t)bytes,
                                                            p.n * (size_t)bytes, hipMemcpyDeviceToHost, s);
                              if (e == hipSuccess) e = hipEventRecord(ev, s);
                              if (e == hipSuccess) e = hipEventSynchronize(ev);
                              if (e == hipSuccess) out(r, p.first, p.n, slot);
                              return e;
                          });
    } catch (...) {
        (void)hipStreamSynchronize(s);
        return hipErrorOutOfMemory;
    }
}

hipError_t write_arrays(const HostWrite *arrays, int count, int device, hipStream_t s)
{
    std::unique_lock<std::mutex> lock(g_staging.mu, std::try_to_lock);
    size_t total = 0;
    for (int k = 0; k < count; k++) total += arrays[k].n;
    const bool small = total <= kSmallWrite;
    char *const staging = lock.owns_lock() && (small || total > kPieceWrite) ? staging_for(small) : nullptr;
    try {
        if (small && staging) {
            hipError_t e = hipSuccess;
            size_t at = 0;
            for (int k = 0; k < count && e == hipSuccess; k++) {
                memcpy(staging + at, arrays[k].src, arrays[k].n);
                e = hipMemcpyAsync(arrays[k].dst, staging + at, arrays[k].n, hipMemcpyHostToDevice, s);
                at += arrays[k].n;
            }
            const hipError_t w = hipStreamSynchronize(s);  // the buffer is idle again, also after an error
            return e != hipSuccess ? e : w;
        }
        if (!staging) {
            hipError_t e = hipSuccess;
            for (int k = 0; k < count && e == hipSuccess; k++)
                e = hipMemcpyAsync(arrays[k].dst, arrays[k].src, arrays[k].n, hipMemcpyHostToDevice, s);
            const hipError_t w = hipStreamSynchronize(s);
            return e != hipSuccess ? e : w;
        }
        std::vector<Piece> pieces;
        const size_t per = piece_bytes(total);
        for (int k = 0; k < count; k++)
            for (size_t i = 0; i < arrays[k].n; i += per) pieces.push_back({k, i, std::min(per, arrays[k].n - i)});
        return for_pieces(pieces, thread_count(total), staging, device, s,
                          [&](const Piece &p, char *slot, hipEvent_t ev) {
                              const HostWrite &w = arrays[p.array];
                              memcpy(slot, (const char *)w.src + p.first, p.n);
                              hipError_t e = hipMemcpyAsync((char *)w.dst + p.first, slot, p.n, hipMemcpyHostToDevice, s);
                              if (e == hipSuccess) e = hipEventRecord(ev, s);
                              return e == hipSuccess ? hipEventSynchronize(ev) : e;
                          });
    } catch (...) {
        (void)hipStreamSynchronize(s);
        return hipErrorOutOfMemory;
    }
}

}  // namespace lbmc
