// Copies between device arrays and a caller's pageable host arrays through
// pinned staging memory, by several threads.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace lbmc {

// The process's staging memory (1 MB with the first small transfer, 16 MB with
// the first larger one): held by every context and every model, whose
// transfers alone use it, freed with the last.
void staging_hold();
void staging_release();

// One array of a read: n elements of `bytes` bytes at device address src to
// host address dst; widen: floats at src, doubles at dst
struct HostRead {
    void *dst;
    const void *src;
    size_t n;
};

// dst[k] <- src[k] for every array, after the work on stream s; returns when
// the data are in place
hipError_t read_arrays(const HostRead *arrays, int count, int bytes, bool widen, int device, hipStream_t s);

// One array of a write: n bytes
struct HostWrite {
    void *dst;
    const void *src;
    size_t n;
};

// dst (device) <- src (host) for every array, ordered on stream s; returns
// when the data are in place
hipError_t write_arrays(const HostWrite *arrays, int count, int device, hipStream_t s);

}  // namespace lbmc
