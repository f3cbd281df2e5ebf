// Reading an object's state back: 3-vectors of device records, gathered into particle order by a kernel that stores
// straight into pinned host memory, then widened (or copied) into the caller's double arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "host_util.h"

namespace spgvbd {

// One 3-vector per particle: components 0 .. 2 of the record at src + stride * slot.
template <class T>
struct Field3 {
    const T *src;
    int32_t stride;  // in T
    double *dst;     // caller's array, 3 per particle; null: not read
};

constexpr int kStateFields = 4;  // fields per read at most

// The largest of the ranges between consecutive offsets.
inline int64_t largestRange(const std::vector<int64_t> &offsets)
{
    int64_t n = 0;
    for (size_t k = 1; k < offsets.size(); ++k) n = std::max(n, offsets[k] - offsets[k - 1]);
    return n;
}

// The pinned staging memory and events of one context's reads (used by one thread at a time, as its context is).
class StateReader {
  public:
    StateReader() = default;
    StateReader(const StateReader &) = delete;
    StateReader &operator=(const StateReader &) = delete;
    ~StateReader();
    // The staging memory for reads of n particles (bounded), so that the first read need not allocate it.
    void reserve(size_t bytesPerParticle, int64_t n);
    // Reads `count` fields of n particles: particle i's record is order[i], or i where order is null. Waits for the
    // work queued on `stream` before it. T: float or double.
    template <class T>
    void read(const Field3<T> *fields, int count, const int32_t *order, int64_t n, hipStream_t stream);

  private:
    void *m_host = nullptr;
    size_t m_bytes = 0;
    std::vector<hipEvent_t> m_events;
};

}  // namespace spgvbd
