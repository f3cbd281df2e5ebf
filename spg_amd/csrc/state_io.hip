// The state read-out of state_io.h.
//
// What bounds it: PCIe (53 GB/s to pinned memory, 17 GB/s to pageable memory, measured), and the host's first touch of
// the caller's arrays. So the device sends only what is asked for: this object's 12 bytes per 32-bit vector, in
// particle order, and not every object's padded float4 records; and several host threads widen them, since a
// freshly allocated array is faulted in page by page while it is written. Step and read-out of a 512x512 cloth: 1.92 ms
// with pageable copies of all records, 1.21 ms now; of 24 objects advanced together (each of whose reads copied all 24):
// 9.2 ms, 1.26 ms now; of a 256x256 rigid-body lattice 1.43 ms, 0.68 ms now.
#include <algorithm>
#include <cstring>

#include "host_threads.h"
#include "state_io.h"

namespace spgvbd {

namespace {

// Bytes gathered by one launch (32,768 particles' positions and velocities in 32 bits): while the host widens one part
// the next is sent. A larger read goes through the staging memory in rounds.
constexpr int64_t kPartBytes = 786432;
constexpr int64_t kParts = 10;  // parts of staging memory at most, 7.9 MB
constexpr int kThreads = 4;     // host threads of a read of several parts

// records of `bytes` bytes per part
int64_t perPart(size_t bytes) { return kPartBytes / static_cast<int64_t>(bytes); }

template <class T>
struct GatherArgs {
    const T *src[kStateFields];
    int32_t stride[kStateFields];
    const int32_t *order;
    int64_t first;
    int32_t n;
    T *out;  // field f at out + 3 n f
};

// A thread per component, so that the stores of a wavefront are one contiguous span (the three threads of a particle
// read the same record). blockIdx.y: the field.
template <class T>
__global__ void __launch_bounds__(256) gatherKernel(GatherArgs<T> a)
{
    const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * a.n) return;
    const int32_t i = k / 3, d = k - 3 * i;
    const int64_t p = a.first + i;
    const int64_t slot = a.order ? a.order[p] : p;
    const int f = blockIdx.y;
    a.out[static_cast<int64_t>(f) * 3 * a.n + k] = a.src[f][slot * a.stride[f] + d];
}

void widen(const float *src, double *dst, int64_t n)
{
    for (int64_t i = 0; i < n; ++i) dst[i] = src[i];
}
void widen(const double *src, double *dst, int64_t n) { std::memcpy(dst, src, n * sizeof(double)); }

}  // namespace

StateReader::~StateReader()
{
    for (hipEvent_t e : m_events) (void)hipEventDestroy(e);
    if (m_host) (void)hipHostFree(m_host);
}

void StateReader::reserve(size_t bytesPerParticle, int64_t n)
{
    if (n <= 0) return;
    const int64_t parts = std::min(kParts, (n + perPart(bytesPerParticle) - 1) / perPart(bytesPerParticle));
    const size_t bytes = parts > 1 ? static_cast<size_t>(parts * kPartBytes) : static_cast<size_t>(n) * bytesPerParticle;
    if (m_bytes < bytes) {
        if (m_host) (void)hipHostFree(m_host);
        m_host = nullptr;
        m_bytes = 0;
        // coherent: the kernels' stores are there once their event is, without a further flush
        hipCheck(hipHostMalloc(&m_host, bytes, hipHostMallocMapped | hipHostMallocCoherent), "hipHostMalloc");
        m_bytes = bytes;
    }
    while (static_cast<int64_t>(m_events.size()) < parts) {
        hipEvent_t e;
        hipCheck(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        m_events.push_back(e);
    }
}

template <class T>
void StateReader::read(const Field3<T> *fields, int count, const int32_t *order, int64_t n, hipStream_t stream)
{
    Field3<T> use[kStateFields];
    int nf = 0;
    for (int f = 0; f < count; ++f)
        if (fields[f].dst) use[nf++] = fields[f];
    if (nf == 0 || n == 0) {
        hipCheck(hipStreamSynchronize(stream), "hipStreamSynchronize");
        return;
    }
    const size_t bytes = 3 * nf * sizeof(T);
    reserve(bytes, n);
    const int64_t part = perPart(bytes), parts = (n + part - 1) / part, inFlight = std::min(kParts, parts);
    T *host = static_cast<T *>(m_host);
    const size_t partValues = kPartBytes / sizeof(T);
    for (int64_t p0 = 0; p0 < parts; p0 += inFlight) {
        const int64_t now = std::min(inFlight, parts - p0);
        for (int64_t k = 0; k < now; ++k) {
            GatherArgs<T> a{};
            for (int f = 0; f < nf; ++f) {
                a.src[f] = use[f].src;
                a.stride[f] = use[f].stride;
            }
            a.order = order;
            a.first = (p0 + k) * part;
            a.n = static_cast<int32_t>(std::min(part, n - a.first));
            a.out = host + k * partValues;
            gatherKernel<T><<<dim3((3 * a.n + 255) / 256, nf), 256, 0, stream>>>(a);
            hipCheck(hipGetLastError(), "state gather launch");
            hipCheck(hipEventRecord(m_events[k], stream), "hipEventRecord");
        }
        hipCheck(hipEventSynchronize(m_events[0]), "hipEventSynchronize");
        forAll(now, kThreads, [&](int64_t k) {
            hipCheck(hipEventSynchronize(m_events[k]), "hipEventSynchronize");
            const int64_t first = (p0 + k) * part, m = std::min(part, n - first);
            for (int f = 0; f < nf; ++f) widen(host + k * partValues + f * 3 * m, use[f].dst + 3 * first, 3 * m);
        });
    }
}

template void StateReader::read<float>(const Field3<float> *, int, const int32_t *, int64_t, hipStream_t);
template void StateReader::read<double>(const Field3<double> *, int, const int32_t *, int64_t, hipStream_t);

}  // namespace spgvbd
