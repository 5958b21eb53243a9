/* The streaming call (cudec_amd/csrc/stream.cpp) over a stand-in for the HIP
 * runtime: TEST INFRASTRUCTURE ONLY. "Device" memory is host memory, a copy
 * is done where it is asked for, and a chunk "decodes" to its own bytes; what
 * the call makes and keeps is counted. Copies above kSkip bytes are left out,
 * so that staging of gigabytes can be asked for. */
#include "../cudec_amd/csrc/stream.cpp"

#include <cstdlib>
#include <unordered_map>

namespace {
constexpr size_t kSkip = size_t{256} << 20;
struct Counts {
    uint64_t streams, events; /* made */
    uint64_t held, most;      /* device bytes, now and at most */
    uint64_t open;            /* streams, events and allocations not given back */
} g_counts;
std::unordered_map<void*, size_t> g_sizes;
int g_device = 0;
hipError_t g_last = hipSuccess; /* the thread's last error */
constexpr size_t kNoMemory = size_t{1} << 40;
}  // namespace

extern "C" {

hipError_t hipGetDevice(int* d) {
    *d = g_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    g_device = d;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) {
    *s = static_cast<hipStream_t>(std::malloc(8));
    g_counts.streams++;
    g_counts.open++;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    g_counts.open--;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    return s == nullptr ? hipErrorInvalidHandle : hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = static_cast<hipEvent_t>(std::malloc(8));
    g_counts.events++;
    g_counts.open++;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    g_counts.open--;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return e == nullptr || s == nullptr ? hipErrorInvalidHandle : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    return e == nullptr ? hipErrorInvalidHandle : hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (n >= kNoMemory) {
        return g_last = hipErrorOutOfMemory;
    }
    *p = std::malloc(n);
    g_sizes[*p] = n;
    g_counts.open++;
    g_counts.held += n;
    g_counts.most = g_counts.held > g_counts.most ? g_counts.held : g_counts.most;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    g_counts.held -= g_sizes[p];
    g_counts.open--;
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
    if (n >= kNoMemory) {
        return g_last = hipErrorOutOfMemory;
    }
    *p = std::malloc(n);
    g_counts.open++;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    g_counts.open--;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (st == nullptr) {
        return hipErrorInvalidHandle;
    }
    if (n <= kSkip) {
        std::memcpy(d, s, n);
    }
    return hipSuccess;
}

cudec_status cudec_lz4_decompress_batch(const void* const* src, const size_t* sizes,
                                        void* const* dst, const size_t* caps, size_t n,
                                        cudec_chunk_result* results, cudec_stream_t) {
    for (size_t i = 0; i < n; i++) {
        const bool fits = sizes[i] <= caps[i];
        results[i].status = fits ? CUDEC_OK : CUDEC_ERR_OUTPUT_TOO_SMALL;
        results[i].reserved = 0;
        results[i].bytes_written = fits ? sizes[i] : 0;
        if (fits) {
            std::memcpy(dst[i], src[i], sizes[i]);
        }
    }
    return CUDEC_OK;
}

void host_stream_most_from_here(void) { g_counts.most = g_counts.held; }

/* What the program's next GPU call would report. */
int host_last_error(void) { return g_last; }

void host_stream_counts(uint64_t* out) { std::memcpy(out, &g_counts, sizeof(g_counts)); }

}  // extern "C"
