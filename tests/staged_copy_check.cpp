// Host-side check of the staged device-to-host copy
// (stencil_benchmarks_amd/csrc/runtime.hip), with the HIP calls it makes
// replaced by host ones: a copy is whole where a worker cannot be started, and
// one that fails says so and leaves no error for the next call to report.
// Exits non-zero on the first that does not.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../stencil_benchmarks_amd/csrc/runtime.hip"

namespace sb {
void vadv_noalloc_setup(Context &) {}
}  // namespace sb

// ---- the host in place of the device ------------------------------------
static thread_local hipError_t t_last = hipSuccess;
static thread_local bool t_fail_copies = false;
static thread_local long t_allocations_left = -1;  // -1: no limit

void *operator new(size_t n) {
    if (t_allocations_left == 0) throw std::bad_alloc();
    if (t_allocations_left > 0) --t_allocations_left;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
int sched_getaffinity(pid_t, size_t, cpu_set_t *set) noexcept {
    for (int c = 0; c < 8; ++c) CPU_SET(c, set);
    return 0;
}
hipError_t hipGetDevice(int *device) { *device = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    std::memset(p, 0, sizeof(*p));
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(1);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) {
    return t_last = hipErrorInvalidValue;  // pageable memory is unknown to the runtime
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    if (t_fail_copies) return t_last = hipErrorUnknown;
    std::memcpy(dst, src, n);
    return hipSuccess;
}
}  // extern "C"

int main() {
    constexpr size_t kBytes = (size_t(41) << 20) + 13;
    char *src = static_cast<char *>(std::malloc(kBytes)), *dst = static_cast<char *>(std::malloc(kBytes));
    for (size_t i = 0; i < kBytes; ++i) src[i] = char(i * 2654435761u >> 13);
    // allocations that may succeed while the workers are started
    for (long left : {-1L, 0L, 1L, 2L, 3L}) {
        std::memset(dst, 0, kBytes);
        if (sb_memcpy_d2h(dst, src, 1)) return 1;  // the device's context, before the limit
        t_allocations_left = left;
        const int status = sb_memcpy_d2h(dst, src, kBytes);
        t_allocations_left = -1;
        if (status || std::memcmp(dst, src, kBytes)) {
            std::printf("copy with %ld allocations: status %d\n", left, status);
            return 1;
        }
    }
    t_fail_copies = true;
    const int status = sb_memcpy_d2h(dst, src, kBytes);
    t_fail_copies = false;
    if (status == 0 || std::strlen(sb_last_error()) == 0) {
        std::printf("a failed copy reported status %d\n", status);
        return 1;
    }
    if (const hipError_t left = hipGetLastError(); left != hipSuccess) {
        std::printf("a failed copy left error %d behind\n", int(left));
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
