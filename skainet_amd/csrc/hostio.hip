// Copies between device memory and this library's page-locked host buffers made by a kernel on the caller's stream, with a
// completion flag the host polls. What they replace is a copy-engine transfer plus hipStreamSynchronize: the hand-over
// between the compute queue and a copy engine and the interrupt-driven wait cost more than a small payload itself.
#include "common.h"

namespace skh {

// 16 bytes per thread and turn where both sides are 16-byte aligned, else bytes. With `flag` the last workgroup to finish
// publishes `ticket` there (page-locked host memory). Stores to page-locked memory are not held in any GPU cache, so a
// workgroup's bytes are out once its waves' store counters have drained; the release of the flag then orders them for the
// host (a system-scope fence per wave instead, which writes back whole L2s, cost 1.5 us more). One workgroup of 1024
// threads moves up to 32 KB: a second one would pay an atomic round trip to agree on who is last. The counter is left at
// zero for the next copy.
constexpr int HC_THREADS = 1024;
__global__ __launch_bounds__(HC_THREADS) void host_copy_kernel(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, int64_t bytes,
                                                               int wide, uint32_t* counter, uint32_t* flag, uint32_t ticket) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, threads = (int64_t)gridDim.x * blockDim.x;
    if (wide) {
        const int64_t n16 = bytes >> 4;
        for (int64_t i = tid; i < n16; i += 2 * threads) {
            const bool more = i + threads < n16;
            const uint4 a = reinterpret_cast<const uint4*>(src)[i], b = reinterpret_cast<const uint4*>(src)[more ? i + threads : i];
            reinterpret_cast<uint4*>(dst)[i] = a;
            if (more) reinterpret_cast<uint4*>(dst)[i + threads] = b;
        }
        for (int64_t i = (n16 << 4) + tid; i < bytes; i += threads) dst[i] = src[i];
    } else {
        for (int64_t i = tid; i < bytes; i += threads) dst[i] = src[i];
    }
    if (!flag) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (gridDim.x > 1) {
            if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1) return;
            __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __hip_atomic_store(flag, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

int launch_host_copy(void* dst, const void* src, size_t bytes, uint32_t* counter, uint32_t* flag, uint32_t ticket) {
    const int wide = ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0;
    const size_t per_group = wide ? 2 * 16 * HC_THREADS : 4 * HC_THREADS;
    size_t grid = (bytes + per_group - 1) / per_group;
    if (grid > 64) grid = 64;
    if (grid < 1) grid = 1;
    // small copies take no more waves than they have pieces
    const size_t items = wide ? (bytes + 15) / 16 : bytes;
    const unsigned threads = items >= HC_THREADS ? HC_THREADS : (unsigned)((items + 63) / 64 * 64);   // at least one item: bytes > 0
    host_copy_kernel<<<dim3((unsigned)grid), dim3(threads), 0, current_stream()>>>(
        static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src), (int64_t)bytes, wide, counter, flag, ticket);
    SKH_CHECK(hipGetLastError());
    return 0;
}

}  // namespace skh
