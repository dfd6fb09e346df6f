// Outputs on their way to the caller's pageable memory.
//
// The runtime copies such memory in parts, each first over the link into pinned memory and then on
// the host, one after the other: 3 MB of outputs 176 us, where the link takes 55 and a core's copy out
// of pinned memory that the GPU has just written 105.  Here a kernel writes the outputs to pinned
// memory chunk by chunk and raises a flag behind each; the host copies a chunk as soon as its flag is
// up, and is what bounds the copy now.  A whole q4_gemm hook, us: 150 rows of 5120 outputs (3 MB)
// 240 -> 179, 400 rows 573 -> 386, 1500 rows 2045 -> 1386.  (The runtime's copies of pinned memory with an
// event behind every 512 KB took 249 at 150 rows, this kernel with an event 194; a second host thread
// gained 10 % at 30 MB and nothing at 3.)
#include <emmintrin.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <new>

#include "device_util.h"
#include "internal.h"

namespace mi355q {

constexpr uint32_t kChunkThreads = 256, kChunkLoads = 4;
constexpr uint32_t kChunkBytes = kChunkThreads * kChunkLoads * 16u;
// The two halves of the pinned memory: one is filled while the other is copied out.
constexpr size_t kHalfBytes = 2u << 20;
constexpr uint32_t kHalfChunks = kHalfBytes / kChunkBytes;
// Below, the runtime's own copy is as fast (a hook with 460 KB of outputs 84 and 82 to 87 us, 768 KB 106 and 100).
constexpr size_t kHostCopyMin = 512u << 10;
// Workgroups: enough to fill the link, few enough that the first chunks arrive well before the last
// (the 150 rows with 4, 8, 16, 32, 64, 128 of them: 242, 183, 179, 182, 194, 218 us).
constexpr uint32_t kCopyGroups = 16;

struct HostOutputs {
    unsigned char *memory;   // two halves, pinned
    uint64_t *flags;         // one a chunk, pinned: the number of the last copy that has filled it
    uint64_t copies[2];      // of each half so far (64 bits: a number never comes again)
};

// bytes <= kHalfBytes from `from` (16-byte aligned) to `to`.
__global__ void __launch_bounds__(kChunkThreads) host_chunks_kernel(unsigned char *to, const unsigned char *from, uint32_t bytes,
                                                                   uint64_t *flags, uint64_t number)
{
    for (uint32_t chunk = blockIdx.x; chunk * kChunkBytes < bytes; chunk += gridDim.x) {
        const uint32_t begin = chunk * kChunkBytes, end = bytes - begin < kChunkBytes ? bytes : begin + kChunkBytes;
        u32x4 piece[kChunkLoads] = {};
#pragma unroll
        for (uint32_t i = 0; i < kChunkLoads; ++i) {
            const uint32_t at = begin + (i * kChunkThreads + threadIdx.x) * 16u;
            if (at + 16u <= end) piece[i] = *(const u32x4 *)(from + at);
        }
#pragma unroll
        for (uint32_t i = 0; i < kChunkLoads; ++i) {
            const uint32_t at = begin + (i * kChunkThreads + threadIdx.x) * 16u;
            if (at + 16u <= end) *(u32x4 *)(to + at) = piece[i];
        }
        const uint32_t rest = end & ~15u;  // (all but the last chunk end at a multiple of 16)
        if (rest + threadIdx.x < end) to[rest + threadIdx.x] = from[rest + threadIdx.x];
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0u) __hip_atomic_store(flags + chunk, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

void host_outputs_free(mi355q_context *ctx)
{
    HostOutputs *const outputs = ctx->host_outputs;
    if (outputs == nullptr) return;
    if (outputs->memory) (void)hipHostFree(outputs->memory);
    if (outputs->flags) (void)hipHostFree(outputs->flags);
    delete outputs;
    ctx->host_outputs = nullptr;
}

// Whether a copy takes this way: a large one, to memory that the runtime does not know (it reaches pinned
// and managed memory directly), outside of a graph's recording, from 16-byte aligned memory (every output's
// place in a staging buffer is).  The pinned memory is made on the first such copy and kept by the context; without
// it the runtime's copy does it.
static bool host_outputs_serve(mi355q_context *ctx, const void *host, const void *device, size_t bytes)
{
    if (bytes < kHostCopyMin || ctx->capturing || (uintptr_t)device % 16u != 0u) return false;
    hipPointerAttribute_t known;
    if (hipPointerGetAttributes(&known, host) != hipSuccess)
        (void)hipGetLastError();
    else if (known.type != hipMemoryTypeUnregistered)
        return false;
    if (ctx->host_outputs != nullptr) return true;
    HostOutputs *const outputs = new (std::nothrow) HostOutputs();
    if (outputs == nullptr) return false;
    ctx->host_outputs = outputs;
    hipError_t status = hipHostMalloc((void **)&outputs->memory, 2u * kHalfBytes, hipHostMallocCoherent);
    if (status == hipSuccess)
        status = hipHostMalloc((void **)&outputs->flags, 2u * kHalfChunks * sizeof(uint64_t), hipHostMallocCoherent);
    if (status == hipSuccess) {
        memset(outputs->flags, 0, 2u * kHalfChunks * sizeof(uint64_t));
        return true;
    }
    (void)hipGetLastError();
    host_outputs_free(ctx);
    return false;
}

// Waits for a chunk's flag; a stream that has ended, or failed, without raising it is an error.
static hipError_t wait_for_flag(hipStream_t stream, const uint64_t *flag, uint64_t number)
{
    for (;;) {
        for (uint32_t poll = 0; poll < 4096u; ++poll) {
            if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == number) return hipSuccess;
            _mm_pause();
        }
        const hipError_t status = hipStreamQuery(stream);
        if (status == hipErrorNotReady) {
            (void)hipGetLastError();
            continue;
        }
        if (status != hipSuccess) return status;
        return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == number ? hipSuccess : hipErrorUnknown;
    }
}

hipError_t copy_outputs(mi355q_context *ctx, void *host, const void *device, size_t bytes)
{
    if (!host_outputs_serve(ctx, host, device, bytes))
        return hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, ctx->stream);
    if (ctx->trace) fprintf(stderr, "mi355q: host outputs, %zu bytes in chunks of %u\n", bytes, kChunkBytes);
    HostOutputs &outputs = *ctx->host_outputs;
    const size_t parts = (bytes + kHalfBytes - 1) / kHalfBytes;  // part i passes through half i % 2
    auto part_bytes = [&](size_t i) { return (uint32_t)std::min(kHalfBytes, bytes - i * kHalfBytes); };
    auto send = [&](size_t i) {
        const size_t half = i % 2u;
        hipLaunchKernelGGL(host_chunks_kernel, dim3(kCopyGroups), dim3(kChunkThreads), 0, ctx->stream,
                           outputs.memory + half * kHalfBytes, (const unsigned char *)device + i * kHalfBytes, part_bytes(i),
                           outputs.flags + half * kHalfChunks, ++outputs.copies[half]);
        return hipGetLastError();
    };
    hipError_t status = send(0);
    if (status == hipSuccess && parts > 1u) status = send(1);
    for (size_t i = 0; i < parts && status == hipSuccess; ++i) {
        const size_t half = i % 2u;
        const uint32_t size = part_bytes(i);
        for (uint32_t at = 0, chunk = 0; at < size && status == hipSuccess; at += kChunkBytes, ++chunk) {
            status = wait_for_flag(ctx->stream, outputs.flags + half * kHalfChunks + chunk, outputs.copies[half]);
            if (status == hipSuccess)
                memcpy((unsigned char *)host + i * kHalfBytes + at, outputs.memory + half * kHalfBytes + at,
                       std::min(kChunkBytes, size - at));
        }
        if (status == hipSuccess && i + 2u < parts) status = send(i + 2u);
    }
    if (status != hipSuccess) (void)hipStreamSynchronize(ctx->stream);  // nothing may land in the halves any more
    return status;
}

}  // namespace mi355q
