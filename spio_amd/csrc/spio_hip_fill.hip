// spio_hip_zero_fill_async, spio_hip_zero_fill_pair_async -- clear one or two device buffers with a kernel.
//
// The weight-gradient kernels add into grad_weight, so the buffer has to hold
// zeros when they start.  Callers without a tensor library clear it through
// this entry point.  It launches a small fill kernel rather than a runtime
// memset: a kernel node behaves the same eagerly and under HIP graph capture,
// so the call may sit inside a captured region.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "spio_hip.h"
#include "spio_hip_internal.h"

namespace {

constexpr int kFillThreads = 256;
constexpr unsigned kMaxFillBlocks = 2048;  // 8 workgroups per CU; the kernel strides over the rest

// A buffer, cut at its 16-byte boundaries: `head` bytes, `vectors` times 16 bytes, the rest.
struct Range {
    unsigned char* ptr;
    size_t bytes, head, vectors;
};

Range make_range(void* ptr, size_t bytes) {
    size_t head = static_cast<size_t>((16 - reinterpret_cast<uintptr_t>(ptr) % 16) % 16);
    if (head > bytes) head = bytes;
    return {static_cast<unsigned char*>(ptr), bytes, head, (bytes - head) / 16};
}

// Bytes before the first and after the last 16-byte boundary are written one by one (by the
// first lanes of block 0); everything between as 16-byte vectors, grid-strided.
__device__ void clear(const Range& r, size_t tid, size_t stride) {
    uint4* body = reinterpret_cast<uint4*>(r.ptr + r.head);
    for (size_t i = tid; i < r.vectors; i += stride) body[i] = uint4{0u, 0u, 0u, 0u};
    const size_t tail_begin = r.head + r.vectors * 16;
    if (tid < r.head) r.ptr[tid] = 0;
    if (tid < r.bytes - tail_begin) r.ptr[tail_begin + tid] = 0;
}

// Bound by its launch: the sums it clears are kilobytes.  Two buffers of one layer (the sums of the weight
// and of the bias gradient) therefore go in one launch; an empty second range costs a few scalar compares.
// 54 KiB and 384 bytes, back to back through the Python driver: two calls 9.0 us, one for both 4.4 us.  Of a
// training step the second launch is 1 to 2 us, which is within what its runs differ by.
__global__ void __launch_bounds__(kFillThreads) zero_fill_kernel(Range a, Range b) {
    const size_t tid = static_cast<size_t>(blockIdx.x) * kFillThreads + threadIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * kFillThreads;
    clear(a, tid, stride);
    clear(b, tid, stride);
}

}  // namespace

extern "C" int spio_hip_zero_fill_pair_async(void* first, size_t first_bytes, void* second, size_t second_bytes,
                                         void* stream) {
    if ((!first && first_bytes) || (!second && second_bytes))
        return spio_hip_set_error(SPIO_HIP_ERR_ARGUMENT, "zero fill: null pointer");
    if (!first_bytes && !second_bytes) return SPIO_HIP_OK;
    const Range a = make_range(first, first_bytes), b = make_range(second, second_bytes);
    // head and tail are shorter than 16 bytes each: the first 16 threads cover them
    const size_t vectors = a.vectors > b.vectors ? a.vectors : b.vectors;
    size_t blocks = (vectors + kFillThreads - 1) / kFillThreads;
    if (blocks < 1) blocks = 1;
    if (blocks > kMaxFillBlocks) blocks = kMaxFillBlocks;
    hipLaunchKernelGGL(zero_fill_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kFillThreads), 0,
                       static_cast<hipStream_t>(stream), a, b);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char buf[256];
        snprintf(buf, sizeof(buf), "HIP error: zero-fill launch failed: %s (%d)", hipGetErrorString(e),
                 static_cast<int>(e));
        return spio_hip_set_error(SPIO_HIP_ERR_HIP_BASE + static_cast<int>(e), buf);
    }
    return SPIO_HIP_OK;
}

extern "C" int spio_hip_zero_fill_async(void* device_ptr, size_t bytes, void* stream) {
    return spio_hip_zero_fill_pair_async(device_ptr, bytes, nullptr, 0, stream);
}
