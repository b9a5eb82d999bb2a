// k_xfer.hip -- the host-pointer entries' transfers between their pinned staging and the
// device: small ones by a kernel in the stream (pinned memory is mapped), large ones by the
// copy engines.
#include "sw_hip.h"

// 16 bytes per thread, then the last dwords
__global__ __launch_bounds__(256) void k_xfer(void *__restrict__ dst, const void *__restrict__ src, size_t n16, size_t n4) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) ((sw_u32x4 *)dst)[i] = ((const sw_u32x4 *)src)[i];
    else if (i - n16 < n4 - 4 * n16) ((uint32_t *)dst)[3 * n16 + i] = ((const uint32_t *)src)[3 * n16 + i];
}

// An engine's copy is ordered against the kernels around it by signals between queues, about
// 5 us a transfer from 64 KB or so on (below, the runtime copies by a kernel of its own); a
// kernel is ordered by the stream.  Beyond some 1 MB the engine's rate over the link is worth
// more.  Whole calls, engine / kernel: a bf16 matmul of 4096 x 4096, 2 tokens (32 KB each
// way) 45 / 34 us, 16 (256 KB) 81 / 71, 64 (1 MB) 206 / 202; an 8-expert int4 group of one row
// each (160 KB) 81 / 70; groups of 96 rows (1.9 MB) 318 / 323, of 256 (5 MB) 1,074 / 1,174.
#define XFER_KERNEL_MAX ((size_t)1 << 20)
hipError_t sw_xfer(hipStream_t st, void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    if (bytes > XFER_KERNEL_MAX || bytes % 4 || ((uintptr_t)dst | (uintptr_t)src) % 16)
        return hipMemcpyAsync(dst, src, bytes, kind, st);
    const size_t n16 = bytes / 16, n4 = bytes / 4, n = n16 + (n4 - 4 * n16);
    if (n) SW_LAUNCH(k_xfer, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dst, src, n16, n4);
    return hipGetLastError();
}
