// Transfers between the engine's device buffers and host memory for calls that work on host arrays.
// A blocking copy of a few kilobytes costs about 13 us whatever its size, and a chunk has four arrays
// and a record: one kernel writes them all into page-locked memory, and the call waits once.
#include <hip/hip_runtime.h>

#include "uw_host.h"

namespace {

constexpr int kCopyThreads = 256;
constexpr size_t kPinnedMax = size_t(16) << 20;  // largest page-locked buffer kept by a context

template <class T>
__device__ __forceinline__ void copy_as(const void* src, void* dst, uint64_t n, uint64_t i, uint64_t step) {
    for (; i < n; i += step) static_cast<T*>(dst)[i] = static_cast<const T*>(src)[i];
}

// Sizes and addresses are multiples of 2 (u16 indices); wider words where all of them allow it.
__global__ void __launch_bounds__(kCopyThreads) k_copy(uw_copies c) {
    const uint64_t i = uint64_t(blockIdx.x) * kCopyThreads + threadIdx.x, step = uint64_t(gridDim.x) * kCopyThreads;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint64_t bits = reinterpret_cast<uint64_t>(c.src[k]) | reinterpret_cast<uint64_t>(c.dst[k]) | c.bytes[k];
        if ((bits & 15u) == 0u) copy_as<uint4>(c.src[k], c.dst[k], c.bytes[k] / 16, i, step);
        else if ((bits & 3u) == 0u) copy_as<uint32_t>(c.src[k], c.dst[k], c.bytes[k] / 4, i, step);
        else copy_as<uint16_t>(c.src[k], c.dst[k], c.bytes[k] / 2, i, step);
    }
}

// One chunk's record and, if they fit `cap` bytes, its arrays behind it (uw_mesh_sections).
__global__ void __launch_bounds__(kCopyThreads) k_chunk_out(const uw_chunk_info* __restrict__ info, uw_mesh_ptrs m,
                                                            uw_mesh_format f, unsigned char* __restrict__ dst, uint64_t cap) {
    const uw_chunk_info ci = *info;
    const uw_mesh_sections s = uw_sections(ci.n_verts, ci.n_inds, f);
    const uint64_t i = uint64_t(blockIdx.x) * kCopyThreads + threadIdx.x, step = uint64_t(gridDim.x) * kCopyThreads;
    if (i == 0) *reinterpret_cast<uw_chunk_info*>(dst) = ci;
    if (kMeshHeader + s.total > cap) return;
    // whole words: the sections start at multiples of 256, and the sources are as long as the worst case
#pragma unroll
    for (int k = 0; k < 4; ++k) copy_as<uint32_t>(m.p[k], dst + kMeshHeader + s.off[k], (s.bytes[k] + 3) / 4, i, step);
}

__global__ void k_set_coord(int32_t* p, int32_t x, int32_t y, int32_t z) {
    if (threadIdx.x == 0) {
        p[0] = x;
        p[1] = y;
        p[2] = z;
    }
}

uint32_t copy_blocks(const uw_ctx* ctx, uint64_t bytes) {
    const uint64_t b = (bytes + 16 * kCopyThreads - 1) / (16 * kCopyThreads), most = uint64_t(ctx->num_cus) * 4;
    return uint32_t(b < 1 ? 1 : b > most ? most : b);
}

}  // namespace

bool uw_pinned(uw_ctx* ctx, size_t bytes, unsigned char** p) {
    *p = nullptr;
    if (bytes > kPinnedMax) return false;
    if (bytes > ctx->pinned_bytes) {
        if (bytes < ctx->pinned_bytes * 2) bytes = ctx->pinned_bytes * 2 < kPinnedMax ? ctx->pinned_bytes * 2 : kPinnedMax;
        if (ctx->h_pinned) (void)hipHostFree(ctx->h_pinned);
        ctx->h_pinned = nullptr;
        ctx->pinned_bytes = 0;
        if (hipHostMalloc(reinterpret_cast<void**>(&ctx->h_pinned), bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            ctx->h_pinned = nullptr;
            return false;
        }
        ctx->pinned_bytes = bytes;
    }
    *p = ctx->h_pinned;
    return true;
}

int uw_copy_launch(uw_ctx* ctx, const uw_copies& c, hipStream_t st) {
    uint64_t most = 0;
    for (int k = 0; k < 4; ++k) most = c.bytes[k] > most ? c.bytes[k] : most;
    if (most == 0) return UW_OK;
    hipLaunchKernelGGL(k_copy, dim3(copy_blocks(ctx, most)), dim3(kCopyThreads), 0, st, c);
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_chunk_out_launch(uw_ctx* ctx, const uw_chunk_info* info, const uw_mesh_ptrs& m, const uw_mesh_format& f,
                        unsigned char* dst, uint64_t cap, hipStream_t st) {
    hipLaunchKernelGGL(k_chunk_out, dim3(32), dim3(kCopyThreads), 0, st, info, m, f, dst, cap);
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_set_coord_launch(uw_ctx* ctx, int32_t* d_coord, int32_t x, int32_t y, int32_t z, hipStream_t st) {
    hipLaunchKernelGGL(k_set_coord, dim3(1), dim3(64), 0, st, d_coord, x, y, z);
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_device_alloc(uw_ctx* ctx, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && uw_blocks_release(ctx)) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    if (e == hipSuccess) return UW_OK;
    *p = nullptr;
    return uw_hip_fail(ctx, e, "hipMalloc");
}

int uw_block_take(uw_ctx* ctx, size_t bytes, void** out, size_t* got) {
    bytes = uw_block_pool::rounded(bytes);
    {
        std::lock_guard<std::mutex> lock(ctx->blocks_lock);
        uw_block b;
        if (ctx->blocks.take(bytes, &b)) {
            *got = b.bytes;
            *out = b.p;
            return UW_OK;
        }
    }
    const int rc = uw_device_alloc(ctx, out, bytes);
    *got = rc == UW_OK ? bytes : 0;
    return rc;
}

void uw_block_give(uw_ctx* ctx, void* p, size_t bytes) {
    if (!p) return;
    std::lock_guard<std::mutex> lock(ctx->blocks_lock);
    ctx->blocks.give(uw_block{p, bytes}, [](const uw_block& b) { (void)hipFree(b.p); });
}

bool uw_blocks_release(uw_ctx* ctx) {
    std::lock_guard<std::mutex> lock(ctx->blocks_lock);
    return ctx->blocks.clear([](const uw_block& b) { (void)hipFree(b.p); });
}

void uw_host_release(uw_ctx* ctx) {
    uw_blocks_release(ctx);
    if (ctx->h_pinned) (void)hipHostFree(ctx->h_pinned);
    ctx->h_pinned = nullptr;
    ctx->pinned_bytes = 0;
}
