// Host transfers (uw_host.hip): a page-locked buffer per context, kernels that gather a call's arrays into
// it (or scatter them out of it), and the context's kept device blocks.
#pragma once

#include "uw_internal.h"

// Up to four arrays copied by one kernel; addresses and sizes multiples of 2, page-locked or device memory.
struct uw_copies {
    const void* src[4];
    void* dst[4];
    uint64_t bytes[4];
};

// Arrays of a mesh: vertices, indices, collision normals, collision cells (null: not asked for).
struct uw_mesh_ptrs {
    const void* p[4];
};
struct uw_mesh_format {
    uint32_t vert_bytes, ind_bytes, normals, cells;  // bytes per vertex and index; whether collision arrays are there
};
struct uw_mesh_sections {
    uint64_t off[4], bytes[4], total;
};
constexpr uint64_t kMeshHeader = 256;
__host__ __device__ inline uw_mesh_sections uw_sections(uint64_t nv, uint64_t ni, const uw_mesh_format& f) {
    uw_mesh_sections s;
    const uint64_t ntri = ni / 3;
    s.bytes[0] = nv * f.vert_bytes;
    s.bytes[1] = ni * f.ind_bytes;
    s.bytes[2] = f.normals ? ntri * 12 : 0;
    s.bytes[3] = f.cells ? ntri * 4 : 0;
    uint64_t o = 0;
    for (int k = 0; k < 4; ++k) {
        s.off[k] = o;
        o += (s.bytes[k] + 255) & ~uint64_t(255);
    }
    s.total = o;
    return s;
}

// Holds ctx->host_lock while a call uses the page-locked buffer. Kernels on the null stream read and write
// the buffer: a call that leaves before it has waited for them (an error) waits here, before the lock is
// given up and the next holder writes the buffer, or grows it.
struct uw_pinned_use {
    std::unique_lock<std::mutex> lock;
    bool pending = false;  // a kernel that uses the buffer may still run
    explicit uw_pinned_use(uw_ctx* ctx) : lock(ctx->host_lock) {}
    ~uw_pinned_use() {
        if (pending) (void)hipStreamSynchronize(nullptr);
    }
};
// The context's page-locked buffer with room for `bytes`, kept and grown to at most 16 MiB; false where
// it can't be had (the caller copies directly). The caller holds a uw_pinned_use while it uses the buffer.
bool uw_pinned(uw_ctx* ctx, size_t bytes, unsigned char** p);
int uw_copy_launch(uw_ctx* ctx, const uw_copies& c, hipStream_t st);
int uw_chunk_out_launch(uw_ctx* ctx, const uw_chunk_info* info, const uw_mesh_ptrs& m, const uw_mesh_format& f,
                        unsigned char* dst, uint64_t cap, hipStream_t st);
int uw_set_coord_launch(uw_ctx* ctx, int32_t* d_coord, int32_t x, int32_t y, int32_t z, hipStream_t st);

// Device blocks kept by the context between uses (uw_blocks.h; freed with it). A block may still be read
// by work queued before it was given back: a taker synchronises the device after the take and before it
// writes.
int uw_block_take(uw_ctx* ctx, size_t bytes, void** out, size_t* got);
void uw_block_give(uw_ctx* ctx, void* p, size_t bytes);
// Frees the kept blocks; whether there were any.
bool uw_blocks_release(uw_ctx* ctx);
void uw_host_release(uw_ctx* ctx);
