// Bulk path of the batched build: chunks of at least `bulk_min` cells per axis (1, the default: all of
// them) leave the persistent queue. One workgroup per chunk runs its density, classification and emission
// as a serial chain; here every phase is spread over the device instead:
//
//   k_bulk_density  one lane per z-line (lanes on consecutive lines t = x L + y of one chunk),
//                   densities into a per-chunk HBM field [z][t], so each sample's store is a row,
//                   and the lines' sign words (uw_rows.h)
//   k_bulk_rows     one wave per chunk: vertex records and triangles of the
//                   chunk's cell rows from the sign words, their scan (first-seen order within the
//                   chunk), its totals and record; the workgroup's chunks reserve their vertex and
//                   index ranges with one atomic on the launch's range counter (the persistent
//                   kernel's reservations use the same counter, so ranges never overlap); the
//                   chunk's tiles with triangles go into a list per size class
//   k_bulk_emit     persistent workgroups over the listed tiles, most triangles first: vertices,
//                   indices and, when requested, tape, colours and collision records (uw_emit_rows)
//
// The queue set-up (k_prep / k_place in uw_batched.hip) sorts chunks by resolution, largest first,
// so the bulk chunks are the first `nbig` queue entries; k_place publishes nbig in the queue state
// and starts the persistent kernel's queue after them. Output (vertex numbering, index order,
// records) is that of the persistent and plain paths, chunk by chunk.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>

#include "uw_mesh.h"
#include "uw_noise.h"
#include "uw_queue.h"
#include "uw_rows.h"
#include "uw_wave.h"

namespace {

constexpr int kMaxN = UW_BATCH_MAX_RESOLUTION;
static_assert(kMaxN <= 32, "one row segment per cell row");
// Launches whose chunks all take the bulk path in at most this many density items each don't need the
// queue's order: k_prep places them by itself and k_place (4.7 us) is left out, at the price of visiting
// the empty items of smaller chunks. 4096 chunks of 12^3 (3 items of 64 lines) take 72.2 us, in queue order
// 76.7 and on the persistent kernel 84.5; 4000 of 3 .. 21 cells 101 and in queue order 105. Chunks of 32^3
// have 9 items: those of smaller chunks are mostly empty, each a dependent load that the order skips.
constexpr int32_t kAnyOrderItems = 4;
constexpr size_t kBulkScratchMax = size_t(8) << 30;  // 8 GiB: about 55,000 chunks at max_res 32
// Distinct x values among `block` consecutive lines t = x L + y of a chunk with L samples per axis, at most.
constexpr int bulk_nx_tab(int32_t L, int block) { return (block - 1) / L + 2; }

struct BulkArgs {
    uw_field f;
    const uw_tables* tab;
    const uw_task* tasks;
    uint32_t* qhead;            // queue state: bulk entry count, range, exit and tile counters
    int32_t max_res;            // largest resolution of the launch (sizes the per-chunk slots)
    int32_t Lm;                 // max_res + 1
    int32_t wpc;                // density workgroup items per chunk: ceil(Lm^2 / the density workgroup's threads)
    int32_t tile_rows;          // row segments per emission tile, about (uw_slab_tiling)
    int32_t max_tiles;          // tiles of a chunk, at most
    uint64_t list_cap;          // tiles per size class, at most
    int32_t any_order;          // 1: entries are not sorted by resolution
    int32_t all;                // 1: no persistent kernel in this launch (the totals are written here)
    const unsigned char* ztab;  // per-chunk z tables written by k_prep
    int32_t zstride;
    int32_t packed;
    float* dens;                  // [j][Lm^3], chunk layout [z][t] with the chunk's own L
    uint32_t* words;              // [j][Lm^2 words(Lm)]: sign words, the chunk's own layout
    unsigned long long* rows;     // [j][max_res^2 + 1]: scanned rows (x n + y) and the totals
    uint32_t* below;              // [j] early-blank bits, zeroed by the queue set-up
    unsigned long long* rec;      // [j][4]: vertex base, index base, vertices, indices
    uint32_t* list;               // [class][list_cap]: j max_tiles + tile
    uw_chunk_info* info;
    uw_totals* totals;
    float* verts;
    uint32_t* inds;
    uw_vertex_tape* tape;
    uw_emit_opts eo;
    uint64_t vcap, icap;
};

__device__ __forceinline__ uint32_t bulk_count(const BulkArgs& a) { return *uw_queue_bulk_count(a.qhead); }
__device__ __forceinline__ float* bulk_dens(const BulkArgs& a, uint32_t j) {
    return a.dens + uint64_t(j) * uint64_t(a.Lm) * a.Lm * a.Lm;
}
__device__ __forceinline__ uint32_t* bulk_words(const BulkArgs& a, uint32_t j) {
    return a.words + uint64_t(j) * uint64_t(a.Lm * a.Lm * uw_sign_words(a.Lm));
}
__device__ __forceinline__ unsigned long long* bulk_rows(const BulkArgs& a, uint32_t j) {
    return a.rows + uint64_t(j) * uint64_t(a.max_res * a.max_res + 1);
}

__device__ __forceinline__ void load_task(const BulkArgs& a, uint32_t j, int32_t* c, int32_t* n, int32_t* cx,
                                          int32_t* cy, int32_t* cz) {
    const int4* p = reinterpret_cast<const int4*>(a.tasks + j);
    const int4 r0 = p[0];
    const int4 r1 = p[1];
    *c = __builtin_amdgcn_readfirstlane(r0.x);
    *n = __builtin_amdgcn_readfirstlane(r0.y);
    *cx = __builtin_amdgcn_readfirstlane(r0.z);
    *cy = __builtin_amdgcn_readfirstlane(r0.w);
    *cz = __builtin_amdgcn_readfirstlane(r1.x);
}

// ---------------------------------------------------------------------------------------------
// Densities and sign words. An item is BLOCK lines of a chunk: 128, or 64 where the launch's largest
// chunks leave a fifth of 128-line items idle (bulk_density_block). Small items leave few lanes idle
// (32^3 has 1089 lines: 18 waves of 64 lines where items of 256 take 20) and let no wave wait for many
// others, against the y entries of the chunk (L per octave) and the x entries of the item's lines,
// which every item computes into LDS by chains of f64 operations. 8192 chunks of 8 .. 32 cells took
// 370 us at 256 lines, 300 at 128 and 321 at 64; 4096 of 12^3 (169 lines) 46.7, 41.1 and 31.8. Bound by
// vector instructions.
template <int OCT, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_bulk_density(BulkArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int32_t O = uw_octaves<OCT>::count(a.f);
    uint2* GH = reinterpret_cast<uint2*>(smem);  // uw_grad_half of every slot
    uint8_t* P = reinterpret_cast<uint8_t*>(GH + 256);
    const int32_t pitch = uw_axis_pitch(O);
    uw_axis* AYs = reinterpret_cast<uw_axis*>(P + 256);  // [L][pitch]: the chunk's y entries
    __shared__ double s_freq[UW_MAX_OCTAVES];
    // item = (BLOCK lines wb of a chunk) nbig + chunk: the first lines of every chunk first, the short
    // or empty last ones at the end. (Chunk-major, a grid that is a multiple of wpc gave every
    // workgroup the same wb throughout: two of five had next to nothing to do.)
    const uint32_t nbig = bulk_count(a), items = nbig * uint32_t(a.wpc);
    if (blockIdx.x >= items) return;
    const int tid = threadIdx.x;
    for (int i = tid; i < 256; i += BLOCK) {
        const uint8_t p = a.tab->perm[i];
        P[i] = p;
        GH[i] = uw_grad_half(p & 15u);
    }
    if (tid < UW_MAX_OCTAVES) s_freq[tid] = a.f.octave_freq[tid];
    const int32_t rw = OCT > 0 ? uw_zrec_words(OCT) : uw_zrec_words(O);
    const float iso = a.f.iso;
    for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
        const uint32_t wb = item / nbig, j = item - wb * nbig;
        int32_t c, n, cx, cy, cz;
        load_task(a, j, &c, &n, &cx, &cy, &cz);
        if (n < 1 || n > a.max_res) continue;
        const int32_t L = n + 1, lines = L * L, t0 = int32_t(wb) * BLOCK;
        if (t0 >= lines) {  // entries come largest first (else any_order): no later one has these lines
            if (!a.any_order) item += (nbig - j - 1) / gridDim.x * gridDim.x;
            continue;
        }
        // (most of a chunk's items find their bits set; read early, its latency is the walk's)
        const uint32_t seen = __hip_atomic_load(a.below + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();  // the previous item's tables are read no more
        const uw_divider dL = uw_make_divider(uint32_t(L));
        const int32_t t = t0 + tid;
        const bool valid = t < lines;
        const int32_t xfirst = int32_t(uw_div(uint32_t(t0), dL));
        const int32_t x = valid ? int32_t(uw_div(uint32_t(t), dL)) : xfirst, y = valid ? t - x * L : 0;
        const int32_t nx = int32_t(uw_div(uint32_t(min(t0 + BLOCK, lines) - 1), dL)) - xfirst + 1;
        const float step = float(a.f.extent) / float(n);
        uw_axis* AXs = AYs + L * pitch;  // [nx][pitch]: the item's x entries
        const uw_divider dnx = uw_make_divider(uint32_t(nx));
        for (int e = tid; e < O * (L + nx); e += BLOCK) {
            if (e < O * L) {
                const int32_t k = int32_t(uw_div(uint32_t(e), dL)), i = e - k * L;
                AYs[i * pitch + k] = uw_axis_of(uw_sample_coord(a.f, 1, cy, i, step), s_freq[k]);
            } else {
                const int32_t q = e - O * L, k = int32_t(uw_div(uint32_t(q), dnx)), i = q - k * nx;
                AXs[i * pitch + k] = uw_hash_x(uw_axis_of(uw_sample_coord(a.f, 0, cx, xfirst + i, step), s_freq[k]), P);
            }
        }
        __syncthreads();
        const uw_ztab Zt = uw_ztab_of(a.ztab, c, O, a.zstride);
        const uw_axis* ax = AXs + (x - xfirst) * pitch;
        const uw_axis* ay = AYs + y * pitch;
        float* out = bulk_dens(a, j) + t;
        float vmin = INFINITY, vmax = -INFINITY;
        const int32_t WL = uw_sign_words(L);
        uint32_t word = 0, first = 0;
        uw_noise_zline<OCT, false>(
            a.f, [=](int k) { return ax[k]; }, [=](int k) { return ay[k]; }, P, GH, Zt.rec, rw, L, vmin,
            vmax, [&](int32_t iz, float rho) {
                if (valid) out[iz * lines] = rho;
                word = uw_push_sign(word, rho, iso);
                if (iz == 31) {  // uniform: the first word of a line of 32 or 33 samples
                    first = word;
                    word = 0;
                }
            });
        const int32_t rest = L & 31;  // samples of the last word (0: 32 of them)
        uint32_t* wout = bulk_words(a, j) + t * WL;
        const uint32_t full = rest ? (1u << rest) - 1u : 0u;
        const uint32_t lt = word | first, ge = (word ^ full) | (L > 31 ? ~first : 0u);
        if (valid) {
            if (L > 31) wout[0] = __brev(first);
            if (rest) wout[WL - 1] = __brev(word) >> (32 - rest);
        }
        const uint32_t bits = (__any(valid && vmin <= iso) ? UW_BELOW_NOT_ABOVE : 0u) | (__any(valid && lt) ? UW_BELOW_LT : 0u) |
                              (__any(valid && ge) ? UW_BELOW_GE : 0u);
        if ((tid & 63) == 0 && (bits & ~seen)) atomicOr(a.below + j, bits);
    }
}

// ---------------------------------------------------------------------------------------------
// Row counts, scans, records and range reservations: one wave per bulk entry; a workgroup's
// chunks reserve their ranges with one atomic for their sum, each chunk's range following from its
// prefix among them. The range counter is the launch's one contended address (the memory-side atomic
// unit serialises it, about 20 ns an atomic). The tiles with triangles are listed by size class, a
// counter per class on a line of its own, one atomic per class and workgroup.
// Workgroups of 4 chunks spread a launch of up to 1024 chunks over the compute units (256 chunks of
// 24^3: 17.9 us on 16 of them); larger launches take 16 per workgroup and a quarter of the atomics.
template <int W>
__global__ void __launch_bounds__(64 * W) k_bulk_rows(BulkArgs a) {
    constexpr int kRowsWaves = W, kRowsBlock = 64 * W;
    extern __shared__ __align__(16) uint32_t s_tiles[];  // [waves][max_tiles]: triangles per tile
    __shared__ uint32_t lut[256];
    __shared__ unsigned long long s_tot[kRowsWaves];  // per wave: its chunk's vertices | indices << 32 (0: none)
    __shared__ unsigned long long s_vo, s_io;
    __shared__ uint32_t s_count[kTileClasses], s_first[kTileClasses];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t nbig = bulk_count(a), j0 = blockIdx.x * uint32_t(kRowsWaves);
    if (j0 >= nbig) return;
    const uint32_t j = __builtin_amdgcn_readfirstlane(j0 + uint32_t(wave));
    unsigned long long* resv = uw_queue_resv(a.qhead);
    const int32_t listed = kRowsWaves * a.max_tiles;
    int32_t c = 0, n = 0, cx, cy, cz;
    uint32_t sb = 0, act = 0;
    if (j < nbig) {  // wave-uniform
        load_task(a, j, &c, &n, &cx, &cy, &cz);
        sb = a.below[j];
    }
    for (int i = tid; i < 256; i += kRowsBlock) lut[i] = a.tab->cell[i];
    if (tid < kTileClasses) s_count[tid] = 0u;
    for (int32_t i = tid; i < listed; i += kRowsBlock) s_tiles[i] = 0u;
    __syncthreads();
    const bool valid = n >= 1 && n <= a.max_res;
    unsigned long long tot = 0;
    if (valid && (sb & UW_BELOW_LT) && (sb & UW_BELOW_GE))
        tot = uw_wave_rows(bulk_words(a, j), n, lut, bulk_rows(a, j), &act, uw_slab_tiling(n, a.tile_rows).planes,
                           s_tiles + wave * a.max_tiles);
    const uint32_t nv = uint32_t(tot), ni = 3u * uint32_t(tot >> 32);
    if (lane == 0) s_tot[wave] = (unsigned long long)nv | ((unsigned long long)ni << 32);
    __syncthreads();
    if (tid == 0) {
        unsigned long long all = 0;
        uint32_t nonblank = 0;
#pragma unroll
        for (int w = 0; w < kRowsWaves; ++w) {
            all += s_tot[w];
            nonblank += s_tot[w] ? 1u : 0u;
        }
        unsigned long long vo = 0, io = 0;
        if (all) {
            const uint32_t av = uint32_t(all & 0xFFFFFFFFull), ai = uint32_t(all >> 32);
            if (a.packed) {
                const unsigned long long old = atomicAdd(resv, all);
                vo = old & 0xFFFFFFFFull;
                io = old >> 32;
            } else {
                vo = atomicAdd(resv, (unsigned long long)av);
                io = atomicAdd(resv + kResvIndsOffset, (unsigned long long)ai);
            }
            atomicAdd(resv + kExitOffset, (unsigned long long)nonblank << 32);  // non-blank chunks of the launch
        }
        s_vo = vo;
        s_io = io;
    }
    for (int32_t i = tid; i < listed; i += kRowsBlock)
        if (s_tiles[i]) atomicAdd(&s_count[uw_tile_class(s_tiles[i])], 1u);
    __syncthreads();
    bool over = false;
    if (j < nbig) {
        unsigned long long pre = 0;
        for (int w = 0; w < wave; ++w) pre += s_tot[w];
        const unsigned long long vo = ni ? s_vo + (pre & 0xFFFFFFFFull) : 0ull, io = ni ? s_io + (pre >> 32) : 0ull;
        over = ni > 0 && (vo + nv > a.vcap || io + ni > a.icap);
        if (lane == 0) {
            uint32_t flags = 0;
            if (!valid) flags = UW_CHUNK_INVALID | UW_CHUNK_BLANK;
            else if (!(sb & UW_BELOW_NOT_ABOVE)) flags = UW_CHUNK_BLANK | UW_CHUNK_EARLY_SKIP;
            else if (ni == 0) flags = UW_CHUNK_BLANK;
            if (over) {
                flags |= UW_CHUNK_OVERFLOW;
                atomicOr(&a.totals->overflow, 1u);
            }
            if (a.eo.ind16 && nv > 65535u) flags |= UW_CHUNK_INDEX_WRAP;
            uw_chunk_info r = {flags, nv, ni, act, vo, io};
            a.info[c] = r;
            unsigned long long* rec = a.rec + 4 * uint64_t(j);
            rec[0] = over ? ~0ull : vo;  // ~0: nothing is emitted
            rec[1] = io;
            rec[2] = nv;
            rec[3] = ni;
        }
    }
    if (tid < kTileClasses) {
        const uint32_t k = s_count[tid];
        s_first[tid] = k ? atomicAdd(uw_queue_tile_count(a.qhead, tid), k) : 0u;
        s_count[tid] = 0u;
    }
    __syncthreads();
    for (int32_t i = tid; i < listed; i += kRowsBlock)
        if (s_tiles[i]) {
            const int k = uw_tile_class(s_tiles[i]);
            const uint64_t at = s_first[k] + atomicAdd(&s_count[k], 1u);
            a.list[uint64_t(k) * a.list_cap + at] = j0 * uint32_t(a.max_tiles) + uint32_t(i);
        }
}

// ---------------------------------------------------------------------------------------------
// Emission of the listed tiles (uw_emit_rows), most triangles first, in rounds of alternating
// direction over the resident workgroups.
template <bool EXTRA>
__global__ void __launch_bounds__(kEmitThreads, EXTRA ? 5 : 6) k_bulk_emit(BulkArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t G = gridDim.x, b = blockIdx.x;
    if (a.all && b == 0 && threadIdx.x == 0) {  // the range counters of k_bulk_rows are the totals
        const unsigned long long* resv = uw_queue_resv(a.qhead);
        const unsigned long long r0 = resv[0];
        a.totals->n_verts = a.packed ? (r0 & 0xFFFFFFFFull) : r0;
        a.totals->n_inds = a.packed ? (r0 >> 32) : resv[kResvIndsOffset];
        a.totals->n_nonblank = uint32_t(resv[kExitOffset] >> 32);
    }
    uint32_t ends[kTileClasses], items = 0;  // listed tiles of the classes up to each
#pragma unroll
    for (int k = 0; k < kTileClasses; ++k) ends[k] = items += *uw_queue_tile_count(a.qhead, k);
    if (b >= items) return;
    uw_emit_tables(a.tab, smem);
    uw_emit_tile e;
    e.eo = a.eo;
    e.iso = a.f.iso;
    e.extent = float(a.f.extent);
    e.T = 1;
    e.Y0 = 0;
    e.tz = 0;
    e.verts = a.verts;
    e.inds = a.inds;
    e.tape = a.tape;
    for (uint32_t r = 0;; ++r) {
        const uint32_t q = r * G + ((r & 1u) ? G - 1u - b : b);
        if (q >= items) return;  // later rounds lie further past the last tile
        const uint32_t item = __builtin_amdgcn_readfirstlane(a.list[uw_list_place(q, ends, a.list_cap)]);
        if (r) __syncthreads();  // the tile's LDS is written again
        const uint32_t j = item / uint32_t(a.max_tiles), tile = item - j * uint32_t(a.max_tiles);
        int32_t c, n, cx, cy, cz;
        load_task(a, j, &c, &n, &cx, &cy, &cz);
        const unsigned long long* rec = a.rec + 4 * uint64_t(j);
        if (rec[0] == ~0ull) continue;  // (block-uniform)
        const uw_slabs g = uw_slab_tiling(n, a.tile_rows);
        e.n = n;
        e.L = n + 1;
        e.WL = uw_sign_words(n + 1);
        e.cells = n;
        e.X0 = int32_t(tile) * g.planes;
        e.X1 = min(n, e.X0 + g.planes);
        e.Y1 = n;
        e.sx = n + 1;
        e.sy = 1;
        e.sz = (n + 1) * (n + 1);
        e.words = bulk_words(a, j);
        e.rows = bulk_rows(a, j);
        e.dens = bulk_dens(a, j);
        const uw_emit_row row = uw_emit_load(e);
        e.vo = rec[0];
        e.io = rec[1];
        e.vlim = e.vo + rec[2];
        e.ilim = e.io + rec[3];
        e.step = float(a.f.extent) / float(n);
        e.ox = float(a.f.extent * cx);
        e.oy = float(a.f.extent * cy);
        e.oz = float(a.f.extent * cz);
        uw_emit_rows<EXTRA>(e, row, smem);
    }
}

using BulkDensityKernel = void (*)(BulkArgs);
template <int BLOCK>
BulkDensityKernel pick_bulk_density(int octaves) {
    switch (octaves) {
        case 1: return k_bulk_density<1, BLOCK>;
        case 2: return k_bulk_density<2, BLOCK>;
        case 3: return k_bulk_density<3, BLOCK>;
        case 4: return k_bulk_density<4, BLOCK>;
        case 5: return k_bulk_density<5, BLOCK>;
        case 6: return k_bulk_density<6, BLOCK>;
        case 7: return k_bulk_density<7, BLOCK>;
        case 8: return k_bulk_density<8, BLOCK>;
        default: return k_bulk_density<0, BLOCK>;
    }
}
BulkDensityKernel pick_bulk_density(int octaves, int block) {
    return block == 64 ? pick_bulk_density<64>(octaves) : pick_bulk_density<128>(octaves);
}
int bulk_density_block(int32_t max_res) {
    const int32_t lines = (max_res + 1) * (max_res + 1), w128 = 2 * ((lines + 127) / 128), w64 = (lines + 63) / 64;
    return 5 * w64 <= 4 * w128 ? 64 : 128;
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

int grid_for(uw_ctx* ctx, const void* k, size_t lds, int* grid, int block) {
    int per_cu = 0;
    if (int rc = uw_resident(ctx, k, block, lds, &per_cu)) return rc;
    if (per_cu < 1) return uw_fail(ctx, UW_ERR_INVALID_ARG, "bulk kernel does not fit on a CU");
    *grid = per_cu * ctx->num_cus;
    return UW_OK;
}

}  // namespace

int uw_bulk_shape_for(uw_ctx* ctx, const uw_batch_tuning& t, int32_t nchunks, uw_bulk_shape* s) {
    memset(s, 0, sizeof(*s));
    s->on = t.bulk_min >= 1 && t.bulk_min <= t.max_res;
    if (!s->on) return UW_OK;
    s->max_res = t.max_res;
    const int32_t Lm = t.max_res + 1;
    const int block = bulk_density_block(t.max_res);
    s->wpc = (Lm * Lm + block - 1) / block;
    s->any_order = t.bulk_min == 1 && s->wpc <= kAnyOrderItems;
    const int32_t O = ctx->params.octaves;
    int32_t entries = 0;  // y and x entries per octave
    for (int32_t L = t.bulk_min + 1; L <= Lm; ++L) entries = std::max(entries, L + bulk_nx_tab(L, block));
    s->lds_density = 256 * sizeof(uint2) + 256 + sizeof(uw_axis) * size_t(uw_axis_pitch(O)) * size_t(entries);
    if (int rc = grid_for(ctx, reinterpret_cast<const void*>(pick_bulk_density(O, block)), s->lds_density, &s->grid_density, block))
        return rc;
    // tiles as deep as the emitter takes (each repeats a halo plane), and shallower while a launch of
    // chunks of max_res has fewer than 30 per compute unit, whose last rounds would be uneven: 1000
    // chunks of 3 .. 32 cells took 30.6 us in tiles of 224 rows and 25.8 of 160, 8192 of 8 .. 32 cells 125
    // and 141. Not below 96 (3 planes of 24: 17.3 us for 256 chunks, one plane each 23.8)
    const size_t nc = size_t(nchunks > 0 ? nchunks : 1);
    s->tile_rows = kTileRows;
    while (s->tile_rows > 96 && int64_t(nc) * uw_slab_tiling(t.max_res, s->tile_rows).tiles < 30 * int64_t(ctx->num_cus))
        s->tile_rows -= 32;
    s->max_tiles = 1;
    int32_t rows = 1;
    for (int32_t n = t.bulk_min; n <= t.max_res; ++n) {
        const uw_slabs g = uw_slab_tiling(n, s->tile_rows);
        s->max_tiles = g.tiles > s->max_tiles ? g.tiles : s->max_tiles;
        rows = g.max_rows > rows ? g.max_rows : rows;
    }
    if (!uw_emit_takes(rows, t.max_res, t.max_res))
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "emission tiles larger than a workgroup takes");
    s->lds_emit = uw_emit_lds_bytes(rows, t.max_res);
    const void* emit[2] = {reinterpret_cast<const void*>(k_bulk_emit<false>), reinterpret_cast<const void*>(k_bulk_emit<true>)};
    for (int extra = 0; extra < 2; ++extra)
        if (int rc = grid_for(ctx, emit[extra], s->lds_emit, &s->grid_emit[extra], kEmitThreads)) return rc;
    s->rows_waves = nc <= 1024 ? 4 : 16;
    s->grid_rows = int((nc + size_t(s->rows_waves) - 1) / size_t(s->rows_waves));
    if (nc * size_t(s->max_tiles) > 0x7FFFFFFFull) return uw_fail(ctx, UW_ERR_INVALID_ARG, "too many chunks for the bulk path");
    // scratch for every chunk of the launch (the resolutions are on the device; a launch's bulk
    // chunks are at most all of them)
    size_t o = 0;
    s->dens_off = o;
    o = align256(o + nc * size_t(Lm) * Lm * Lm * sizeof(float));
    s->words_off = o;
    o = align256(o + nc * size_t(Lm) * Lm * size_t(uw_sign_words(Lm)) * sizeof(uint32_t));
    s->rows_off = o;
    o = align256(o + nc * (size_t(t.max_res) * t.max_res + 1) * sizeof(unsigned long long));
    s->below_off = o;
    o = align256(o + nc * sizeof(uint32_t));
    s->rec_off = o;
    o = align256(o + nc * 4 * sizeof(unsigned long long));
    s->list_off = o;
    s->list_cap = uint64_t(nc) * uint64_t(s->max_tiles);
    o = align256(o + size_t(kTileClasses) * size_t(s->list_cap) * sizeof(uint32_t));
    s->bytes = o;
    // a launch whose worst case would need more scratch than this keeps every chunk on the
    // persistent kernel (same output, no per-chunk density slots)
    if (s->bytes > kBulkScratchMax) memset(s, 0, sizeof(*s));
    return UW_OK;
}

namespace {
BulkArgs bulk_args(uw_ctx* ctx, const uw_bulk_shape& s, const uw_bulk_io& io) {
    BulkArgs a;
    memset(&a, 0, sizeof(a));
    a.f = uw_make_field(ctx->params);
    a.tab = ctx->d_tables;
    a.tasks = io.tasks;
    a.all = io.all ? 1 : 0;
    a.any_order = s.any_order ? 1 : 0;
    a.qhead = io.qhead;
    a.max_res = s.max_res;
    a.Lm = s.max_res + 1;
    a.wpc = s.wpc;
    a.tile_rows = s.tile_rows;
    a.max_tiles = s.max_tiles;
    a.list_cap = s.list_cap;
    a.ztab = io.ztab;
    a.zstride = io.zstride;
    a.packed = io.packed;
    a.dens = reinterpret_cast<float*>(io.scratch + s.dens_off);
    a.words = reinterpret_cast<uint32_t*>(io.scratch + s.words_off);
    a.rows = reinterpret_cast<unsigned long long*>(io.scratch + s.rows_off);
    a.below = reinterpret_cast<uint32_t*>(io.scratch + s.below_off);
    a.rec = reinterpret_cast<unsigned long long*>(io.scratch + s.rec_off);
    a.list = reinterpret_cast<uint32_t*>(io.scratch + s.list_off);
    a.info = io.out->info;
    a.totals = io.out->totals;
    a.verts = io.out->verts;
    a.inds = io.out->inds;
    a.tape = io.tape;
    a.eo = uw_make_emit_opts(io.out);
    a.vcap = io.out->vert_cap;
    a.icap = io.out->ind_cap;
    return a;
}
}  // namespace

int uw_bulk_launch_front(uw_ctx* ctx, const uw_bulk_shape& s, const uw_bulk_io& io, hipStream_t st) {
    if (!s.on) return UW_OK;
    const BulkArgs a = bulk_args(ctx, s, io);
    const int block = bulk_density_block(s.max_res);
    const BulkDensityKernel kd = pick_bulk_density(ctx->params.octaves, block);
    // a launch of bulk chunks alone has its dominant kernel here, one with the persistent kernel has it there
    if (int rc = uw_prof_start(ctx, st, io.all ? UW_STAGE_DOMINANT : UW_STAGE_BULK_FRONT)) return rc;
    hipLaunchKernelGGL(kd, dim3(uint32_t(s.grid_density)), dim3(uint32_t(block)), s.lds_density, st, a);
    if (io.all) {
        if (int rc = uw_prof_end(ctx, st)) return rc;
        if (int rc = uw_prof_start(ctx, st, UW_STAGE_BULK_FRONT)) return rc;
    }
    hipLaunchKernelGGL(s.rows_waves == 4 ? k_bulk_rows<4> : k_bulk_rows<16>, dim3(uint32_t(s.grid_rows)),
                       dim3(uint32_t(64 * s.rows_waves)), size_t(s.rows_waves) * size_t(s.max_tiles) * sizeof(uint32_t), st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_bulk_launch_back(uw_ctx* ctx, const uw_bulk_shape& s, const uw_bulk_io& io, hipStream_t st) {
    if (!s.on) return UW_OK;
    const BulkArgs a = bulk_args(ctx, s, io);
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_BULK_EMIT)) return rc;
    const bool extra = uw_emit_extra(a.eo);
    hipLaunchKernelGGL(extra ? k_bulk_emit<true> : k_bulk_emit<false>, dim3(uint32_t(s.grid_emit[extra])), dim3(kEmitThreads),
                       s.lds_emit, st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}
