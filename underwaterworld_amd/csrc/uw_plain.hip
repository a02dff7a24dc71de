// Plain path: the stages of the chunk builder as kernel launches over every chunk, in chunk order.
//
//   k_plain_setup  per-chunk z tables; the launch's counters cleared
//   k_lines        density of every sample (Chunk::build_iso, chunk.rs:105-129) and its sign words
//                  (rho < iso, chunk.rs:155-162)
//   k_rows         vertex records and triangles of every row segment and their scan
//                  (chunk.rs:141-164): one wave per chunk, or one workgroup above 32 cells per axis
//   k_emit         one workgroup per (chunk, tile): the chunk's place in the output (sum of the sizes
//                  before it), then vertices, indices and collision records (chunk.rs:164-250); the
//                  first workgroups write the chunks' records and the totals, and the cube cases of
//                  every cell where the caller asks for them
//
// HBM layout (scratch, per chunk c of resolution n, L = n + 1):
//   dens   [c][L^3] f32     sample (x, y, z) at z L^2 + x L + y: a wave's store is one row of lines
//   words  [c][L^2][WL] u32 sign words (uw_rows.h)
//   rows   [c][R + 1] u64   scanned row segments and totals (uw_rows.h)
//   sizes  [c] u64          vertices | triangles << 32
//   groups [ceil(n_chunks / 256)][2] u64  vertices and triangles of 256 chunks; then the number of
//          non-blank chunks, and the number of listed tiles of each size class
//   list   [kTileClasses][n_chunks x tiles] u32   tiles with triangles (chunk x tiles + tile) by size
//          class, in any order
#include <hip/hip_runtime.h>
#include <string.h>

#include "uw_host.h"
#include "uw_mesh.h"
#include "uw_noise.h"
#include "uw_rows.h"
#include "uw_wave.h"

namespace {

constexpr int kThreads = 256;
constexpr int kGroup = 256;  // chunks per size group
__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// The z tables of a launch (uw_ztab_block, one thread per record) and its counters cleared: `below`
// (one word per chunk) and the size groups.
__global__ void __launch_bounds__(kThreads) k_plain_setup(uw_field f, const int32_t* __restrict__ coords, int32_t n,
                                                          int32_t nchunks, unsigned char* __restrict__ ztab,
                                                          uint32_t* __restrict__ below,
                                                          unsigned long long* __restrict__ groups, int32_t ngroup_words) {
    extern __shared__ uint32_t zstage[];
    const int64_t g = int64_t(blockIdx.x) * kThreads + threadIdx.x;  // at least one thread per chunk and group word
    if (g < nchunks) below[g] = 0u;
    if (g < ngroup_words) groups[g] = 0ull;
    uw_ztab_block<kThreads>(f, coords, nullptr, n, nchunks, n + 1, ztab, uint64_t(blockIdx.x) * kThreads, zstage);
}

struct PlainArgs {
    uw_field f;
    const uw_tables* tab;
    const int32_t* coords;
    int32_t nchunks, n, L, WL, T;
    int32_t ngroups;  // size groups
    int32_t packed;   // 1: every launch total fits 32 bits
    int32_t listed;   // 1: the emission takes the listed tiles
    int32_t wpc;     // workgroups of 256 lines per chunk
    int32_t nx_tab;  // distinct x among a workgroup's lines, at most
    int32_t zseg, zlen;  // z segments of a line (sample_density) and samples of each
    float step;
    const unsigned char* ztab;
    float* dens;
    uint32_t* words;
    unsigned long long* rows;
    unsigned long long* sizes;
    unsigned long long* groups;
    uint32_t* list;
    uint64_t list_cap;  // entries per class
    uint32_t* below;
    uw_chunk_info* info;
    uw_totals* totals;
    uint64_t vcap, icap;
    float* verts;
    uint32_t* inds;
    uw_emit_opts eo;
    uw_tiling tiling;
    uint8_t* cases;     // cube cases of every cell (null: not asked for)
    int32_t ncase;      // workgroups of the emission that write them
};

// A chunk's record (its offsets are the emission's) and its sizes, by one thread.
__device__ __forceinline__ void put_sizes(const PlainArgs& a, int32_t chunk, bool early, unsigned long long total,
                                          uint32_t act) {
    const uint32_t nv = uint32_t(total), nt = uint32_t(total >> 32);
    const uint32_t flags = early ? uint32_t(UW_CHUNK_BLANK | UW_CHUNK_EARLY_SKIP) : nt == 0u ? uint32_t(UW_CHUNK_BLANK) : 0u;
    uw_chunk_info r = {flags, nv, 3u * nt, act, 0, 0};
    a.info[chunk] = r;
    a.sizes[chunk] = total;
}
// Adds the sizes of some non-blank chunks of group g (one thread).
__device__ __forceinline__ void add_group(const PlainArgs& a, int32_t g, uint64_t nv, uint64_t nt) {
    atomicAdd(a.groups + 2 * g, (unsigned long long)nv);
    atomicAdd(a.groups + 2 * g + 1, (unsigned long long)nt);
}
// The launch's counters, 128 bytes apart (atomics on one line are served one after another).
constexpr int kLine = 16;
__device__ __forceinline__ unsigned long long* nonblank_count(const PlainArgs& a) {
    return a.groups + kLine * ((2 * a.ngroups + kLine - 1) / kLine);
}
__device__ __forceinline__ unsigned long long* class_count(const PlainArgs& a, int k) { return nonblank_count(a) + kLine * (k + 1); }

// Enters the tiles with triangles of `chunks` consecutive chunks from `chunk` on into the list (the
// whole workgroup; nt: triangles per chunk and tile, LDS). One atomic per class and workgroup: one per
// chunk, on one address, took 25 us for 4096 chunks.
template <int BLOCK>
__device__ __forceinline__ void list_tiles(const PlainArgs& a, int32_t chunk, int32_t chunks, const uint32_t* nt) {
    __shared__ uint32_t s_count[kTileClasses], s_first[kTileClasses];
    const int tid = threadIdx.x;
    const int32_t tiles = a.tiling.tiles(), total = chunks * tiles;
    if (tid < kTileClasses) s_count[tid] = 0u;
    __syncthreads();
    for (int32_t i = tid; i < total; i += BLOCK)
        if (nt[i]) atomicAdd(&s_count[uw_tile_class(nt[i])], 1u);
    __syncthreads();
    if (tid < kTileClasses) {
        const uint32_t c = s_count[tid];
        s_first[tid] = c ? uint32_t(atomicAdd(class_count(a, tid), (unsigned long long)c)) : 0u;
        s_count[tid] = 0u;
    }
    __syncthreads();
    for (int32_t i = tid; i < total; i += BLOCK)
        if (nt[i]) {
            const int k = uw_tile_class(nt[i]);
            a.list[uint64_t(k) * a.list_cap + s_first[k] + atomicAdd(&s_count[k], 1u)] = uint32_t(chunk * tiles + i);
        }
}

// ---------------------------------------------------------------------------------------------
// Densities. Workgroup b takes 256 consecutive z-lines t = x L + y of chunk b / wpc, one per lane,
// whatever the resolution (x-planes of their own leave 207 of 256 lanes idle at 49 samples per axis:
// 73 -> 33 us for 48 chunks of 48^3 at 6 octaves); the x and y entries of its lines are in LDS.
// BUILD: densities to the scratch layout, and sign words. !BUILD: densities to the caller's layout (z fastest),
// through an LDS tile of 16 samples per line so that stores are 64-byte runs, and the sign summary. There a
// workgroup may take a z segment of its lines (zseg > 1, uw_sample_density): a line's samples and tile
// flushes are one chain, which is the launch's time while compute units stand idle.
constexpr int kTileZ = 16, kTilePitch = kTileZ + 1;
// Segments are cut while a launch has fewer than 2 workgroups per compute unit, to 8 samples at least:
// each segment repeats the x and y entries of its lines and builds every octave's lattice faces at its
// first sample (6 octaves: 8 chunks of 64^3 41.9 -> 24.6 us, 64 of 32^3 32.5 -> 25.2, 64 of 8^3 19.6 ->
// 15.8; cut up to 4 per unit, 24 of 64^3 took 42.9 where 2 take 33.1, and 256 of 24^3 37.2 where uncut
// lines take 30.6).
constexpr int kSegPerCu = 2, kSegSamples = 8;

template <int OCT, bool BUILD>
__global__ void __launch_bounds__(kThreads) k_lines(PlainArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int32_t O = uw_octaves<OCT>::count(a.f), L = a.L, lines = L * L;
    uint2* GH = reinterpret_cast<uint2*>(smem);            // uw_grad_half of every slot
    uint8_t* P = reinterpret_cast<uint8_t*>(GH + 256);  // 256 B
    const int32_t pitch = uw_axis_pitch(O);
    uw_axis* AY = reinterpret_cast<uw_axis*>(P + 256);   // [L][pitch]
    uw_axis* AX = AY + L * pitch;                        // [nx_tab][pitch]
    float* TILE = reinterpret_cast<float*>(AX + a.nx_tab * pitch);  // !BUILD: [4 waves][64 lines][kTilePitch]
    __shared__ double s_freq[UW_MAX_OCTAVES];
    __shared__ uint32_t s_bits;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nthr = int(blockDim.x);  // 256, or the waves that one chunk's lines fill
    int32_t item = int32_t(blockIdx.x), seg = 0;
    if (!BUILD) {
        item = int32_t(blockIdx.x) / a.zseg;
        seg = int32_t(blockIdx.x) - item * a.zseg;
    }
    const int32_t chunk = item / a.wpc, t0 = (item - chunk * a.wpc) * nthr;
    const int32_t cx = a.coords[3 * chunk], cy = a.coords[3 * chunk + 1];
    if (tid == 0) s_bits = 0u;
    if (tid < UW_MAX_OCTAVES) s_freq[tid] = a.f.octave_freq[tid];
    for (int i = tid; i < 256; i += nthr) {
        const uint8_t p = a.tab->perm[i];
        P[i] = p;
        GH[i] = uw_grad_half(p & 15u);
    }
    __syncthreads();
    const uw_divider dL = uw_make_divider(uint32_t(L));
    const int32_t t = t0 + tid, xfirst = int32_t(uw_div(uint32_t(t0), dL));
    const int32_t nx = int32_t(uw_div(uint32_t(min(t0 + nthr, lines) - 1), dL)) - xfirst + 1;
    const bool valid = t < lines;
    const int32_t x = valid ? int32_t(uw_div(uint32_t(t), dL)) : xfirst, y = valid ? t - x * L : 0;
    const int32_t ne = O * (L + nx);
    const uw_divider dnx = uw_make_divider(uint32_t(nx));
    for (int e = tid; e < ne; e += nthr) {
        if (e < O * L) {
            const int32_t k = int32_t(uw_div(uint32_t(e), dL)), i = e - k * L;
            AY[i * pitch + k] = uw_axis_of(uw_sample_coord(a.f, 1, cy, i, a.step), s_freq[k]);
        } else {
            const int32_t q = e - O * L, k = int32_t(uw_div(uint32_t(q), dnx)), i = q - k * nx;
            AX[i * pitch + k] = uw_hash_x(uw_axis_of(uw_sample_coord(a.f, 0, cx, xfirst + i, a.step), s_freq[k]), P);
        }
    }
    __syncthreads();
    const uw_ztab Zt = uw_ztab_of(a.ztab, chunk, O, L);
    const int32_t rw = OCT > 0 ? uw_zrec_words(OCT) : Zt.rw;
    const uw_axis* ax = AX + (x - xfirst) * pitch;
    const uw_axis* ay = AY + y * pitch;
    const float iso = a.f.iso;
    float vmin = INFINITY, vmax = -INFINITY;
    uint32_t bits = 0;
    if (__any(valid)) {  // a wave with no line of the chunk leaves its SIMD to the others
        if (BUILD) {
            float* out = a.dens + uint64_t(chunk) * uint64_t(lines) * uint64_t(L) + t;
            uint32_t* wout = a.words + (uint64_t(chunk) * uint64_t(lines) + t) * a.WL;
            uint32_t word = 0, any = 0, all = 0xFFFFFFFFu;
            uw_noise_zline<OCT, false>(
                a.f, [=](int k) { return ax[k]; }, [=](int k) { return ay[k]; }, P, GH, Zt.rec, rw, L, vmin,
                vmax, [&](int32_t iz, float rho) {
                    if (valid) out[iz * lines] = rho;
                    word = uw_push_sign(word, rho, iso);
                    if ((iz & 31) == 31) {  // uniform: a full word (chunks of 31 cells per axis and up)
                        any |= word;
                        all &= word;
                        if (valid) wout[iz >> 5] = __brev(word);
                        word = 0;
                    }
                });
            const int32_t rest = L & 31;
            if (rest) {
                const uint32_t full = (1u << rest) - 1u;
                any |= word;
                all &= word | ~full;
                word = __brev(word) >> (32 - rest);
                if (valid) wout[a.WL - 1] = word;
            }
            bits = (vmin <= iso ? UW_BELOW_NOT_ABOVE : 0u) | (any ? UW_BELOW_LT : 0u) | (~all ? UW_BELOW_GE : 0u);
        } else {
            const int32_t z0 = seg * a.zlen, count = min(L - z0, a.zlen);
            float* dst = a.dens + (uint64_t(chunk) * uint64_t(lines) + uint64_t(t0 + 64 * wave)) * uint64_t(L) + z0;
            float* tile = TILE + wave * 64 * kTilePitch;
            const int32_t left = lines - (t0 + 64 * wave);  // lines of the wave
            // samples [z, z + nz) of the segment from the wave's tile, 64 at a time over its lines (LDS
            // operations of a wave stay in order)
            auto flush = [&](int32_t z, int32_t nz, const uw_divider& dn) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll 4
                for (int32_t i = 0; i < nz; ++i) {
                    const uint32_t e = uint32_t(64 * i + lane);
                    const int32_t q = int32_t(uw_div(e, dn)), k = int32_t(e) - q * nz;
                    if (q < left) dst[q * L + z + k] = tile[q * kTilePitch + k];
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            };
            const uw_divider dfull = uw_make_divider(kTileZ);
            uw_noise_zline<OCT, true>(
                a.f, [=](int k) { return ax[k]; }, [=](int k) { return ay[k]; }, P, GH, Zt.rec + z0 * rw, rw, count, vmin,
                vmax, [&](int32_t iz, float rho) {
                    tile[lane * kTilePitch + (iz & (kTileZ - 1))] = rho;
                    if ((iz & (kTileZ - 1)) == kTileZ - 1) flush(iz - (kTileZ - 1), kTileZ, dfull);
                });
            const int32_t rest = count & (kTileZ - 1);
            if (rest) flush(count - rest, rest, uw_make_divider(uint32_t(rest)));
            bits = uint32_t(uw_below_bits(vmin, vmax, iso));
        }
    }
    if (valid && bits) atomicOr(&s_bits, bits);
    __syncthreads();
    if (tid == 0 && s_bits) atomicOr(&a.below[chunk], s_bits);
}

// Row counts, one wave per chunk; a workgroup adds its chunks to their group at once. 4 chunks per
// workgroup spread a launch of up to 1024 chunks over the compute units; larger launches take 16 and a
// quarter of the atomics.
template <int W>
__global__ void __launch_bounds__(64 * W) k_rows_wave(PlainArgs a) {
    constexpr int kBlock = 64 * W;
    static_assert(kGroup % W == 0, "a workgroup's chunks lie in one group");
    extern __shared__ __align__(16) uint32_t s_tiles[];  // [W][tiles]
    __shared__ uint32_t lut[256];
    __shared__ unsigned long long s_size[W];
    const int tid = threadIdx.x, wave = tid >> 6;
    const int32_t chunk0 = int32_t(blockIdx.x) * W, chunk = __builtin_amdgcn_readfirstlane(chunk0 + wave);
    const int32_t tiles = a.tiling.tiles();
    const uint32_t sb = chunk < a.nchunks ? a.below[chunk] : 0u;
    for (int32_t i = tid; i < 256; i += kBlock) lut[i] = a.tab->cell[i];
    for (int32_t i = tid; i < W * tiles; i += kBlock) s_tiles[i] = 0u;
    __syncthreads();
    unsigned long long total = 0;
    uint32_t act = 0;
    if ((sb & UW_BELOW_LT) && (sb & UW_BELOW_GE))  // wave-uniform
        total = uw_wave_rows(a.words + uint64_t(chunk) * uint64_t(a.L * a.L) * a.WL, a.n, lut,
                             a.rows + uint64_t(chunk) * uint64_t(a.n * a.n * a.T + 1), &act, a.tiling.planes,
                             s_tiles + wave * tiles);
    if ((tid & 63) == 0) {
        if (chunk < a.nchunks) put_sizes(a, chunk, !(sb & UW_BELOW_NOT_ABOVE), total, act);
        s_size[wave] = total;
    }
    __syncthreads();
    if (tid == 0) {
        uint64_t nv = 0, nt = 0;
        uint32_t nb = 0;
        for (int w = 0; w < W; ++w) {
            nv += uint32_t(s_size[w]);
            nt += s_size[w] >> 32;
            nb += s_size[w] ? 1u : 0u;
        }
        if (nb) {
            add_group(a, chunk0 / kGroup, nv, nt);
            atomicAdd(nonblank_count(a), (unsigned long long)nb);
        }
    }
    if (a.listed) list_tiles<kBlock>(a, chunk0, min(W, a.nchunks - chunk0), s_tiles);
}

// Row counts of chunks of more than 32 cells per axis: one workgroup of 1024 threads per chunk (at
// most 8 segments per thread), sign words staged in LDS.
constexpr int kRowsBlock = 1024;
__global__ void __launch_bounds__(kRowsBlock) k_rows_block(PlainArgs a) {
    extern __shared__ __align__(16) uint32_t lwords[];  // sign words, then triangles per tile
    __shared__ uint32_t lut[256];
    const int32_t chunk = blockIdx.x, tid = threadIdx.x;
    const uint32_t sb = a.below[chunk];
    if (!((sb & UW_BELOW_LT) && (sb & UW_BELOW_GE))) {  // block-uniform
        if (tid == 0) put_sizes(a, chunk, !(sb & UW_BELOW_NOT_ABOVE), 0ull, 0u);
        return;
    }
    const int32_t nw = a.L * a.L * a.WL, tiles = a.tiling.tiles();
    uint32_t* s_tiles = lwords + nw;
    const uint32_t* src = a.words + uint64_t(chunk) * uint64_t(nw);
    if (tid < 256) lut[tid] = a.tab->cell[tid];
    for (int32_t i = tid; i < tiles; i += kRowsBlock) s_tiles[i] = 0u;
#pragma unroll 8
    for (int32_t i = tid; i < nw; i += kRowsBlock) lwords[i] = src[i];
    __syncthreads();
    static_assert(2 * UW_MAX_RESOLUTION * UW_MAX_RESOLUTION <= 8 * kRowsBlock, "segments per thread");
    uint32_t act = 0;
    const unsigned long long total = uw_block_rows<kRowsBlock, 8>(
        lwords, a.n, lut, a.rows + uint64_t(chunk) * uint64_t(a.n * a.n * a.T + 1), &act, a.tiling, s_tiles);
    if (tid == 0) {
        put_sizes(a, chunk, !(sb & UW_BELOW_NOT_ABOVE), total, act);
        if (total) {
            add_group(a, chunk / kGroup, uint32_t(total), total >> 32);
            atomicAdd(nonblank_count(a), 1ull);
        }
    }
    if (a.listed) list_tiles<kRowsBlock>(a, chunk, 1, s_tiles);
}

// ---------------------------------------------------------------------------------------------
// Sum over the workgroup of one u64 per thread (every thread).
__device__ __forceinline__ unsigned long long block_sum(unsigned long long v, unsigned long long* lds) {
    v = uw_wave_last(uw_wave_incl_scan(v));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long s = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) s += lds[w];
    return s;
}

// Records of the 256 chunks of group g: their offsets (the groups before it, then a scan of its
// sizes) and the flags that depend on them; the last group's workgroup writes the totals.
__device__ __forceinline__ void group_records(const PlainArgs& a, int32_t grp) {
    __shared__ unsigned long long s_sum[2][kThreads / 64], s_scan[2][kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    unsigned long long gv = 0, gt = 0;
    for (int32_t g = tid; g < grp; g += kThreads) {
        gv += a.groups[2 * g];
        gt += a.groups[2 * g + 1];
    }
    const int32_t chunk = grp * kGroup + tid;
    const bool has = chunk < a.nchunks;
    const unsigned long long size = has ? a.sizes[chunk] : 0ull;
    const uint32_t nv = uint32_t(size), nt = uint32_t(size >> 32);
    const unsigned long long iv = uw_wave_incl_scan((unsigned long long)nv), it = uw_wave_incl_scan((unsigned long long)nt);
    if (lane == 63) {
        s_scan[0][wave] = iv;
        s_scan[1][wave] = it;
    }
    unsigned long long vo = block_sum(gv, s_sum[0]), to = block_sum(gt, s_sum[1]);
    for (int w = 0; w < wave; ++w) {
        vo += s_scan[0][w];
        to += s_scan[1][w];
    }
    vo += iv - nv;
    const unsigned long long io = 3ull * (to + it - nt);
    const uint32_t ni = 3u * nt;
    const bool over = vo + nv > a.vcap || io + ni > a.icap;
    if (has) {
        uw_chunk_info r = a.info[chunk];
        r.vert_off = vo;
        r.ind_off = io;
        if (over) r.flags |= UW_CHUNK_OVERFLOW;
        if (a.eo.ind16 && nv > 65535u) r.flags |= UW_CHUNK_INDEX_WRAP;
        a.info[chunk] = r;
    }
    if (chunk == a.nchunks - 1) {
        // the launch overflows exactly when some chunk does: the last chunk's end is the largest
        uw_totals tot = {vo + nv, io + ni, uint32_t(*nonblank_count(a)), over ? 1u : 0u};
        *a.totals = tot;
    }
}

// Cube cases of every cell (chunk.rs:155-162), a row segment per thread and step, by workgroup b of
// a.ncase: a launch of its own, one cell per thread, cost 1024 chunks of 8^3 cells 4.0 us and could not
// hold 2^32 cells. Rows of a multiple of four cells are written in words.
__device__ __forceinline__ void write_cases(const PlainArgs& a, uint32_t b) {
    const uint32_t per = uint32_t(a.n) * uint32_t(a.n) * uint32_t(a.T);
    const uint64_t rows = uint64_t(per) * uint64_t(a.nchunks);
    const bool aligned = ((reinterpret_cast<uint64_t>(a.cases) | uint64_t(a.n)) & 3u) == 0u;
    for (uint64_t r = uint64_t(b) * kThreads + threadIdx.x; r < rows; r += uint64_t(a.ncase) * kThreads) {
        const uint64_t chunk = r / per;
        const uint32_t s = uint32_t(r - chunk * per), q = s / uint32_t(a.T), x = q / uint32_t(a.n);
        const int32_t tz = int32_t(s - q * uint32_t(a.T)), y = int32_t(q - x * uint32_t(a.n));
        uw_row_bits w;
        w.load(a.words + chunk * uint64_t(a.L * a.L) * a.WL, int32_t(x), y, tz, a.n, a.L, a.WL);
        uint8_t* out = a.cases + (chunk * uint64_t(a.n * a.n) + q) * uint64_t(a.n) + 32 * tz;
        const uint32_t nz = uint32_t(min(32, a.n - 32 * tz));
        if (aligned) {
            for (uint32_t z = 0; z < nz; z += 4) {
                uint32_t v = 0;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) v |= uw_case_of_index(w.index(z + i)) << (8 * i);
                *reinterpret_cast<uint32_t*>(out + z) = v;
            }
        } else {
            for (uint32_t z = 0; z < nz; ++z) out[z] = uint8_t(uw_case_of_index(w.index(z)));
        }
    }
}

// Emission. Workgroups [0, groups) write the records, the next ncase the cube cases. The others take
// tiles: LISTED, as many workgroups as stay resident take the listed tiles (those with triangles), most
// triangles first, in rounds of alternating direction so that the workgroups' sums stay even (a queue's claims, one atomic
// per tile on one address, cost more than the balance they bring: 40 -> 54 us for 4096 chunks of
// 12^3); else, for launches whose tiles all fit the device at once, workgroup b takes tile b, which
// saves the look-ups. A chunk's first vertex and index are summed from the sizes before it (the groups
// before its own, then the chunks of its group) by the workgroup itself, so no launch scans the chunks.
template <bool LISTED, bool EXTRA, bool CASES>
__global__ void __launch_bounds__(kThreads, EXTRA ? 5 : 6) k_emit(PlainArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ unsigned long long s_sum[2][kThreads / 64];
    if (int32_t(blockIdx.x) < a.ngroups) {
        group_records(a, int32_t(blockIdx.x));
        return;
    }
    if (CASES && int32_t(blockIdx.x) < a.ngroups + a.ncase) {
        write_cases(a, blockIdx.x - uint32_t(a.ngroups));
        return;
    }
    const int tid = threadIdx.x;
    const uint32_t before = uint32_t(a.ngroups) + (CASES ? uint32_t(a.ncase) : 0u);
    const uint32_t tiles = uint32_t(a.tiling.tiles()), G = gridDim.x - before, b = blockIdx.x - before;
    uint32_t ends[kTileClasses], items = 0;  // listed tiles of the classes up to each
    if (LISTED) {
#pragma unroll
        for (int k = 0; k < kTileClasses; ++k) ends[k] = items += uint32_t(*class_count(a, k));
        if (b >= items) return;
    } else if (a.sizes[b / tiles] == 0ull) {
        return;
    }
    uw_emit_tables(a.tab, smem);
    uw_emit_tile e;
    e.eo = a.eo;
    e.iso = a.f.iso;
    e.step = a.step;
    e.extent = float(a.f.extent);
    e.n = a.n;
    e.L = a.L;
    e.T = a.T;
    e.WL = a.WL;
    e.cells = a.tiling.cells;
    e.verts = a.verts;
    e.inds = a.inds;
    e.tape = nullptr;
    const int32_t lines = a.L * a.L, yz = a.tiling.yt * a.tiling.T;
    e.sx = a.L;
    e.sy = 1;
    e.sz = lines;
    for (uint32_t r = 0;; ++r) {
        uint32_t item = b;
        if (LISTED) {
            const uint32_t q = r * G + ((r & 1u) ? G - 1u - b : b);
            if (q >= items) return;  // later rounds lie further past the last tile
            item = __builtin_amdgcn_readfirstlane(a.list[uw_list_place(q, ends, a.list_cap)]);
            if (r) __syncthreads();  // the tile's LDS is written again
        }
        const int32_t chunk = int32_t(item / tiles), tile = int32_t(item - uint32_t(chunk) * tiles);
        const int32_t xt = tile / yz, rem = tile - xt * yz, yt = rem / a.tiling.T;
        e.X0 = xt * a.tiling.planes;
        e.X1 = min(a.n, e.X0 + a.tiling.planes);
        e.Y0 = yt * 32;
        e.Y1 = min(a.n, e.Y0 + 32);
        e.tz = rem - yt * a.tiling.T;
        e.words = a.words + uint64_t(chunk) * uint64_t(lines) * a.WL;
        e.rows = a.rows + uint64_t(chunk) * uint64_t(a.n * a.n * a.T + 1);
        e.dens = a.dens + uint64_t(chunk) * uint64_t(lines) * uint64_t(a.L);
        // one memory round trip: the tile's rows, and the sizes before the chunk
        const uw_emit_row row = uw_emit_load(e);
        const int32_t grp = chunk / kGroup, mate = grp * kGroup + tid;
        const unsigned long long size = a.sizes[chunk], msize = mate < chunk ? a.sizes[mate] : 0ull;
        const int32_t cx = a.coords[3 * chunk], cy = a.coords[3 * chunk + 1], cz = a.coords[3 * chunk + 2];
        unsigned long long sv = uint32_t(msize), st = msize >> 32;
        for (int32_t g = tid; g < grp; g += kThreads) {
            sv += a.groups[2 * g];
            st += a.groups[2 * g + 1];
        }
        if (a.packed) {  // every launch total below 2^32: one sum of both
            const unsigned long long s = block_sum(sv | (st << 32), s_sum[0]);
            e.vo = s & 0xFFFFFFFFull;
            e.io = 3ull * (s >> 32);
        } else {
            e.vo = block_sum(sv, s_sum[0]);
            e.io = 3ull * block_sum(st, s_sum[1]);
        }
        e.vlim = e.vo + uint32_t(size);
        e.ilim = e.io + 3u * uint32_t(size >> 32);
        e.ox = float(a.f.extent * cx);
        e.oy = float(a.f.extent * cy);
        e.oz = float(a.f.extent * cz);
        if (e.vlim <= a.vcap && e.ilim <= a.icap) uw_emit_rows<EXTRA>(e, row, smem);  // (block-uniform)
        if (!LISTED) return;
    }
}

using EmitKernel = void (*)(PlainArgs);
template <bool LISTED>
EmitKernel pick_emit(bool extra, bool cases) {
    if (cases) return extra ? k_emit<LISTED, true, true> : k_emit<LISTED, false, true>;
    return extra ? k_emit<LISTED, true, false> : k_emit<LISTED, false, false>;
}

// Page-locked room for a host build's record and arrays (a full 12^3 chunk has 0.3 MB)
constexpr uint64_t kChunkPinned = uint64_t(2) << 20;

// LDS bytes of k_lines.
size_t lines_lds_bytes(int32_t O, int32_t L, int32_t nx_tab, bool build) {
    return 256 * sizeof(uint2) + 256 + sizeof(uw_axis) * size_t(uw_axis_pitch(O)) * size_t(L + nx_tab) +
           (build ? 0 : size_t(kThreads) * kTilePitch * sizeof(float));
}

using LinesKernel = void (*)(PlainArgs);

template <bool BUILD>
LinesKernel pick_lines(int octaves) {
    switch (octaves) {
        case 1: return k_lines<1, BUILD>;
        case 2: return k_lines<2, BUILD>;
        case 3: return k_lines<3, BUILD>;
        case 4: return k_lines<4, BUILD>;
        case 5: return k_lines<5, BUILD>;
        case 6: return k_lines<6, BUILD>;
        case 7: return k_lines<7, BUILD>;
        case 8: return k_lines<8, BUILD>;
        default: return k_lines<0, BUILD>;
    }
}

// Words of the size groups and the launch's counters.
int32_t group_words(int32_t ngroups) { return kLine * ((2 * ngroups + kLine - 1) / kLine + 1 + kTileClasses); }

// Scratch of one plain launch, in one context-owned buffer: byte offsets of the arrays.
struct PlainLayout {
    size_t ztab, below, groups, sizes, list, words, rows, dens, bytes;
    int32_t ngroups;
};
PlainLayout plain_layout(int32_t nchunks, int32_t n, int32_t octaves, int32_t tiles) {  // tiles 0: densities only
    auto align = [](size_t v) { return (v + 255) & ~size_t(255); };
    const size_t nc = size_t(nchunks), L = size_t(n) + 1, WL = size_t(uw_sign_words(n + 1));
    PlainLayout l;
    l.ngroups = int32_t((nc + kGroup - 1) / kGroup);
    size_t o = 0;
    l.ztab = o;
    o = align(o + nc * uw_ztab_bytes(octaves, n + 1));
    l.below = o;
    o = align(o + nc * sizeof(uint32_t));
    l.groups = o;
    o = align(o + size_t(group_words(l.ngroups)) * sizeof(unsigned long long));
    l.sizes = o;
    l.list = l.words = l.rows = l.dens = o;
    if (tiles > 0) {
        o = align(o + nc * sizeof(unsigned long long));
        l.list = o;
        o = align(o + nc * size_t(tiles) * kTileClasses * sizeof(uint32_t));
        l.words = o;
        o = align(o + nc * L * L * WL * sizeof(uint32_t));
        l.rows = o;
        o = align(o + nc * (size_t(n) * n * uw_row_segs(n) + 1) * sizeof(unsigned long long));
        l.dens = o;
        o = align(o + nc * L * L * L * sizeof(float));
    }
    l.bytes = o;
    return l;
}

// Arguments shared by the launches of one call, over the context's scratch (grown as needed).
int plain_args(uw_ctx* ctx, const int32_t* coords, int32_t nchunks, int32_t n, int32_t tiles, PlainArgs* a, PlainLayout* lay) {
    *lay = plain_layout(nchunks, n, ctx->params.octaves, tiles);
    if (lay->bytes > ctx->plain_bytes) {
        (void)hipFree(ctx->d_plain);
        ctx->d_plain = nullptr;
        ctx->plain_bytes = 0;
        UW_ALLOC(ctx, ctx->d_plain, lay->bytes);
        ctx->plain_bytes = lay->bytes;
    }
    unsigned char* base = ctx->d_plain;
    memset(a, 0, sizeof(*a));
    a->f = uw_make_field(ctx->params);
    a->tab = ctx->d_tables;
    a->coords = coords;
    a->nchunks = nchunks;
    a->n = n;
    a->L = n + 1;
    a->WL = uw_sign_words(n + 1);
    a->T = uw_row_segs(n);
    a->wpc = (a->L * a->L + kThreads - 1) / kThreads;
    a->nx_tab = (kThreads - 1) / a->L + 2;
    if (a->nx_tab > a->L) a->nx_tab = a->L;
    a->zseg = 1;
    a->zlen = a->L;
    a->step = float(a->f.extent) / float(n);
    a->ztab = base + lay->ztab;
    a->ngroups = lay->ngroups;
    a->packed = uint64_t(nchunks) * uw_max_verts(n) < (1ull << 32) && uint64_t(nchunks) * uw_max_inds(n) < (1ull << 32) ? 1 : 0;
    a->below = reinterpret_cast<uint32_t*>(base + lay->below);
    a->groups = reinterpret_cast<unsigned long long*>(base + lay->groups);
    a->sizes = reinterpret_cast<unsigned long long*>(base + lay->sizes);
    a->list = reinterpret_cast<uint32_t*>(base + lay->list);
    a->list_cap = uint64_t(nchunks) * uint64_t(tiles);
    a->words = reinterpret_cast<uint32_t*>(base + lay->words);
    a->rows = reinterpret_cast<unsigned long long*>(base + lay->rows);
    a->dens = reinterpret_cast<float*>(base + lay->dens);
    return UW_OK;
}

int launch_lines(uw_ctx* ctx, const PlainArgs& a, const PlainLayout& lay, LinesKernel k, bool build, hipStream_t st) {
    const int32_t O = a.f.octaves;
    const uint64_t zblocks = (uint64_t(a.nchunks) * uint64_t(a.L + 1) + kThreads - 1) / kThreads;
    const uint64_t blocks = uint64_t(a.nchunks) * uint64_t(a.wpc) * uint64_t(a.zseg);
    if (zblocks > 0x7FFFFFFFull || blocks > 0x7FFFFFFFull) return uw_fail(ctx, UW_ERR_INVALID_ARG, "too many chunks for one launch");
    const size_t lds = lines_lds_bytes(O, a.L, a.nx_tab, build);
    UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    // one thread per z record, 256 per workgroup: at least one per chunk and per group word
    hipLaunchKernelGGL(k_plain_setup, dim3(uint32_t(zblocks)), dim3(kThreads),
                       size_t(kThreads) * size_t(uw_zrec_words(O) + 1) * sizeof(uint32_t), st, a.f, a.coords, a.n, a.nchunks,
                       const_cast<unsigned char*>(a.ztab), a.below, a.groups, group_words(lay.ngroups));
    if (int rc = uw_prof_start(ctx, st)) return rc;
    const int32_t lines = a.L * a.L, block = lines < kThreads ? (lines + 63) & ~63 : kThreads;
    hipLaunchKernelGGL(k, dim3(uint32_t(blocks)), dim3(uint32_t(block)), lds, st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

}  // namespace

extern "C" {

int uw_sample_density(uw_ctx* ctx, const int32_t* coords, int32_t nchunks, int32_t n, float* dens, uint32_t* below,
                      void* stream) {
    if (!ctx) return UW_ERR_INVALID_ARG;
    if (int rc = uw_check_resolution(ctx, n)) return rc;
    if (nchunks < 0 || (nchunks > 0 && (!coords || !dens))) return uw_fail(ctx, UW_ERR_INVALID_ARG, "bad arguments");
    if (nchunks == 0) return UW_OK;
    UW_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = uw_refuse_capture(ctx, st)) return rc;
    PlainArgs a;
    PlainLayout lay;
    if (int rc = plain_args(ctx, coords, nchunks, n, 0, &a, &lay)) return rc;
    a.dens = dens;
    if (below) a.below = below;
    const int64_t want = int64_t(kSegPerCu) * ctx->num_cus, have = int64_t(nchunks) * a.wpc;
    if (have < want) {
        const int64_t most = (a.L + kSegSamples - 1) / kSegSamples, segs = (want + have - 1) / have;
        a.zseg = int32_t(segs < most ? segs : most);
        a.zlen = (a.L + a.zseg - 1) / a.zseg;
        a.zseg = (a.L + a.zlen - 1) / a.zlen;
    }
    return launch_lines(ctx, a, lay, pick_lines<false>(a.f.octaves), false, st);
}

int uw_build_chunks_plain(uw_ctx* ctx, const int32_t* coords, int32_t nchunks, int32_t n, const uw_mesh_out* out,
                          uint8_t* cases, void* stream) {
    if (!ctx) return UW_ERR_INVALID_ARG;
    if (int rc = uw_check_resolution(ctx, n)) return rc;
    if (nchunks < 0 || !out || !out->info || !out->totals || (nchunks > 0 && !coords) ||
        (out->vert_cap > 0 && !out->verts) || (out->ind_cap > 0 && !out->inds) || out->vertex_format > 1 ||
        out->index_format > 1)
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "bad arguments");
    UW_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = uw_refuse_capture(ctx, st)) return rc;
    if (nchunks == 0) {
        hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, reinterpret_cast<uint32_t*>(out->totals),
                           uint64_t(sizeof(uw_totals) / 4), 0u);
        UW_HIP(ctx, hipGetLastError());
        return UW_OK;
    }
    // slabs as deep as a tile takes (each repeats a halo plane and the fixed chain of passes), and
    // shallower while a launch has too few tiles to even out: most tiles hold no surface, and then the
    // fullest tile's time is the launch's (48 chunks of 48^3: 32.1 us at 64 tiles per chunk, 24.8 at 192;
    // now 24.2 at 64, 20.6 at 128 and 17.5 at 192). 16 per compute unit for tiles of many rows and for
    // chunks of more than one row segment, a part of whose tiles is next to empty (64 chunks of 33^3: the
    // launch 53.6 us at 8 per unit, 49.7 at 16); 8 for tiles of up to 150 rows, whose fixed chain outweighs
    // their own share (1024 chunks: 4^3 36.7 us at 16 per unit, 30.9 at 8, 8^3 43.6 and 36.1, 12^3 50.3
    // and 43.9; 512 of 12^3 44.6 and 35.4)
    int32_t planes = uw_tile_planes(n);
    uw_tiling tiling = uw_tiling_for(n, planes);
    while (planes > 1) {
        const int64_t want = (tiling.T > 1 || tiling.max_rows > 150 ? 16 : 8) * int64_t(ctx->num_cus);
        if (int64_t(nchunks) * tiling.tiles() >= want) break;
        planes = (planes + 1) / 2;
        tiling = uw_tiling_for(n, planes);
    }
    if (!uw_emit_takes(tiling.max_rows, tiling.cells + (tiling.yt > 1 ? 1 : 0), tiling.cells))
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "emission tiles larger than a workgroup takes");
    const uint64_t items = uint64_t(nchunks) * uint64_t(tiling.tiles());
    if (items > 0x7FFFFFFFull) return uw_fail(ctx, UW_ERR_INVALID_ARG, "too many chunks for one launch");
    PlainArgs a;
    PlainLayout lay;
    if (int rc = plain_args(ctx, coords, nchunks, n, tiling.tiles(), &a, &lay)) return rc;
    a.tiling = tiling;
    a.info = out->info;
    a.totals = out->totals;
    a.vcap = out->vert_cap;
    a.icap = out->ind_cap;
    a.verts = out->verts;
    a.inds = out->inds;
    a.eo = uw_make_emit_opts(out);
    const size_t elds = uw_emit_lds_bytes(tiling.max_rows, tiling.cells);
    const bool extra = uw_emit_extra(a.eo);
    const EmitKernel listed = pick_emit<true>(extra, cases != nullptr), all = pick_emit<false>(extra, cases != nullptr);
    UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(listed), hipFuncAttributeMaxDynamicSharedMemorySize, int(elds)));
    UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(all), hipFuncAttributeMaxDynamicSharedMemorySize, int(elds)));
    int per_cu = 0;
    if (int rc = uw_resident(ctx, reinterpret_cast<const void*>(listed), kThreads, elds, &per_cu)) return rc;
    if (per_cu < 1) return uw_fail(ctx, UW_ERR_INVALID_ARG, "emit kernel does not fit on a CU");
    const uint64_t resident = uint64_t(per_cu) * uint64_t(ctx->num_cus);
    a.listed = items > resident ? 1 : 0;
    if (int rc = launch_lines(ctx, a, lay, pick_lines<true>(a.f.octaves), true, st)) return rc;
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_PLAIN_CLASSIFY)) return rc;
    if (a.T == 1) {  // up to 32 cells per axis
        const int waves = nchunks <= 1024 ? 4 : 16;
        hipLaunchKernelGGL(waves == 4 ? k_rows_wave<4> : k_rows_wave<16>, dim3(uint32_t((nchunks + waves - 1) / waves)),
                           dim3(uint32_t(64 * waves)), size_t(waves) * size_t(tiling.tiles()) * sizeof(uint32_t), st, a);
    } else {
        const size_t lds = (size_t(a.L) * a.L * a.WL + size_t(tiling.tiles())) * sizeof(uint32_t);
        UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(k_rows_block),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        hipLaunchKernelGGL(k_rows_block, dim3(uint32_t(nchunks)), dim3(kRowsBlock), lds, st, a);
    }
    if (int rc = uw_prof_end(ctx, st)) return rc;
    if (cases) {  // as many workgroups as the cases fill, at most 4 per compute unit
        const uint64_t blocks = (uint64_t(nchunks) * uint64_t(n) * n * a.T + kThreads - 1) / kThreads, most = 4 * uint64_t(ctx->num_cus);
        a.cases = cases;
        a.ncase = int32_t(blocks < most ? blocks : most);
    }
    const uint32_t first = uint32_t(lay.ngroups) + uint32_t(a.ncase);  // workgroups before the tiles'
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_PLAIN_EMIT)) return rc;
    if (!a.listed)
        hipLaunchKernelGGL(all, dim3(first + uint32_t(items)), dim3(kThreads), elds, st, a);
    else
        hipLaunchKernelGGL(listed, dim3(first + uint32_t(resident)), dim3(kThreads), elds, st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_chunk_build_host_out(uw_ctx* ctx, int32_t cx, int32_t cy, int32_t cz, int32_t n, const uw_host_out* ho,
                            uw_chunk_info* info) {
    if (!ctx || !info || !ho) return UW_ERR_INVALID_ARG;
    if (int rc = uw_check_resolution(ctx, n)) return rc;
    if ((ho->vert_cap > 0 && !ho->verts) || (ho->ind_cap > 0 && !ho->inds) || ho->vertex_format > 1 ||
        ho->index_format > 1)
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "bad arguments");
    UW_HIP(ctx, hipSetDevice(ctx->device));
    const uint64_t vmax = uw_max_verts(n), imax = uw_max_inds(n);
    if (!ctx->d_coord1) {
        UW_ALLOC(ctx, ctx->d_coord1, 3 * sizeof(int32_t));
        UW_ALLOC(ctx, ctx->d_info1, sizeof(uw_chunk_info));
        UW_ALLOC(ctx, ctx->d_totals1, sizeof(uw_totals));
    }
    if (ctx->verts1_cap < vmax || ctx->inds1_cap < imax) {
        (void)hipFree(ctx->d_verts1);
        (void)hipFree(ctx->d_inds1);
        (void)hipFree(ctx->d_norm1);
        (void)hipFree(ctx->d_cells1);
        ctx->d_verts1 = nullptr;
        ctx->d_inds1 = nullptr;
        ctx->d_norm1 = nullptr;
        ctx->d_cells1 = nullptr;
        ctx->verts1_cap = ctx->inds1_cap = 0;
        UW_ALLOC(ctx, ctx->d_verts1, vmax * 6 * sizeof(float));
        UW_ALLOC(ctx, ctx->d_inds1, imax * sizeof(uint32_t));
        ctx->verts1_cap = vmax;
        ctx->inds1_cap = imax;
    }
    const bool want_norm = ho->tri_normals != nullptr, want_cells = ho->tri_cells != nullptr;
    if (want_norm && !ctx->d_norm1) UW_ALLOC(ctx, ctx->d_norm1, ctx->inds1_cap * sizeof(float));
    if (want_cells && !ctx->d_cells1) UW_ALLOC(ctx, ctx->d_cells1, ctx->inds1_cap / 3 * sizeof(uint32_t));
    if (int rc = uw_set_coord_launch(ctx, ctx->d_coord1, cx, cy, cz, nullptr)) return rc;
    uw_mesh_out out = {ctx->d_verts1, ctx->d_inds1, ctx->d_info1, ctx->d_totals1, ctx->verts1_cap, ctx->inds1_cap,
                       ho->vertex_format, ho->index_format, want_norm ? ctx->d_norm1 : nullptr,
                       want_cells ? ctx->d_cells1 : nullptr};
    if (int rc = uw_build_chunks_plain(ctx, ctx->d_coord1, 1, n, &out, nullptr, nullptr)) return rc;
    const size_t vfl = ho->vertex_format == UW_VERTEX_XYZ_RGB ? 6 : 3;
    const size_t isz = ho->index_format == UW_INDEX_U16 ? sizeof(uint16_t) : sizeof(uint32_t);
    {  // the record and the arrays together, if they fit
        uw_pinned_use use(ctx);
        unsigned char* pin;
        if (uw_pinned(ctx, kChunkPinned, &pin)) {
            const uw_mesh_ptrs m = {{ctx->d_verts1, ctx->d_inds1, ctx->d_norm1, ctx->d_cells1}};
            const uw_mesh_format f = {uint32_t(vfl * sizeof(float)), uint32_t(isz), want_norm ? 1u : 0u, want_cells ? 1u : 0u};
            use.pending = true;
            if (int rc = uw_chunk_out_launch(ctx, ctx->d_info1, m, f, pin, kChunkPinned, nullptr)) return rc;
            UW_HIP(ctx, hipStreamSynchronize(nullptr));
            use.pending = false;
            memcpy(info, pin, sizeof(*info));
            if (info->n_verts > ho->vert_cap || info->n_inds > ho->ind_cap)
                return uw_fail(ctx, UW_ERR_OVERFLOW, "output capacity too small for this chunk");
            const uw_mesh_sections s = uw_sections(info->n_verts, info->n_inds, f);
            if (kMeshHeader + s.total <= kChunkPinned) {
                void* dst[4] = {ho->verts, ho->inds, ho->tri_normals, ho->tri_cells};
                for (int k = 0; k < 4; ++k)
                    if (s.bytes[k]) memcpy(dst[k], pin + kMeshHeader + s.off[k], s.bytes[k]);
                return UW_OK;
            }
        }
    }
    UW_HIP(ctx, hipMemcpy(info, ctx->d_info1, sizeof(uw_chunk_info), hipMemcpyDeviceToHost));
    if (info->n_verts > ho->vert_cap || info->n_inds > ho->ind_cap)
        return uw_fail(ctx, UW_ERR_OVERFLOW, "output capacity too small for this chunk");
    const size_t ntri = info->n_inds / 3;
    if (info->n_verts)
        UW_HIP(ctx, hipMemcpy(ho->verts, ctx->d_verts1, size_t(info->n_verts) * vfl * sizeof(float),
                              hipMemcpyDeviceToHost));
    if (info->n_inds) UW_HIP(ctx, hipMemcpy(ho->inds, ctx->d_inds1, size_t(info->n_inds) * isz, hipMemcpyDeviceToHost));
    if (ntri && want_norm)
        UW_HIP(ctx, hipMemcpy(ho->tri_normals, ctx->d_norm1, ntri * 3 * sizeof(float), hipMemcpyDeviceToHost));
    if (ntri && want_cells)
        UW_HIP(ctx, hipMemcpy(ho->tri_cells, ctx->d_cells1, ntri * sizeof(uint32_t), hipMemcpyDeviceToHost));
    return UW_OK;
}

int uw_chunk_build_host(uw_ctx* ctx, int32_t cx, int32_t cy, int32_t cz, int32_t n, float* verts, uint64_t vert_cap,
                        uint32_t* inds, uint64_t ind_cap, uw_chunk_info* info) {
    const uw_host_out ho = {verts, vert_cap, inds, ind_cap, UW_VERTEX_XYZ, UW_INDEX_U32, nullptr, nullptr};
    return uw_chunk_build_host_out(ctx, cx, cy, cz, n, &ho, info);
}

}  // extern "C"
