// Sign words, row counts and the tile emitter shared by the plain, bulk and volume paths.
//
// The density kernels leave, beside the densities, one bit per sample: rho < iso, the only thing the
// cube cases depend on (chunk.rs:155-162). The samples of a z-line (x, y) are packed along z, word s
// of the line holding samples 32 s .. 32 s + 31 at bits 0 .. 31, uw_sign_words(L) words per line,
// lines in order t = x L + y. Counting and classification read these words (a 32nd of the density
// bytes); the densities themselves are read only at the ends of the edges that carry a vertex.
//
// Row segments. A cell row (x, y) is cut along z into segments of 32 cells; segment tz of row
// (x, y) is row number (x n + y) T + tz, T = ceil(n / 32), which is the reference's scan order
// (chunk.rs:141-143). One thread takes one segment: the vertex records it owns are population counts
// of its edge masks, and only its active cells are visited one by one (for their triangles).
#pragma once

#include <stddef.h>

#include "uw_mesh.h"
#include "uw_wave.h"

__host__ __device__ constexpr int32_t uw_sign_words(int32_t L) { return (L + 31) / 32; }
__host__ __device__ constexpr int32_t uw_row_segs(int32_t n) { return (n + 31) / 32; }

// Packed corner bits of a cell: A | B << 2 | C << 4 | D << 6 with two bits (sample z, sample z + 1)
// from each of the lines (x, y), (x + 1, y), (x, y + 1), (x + 1, y + 1); the index of uw_tables::cell.
__host__ __device__ constexpr uint32_t uw_case_of_index(uint32_t i) {
    // corner order of chunk.rs:144-153: A0 B0 B1 A1 C0 D0 D1 C1
    return (i & 1u) | (((i >> 2) & 1u) << 1) | (((i >> 3) & 1u) << 2) | (((i >> 1) & 1u) << 3) |
           (((i >> 4) & 1u) << 4) | (((i >> 6) & 1u) << 5) | (((i >> 7) & 1u) << 6) | (((i >> 5) & 1u) << 7);
}

// Tiling of a chunk of n cells per axis: segments of 32 cells along z, at most 32 rows along y, and
// x-slabs of at most `planes` cell planes, as even as they come.
struct uw_tiling {
    int32_t planes, xt, yt, T, cells, max_rows;  // cells: of a row segment, at most
    __host__ __device__ int32_t tiles() const { return xt * yt * T; }
};
inline uw_tiling uw_tiling_for(int32_t n, int32_t planes) {
    uw_tiling g;
    const int32_t ny = n < 32 ? n : 32;
    g.yt = (n + 31) / 32;
    g.T = uw_row_segs(n);
    g.xt = (n + planes - 1) / planes;
    g.planes = (n + g.xt - 1) / g.xt;
    g.xt = (n + g.planes - 1) / g.planes;
    g.cells = ny;
    const int32_t rows_y = ny + (g.yt > 1 ? 1 : 0);
    g.max_rows = (g.planes + (g.xt > 1 ? 1 : 0)) * rows_y;
    return g;
}
// The sign words of one row segment: its four lines, each with the word after it (whose bit 0 is the
// sample above the segment's last cell).
struct uw_row_bits {
    uint32_t a, b, c, d;      // lines (x, y), (x + 1, y), (x, y + 1), (x + 1, y + 1)
    uint32_t an, bn, cn, dn;  // next words
    uint32_t valid;           // cells of the segment

    template <class Words>
    __device__ __forceinline__ void load(Words w, int32_t x, int32_t y, int32_t tz, int32_t n, int32_t L, int32_t WL) {
        const int32_t ia = (x * L + y) * WL + tz, ib = ia + L * WL, ic = ia + WL, id = ib + WL;
        a = w[ia];
        b = w[ib];
        c = w[ic];
        d = w[id];
        const bool more = tz + 1 < WL;
        an = more ? w[ia + 1] : 0u;
        bn = more ? w[ib + 1] : 0u;
        cn = more ? w[ic + 1] : 0u;
        dn = more ? w[id + 1] : 0u;
        const int32_t nz = n - 32 * tz;
        valid = nz >= 32 ? 0xFFFFFFFFu : (1u << nz) - 1u;
    }
    __device__ __forceinline__ static uint32_t up(uint32_t w, uint32_t next) {
        return __builtin_amdgcn_alignbit(next, w, 1u);
    }
    // cells whose corners are neither all below iso nor all at or above it
    __device__ __forceinline__ uint32_t active() const {
        const uint32_t ah = up(a, an), bh = up(b, bn), ch = up(c, cn), dh = up(d, dn);
        const uint32_t any = a | b | c | d | ah | bh | ch | dh, all = a & b & c & d & ah & bh & ch & dh;
        return any & ~all & valid;
    }
    // packed corner bits of cell z of the segment
    __device__ __forceinline__ uint32_t index(uint32_t z) const {
        const uint32_t A = __builtin_amdgcn_alignbit(an, a, z) & 3u, B = __builtin_amdgcn_alignbit(bn, b, z) & 3u;
        const uint32_t C = __builtin_amdgcn_alignbit(cn, c, z) & 3u, D = __builtin_amdgcn_alignbit(dn, d, z) & 3u;
        return A | (B << 2) | (C << 4) | (D << 6);
    }
};

// Owned records (bits 0-9), triangles (10-19) and active cells (20-) of a row segment, from its edge
// masks (bit z: edge e of cell z joins a sample below iso and one that is not; chunk.rs:144-153 for
// the corners). Records are counts of the owned edges (uw_owned_mask, edge by edge). A cell's case
// is drawn as loops around its active edges, a loop of k edges giving k - 2 triangles, so its
// triangles are its active edges less two per loop, and every case has one loop except those with a
// face whose four edges are all active or with two opposite corners cut off alone (all 256 rows of
// the table, tests/test_row_counts.py): only those cells are looked up, one by one. The count is a
// straight line of about 110 operations for 32 cells; looking up every active cell instead took
// 21.9 us where this takes 14.7 for 48 chunks of 48^3.
__device__ __forceinline__ uint32_t uw_row_counts(const uw_row_bits& r, int32_t x, int32_t y, int32_t tz,
                                                  const uint32_t* lut) {
    const uint32_t act = r.active();
    if (act == 0u) return 0u;
    const uint32_t ah = uw_row_bits::up(r.a, r.an), bh = uw_row_bits::up(r.b, r.bn), ch = uw_row_bits::up(r.c, r.cn),
                   dh = uw_row_bits::up(r.d, r.dn);
    const uint32_t v = r.valid;
    const uint32_t e0 = (r.a ^ r.b) & v, e1 = (r.b ^ bh) & v, e2 = (ah ^ bh) & v, e3 = (r.a ^ ah) & v;
    const uint32_t e4 = (r.c ^ r.d) & v, e5 = (r.d ^ dh) & v, e6 = (ch ^ dh) & v, e7 = (r.c ^ ch) & v;
    const uint32_t e8 = (r.a ^ r.c) & v, e9 = (r.b ^ r.d) & v, e10 = (bh ^ dh) & v, e11 = (ah ^ ch) & v;
    const uint32_t top = __popc(e4) + __popc(e5) + __popc(e6) + __popc(e7), bottom = __popc(e0) + __popc(e1) + __popc(e2) + __popc(e3);
    const uint32_t n10 = __popc(e10), n11 = __popc(e11), nact = __popc(act);
    uint32_t nv = top + n10 + (y == 0 ? bottom : 0u) + (x == 0 ? n11 : 0u);
    if (tz == 0) nv += (e9 & 1u) + (x == 0 ? (e8 & 1u) : 0u);
    uint32_t nt = top + bottom + n10 + n11 + __popc(e8) + __popc(e9) - 2u * nact;
    uint32_t odd = (e0 & e1 & e2 & e3) | (e4 & e5 & e6 & e7) | (e0 & e9 & e4 & e8) | (e1 & e10 & e5 & e9) |
                   (e2 & e11 & e6 & e10) | (e3 & e8 & e7 & e11) | (e0 & e3 & e8 & e5 & e6 & e10) |
                   (e0 & e1 & e9 & e6 & e7 & e11) | (e1 & e2 & e10 & e4 & e7 & e8) | (e2 & e3 & e11 & e4 & e5 & e9);
    for (; odd; odd &= odd - 1u) {
        const uint32_t w = lut[r.index(uint32_t(__builtin_ctz(odd)))];
        nt += ((w >> 12) & 15u) + 2u - uint32_t(__popc(w & 0xFFFu));
    }
    return nv | (nt << 10) | (nact << 20);
}

// Counts of every row segment of one chunk, and their exclusive scan in scan order: rows[r] = vertex
// records | triangles << 32 of the segments before r (chunk-local), and the chunk's totals at
// rows[n n T]. Returns the totals; act: the chunk's active cells. Two forms:
//
// one wave per chunk (up to 32 cells per axis: at most 16 segments per lane), 64 segments at a time;
// tiles (LDS, one per x-slab of `planes` cell planes): the triangles of each.
__device__ __forceinline__ unsigned long long uw_wave_rows(const uint32_t* __restrict__ words, int32_t n,
                                                           const uint32_t* lut, unsigned long long* __restrict__ rows,
                                                           uint32_t* act, int32_t planes, uint32_t* tiles) {
    const int lane = threadIdx.x & 63;
    const int32_t L = n + 1, T = uw_row_segs(n), WL = uw_sign_words(L), R = n * n * T;
    const uw_divider dT = uw_make_divider(uint32_t(T)), dn = uw_make_divider(uint32_t(n));
    // the sign words of the next 64 segments are fetched while these are counted
    auto load = [&](int32_t r, int32_t* x, int32_t* y, int32_t* tz) {
        const uint32_t q = uw_div(uint32_t(r), dT);
        *tz = r - int32_t(q) * T;
        *x = int32_t(uw_div(q, dn));
        *y = int32_t(q) - *x * n;
        uw_row_bits b;
        b.load(words, *x, *y, *tz, n, L, WL);
        return b;
    };
    unsigned long long carry = 0;
    uint32_t nact = 0;
    int32_t x = 0, y = 0, tz = 0;
    uw_row_bits b = load(min(lane, R - 1), &x, &y, &tz);
    for (int32_t r0 = 0; r0 < R; r0 += 64) {
        const int32_t r = r0 + lane;
        int32_t xn, yn, tn;
        const uw_row_bits bn = load(min(r + 64, R - 1), &xn, &yn, &tn);
        uint32_t c = 0;
        if (r < R) {
            c = uw_row_counts(b, x, y, tz, lut);
            if (c && planes < n) atomicAdd(tiles + uint32_t(x) / uint32_t(planes), (c >> 10) & 0x3FFu);
        }
        b = bn;
        x = xn;
        y = yn;
        tz = tn;
        // 64 segments hold fewer than 2^16 records and triangles
        const uint32_t v = (c & 0x3FFu) | (((c >> 10) & 0x3FFu) << 16);
        const uint32_t inc = uw_wave_incl_scan(v), ex = inc - v, tot = uw_wave_last(inc);
        if (r < R) rows[r] = carry + ((unsigned long long)(ex & 0xFFFFu) | ((unsigned long long)(ex >> 16) << 32));
        carry += (unsigned long long)(tot & 0xFFFFu) | ((unsigned long long)(tot >> 16) << 32);
        nact += c >> 20;
    }
    if (lane == 0) {
        rows[R] = carry;
        if (planes >= n) tiles[0] = uint32_t(carry >> 32);
    }
    *act = uw_wave_last(uw_wave_incl_scan(nact));
    return carry;
}

// or one workgroup of BLOCK threads per chunk, PER consecutive segments per thread (BLOCK PER >= n n T);
// words in LDS. act is thread 0's.
template <int BLOCK, int PER>
__device__ __forceinline__ unsigned long long uw_block_rows(const uint32_t* words, int32_t n, const uint32_t* lut,
                                                            unsigned long long* __restrict__ rows, uint32_t* act,
                                                            const uw_tiling& g, uint32_t* tiles) {
    constexpr int W = BLOCK / 64;
    __shared__ unsigned long long s_scan[W];
    __shared__ uint32_t s_act;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t L = n + 1, T = uw_row_segs(n), WL = uw_sign_words(L), R = n * n * T;
    const int32_t per = (R + BLOCK - 1) / BLOCK;
    const uw_divider dT = uw_make_divider(uint32_t(T)), dn = uw_make_divider(uint32_t(n));
    if (tid == 0) s_act = 0u;
    unsigned long long sum = 0;
    uint32_t nact = 0, c[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int32_t r = tid * per + k;
        c[k] = 0u;
        if (k < per && r < R) {
            const uint32_t q = uw_div(uint32_t(r), dT);
            const int32_t tz = r - int32_t(q) * T, x = int32_t(uw_div(q, dn)), y = int32_t(q) - x * n;
            uw_row_bits b;
            b.load(words, x, y, tz, n, L, WL);
            c[k] = uw_row_counts(b, x, y, tz, lut);
            if (c[k]) atomicAdd(tiles + ((x / g.planes) * g.yt + (y >> 5)) * g.T + tz, (c[k] >> 10) & 0x3FFu);
        }
        sum += (unsigned long long)(c[k] & 0x3FFu) | ((unsigned long long)((c[k] >> 10) & 0x3FFu) << 32);
        nact += c[k] >> 20;
    }
    const unsigned long long inc = uw_wave_incl_scan(sum);
    if (lane == 63) s_scan[wave] = inc;
    __syncthreads();
    unsigned long long base = inc - sum, total = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        base += w < wave ? s_scan[w] : 0ull;
        total += s_scan[w];
    }
    if (nact) atomicAdd(&s_act, nact);
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int32_t r = tid * per + k;
        if (k < per && r < R) rows[r] = base;
        base += (unsigned long long)(c[k] & 0x3FFu) | ((unsigned long long)((c[k] >> 10) & 0x3FFu) << 32);
    }
    if (tid == 0) rows[R] = total;
    __syncthreads();
    *act = s_act;
    return total;
}

// ---------------------------------------------------------------------------------------------
// Emission of one tile: cells [X0, X1) x [Y0, Y1) x row segment tz of a chunk, by one workgroup of
// kEmitThreads threads. The row segments of the tile, and the halo on its low sides (plane X0 - 1,
// row Y0 - 1, and the cell below the segment), are read once, one thread each:
//   1. the row threads list their active cells, in scan order (LIST, u32 per cell);
//   2. a thread per listed cell finds its case and its record count within the row segment (a
//      population count of the row's edge masks below the cell), which the triangles of other cells
//      need to name its records;
//   3. each wave takes 64 listed cells at a time on its own: it maps their owned records and triangles
//      to lanes (V2C, T2C), then writes one vertex per lane and one triangle per lane. The ids of a
//      triangle come from the owner cells' list entries, found by a population count of the owner
//      row's activity below its z.
// What bounds it: vector instructions (about 700 per 64 vertices and their 75 triangles) and the latency
// of the chain, for the largest grid also the stores (1.5 GB for 512^3 cells with the tape, in 918 us); a
// barrier follows steps 1 and 2 only. Windows of 256 cells that the whole workgroup took together, with
// dense per-cell state, three workgroups a unit and the three corners of a triangle found one after the
// other, took 1174 us there, 57 (now 36) for 150^3, 164 (now 122) for 8192 chunks of 8 .. 32 cells, 25 (now
// 17) for 48 chunks of 48^3 and as much for 4096 of 12^3 (28). Fetching a tile's row segments a round ahead
// was slower for chunks (147 where it was 141). A list of at most kListCap cells, whatever the tile, lets five
// workgroups share a compute unit's 160 KB of LDS (29 KB each for tiles of 200 to 224 row segments), six for
// tiles of up to 157 (27 KB); a tile with more active cells (more than half of its cells, for 32 cells per
// axis) is emitted one plane at a time, which always fits.
constexpr int kEmitThreads = 256;
constexpr uint32_t kListCap = 2112;            // listed cells: two planes (one and its halo) of 33 rows of 32
constexpr uint32_t kVertMap = 128, kTriMap = 192;  // map entries per wave
constexpr int kEmitMaxRows = kEmitThreads;  // row segments of a tile, halo included: one thread each

struct uw_emit_tile {
    uw_emit_opts eo;
    float iso, step, ox, oy, oz, extent;
    int32_t n, L, T, WL;
    int32_t X0, X1, Y0, Y1, tz;
    int32_t cells;                   // of a row segment, at most
    const float* dens;               // density of sample (x, y, z) at x sx + y sy + z sz
    int32_t sx, sy, sz;
    const uint32_t* words;           // the chunk's sign words
    const unsigned long long* rows;  // the chunk's scanned row segments, and its totals after the last
    uint64_t vo, io, vlim, ilim;     // first vertex and index of the chunk's ranges, and their ends
    float* verts;
    uint32_t* inds;
    uw_vertex_tape* tape;
};

constexpr size_t kEmitTableBytes = 256 * 8 + 256 * 12 * 2 + 256 * 4 + 256 * 2;  // uw_tables::tri, before, cell, used
static_assert(offsetof(uw_tables, before) == 2048 && offsetof(uw_tables, cell) == 8192 && offsetof(uw_tables, used) == 9216 &&
              kEmitTableBytes % 16 == 0 && kEmitTableBytes / 16 <= 3 * kEmitThreads, "tables copied as one block");
constexpr size_t kEmitWaveBytes = (kEmitThreads / 64) * (kVertMap + kTriMap) * 2;  // V2C, T2C
__host__ __device__ constexpr uint32_t uw_emit_list_cap(int32_t rows, int32_t cells) {
    return uint32_t(rows) * uint32_t(cells) < kListCap ? uint32_t(rows) * uint32_t(cells) : kListCap;
}
// Whether the emitter takes tiles of `rows` row segments (halo included) of `cells` cells: a thread per row
// segment, and a plane with its halo (at most two rows of `line` segments) always fits the list.
__host__ __device__ constexpr bool uw_emit_takes(int32_t rows, int32_t line, int32_t cells) {
    return rows <= kEmitMaxRows && 2u * uint32_t(line) * uint32_t(cells) <= kListCap;
}
// Bytes of dynamic LDS for tiles of `rows` row segments (halo included) of `cells` cells.
__host__ __device__ constexpr size_t uw_emit_lds_bytes(int32_t rows, int32_t cells) {
    return kEmitTableBytes + kEmitWaveBytes + (kListCap / 33 + 1) * 4 /*TAIL*/ + size_t(rows) * (16 + 16 + 4) /*ROW, BITS, XY*/ +
           (size_t(uw_emit_list_cap(rows, cells)) + size_t(rows)) * 4 /*LIST*/;
}

// The tables of the emission into LDS (once per workgroup, 16-byte loads, all issued before the first
// store); a barrier must follow before they are read (the one in uw_emit_rows does).
__device__ __forceinline__ void uw_emit_tables(const uw_tables* __restrict__ tab, unsigned char* smem) {
    const int tid = threadIdx.x;
    constexpr int kTabWords = int(kEmitTableBytes / 16);
    const uint4* src = reinterpret_cast<const uint4*>(tab);
    uint4 w[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        w[i] = tid + i * kEmitThreads < kTabWords ? src[tid + i * kEmitThreads] : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (tid + i * kEmitThreads < kTabWords) reinterpret_cast<uint4*>(smem)[tid + i * kEmitThreads] = w[i];
}

// What a thread of the emission reads of its row segment.
struct uw_emit_row {
    uw_row_bits b;
    uint32_t act;    // active cells
    uint32_t halo;   // packed corner bits of the cell below the segment (tz > 0)
    uint32_t count;  // vertices | triangles << 16 (0 in the halo)
    int32_t x, y;
    unsigned long long base;
};
__device__ __forceinline__ uw_emit_row uw_emit_load(const uw_emit_tile& t) {
    const int tid = threadIdx.x;
    const int32_t xs = t.X0 > 0 ? t.X0 - 1 : 0, ys = t.Y0 > 0 ? t.Y0 - 1 : 0;
    const int32_t ny = t.Y1 - ys, nrows = (t.X1 - xs) * ny;
    uw_emit_row r;
    r.act = r.halo = r.count = 0u;
    r.x = r.y = 0;
    r.base = 0ull;
    if (tid < nrows) {
        const int32_t pl = tid / ny, x = xs + pl, y = ys + tid - pl * ny;
        const int32_t i = (x * t.n + y) * t.T + t.tz;
        r.x = x;
        r.y = y;
        r.base = t.rows[i];
        const unsigned long long size = t.rows[i + 1] - r.base;
        r.b.load(t.words, x, y, t.tz, t.n, t.L, t.WL);
        if (t.tz > 0) {  // corner bits of the cell below the segment: sample 31 of the words before
            const uint32_t* w = t.words + (x * t.L + y) * t.WL + t.tz - 1;
            r.halo = (w[0] >> 31) | ((r.b.a & 1u) << 1) | ((w[t.L * t.WL] >> 31) << 2) | ((r.b.b & 1u) << 3) |
                     ((w[t.WL] >> 31) << 4) | ((r.b.c & 1u) << 5) | ((w[(t.L + 1) * t.WL] >> 31) << 6) | ((r.b.d & 1u) << 7);
        }
        r.act = r.b.active();
        if (x >= t.X0 && y >= t.Y0) r.count = uint32_t(size) | (uint32_t(size >> 32) << 16);
    }
    return r;
}

// One tile, or false (for the whole workgroup) if it has more active cells than the list takes.
// EXTRA: uw_emit_extra(t.eo).
template <bool EXTRA>
__device__ __forceinline__ bool uw_emit_part(const uw_emit_tile& t, const uw_emit_row& r, unsigned char* smem) {
    __shared__ uint32_t s_act[kEmitThreads / 64], s_any[kEmitThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t xs = t.X0 > 0 ? t.X0 - 1 : 0, ys = t.Y0 > 0 ? t.Y0 - 1 : 0;
    const int32_t ny = t.Y1 - ys, nrows = (t.X1 - xs) * ny;
    const int32_t Z0 = 32 * t.tz, n = t.n, L = t.L;
    const uint64_t* TRI = reinterpret_cast<const uint64_t*>(smem);
    const uint16_t* BEF = reinterpret_cast<const uint16_t*>(TRI + 256);
    const uint32_t* LUT = reinterpret_cast<const uint32_t*>(BEF + 256 * 12);
    const uint16_t* USED = reinterpret_cast<const uint16_t*>(LUT + 256);
    uint16_t* V2C = reinterpret_cast<uint16_t*>(smem + kEmitTableBytes) + wave * (kVertMap + kTriMap);  // lane | edge << 6
    uint16_t* T2C = V2C + kVertMap;                                                                     // lane | triangle << 6
    // active cells, list position of the first of them | owned edges (above the chunk's first cell) << 16,
    // first vertex id, first triangle
    uint4* ROW = reinterpret_cast<uint4*>(smem + kEmitTableBytes + kEmitWaveBytes);
    uint4* BITS = ROW + nrows;                             // the row segment's sign words
    uint32_t* XY = reinterpret_cast<uint32_t*>(BITS + nrows);  // x | y << 10 | bit 0 of the next words << 20 | halo << 24
    uint32_t* TAIL = XY + nrows;  // per window of listed cells: triangles of the last row segment's cells among them
    // record count of the row segment before the cell (10 bits, negative in the halo column) | case << 10 |
    // z << 18 | row << 23; the halo column's cells follow the list, one per row
    uint32_t* LIST = TAIL + kListCap / 33 + 1;
    const uint32_t cap = uw_emit_list_cap(nrows, t.cells);
    const uint32_t nact = uint32_t(__popc(r.act));
    const uint32_t inc = uw_wave_incl_scan(nact);
    const bool any = __any(r.count != 0u);
    if (lane == 63) {
        s_act[wave] = inc;
        s_any[wave] = any;
    }
    __syncthreads();
    uint32_t pos = inc - nact, total = 0, some = 0;
#pragma unroll
    for (int w = 0; w < kEmitThreads / 64; ++w) {
        pos += w < wave ? s_act[w] : 0u;
        total += s_act[w];
        some |= s_any[w];
    }
    if (!some) return true;
    if (total > cap) return false;
    if (tid < nrows) {
        const bool halo = r.x < t.X0 || r.y < t.Y0;
        ROW[tid] = make_uint4(r.act, pos | (uw_owned_mask(r.x, r.y, 1) << 16), uint32_t(r.base), uint32_t(r.base >> 32));
        BITS[tid] = make_uint4(r.b.a, r.b.b, r.b.c, r.b.d);
        XY[tid] = uint32_t(r.x) | (uint32_t(r.y) << 10) | ((r.b.an & 1u) << 20) | ((r.b.bn & 1u) << 21) |
                  ((r.b.cn & 1u) << 22) | ((r.b.dn & 1u) << 23) | (halo ? 1u << 24 : 0u);
        if (t.tz > 0) {
            const uint32_t w = LUT[r.halo];
            LIST[cap + tid] = (uint32_t(-int32_t(__popc(w & 0xFFFu & uw_owned_mask(r.x, r.y, 1)))) & 0x3FFu) | ((w >> 16) << 10);
        }
        for (uint32_t left = r.act; left; left &= left - 1u)
            LIST[pos++] = (uint32_t(__builtin_ctz(left)) << 18) | (uint32_t(tid) << 23);
    }
    __syncthreads();
    // windows of at most 64 cells, as many for every wave; at least 33, so that a row segment that ends
    // in a full window began in it or in the one before
    const uint32_t rounds = (total + kEmitThreads - 1) / kEmitThreads;
    uint32_t span = (total + rounds * (kEmitThreads / 64) - 1) / (rounds * (kEmitThreads / 64));
    if (span < 33u) span = 33u;
    const uint32_t windows = (total + span - 1) / span;
    // cases and records before each cell
    for (uint32_t win = wave; win < windows; win += kEmitThreads / 64) {
        const uint32_t i = win * span + lane;
        uint32_t nt = 0, first = 0;
        if (lane < int(span) && i < total) {
            const uint32_t ent = LIST[i], z = (ent >> 18) & 31u, row = ent >> 23, xy = XY[row];
            const uint4 q = BITS[row];
            const int32_t x = int32_t(xy & 1023u), y = int32_t((xy >> 10) & 1023u);
            uw_row_bits b;
            b.a = q.x;
            b.b = q.y;
            b.c = q.z;
            b.d = q.w;
            b.an = (xy >> 20) & 1u;
            b.bn = (xy >> 21) & 1u;
            b.cn = (xy >> 22) & 1u;
            b.dn = (xy >> 23) & 1u;
            const uint32_t w = LUT[b.index(z)], m = (1u << z) - 1u;
            const uint32_t bh = b.up(b.b, b.bn), ch = b.up(b.c, b.cn), dh = b.up(b.d, b.dn);
            // the owned edges (uw_owned_mask) of the cells below z: e4 e5 e6 e7 e10
            uint32_t pre = __popc((b.c ^ b.d) & m) + __popc((b.d ^ dh) & m) + __popc((ch ^ dh) & m) + __popc((b.c ^ ch) & m) +
                           __popc((bh ^ dh) & m);
            if (x == 0 || y == 0 || t.tz == 0) {
                const uint32_t ah = b.up(b.a, b.an);
                if (y == 0)  // e0 e1 e2 e3
                    pre += __popc((b.a ^ b.b) & m) + __popc((b.b ^ bh) & m) + __popc((ah ^ bh) & m) + __popc((b.a ^ ah) & m);
                if (x == 0) pre += __popc((ah ^ ch) & m);  // e11
                if (t.tz == 0) pre += ((b.b ^ b.d) & m & 1u) + (x == 0 ? (b.a ^ b.c) & m & 1u : 0u);  // e9, e8
            }
            LIST[i] = ent | pre | ((w >> 16) << 10);
            nt = xy >> 24 ? 0u : (w >> 12) & 15u;
            first = ROW[row].y & 0xFFFFu;
        }
        // (a row segment has at most 32 cells, so the last one of a full window begins in it)
        const uint32_t sum = uw_wave_incl_scan(nt);
        const uint32_t at = uint32_t(__builtin_amdgcn_readlane(int(first), int(span - 1u))) - win * span;
        if (win + 1 < windows) {
            const uint32_t before = uint32_t(__builtin_amdgcn_readlane(int(sum - nt), int(at & 63u)));
            if (lane == 63) TAIL[win] = sum - before;
        }
    }
    __syncthreads();
    const bool coll = EXTRA && (t.eo.tri_normals || t.eo.tri_cells);
    const uint32_t vstride = EXTRA ? t.eo.vstride : 3u, ind16 = EXTRA ? t.eo.ind16 : 0u;
    auto density = [&](int32_t px, int32_t py, int32_t pz) { return t.dens[px * t.sx + py * t.sy + pz * t.sz]; };
    // densities at the ends of edge ed of cell (cx, cy, cz)
    auto ends = [&](uint32_t ed, int32_t cx, int32_t cy, int32_t cz, float* ra, float* rbv) {
        const uint32_t ca = uw_edge_ofs_a(ed), cb = uw_edge_ofs_b(ed);
        *ra = density(cx + int32_t(ca & 1u), cy + int32_t((ca >> 1) & 1u), cz + int32_t(ca >> 2));
        *rbv = density(cx + int32_t(cb & 1u), cy + int32_t((cb >> 1) & 1u), cz + int32_t(cb >> 2));
    };
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto from = [](uint32_t v, uint32_t src) { return uint32_t(__builtin_amdgcn_ds_bpermute(int(src << 2), int(v))); };
    // owned edges of the cell at z of a row segment (uw_owned_mask), from the row's second word
    const bool bottom = t.tz == 0;
    auto owned = [&](uint32_t w, uint32_t z) {
        const uint32_t low = 0x200u | ((w >> 19) & 0x100u);
        return (w >> 16) | ((bottom & (z == 0u)) ? low : 0u);
    };
    for (uint32_t win = wave; win < windows; win += kEmitThreads / 64) {
        const uint32_t i = win * span + lane;
        uint32_t ent = 0, xyz = 0, own = 0, idb = 0, tb = 0, vm = 0, nt = 0, first = 0;
        if (lane < int(span) && i < total) {
            ent = LIST[i];
            const uint32_t z = (ent >> 18) & 31u, row = ent >> 23, xy = XY[row], cs = (ent >> 10) & 255u;
            const uint4 q = ROW[row];
            xyz = (xy & 0xFFFFFu) | ((uint32_t(Z0) + z) << 20);
            own = owned(q.y, z);
            idb = q.z + (ent & 0x3FFu);
            tb = q.w;
            first = q.y & 0xFFFFu;
            if (!(xy >> 24)) {
                vm = USED[cs] & own;
                nt = uint32_t(TRI[cs]) & 15u;
            }
            own |= cs << 12;
        }
        const uint32_t v = uint32_t(__popc(vm)) | (nt << 16), vinc = uw_wave_incl_scan(v), vex = vinc - v;
        const uint32_t ends_at = uw_wave_last(vinc), nvw = ends_at & 0xFFFFu, ntw = ends_at >> 16;
        if (ends_at == 0u) continue;  // (a window of the halo)
        // triangle number of the lane's first triangle, less its map position: those of the row segment's
        // cells before it are in this window, or (its tail) in the one before
        {
            const uint32_t base = from(vex >> 16, (first - win * span) & 63u);
            tb -= first >= win * span ? base : win ? 0u - TAIL[win - 1] : 0u;
        }
        uint32_t vat = vex & 0xFFFFu, tat = vex >> 16;
        for (uint32_t m0 = 0; m0 < nvw; m0 += kVertMap) {  // one pass, unless the cells are dense
            uint32_t at = vat - m0;
            for (uint32_t left = vm; left; left &= left - 1u, ++at)
                if (at < kVertMap) V2C[at] = uint16_t(uint32_t(lane) | (uint32_t(__builtin_ctz(left)) << 6));
            wave_sync();
            const uint32_t end = min(nvw - m0, kVertMap);
            for (uint32_t j = 0; j < end; j += 64) {
                const uint32_t code = j + lane < end ? V2C[j + lane] : 0u, src = code & 63u, ed = code >> 6;
                const uint32_t c = from(xyz, src), o = from(own, src), base = from(idb, src);
                if (j + lane >= end) continue;
                const int32_t cx = int32_t(c & 1023u), cy = int32_t((c >> 10) & 1023u), cz = int32_t(c >> 20);
                float ra, rbv, p[3];
                ends(ed, cx, cy, cz, &ra, &rbv);
                const uint64_t id = t.vo + (base + uint32_t(__popc(uint32_t(BEF[(o >> 12) * 12u + ed]) & o)));
                if (id >= t.vlim) continue;
                uw_edge_vertex_ab(ed, cx, cy, cz, ra, rbv, t.iso, t.step, t.ox, t.oy, t.oz, p);
                float* dst = t.verts + vstride * id;
                dst[0] = p[0];
                dst[1] = p[1];
                dst[2] = p[2];
                if (vstride == 6) uw_vertex_color(p[2], uw_edge_b(ed), t.extent, dst + 3);
                if (t.tape) {
                    const uint32_t ca = uw_edge_ofs_a(ed), cb = uw_edge_ofs_b(ed);
                    uw_vertex_tape tv;
                    tv.a = uint32_t(((cx + int32_t(ca & 1u)) * L + cy + int32_t((ca >> 1) & 1u)) * L + cz + int32_t(ca >> 2));
                    tv.b = uint32_t(((cx + int32_t(cb & 1u)) * L + cy + int32_t((cb >> 1) & 1u)) * L + cz + int32_t(cb >> 2));
                    tv.rho_a = ra;
                    tv.rho_b = rbv;
                    t.tape[id] = tv;
                }
            }
            wave_sync();
        }
        for (uint32_t m0 = 0; m0 < ntw; m0 += kTriMap) {
            for (uint32_t j = 0; j < nt; ++j)
                if (tat + j - m0 < kTriMap) T2C[tat + j - m0] = uint16_t(uint32_t(lane) | (j << 6));
            wave_sync();
            const uint32_t end = min(ntw - m0, kTriMap);
            for (uint32_t j = 0; j < end; j += 64) {
                const uint32_t code = j + lane < end ? T2C[j + lane] : 0u, src = code & 63u, tj = code >> 6;
                const uint32_t o = from(own, src), e = from(ent, src), base = from(tb, src), c = coll ? from(xyz, src) : 0u;
                if (j + lane >= end) continue;
                const uint32_t row = e >> 23, z = (e >> 18) & 31u, below = (1u << z) - 1u;
                const uint32_t edges = uint32_t(TRI[o >> 12] >> (4 + 12 * tj));
                const uint64_t gi = t.io + 3ull * (base + m0 + j + lane);
                // The record's owner (uw_edge_owner): the cell itself, or one step back along x, y, z. The
                // three edges go through each of the dependent LDS reads together, without branches.
                const uint32_t fx = ~(o >> 11) & 1u, fz = ~(o >> 9) & 1u;  // not in the chunk's first plane, first cell
                uint32_t qe[3], qrow[3], at[3], id[3], bz[3];
                uint4 R[3];
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    const uint32_t ed = (edges >> (4 * k)) & 15u, other = ~(o >> ed) & 1u;
                    const uint32_t bx = other & (0x900u >> ed) & fx, by = other & (0xFu >> ed);
                    bz[k] = other & (0x300u >> ed) & fz;
                    uint32_t q = by ? ed + 4u : 10u;
                    q = ((ed == 8u) & !bz[k]) ? 9u : q;
                    q = ((ed == 8u) & !bx) ? 11u : q;
                    qe[k] = other ? q : ed;
                    qrow[k] = row - (uint32_t(ny) & (0u - bx)) - by;
                    R[k] = ROW[qrow[k]];
                }
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    const uint32_t listed = (R[k].y & 0xFFFFu) + uint32_t(__popc(R[k].x & (below >> bz[k])));
                    const uint32_t halo = cap + qrow[k], under = bz[k] & (z == 0u);
                    at[k] = LIST[listed + ((halo - listed) & (0u - under))];
                }
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    const uint32_t w = at[k], before = BEF[((w >> 10) & 255u) * 12u + qe[k]];
                    id[k] = R[k].z + uint32_t(int32_t(w << 22) >> 22) +
                            uint32_t(__popc(before & owned(R[k].y, z - bz[k])));
                }
                if (gi + 2 < t.ilim && !ind16) {  // 12 bytes in one store
                    *reinterpret_cast<uint3*>(t.inds + gi) = make_uint3(id[0], id[1], id[2]);
                } else {
#pragma unroll
                    for (uint32_t k = 0; k < 3; ++k)
                        if (gi + k < t.ilim) uw_store_index(t.inds, ind16, gi + k, id[k]);
                }
                if (coll && gi + 2 < t.ilim) {
                    const int32_t cx = int32_t(c & 1023u), cy = int32_t((c >> 10) & 1023u), cz = int32_t(c >> 20);
                    const uint64_t tri = gi / 3;
                    if (t.eo.tri_normals) {
                        float nm[3], q[3][3];
#pragma unroll
                        for (uint32_t k = 0; k < 3; ++k) {
                            const uint32_t ed = (edges >> (4 * k)) & 15u;
                            float ra, rbv;
                            ends(ed, cx, cy, cz, &ra, &rbv);
                            uw_edge_vertex_ab(ed, cx, cy, cz, ra, rbv, t.iso, t.step, t.ox, t.oy, t.oz, q[k]);
                        }
                        uw_tri_normal(q[0], q[1], q[2], nm);
                        t.eo.tri_normals[3 * tri] = nm[0];
                        t.eo.tri_normals[3 * tri + 1] = nm[1];
                        t.eo.tri_normals[3 * tri + 2] = nm[2];
                    }
                    if (t.eo.tri_cells)
                        t.eo.tri_cells[tri] = (uint32_t(cx) * uint32_t(n) + uint32_t(cy)) * uint32_t(n) + uint32_t(cz);
                }
            }
            wave_sync();
        }
    }
    return true;
}

// One tile, its tables loaded by uw_emit_tables and its row segments by uw_emit_load. A workgroup
// that emits several tiles puts a barrier between them.
template <bool EXTRA>
__device__ __forceinline__ void uw_emit_rows(const uw_emit_tile& tile, const uw_emit_row& row, unsigned char* smem) {
    uw_emit_tile t = tile;
    uw_emit_row r = row;
    for (;;) {
        if (uw_emit_part<EXTRA>(t, r, smem)) {
            if (t.X1 >= tile.X1) return;
            t.X0 = t.X1;
        }
        t.X1 = t.X0 + 1;  // plane by plane
        r = uw_emit_load(t);
        __syncthreads();  // the LDS is written again
    }
}

// The same for chunks of at most 32 cells per axis, whose tiles are x-slabs of whole planes, at about
// `rows` row segments per tile (on the device: the resolutions of a batched launch are there).
struct uw_slabs {
    int32_t planes, tiles, max_rows;
};
__host__ __device__ inline uw_slabs uw_slab_tiling(int32_t n, int32_t rows) {
    int32_t p = n * n <= rows ? n : rows / n - 1;
    if (p < 1) p = 1;
    uw_slabs g;
    g.tiles = (n + p - 1) / p;
    g.planes = (n + g.tiles - 1) / g.tiles;
    g.tiles = (n + g.planes - 1) / g.planes;
    g.max_rows = (g.planes + (g.tiles > 1 ? 1 : 0)) * n;
    return g;
}

// Size classes of the tiles to emit, most triangles first. Emission time follows the surface: in
// arbitrary order, the last workgroups of 4096 chunks of 12^3 were busy for 37 us where the mean
// ended after 23. uw_list_place: the list entry of the q-th tile, given the running totals of the
// classes (`cap` entries per class).
constexpr int kTileClasses = 4;
__device__ __forceinline__ int uw_tile_class(uint32_t nt) { return nt > 768u ? 0 : nt > 512u ? 1 : nt > 256u ? 2 : 3; }
__device__ __forceinline__ uint64_t uw_list_place(uint32_t q, const uint32_t (&ends)[kTileClasses], uint64_t cap) {
    uint32_t cls = 0, first = 0;
#pragma unroll
    for (int k = 0; k + 1 < kTileClasses; ++k)
        if (q >= ends[k]) {
            cls = uint32_t(k + 1);
            first = ends[k];
        }
    return uint64_t(cls) * cap + (q - first);
}

// Slab depth of the tile emitter at n cells per axis: rows near kTileRows, halo plane included (512^3: 972 us
// at 160 rows, 1303 at 96).
constexpr int32_t kTileRows = 224;
inline int32_t uw_tile_planes(int32_t n) {
    const int32_t ny = n < 32 ? n : 33;
    if (n * ny <= kTileRows) return n;
    const int32_t p = kTileRows / ny - 1;
    return p < 1 ? 1 : p;
}
