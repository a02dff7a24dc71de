// Large single volume: ONE chunk of n cells per axis (n up to UW_VOLUME_MAX_RESOLUTION) meshed as
// one grid with one index space -- Chunk::new(pos) + build_full (chunk.rs:89-103,266-313) for a
// chunk too large for the per-chunk paths. Output equals the reference's builder run on that
// chunk: densities of chunk.rs:105-129, cases of chunk.rs:141-164, lerps of chunk.rs:178-231 and
// first-seen vertex numbering over the whole grid (chunk.rs:233-243).
//
// Kernels (one launch each, no host synchronisation between them):
//   k_vol_tables   per-axis octave entries of the whole grid (x hashed), fade derivatives, the z
//                  records of the line evaluator, and the launch's counters reset
//   k_vol_density  densities of every sample into HBM, and their sign words (uw_rows.h); one lane per
//                  z-line, lanes of a wave on consecutive lines, so each sample's store is one
//                  coalesced row
//   k_vol_rows     owned vertex records and triangles of every row segment (x, y, 32-cell z range)
//                  from the sign words, and their sums per scan block
//   k_vol_scan_*   exclusive scan of the row-segment counts in scan order (x, y, z range): the
//                  first vertex id and first triangle of every row segment; totals and the record
//   k_vol_emit     persistent workgroups over the tiles (uw_emit_rows): vertices, indices, optional
//                  tape / colour / collision; a tile's halo gives the ids of records owned by cells of
//                  neighbouring tiles
//
// HBM layout: densities f32 [(x L + z) L + y] (L = n + 1, y fastest: a wave's store covers 64
// consecutive y); sign words u32 [(x L + y) WL + w] (WL = ceil(L / 32)); row-segment counts u32 and
// scanned bases u64 [(x n + y) T + tz] (T = ceil(n / 32)) holding vertex records | triangles << 32.
#include <hip/hip_runtime.h>
#include <string.h>

#include "uw_mesh.h"
#include "uw_noise.h"
#include "uw_rows.h"
#include "uw_wave.h"

namespace {

constexpr int kVolBlock = 256;
constexpr int kScanPer = 4;         // row segments per thread in the scan's block passes
constexpr int kVolScanThreads = 1024;  // of the one workgroup that scans the block sums
constexpr int kScanBlock = kVolBlock * kScanPer;

// Counters of one build (device): whether some density is not above the threshold (else the early
// skip of chunk.rs:127-129 applies).
struct VolCounters {
    uint32_t below;
};

struct VolArgs {
    uw_field f;
    const uw_tables* tab;
    int32_t c[3];      // chunk coordinate
    int32_t n, L, T;   // cells, samples per axis, row segments per cell row
    int32_t WL;        // sign words per line
    int32_t live;      // octaves that are not zero on every sample (uw_live_octaves)
    float step;
    const uw_axis* axis;  // [3][O][L] (x hashed)
    const float* dfade;   // [3][O][L] fade derivative 30 d^2 (d - 1)^2
    const uint32_t* zrec; // L + 1 z records (uw_zrec_words(live) words each)
    float* dens;          // [(x L + z) L + y]
    uint32_t* words;           // sign words
    uint32_t* counts;          // [(x n + y) T + tz]: records | triangles << 10
    unsigned long long* rows;  // their exclusive scan, and the totals
    unsigned long long* bsum;  // per scan block
    uint32_t* bact;            // active cells per scan block
    VolCounters* cnt;
    uw_chunk_info* info;
    uw_totals* totals;
    float* verts;
    uint32_t* inds;
    uw_vertex_tape* tape;
    uw_emit_opts eo;
    uint64_t vcap, icap;
    int32_t zseg, zwords;  // z segments per line in the density kernel, sign words of each
    int32_t nx_tab;        // x entries per workgroup in the density kernel's LDS table
    uw_tiling tiling;      // emission tiles
};

// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(kVolBlock) k_vol_tables(VolArgs a, uw_axis* axis, float* dfade, uint32_t* zrec) {
    const int32_t O = a.f.octaves, L = a.L;
    const int64_t nent = int64_t(3) * O * L;
    const int64_t g = int64_t(blockIdx.x) * kVolBlock + threadIdx.x;
    if (g == 0) a.cnt->below = 0u;
    if (g < nent) {
        const int32_t ax = int32_t(g / (int64_t(O) * L));
        const int32_t r = int32_t(g - int64_t(ax) * O * L);
        const int32_t k = r / L, i = r - k * L;
        const double p = uw_sample_coord(a.f, ax, a.c[ax], i, a.step);
        uw_axis e = uw_axis_of(p, a.f.octave_freq[k]);
        if (ax == 0) {
            const uint32_t lo = e.bits & 255u, hi = (e.bits >> 8) & 255u;
            e.bits = uint32_t(a.tab->perm[lo]) | (uint32_t(a.tab->perm[hi]) << 8);
        }
        axis[g] = e;
        const double pk = p * a.f.octave_freq[k];
        const double d = pk - floor(pk);
        dfade[g] = float(30.0 * d * d * (d - 1.0) * (d - 1.0));
    } else if (g < nent + L + 1) {
        const int32_t i = int32_t(g - nent);
        uw_field f = a.f;
        f.octaves = a.live;
        uw_fill_zrec(f, a.c[2], L, a.step, i, zrec + size_t(i) * uw_zrec_words(a.live));
    }
}

// ---------------------------------------------------------------------------------------------
// Densities: lines t = x L + y, one per lane, workgroup b takes lines [256 b, 256 b + 256) over
// z segment s (whole sign words). The line's y entries are copied per lane into LDS, its x entries per
// distinct x of the workgroup. Only the octaves that are not zero on the whole grid are evaluated
// (uw_live_octaves): at the volume presets' one sample per world unit and base frequency 1/32, the
// sixth octave and those above have every sample on a lattice point, and they are the ones that build
// new lattice faces at every sample.
template <int OCT>
__global__ void __launch_bounds__(kVolBlock) k_vol_density(VolArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int32_t O = OCT > 0 ? OCT : a.live, OF = a.f.octaves;
    const int32_t L = a.L;
    uint2* GH = reinterpret_cast<uint2*>(smem);  // uw_grad_half of every permutation slot
    uint8_t* P = reinterpret_cast<uint8_t*>(GH + 256);
    uw_axis* AYs = reinterpret_cast<uw_axis*>(P + 256);  // [O][256] per line
    uw_axis* AXs = AYs + O * kVolBlock;                  // [nx_tab][pitch] per distinct x
    const int32_t pitch = uw_axis_pitch(O);
    const int tid = threadIdx.x;
    const int32_t seg = int32_t(blockIdx.x % uint32_t(a.zseg));
    const int64_t blk = int64_t(blockIdx.x / uint32_t(a.zseg));
    const int64_t lines = int64_t(L) * L;
    const int64_t t0 = blk * kVolBlock;
    const int64_t t = t0 + tid;
    const bool valid = t < lines;
    const int32_t xfirst = int32_t(t0 / L);
    const int32_t x = valid ? int32_t(t / L) : xfirst, y = valid ? int32_t(t - int64_t(x) * L) : 0;
    for (int i = tid; i < 256; i += kVolBlock) {
        const uint8_t p = a.tab->perm[i];
        P[i] = p;
        GH[i] = uw_grad_half(p & 15u);
    }
    for (int k = 0; k < O; ++k) AYs[k * kVolBlock + tid] = a.axis[(size_t(OF) + k) * L + y];
    for (int e = tid; e < O * a.nx_tab; e += kVolBlock) {
        const int k = e / a.nx_tab, j = e - k * a.nx_tab;
        const int32_t xx = min(xfirst + j, L - 1);  // entries past the grid are never read
        AXs[j * pitch + k] = a.axis[size_t(k) * L + xx];
    }
    __syncthreads();
    const int32_t w0 = seg * a.zwords, z0 = 32 * w0, z1 = min(L, z0 + 32 * a.zwords);
    float vmin = INFINITY, vmax = -INFINITY;
    if (z0 < z1 && __any(valid)) {
        const int32_t rw = OCT > 0 ? uw_zrec_words(OCT) : uw_zrec_words(O);
        const uw_axis* ax = AXs + (x - xfirst) * pitch;
        const uw_axis* ay = AYs + tid;
        float* out = a.dens + (size_t(x) * L + z0) * L + y;
        uint32_t* wout = a.words + size_t(t) * a.WL + w0;
        const size_t zstride = size_t(L);
        const float iso = a.f.iso;
        uint32_t word = 0;
        uw_field f = a.f;
        f.octaves = O;
        uw_noise_zline<OCT, true>(
            f, [=](int k) { return ax[k]; }, [=](int k) { return ay[k * kVolBlock]; }, P, GH,
            a.zrec + size_t(z0) * rw, rw, z1 - z0, vmin, vmax, [&](int32_t iz, float rho) {
                if (valid) out[size_t(iz) * zstride] = rho;
                word = uw_push_sign(word, rho, iso);
                if ((iz & 31) == 31) {  // uniform
                    if (valid) wout[iz >> 5] = __brev(word);
                    word = 0;
                }
            });
        const int32_t rest = (z1 - z0) & 31;
        if (rest && valid) wout[(z1 - z0) >> 5] = __brev(word) >> (32 - rest);
    }
    // one plain store of the same value by every workgroup that has such a sample: atomics of thousands
    // of workgroups on one address would queue
    if (__syncthreads_or(valid && uw_below_bits(vmin, vmax, a.f.iso) & UW_BELOW_NOT_ABOVE) && tid == 0) a.cnt->below = 1u;
}

// ---------------------------------------------------------------------------------------------
// Row-segment counts, one segment per thread and step, and their sums per scan block.
template <int THREADS>
__device__ __forceinline__ unsigned long long vol_block_scan(unsigned long long v, unsigned long long* total) {
    __shared__ unsigned long long ws[THREADS / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long inc = uw_wave_incl_scan(v);
    if (lane == 63) ws[wave] = inc;
    __syncthreads();
    unsigned long long base = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) {
        base += w < wave ? ws[w] : 0ull;
        sum += ws[w];
    }
    __syncthreads();
    *total = sum;
    return base + inc - v;
}

__global__ void __launch_bounds__(kVolBlock) k_vol_rows(VolArgs a, uint64_t nrows) {
    __shared__ uint32_t lut[256];
    const int tid = threadIdx.x;
    lut[tid] = a.tab->cell[tid];
    __syncthreads();
    const uint64_t b0 = uint64_t(blockIdx.x) * kScanBlock;
    unsigned long long s = 0;
    uint32_t act = 0;
#pragma unroll 2
    for (int j = 0; j < kScanPer; ++j) {
        const uint64_t r = b0 + uint64_t(j) * kVolBlock + tid;
        if (r < nrows) {
            const uint32_t q = uint32_t(r) / uint32_t(a.T);  // fewer than 2^23 row segments
            const int32_t tz = int32_t(uint32_t(r) - q * uint32_t(a.T));
            const int32_t x = int32_t(q / uint32_t(a.n)), y = int32_t(q - uint32_t(x) * uint32_t(a.n));
            uw_row_bits b;
            b.load(a.words, x, y, tz, a.n, a.L, a.WL);
            const uint32_t c = uw_row_counts(b, x, y, tz, lut);
            a.counts[r] = c & 0xFFFFFu;
            s += (unsigned long long)(c & 0x3FFu) | ((unsigned long long)((c >> 10) & 0x3FFu) << 32);
            act += c >> 20;
        }
    }
    unsigned long long tot, atot;
    (void)vol_block_scan<kVolBlock>(s, &tot);
    (void)vol_block_scan<kVolBlock>(act, &atot);
    if (tid == 0) {
        a.bsum[blockIdx.x] = tot;
        a.bact[blockIdx.x] = uint32_t(atot);
    }
}

// ---------------------------------------------------------------------------------------------
// Exclusive scan of the row-segment counts (u64 pairs that never carry between halves: both
// totals stay below 2^32 for n <= UW_VOLUME_MAX_RESOLUTION).

// One workgroup: exclusive scan of the block sums; the totals, the chunk record and the overflow
// flag (the emit kernel reads them).
__global__ void __launch_bounds__(kVolScanThreads) k_vol_scan_blocks(VolArgs a, uint32_t nblocks) {
    unsigned long long carry = 0, active = 0;
    for (uint32_t b0 = 0; b0 < nblocks; b0 += kVolScanThreads) {
        const uint32_t b = b0 + threadIdx.x;
        const unsigned long long v = b < nblocks ? a.bsum[b] : 0ull;
        const unsigned long long ac = b < nblocks ? a.bact[b] : 0ull;
        unsigned long long tot;
        const unsigned long long ex = vol_block_scan<kVolScanThreads>(v, &tot);
        if (b < nblocks) a.bsum[b] = carry + ex;
        carry += tot;
        (void)vol_block_scan<kVolScanThreads>(ac, &tot);
        active += tot;
    }
    if (threadIdx.x == 0) {
        const VolCounters cn = *a.cnt;
        const uint64_t nv = carry & 0xFFFFFFFFull, ni = 3ull * (carry >> 32);
        uint32_t flags = 0;
        if (!cn.below) flags = UW_CHUNK_BLANK | UW_CHUNK_EARLY_SKIP;
        else if (ni == 0) flags = UW_CHUNK_BLANK;
        const bool ovf = nv > a.vcap || ni > a.icap;
        if (ovf) flags |= UW_CHUNK_OVERFLOW;
        if (a.eo.ind16 && nv > 65535u) flags |= UW_CHUNK_INDEX_WRAP;
        uw_chunk_info r = {flags, uint32_t(nv), uint32_t(ni), uint32_t(active), 0, 0};
        *a.info = r;
        uw_totals t;
        t.n_verts = nv;
        t.n_inds = ni;
        t.n_nonblank = ni > 0 ? 1u : 0u;
        t.overflow = ovf ? 1u : 0u;
        *a.totals = t;
    }
}

__global__ void __launch_bounds__(kVolBlock) k_vol_scan_apply(const uint32_t* __restrict__ counts,
                                                              unsigned long long* __restrict__ rows, uint64_t nrows,
                                                              const unsigned long long* __restrict__ bsum) {
    const uint64_t b0 = uint64_t(blockIdx.x) * kScanBlock;
    unsigned long long carry = bsum[blockIdx.x];
    uint32_t c[kScanPer];
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
        const uint64_t i = b0 + uint64_t(j) * kVolBlock + threadIdx.x;
        c[j] = i < nrows ? counts[i] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
        const uint64_t i = b0 + uint64_t(j) * kVolBlock + threadIdx.x;
        const unsigned long long v = (unsigned long long)(c[j] & 0x3FFu) | ((unsigned long long)(c[j] >> 10) << 32);
        unsigned long long tot;
        const unsigned long long ex = vol_block_scan<kVolBlock>(v, &tot);
        if (i < nrows) rows[i] = carry + ex;
        if (i + 1 == nrows) rows[nrows] = carry + ex + v;
        carry += tot;
    }
}

// ---------------------------------------------------------------------------------------------
// Emission: persistent workgroups over the tiles (uw_emit_rows), z segments of one tile row next to
// each other.
template <bool EXTRA>
__global__ void __launch_bounds__(kEmitThreads, EXTRA ? 5 : 6) k_vol_emit(VolArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uw_totals tot = *a.totals;
    if (tot.overflow || tot.n_inds == 0) return;
    uw_emit_tables(a.tab, smem);
    uw_emit_tile e;
    e.eo = a.eo;
    e.iso = a.f.iso;
    e.step = a.step;
    e.ox = float(a.f.extent * a.c[0]);
    e.oy = float(a.f.extent * a.c[1]);
    e.oz = float(a.f.extent * a.c[2]);
    e.extent = float(a.f.extent);
    e.n = a.n;
    e.L = a.L;
    e.T = a.T;
    e.WL = a.WL;
    e.cells = a.tiling.cells;
    e.dens = a.dens;
    e.sx = a.L * a.L;
    e.sy = 1;
    e.sz = a.L;
    e.words = a.words;
    e.rows = a.rows;
    e.vo = e.io = 0;
    e.vlim = tot.n_verts;
    e.ilim = tot.n_inds;
    e.verts = a.verts;
    e.inds = a.inds;
    e.tape = a.tape;
    // Workgroups go to the eight XCDs in turn: XCD q takes the tile rows (x slab, y range) q, q + 8, ...
    // and its workgroups their z segments side by side, whose mesh ranges interleave row by row: the
    // partly written lines meet in that XCD's L2.
    const uint32_t T = uint32_t(a.tiling.T), yt = uint32_t(a.tiling.yt), strips = uint32_t(a.tiling.xt) * yt;
    const uint32_t nx = gridDim.x < 8u ? gridDim.x : 8u, xcd = blockIdx.x % nx, per = (gridDim.x - xcd + nx - 1u) / nx;
    const uint32_t mine = (strips > xcd ? (strips - xcd + nx - 1u) / nx : 0u) * T;  // tiles of this XCD
    auto place = [&](uint32_t i) {
        const uint32_t s = i / T, strip = s * nx + xcd, xt = strip / yt;
        e.X0 = int32_t(xt) * a.tiling.planes;
        e.X1 = min(a.n, e.X0 + a.tiling.planes);
        e.Y0 = int32_t(strip - xt * yt) * 32;
        e.Y1 = min(a.n, e.Y0 + 32);
        e.tz = int32_t(i - s * T);
    };
    uint32_t i = blockIdx.x / nx;
    if (i >= mine) return;
    place(i);
    uw_emit_row row = uw_emit_load(e);
    for (;;) {
        const uw_emit_tile cur = e;
        const uw_emit_row r = row;
        i += per;
        if (i < mine) {  // the next tile's row segments arrive during this one
            place(i);
            row = uw_emit_load(e);
        }
        uw_emit_rows<EXTRA>(cur, r, smem);
        if (i >= mine) return;
        __syncthreads();  // the tile's LDS is written again
    }
}

// ---------------------------------------------------------------------------------------------
// Backward over the volume's vertices (the adjoint of uw_adjoint.hip for one grid): the octave
// values and gradients at each vertex's endpoint samples are recomputed from the per-axis tables of the
// grid (read through the cache; 3 O L entries). Per-workgroup parameter sums in f64, added in
// workgroup order by k_vol_backward_sum.
//
// A sample is an endpoint of several vertices: of the 128 endpoints of 64 consecutive vertices, 73 are
// different samples (96^3 cells of the volume preset). A wave adds up the weights of each of its
// batch's samples first, in a hash table of its own in LDS (a wave's LDS operations run in order, so
// runs agree), moves the samples on to a queue, and evaluates 64 of the queue at a time. The density
// gradient takes one atomic per sample and batch; the hash leaves samples that are neighbours along z in
// neighbouring slots, so that their atomics share a request. Octaves that are zero on every sample
// (uw_live_octaves) have value 0 and, all fades and their derivatives being 0 there, the gradient of
// the lattice point itself. 31 M vertices of 512^3 cells: 1320 us where one endpoint at a time took 2480
// (without the density gradient 1110; atomics in a scattering hash's order alone took 1550).
constexpr int kVolBwdParts = 19;   // UW_MAX_OCTAVES + 3
constexpr int kVolBwdPerCu = 6;    // workgroups per compute unit at most: LDS
constexpr uint32_t kSampleSlots = 256, kSampleNone = 0xFFFFFFFFu;  // hash slots, at most 128 taken
constexpr uint32_t kSampleQueue = 192;  // 63 left over and 128 new ones

template <int LIVE>
__global__ void __launch_bounds__(kVolBlock) k_vol_backward(VolArgs a, const uw_chunk_info* __restrict__ info,
                                                            const uw_vertex_tape* __restrict__ tape,
                                                            const float* __restrict__ grad_verts, float* grad_dens,
                                                            int want_params, double* __restrict__ part) {
    constexpr int OMAX = LIVE > 0 ? LIVE : UW_MAX_OCTAVES;
    constexpr int kWaves = kVolBlock / 64;
    __shared__ uint2 GH[256];
    __shared__ uint8_t P[256];
    __shared__ double HW[kWaves][kSampleSlots], QW[kWaves][kSampleQueue];
    __shared__ uint32_t HK[kWaves][kSampleSlots], QK[kWaves][kSampleQueue];
    __shared__ double red[kWaves][OMAX + kParamExtra], sums[UW_MAX_OCTAVES + kParamExtra];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < 256; i += kVolBlock) {
        const uint8_t p = a.tab->perm[i];
        P[i] = p;
        GH[i] = uw_grad_half(p & 15u);
    }
    double* hw = HW[wave];
    double* qw = QW[wave];
    uint32_t* hk = HK[wave];
    uint32_t* qk = QK[wave];
    for (uint32_t i = lane; i < kSampleSlots; i += 64) {
        hk[i] = kSampleNone;
        hw[i] = 0.0;
    }
    __syncthreads();
    const uw_chunk_info ci = *info;
    const bool skip = (ci.flags & (UW_CHUNK_OVERFLOW | UW_CHUNK_INVALID)) != 0;
    const int32_t O = a.f.octaves, live = LIVE > 0 ? LIVE : a.live, L = a.L;
    const uint32_t uL = uint32_t(L);
    const float iso = a.f.iso;
    double acc[OMAX + kParamExtra];  // uw_param_grad's N (the live octaves), G, W, T
#pragma unroll
    for (int k = 0; k < OMAX + kParamExtra; ++k) acc[k] = 0.0;
    auto evaluate = [&](uint32_t s, double we) {
        const uint32_t xy = s / uL, zz = s - xy * uL, xx = xy / uL, yy = xy - xx * uL;
        // octave k's entry of an axis: a scalar base per octave, one offset per lane
        auto entry = [&](int ax, int k, uint32_t i) { return *(a.axis + (size_t(ax) * O + k) * L + i); };
        auto dfade = [&](int ax, int k, uint32_t i) { return *(a.dfade + (size_t(ax) * O + k) * L + i); };
        float total = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
#pragma unroll
        for (int k = 0; k < OMAX; ++k) {
            if (k < live) {
                float g[3];
                const float nk = uw_octave_grad(entry(0, k, xx), entry(1, k, yy), entry(2, k, zz), dfade(0, k, xx),
                                                dfade(1, k, yy), dfade(2, k, zz), P, GH, g);
                const float af = a.f.amp[k] * float(a.f.octave_freq[k]);
                acc[k] = fma(we, double(nk), acc[k]);
                total = fmaf(a.f.amp[k], nk, total);
                gx = fmaf(af, g[0], gx);
                gy = fmaf(af, g[1], gy);
                gz = fmaf(af, g[2], gz);
            }
        }
        for (int k = live; k < O; ++k) {
            const uint32_t b = P[(entry(0, k, xx).bits ^ entry(1, k, yy).bits) & 255u];
            const uint2 g = GH[b ^ (entry(2, k, zz).bits & 255u)];
            const float af = a.f.amp[k] * float(a.f.octave_freq[k]);
            gx = fmaf(af, uw_mix_mul_x(g.x, UW_PERLIN_SCALE), gx);
            gy = fmaf(af, uw_mix_mul_x(g.x >> 16, UW_PERLIN_SCALE), gy);
            gz = fmaf(af, uw_mix_mul_x(g.y, UW_PERLIN_SCALE), gz);
        }
        acc[OMAX + 0] = fma(we, double(gx), acc[OMAX + 0]);
        acc[OMAX + 1] = fma(we, double(gy), acc[OMAX + 1]);
        acc[OMAX + 2] = fma(we, double(gz), acc[OMAX + 2]);
        acc[OMAX + 3] += we;
        acc[OMAX + 4] = fma(we, double(total), acc[OMAX + 4]);
    };
    auto add = [&](uint32_t s, float w) {  // (128 samples at most in 256 slots: a free one is found)
        uint32_t h = (s + 64u * (s >> 9)) & (kSampleSlots - 1u);
        for (;;) {
            const uint32_t was = atomicCAS(hk + h, kSampleNone, s);
            if (was == kSampleNone || was == s) break;
            h = (h + 1u) & (kSampleSlots - 1u);
        }
        __hip_atomic_fetch_add(hw + h, double(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const uint64_t nv = skip ? 0 : ci.n_verts, batches = (nv + 63) / 64;
    uint32_t queued = 0;  // wave-uniform
    const uint64_t b0 = uint64_t(blockIdx.x) * kWaves + wave, stride = uint64_t(gridDim.x) * kWaves;
    uw_vertex_tape next = {0u, 0u, 0.0f, 0.0f};  // the next batch's records, fetched a batch ahead
    if (b0 * 64 + lane < nv) next = tape[b0 * 64 + lane];
    for (uint64_t b = b0; b < batches; b += stride) {
        const uint64_t v = b * 64 + lane;
        const uw_vertex_tape tv = next;
        if (v + 64 * stride < nv) next = tape[v + 64 * stride];
        if (v < nv) {
            const int64_t diff = int64_t(tv.b) - int64_t(tv.a);
            const int axis = (diff == 1 || diff == -1) ? 2 : ((diff == L || diff == -L) ? 1 : 0);
            const float dir = diff > 0 ? a.step : -a.step;
            const float gv = grad_verts[3 * v + axis] * dir;
            const float D = tv.rho_b - tv.rho_a;
            const float inv_d2 = 1.0f / (D * D);
            add(tv.a, gv * (iso - tv.rho_b) * inv_d2);
            add(tv.b, gv * (tv.rho_a - iso) * inv_d2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t j = 0; j < kSampleSlots; j += 64) {
            const uint32_t s = hk[j + lane];
            const bool taken = s != kSampleNone;
            const uint64_t m = __ballot(taken);
            if (taken) {
                const double w = hw[j + lane];
                hk[j + lane] = kSampleNone;
                hw[j + lane] = 0.0;
                if (grad_dens) unsafeAtomicAdd(grad_dens + s, float(w));
                if (want_params) {
                    const uint32_t at = queued + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
                    qk[at] = s;
                    qw[at] = w;
                }
            }
            if (want_params) queued += uint32_t(__popcll(m));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        while (queued >= 64) {
            queued -= 64;
            evaluate(qk[queued + lane], qw[queued + lane]);
        }
    }
    if (!want_params) return;
    if (uint32_t(lane) < queued) evaluate(qk[lane], qw[lane]);
#pragma unroll
    for (int k = 0; k < OMAX + kParamExtra; ++k) {
        const double t = uw_wave_sum_f64(acc[k]);
        if (lane == 0) red[wave][k] = t;
    }
    __syncthreads();
    // sums: N of every octave (0 from the first one that is zero everywhere on), G, W, T
    if (tid < UW_MAX_OCTAVES + kParamExtra) {
        const int src = tid < O ? (tid < live ? tid : -1) : OMAX + tid - O;
        double t = 0.0;
        if (src >= 0 && src < OMAX + kParamExtra)
            for (int w = 0; w < kWaves; ++w) t += red[w][src];
        sums[tid] = t;
    }
    __syncthreads();
    if (tid < O + 3) part[size_t(blockIdx.x) * kVolBwdParts + tid] = uw_param_grad(a.f, sums, O, tid);
}

// One workgroup per parameter: each thread adds a stride of the workgroup sums, then the waves'
// totals are added in wave order (a fixed order, so runs agree). A single thread walking all
// workgroups' sums in turn waited on one load per sum: 0.64 ms for 2048 workgroups.
__global__ void __launch_bounds__(kVolBlock) k_vol_backward_sum(const double* __restrict__ part, int32_t nblocks,
                                                                int32_t O, double* grad_amp, double* grad_off) {
    __shared__ double ws[kVolBlock / 64];
    const int k = int(blockIdx.x), tid = threadIdx.x;
    double t = 0.0;
    for (int32_t b = tid; b < nblocks; b += kVolBlock) t += part[size_t(b) * kVolBwdParts + k];
    t = uw_wave_sum_f64(t);
    if ((tid & 63) == 0) ws[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < kVolBlock / 64; ++w) s += ws[w];
        if (k < O) {
            if (grad_amp) grad_amp[k] = s;
        } else if (grad_off) {
            grad_off[k - O] = s;
        }
    }
}

// ---------------------------------------------------------------------------------------------
struct VolLayout {
    size_t axis_off, df_off, zrec_off, dens_off, words_off, counts_off, rows_off, bsum_off, bact_off, cnt_off, part_off, bytes;
    uint64_t nrows;
    uint32_t nscan;
};

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

VolLayout vol_layout(int32_t n, int32_t octaves, int32_t bwd_blocks) {
    VolLayout l;
    const size_t L = size_t(n) + 1;
    const size_t T = size_t(uw_row_segs(n));
    l.nrows = uint64_t(n) * uint64_t(n) * T;
    l.nscan = uint32_t((l.nrows + kScanBlock - 1) / kScanBlock);
    size_t o = 0;
    l.axis_off = o;
    o = align256(o + 3 * size_t(octaves) * L * sizeof(uw_axis));
    l.df_off = o;
    o = align256(o + 3 * size_t(octaves) * L * sizeof(float));
    l.zrec_off = o;
    o = align256(o + (L + 1) * size_t(uw_zrec_words(octaves)) * sizeof(uint32_t));
    l.dens_off = o;
    o = align256(o + L * L * L * sizeof(float));
    l.words_off = o;
    o = align256(o + L * L * size_t(uw_sign_words(n + 1)) * sizeof(uint32_t));
    l.counts_off = o;
    o = align256(o + size_t(l.nrows) * sizeof(uint32_t));
    l.rows_off = o;
    o = align256(o + size_t(l.nrows + 1) * sizeof(unsigned long long));
    l.bsum_off = o;
    o = align256(o + size_t(l.nscan) * sizeof(unsigned long long));
    l.bact_off = o;
    o = align256(o + size_t(l.nscan) * sizeof(uint32_t));
    l.cnt_off = o;
    o = align256(o + sizeof(VolCounters));
    l.part_off = o;
    o = align256(o + size_t(bwd_blocks) * kVolBwdParts * sizeof(double));
    l.bytes = o;
    return l;
}

int vol_backward_blocks(const uw_ctx* ctx) { return ctx->num_cus * kVolBwdPerCu; }  // at most

// Fills the launch arguments over the context's volume scratch (grown as needed).
int vol_prepare(uw_ctx* ctx, int32_t cx, int32_t cy, int32_t cz, int32_t n, VolArgs* a, VolLayout* lay) {
    const int32_t O = ctx->params.octaves;
    *lay = vol_layout(n, O, vol_backward_blocks(ctx));
    if (lay->bytes > ctx->vol_bytes) {
        (void)hipFree(ctx->d_vol);
        ctx->d_vol = nullptr;
        ctx->vol_bytes = 0;
        UW_ALLOC(ctx, ctx->d_vol, lay->bytes);
        ctx->vol_bytes = lay->bytes;
    }
    unsigned char* base = ctx->d_vol;
    memset(a, 0, sizeof(*a));
    a->f = uw_make_field(ctx->params);
    a->tab = ctx->d_tables;
    a->c[0] = cx;
    a->c[1] = cy;
    a->c[2] = cz;
    a->n = n;
    a->L = n + 1;
    a->T = uw_row_segs(n);
    a->WL = uw_sign_words(n + 1);
    a->live = uw_live_octaves(a->f, a->c, n, float(a->f.extent) / float(n));
    a->step = float(a->f.extent) / float(n);
    a->axis = reinterpret_cast<const uw_axis*>(base + lay->axis_off);
    a->dfade = reinterpret_cast<const float*>(base + lay->df_off);
    a->zrec = reinterpret_cast<const uint32_t*>(base + lay->zrec_off);
    a->dens = reinterpret_cast<float*>(base + lay->dens_off);
    a->words = reinterpret_cast<uint32_t*>(base + lay->words_off);
    a->counts = reinterpret_cast<uint32_t*>(base + lay->counts_off);
    a->bact = reinterpret_cast<uint32_t*>(base + lay->bact_off);
    a->rows = reinterpret_cast<unsigned long long*>(base + lay->rows_off);
    a->bsum = reinterpret_cast<unsigned long long*>(base + lay->bsum_off);
    a->cnt = reinterpret_cast<VolCounters*>(base + lay->cnt_off);
    const int32_t L = n + 1;
    // z segments of whole sign words: as many as give every SIMD kDensityWaves waves (each forces a
    // set-up of every octave's lattice cell at its first sample)
    constexpr int64_t kDensityWaves = 12;
    const int64_t line_waves = (int64_t(L) * L + 63) / 64, want = kDensityWaves * 4 * ctx->num_cus;
    int64_t segs = (want + line_waves - 1) / line_waves;
    segs = segs < 1 ? 1 : segs > a->WL ? a->WL : segs;
    a->zwords = int32_t((a->WL + segs - 1) / segs);
    a->zseg = (a->WL + a->zwords - 1) / a->zwords;
    a->nx_tab = kVolBlock / L + 2;
    if (a->nx_tab > L) a->nx_tab = L;
    return UW_OK;
}

using VolDensityKernel = void (*)(VolArgs);
VolDensityKernel pick_vol_density(int octaves) {
    switch (octaves) {
        case 1: return k_vol_density<1>;
        case 2: return k_vol_density<2>;
        case 3: return k_vol_density<3>;
        case 4: return k_vol_density<4>;
        case 5: return k_vol_density<5>;
        case 6: return k_vol_density<6>;
        case 7: return k_vol_density<7>;
        case 8: return k_vol_density<8>;
        default: return k_vol_density<0>;
    }
}

using VolBackwardKernel = void (*)(VolArgs, const uw_chunk_info*, const uw_vertex_tape*, const float*, float*, int, double*);
VolBackwardKernel pick_vol_backward(int octaves) {
    switch (octaves) {
        case 1: return k_vol_backward<1>;
        case 2: return k_vol_backward<2>;
        case 3: return k_vol_backward<3>;
        case 4: return k_vol_backward<4>;
        case 5: return k_vol_backward<5>;
        case 6: return k_vol_backward<6>;
        case 7: return k_vol_backward<7>;
        case 8: return k_vol_backward<8>;
        default: return k_vol_backward<0>;
    }
}

// The tables kernel (per-axis entries, z records, counters reset); shared by forward and backward.
int vol_launch_tables(uw_ctx* ctx, VolArgs& a, const VolLayout& lay, hipStream_t st) {
    unsigned char* base = ctx->d_vol;
    const int64_t work = int64_t(3) * a.f.octaves * a.L + a.L + 1;
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_VOLUME_TABLES)) return rc;
    hipLaunchKernelGGL(k_vol_tables, dim3(uint32_t((work + kVolBlock - 1) / kVolBlock)), dim3(kVolBlock), 0, st, a,
                       reinterpret_cast<uw_axis*>(base + lay.axis_off), reinterpret_cast<float*>(base + lay.df_off),
                       reinterpret_cast<uint32_t*>(base + lay.zrec_off));
    return uw_prof_end(ctx, st);
}

bool vol_args_ok(int32_t n, const uw_mesh_out* out) {
    return n >= 1 && n <= UW_VOLUME_MAX_RESOLUTION && out && out->info && out->totals && out->vertex_format <= 1 &&
           out->index_format <= 1 && (out->vert_cap == 0 || out->verts) && (out->ind_cap == 0 || out->inds);
}

}  // namespace

extern "C" {

int uw_build_volume(uw_ctx* ctx, int32_t cx, int32_t cy, int32_t cz, int32_t n, const uw_mesh_out* out,
                    uw_vertex_tape* tape, void* stream) {
    if (!ctx) return UW_ERR_INVALID_ARG;
    if (!vol_args_ok(n, out)) return uw_fail(ctx, UW_ERR_INVALID_ARG, "bad arguments (1 <= n <= UW_VOLUME_MAX_RESOLUTION)");
    UW_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = uw_refuse_capture(ctx, st)) return rc;
    VolArgs a;
    VolLayout lay;
    if (int rc = vol_prepare(ctx, cx, cy, cz, n, &a, &lay)) return rc;
    a.info = out->info;
    a.totals = out->totals;
    a.verts = out->verts;
    a.inds = out->inds;
    a.tape = tape;
    a.eo = uw_make_emit_opts(out);
    a.vcap = out->vert_cap;
    a.icap = out->ind_cap;
    if (int rc = vol_launch_tables(ctx, a, lay, st)) return rc;
    // densities
    const VolDensityKernel dk = pick_vol_density(a.live);
    const size_t lds = 256 * sizeof(uint2) + 256 +
                       sizeof(uw_axis) * (size_t(a.live) * kVolBlock + size_t(uw_axis_pitch(a.live)) * size_t(a.nx_tab));
    UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(dk), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds)));
    const uint64_t lines = uint64_t(a.L) * uint64_t(a.L);
    const uint64_t dblocks = (lines + kVolBlock - 1) / kVolBlock * uint64_t(a.zseg);
    if (int rc = uw_prof_start(ctx, st)) return rc;
    hipLaunchKernelGGL(dk, dim3(uint32_t(dblocks)), dim3(kVolBlock), lds, st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_VOLUME_COUNT)) return rc;
    hipLaunchKernelGGL(k_vol_rows, dim3(lay.nscan), dim3(kVolBlock), 0, st, a, lay.nrows);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_VOLUME_SCAN)) return rc;
    hipLaunchKernelGGL(k_vol_scan_blocks, dim3(1), dim3(kVolScanThreads), 0, st, a, lay.nscan);
    hipLaunchKernelGGL(k_vol_scan_apply, dim3(lay.nscan), dim3(kVolBlock), 0, st, a.counts, a.rows, lay.nrows, a.bsum);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    // tiles as deep as the emitter takes (5 planes of 33 rows: 922 us for 512^3, 3 planes 979), shallower
    // while there are fewer than 4 per compute unit (150^3: 37.5 us in 3 planes, 42.5 in one, whose halo is
    // as large as itself)
    int32_t planes = uw_tile_planes(n);
    a.tiling = uw_tiling_for(n, planes);
    while (planes > 1 && int64_t(a.tiling.tiles()) < 4 * int64_t(ctx->num_cus)) {
        planes = (planes + 1) / 2;
        a.tiling = uw_tiling_for(n, planes);
    }
    if (!uw_emit_takes(a.tiling.max_rows, a.tiling.cells + (a.tiling.yt > 1 ? 1 : 0), a.tiling.cells))
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "emission tiles larger than a workgroup takes");
    const size_t elds = uw_emit_lds_bytes(a.tiling.max_rows, a.tiling.cells);
    using VolEmitKernel = void (*)(VolArgs);
    const VolEmitKernel ek = uw_emit_extra(a.eo) ? k_vol_emit<true> : k_vol_emit<false>;
    UW_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(ek), hipFuncAttributeMaxDynamicSharedMemorySize, int(elds)));
    int per_cu = 0;
    if (int rc = uw_resident(ctx, reinterpret_cast<const void*>(ek), kEmitThreads, elds, &per_cu)) return rc;
    if (per_cu < 1) return uw_fail(ctx, UW_ERR_INVALID_ARG, "emit kernel does not fit on a CU");
    const int resident = per_cu * ctx->num_cus;
    if (int rc = uw_prof_start(ctx, st, UW_STAGE_VOLUME_EMIT)) return rc;
    hipLaunchKernelGGL(ek, dim3(uint32_t(resident < a.tiling.tiles() ? resident : a.tiling.tiles())), dim3(kEmitThreads),
                       elds, st, a);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

int uw_volume_backward(uw_ctx* ctx, int32_t cx, int32_t cy, int32_t cz, int32_t n, const uw_chunk_info* info,
                       const uw_vertex_tape* tape, const float* grad_verts, float* grad_dens, double* grad_amp,
                       double* grad_off, void* stream) {
    if (!ctx) return UW_ERR_INVALID_ARG;
    if (n < 1 || n > UW_VOLUME_MAX_RESOLUTION || !info || !tape || !grad_verts)
        return uw_fail(ctx, UW_ERR_INVALID_ARG, "bad arguments");
    UW_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = uw_refuse_capture(ctx, st)) return rc;
    VolArgs a;
    VolLayout lay;
    if (int rc = vol_prepare(ctx, cx, cy, cz, n, &a, &lay)) return rc;
    if (int rc = vol_launch_tables(ctx, a, lay, st)) return rc;
    const int want = (grad_amp || grad_off) ? 1 : 0;
    // as many workgroups as are resident (registers: 3 to 6 per compute unit by octave count), so that
    // all take the same number of batches
    const VolBackwardKernel bk = pick_vol_backward(a.live);
    int per_cu = 0;
    if (int rc = uw_resident(ctx, reinterpret_cast<const void*>(bk), kVolBlock, 0, &per_cu)) return rc;
    if (per_cu < 1) return uw_fail(ctx, UW_ERR_INVALID_ARG, "backward kernel does not fit on a CU");
    const int blocks = (per_cu < kVolBwdPerCu ? per_cu : kVolBwdPerCu) * ctx->num_cus;
    double* part = reinterpret_cast<double*>(ctx->d_vol + lay.part_off);
    const int O = a.f.octaves;
    if (int rc = uw_prof_start(ctx, st)) return rc;
    hipLaunchKernelGGL(bk, dim3(blocks), dim3(kVolBlock), 0, st, a, info, tape, grad_verts, grad_dens,
                       want, part);
    if (want) hipLaunchKernelGGL(k_vol_backward_sum, dim3(O + 3), dim3(kVolBlock), 0, st, part, blocks, O, grad_amp, grad_off);
    if (int rc = uw_prof_end(ctx, st)) return rc;
    UW_HIP(ctx, hipGetLastError());
    return UW_OK;
}

uint64_t uw_volume_scratch_bytes(const uw_ctx* ctx, int32_t n) {
    if (!ctx || n < 1 || n > UW_VOLUME_MAX_RESOLUTION) return 0;
    return vol_layout(n, ctx->params.octaves, vol_backward_blocks(ctx)).bytes;
}

}  // extern "C"
