// Device-side density field: sample coordinates, Perlin octaves and the z-bias.
//
// Restates, for FP32 VALU execution, the reference's density:
//   Chunk::build_iso coordinates           underwater_world/src/chunk.rs:107-116
//   perlin_util::perlin_3d_octaves          underwater_world/src/perlin_util.rs:6-22
//   perlin_util::iso_at (bias)              underwater_world/src/perlin_util.rs:24-29
//   noise 0.8.2 core::perlin::perlin_3d     (external crate, call site perlin_util.rs:13)
//
// Numerics. Sample coordinates are formed in f64 exactly as the reference does, and per axis the
// lattice index, the fraction d, d - 1 and the quintic fade s(d) are derived in f64 and rounded
// once to f32. These per-axis quantities are shared by every sample of a grid line, so they are
// computed once per (axis index, octave) into LDS. Only the per-sample combination runs in f32:
// eight gradient dots (one rounding each: the gradients are {-1,0,1} vectors with two nonzero
// components) and seven FMA lerps, which equal the crate's 8-term multilinear polynomial
// k0 + k1 a + ... + k7 a b c in exact arithmetic.
#pragma once

#include "uw_internal.h"

// One axis of one octave: hashed/low lattice bytes and the f32-rounded fraction data.
struct __align__(16) uw_axis {
    uint32_t bits;  // x axis: P[L & 255] | P[(L+1) & 255] << 8; y, z axes: (L & 255) | ((L+1) & 255) << 8
    float d;        // p - floor(p)
    float dm1;      // d - 1
    float fade;     // d^3 (d (6 d - 15) + 10)
};

// LDS tables of axis entries keep a sample's octaves together, [sample][octave], so that an octave's
// entry is at a constant offset from the lane's; an odd pitch spreads the 16-byte reads of consecutive
// samples over all banks.
__host__ __device__ constexpr int32_t uw_axis_pitch(int32_t octaves) { return octaves | 1; }

// 1/(sqrt(3)/2), noise 0.8.2 perlin_3d SCALE_FACTOR, rounded to f32.
#define UW_PERLIN_SCALE 1.1547005383792515f

// Noise coordinate of sample i of chunk c along `axis` (chunk.rs:107-108): all f64; the product
// by a power-of-two frequency equals the reference's division by CHUNK_SIZE, and the world-space
// offset (0 for the reference, where adding it is exact) shifts every sample.
__device__ __forceinline__ double uw_sample_coord(const uw_field& f, int axis, int32_t c, int32_t i, float step) {
    const double local = double(i) * double(step);
    return ((local + double(f.extent * c)) + f.offset[axis]) * f.frequency;
}

__device__ __forceinline__ double uw_quintic64(double t) { return t * t * t * (t * (t * 6.0 - 15.0) + 10.0); }

__device__ __forceinline__ uw_axis uw_axis_of(double p, double fk) {
    const double pk = p * fk;
    const double fl = floor(pk);
    const int64_t L = int64_t(fl);
    const double d = pk - fl;
    uw_axis a;
    a.bits = uint32_t(L & 255) | (uint32_t((L + 1) & 255) << 8);
    a.d = float(d);
    a.dm1 = float(d - 1.0);
    a.fade = float(uw_quintic64(d));
    return a;
}

// Fold the first hash level into an x-axis entry.
__device__ __forceinline__ uw_axis uw_hash_x(uw_axis a, const uint8_t* perm) {
    a.bits = uint32_t(perm[a.bits & 255]) | (uint32_t(perm[(a.bits >> 8) & 255]) << 8);
    return a;
}

__device__ __forceinline__ float uw_gdot(float4 g, float x, float y, float z) {
    return fmaf(g.z, z, fmaf(g.y, y, g.x * x));
}

__device__ __forceinline__ float uw_lerp(float t, float a, float b) { return fmaf(t, b - a, a); }

// Gradient of permutation slot j (components exactly -1, 0 or 1) from an LDS table of three floats per
// slot: the 12-byte stride spreads the slots of a gather over all LDS banks.
__device__ __forceinline__ float4 uw_grad3(const float* G3, uint32_t j) {
    const float* g = G3 + 3u * j;
    return make_float4(g[0], g[1], g[2], 0.0f);
}

// Gradient vector of hash code h (0..15) from the packed constants: no table load, so filling a
// per-slot LDS table costs one memory round trip (the permutation) instead of two.
__device__ __forceinline__ float4 uw_grad_vec(uint32_t h) {
    constexpr uint32_t kx = uw_grad_pack(0), ky = uw_grad_pack(1), kz = uw_grad_pack(2);
    const uint32_t sh = 2u * h;
    const int gx = __builtin_amdgcn_sbfe(int(kx), sh, 2u);
    const int gy = __builtin_amdgcn_sbfe(int(ky), sh, 2u);
    const int gz = __builtin_amdgcn_sbfe(int(kz), sh, 2u);
    return make_float4(float(gx), float(gy), float(gz), 0.0f);
}

// One octave of improved Perlin noise at the lattice cell / fractions given by X (hashed), Y, Z.
// P: permutation table; G3: gradient source (uw_grad3).
template <class GT>
__device__ __forceinline__ float uw_perlin_octave(const uw_axis& X, const uw_axis& Y, const uw_axis& Z,
                                                  const uint8_t* P, GT G3) {
    const uint32_t a0 = X.bits & 255, a1 = X.bits >> 8;
    const uint32_t y0 = Y.bits & 255, y1 = Y.bits >> 8;
    const uint32_t z0 = Z.bits & 255, z1 = Z.bits >> 8;
    const uint32_t b00 = P[a0 ^ y0], b01 = P[a0 ^ y1], b10 = P[a1 ^ y0], b11 = P[a1 ^ y1];
    const float g000 = uw_gdot(uw_grad3(G3, b00 ^ z0), X.d, Y.d, Z.d);
    const float g100 = uw_gdot(uw_grad3(G3, b10 ^ z0), X.dm1, Y.d, Z.d);
    const float g010 = uw_gdot(uw_grad3(G3, b01 ^ z0), X.d, Y.dm1, Z.d);
    const float g110 = uw_gdot(uw_grad3(G3, b11 ^ z0), X.dm1, Y.dm1, Z.d);
    const float g001 = uw_gdot(uw_grad3(G3, b00 ^ z1), X.d, Y.d, Z.dm1);
    const float g101 = uw_gdot(uw_grad3(G3, b10 ^ z1), X.dm1, Y.d, Z.dm1);
    const float g011 = uw_gdot(uw_grad3(G3, b01 ^ z1), X.d, Y.dm1, Z.dm1);
    const float g111 = uw_gdot(uw_grad3(G3, b11 ^ z1), X.dm1, Y.dm1, Z.dm1);
    const float x00 = uw_lerp(X.fade, g000, g100);
    const float x10 = uw_lerp(X.fade, g010, g110);
    const float x01 = uw_lerp(X.fade, g001, g101);
    const float x11 = uw_lerp(X.fade, g011, g111);
    const float y0v = uw_lerp(Y.fade, x00, x10);
    const float y1v = uw_lerp(Y.fade, x01, x11);
    const float r = uw_lerp(Z.fade, y0v, y1v) * UW_PERLIN_SCALE;
    return fminf(fmaxf(r, -1.0f), 1.0f);
}

// Bias split: rho = (adj + p) + post.  Terrace (perlin_util.rs:27-28): adj = (z * a) / b,
// post = -fmod(adj, c) (u - m == u + (-m) exactly). Linear: adj = z * a, post = b.
__device__ __forceinline__ void uw_bias_terms(const uw_field& f, double pz, float* adj, float* post) {
    const float z32 = float(pz);
    if (f.bias_kind == UW_BIAS_TERRACE) {
        const float a = (z32 * f.bias_a) / f.bias_b;
        *adj = a;
        *post = -fmodf(a, f.bias_c);
    } else {
        *adj = z32 * f.bias_a;
        *post = f.bias_b;
    }
}

__device__ __forceinline__ float uw_density_from(float total, float amp_sum, float adj, float post) {
    const float p = total / amp_sum;
    return (adj + p) + post;
}

// ---------------------------------------------------------------------------------------------
// Line evaluation. Along a grid line of fixed (x, y) only z varies, and within one lattice cell of
// octave k the eight corner gradients are fixed, so each corner term is affine in dz:
//   g_ijl(dz) = Gx dx_i + Gy dy_j + Gz (dz - l) = P_ijl + Gz_ijl dz_l.
// The x and y lerps are linear, so the two z faces of the cell reduce to
//   N_l(dz) = A_l + B_l dz_l,  A_l = lerp_y(lerp_x(P_.. l)),  B_l = lerp_y(lerp_x(Gz_.. l)),
// and a sample is N0 + s(dz) (N1 - N0) with N1 - N0 = C + D dz: three FMAs, the clamp and the
// octave accumulation. The A/B setup (gradient fetches and ~20 FLOPs per face) is redone only when
// the line enters a new lattice cell of that octave, which is wave-uniform because every lane of a
// wave walks its own line at the same z index.

struct uw_line_oct {
    float A0, B0, A1, B1;
    float C, D;  // N1 - N0 = C + D dz with C = (A1 - B1) - A0, D = B1 - B0
};

__device__ __forceinline__ void uw_line_diff(uw_line_oct& s) {
    s.C = (s.A1 - s.B1) - s.A0;
    s.D = s.B1 - s.B0;
}

// Gradient of each permutation slot as f16 (components exactly -1, 0 or 1): x | y << 16, then z. The
// line evaluator reads it with one 8-byte LDS read and uses the halves as they are, as f16 operands of
// mixed-precision FMAs (f32 arithmetic and results, so the products are those of the f32 components).
__device__ __forceinline__ uint2 uw_grad_half(uint32_t code) {
    constexpr uint32_t kx = uw_grad_pack(0), ky = uw_grad_pack(1), kz = uw_grad_pack(2);
    auto half = [](uint32_t f) { return (f & 1u ? 0x3C00u : 0u) | ((f & 2u) << 14); };  // 2-bit two's complement
    const uint32_t sh = 2u * code;
    return make_uint2(half(kx >> sh) | (half(ky >> sh) << 16), half(kz >> sh));
}
// g.x v (f16 in the low half of g), and g.y v + c (high half): each one rounding, as fmaf.
__device__ __forceinline__ float uw_mix_mul_x(uint32_t g, float v) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(g), "v"(v));
    return r;
}
__device__ __forceinline__ float uw_mix_fma_y(uint32_t g, float v, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(g), "v"(v), "v"(c));
    return r;
}
// g.z v + c (low half)
__device__ __forceinline__ float uw_mix_fma_z(uint32_t g, float v, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(g), "v"(v), "v"(c));
    return r;
}
// uw_lerp(t, a, b) of two f16 values in high halves, and in low halves
__device__ __forceinline__ float uw_mix_lerp_hi(float t, uint32_t a, uint32_t b) {
    float d, r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(b), "v"(a));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(t), "v"(d), "v"(a));
    return r;
}
__device__ __forceinline__ float uw_mix_lerp(float t, uint32_t a, uint32_t b) {
    float d, r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(d) : "v"(b), "v"(a));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(r) : "v"(t), "v"(d), "v"(a));
    return r;
}

// Second-level hashes of a line's x / y corners, as byte offsets of their gradient slots (8 hash):
// (b00 | b10 << 16, b01 | b11 << 16). A z lattice byte moves a slot by xor, so a face's four slot
// addresses are one operation each.
__device__ __forceinline__ uint2 uw_line_hash(uint32_t xbits, uint32_t ybits, const uint8_t* P) {
    const uint32_t a0 = xbits & 255u, a1 = xbits >> 8, y0 = ybits & 255u, y1 = ybits >> 8;
    return make_uint2((uint32_t(P[a0 ^ y0]) << 3) | (uint32_t(P[a1 ^ y0]) << 19),
                      (uint32_t(P[a0 ^ y1]) << 3) | (uint32_t(P[a1 ^ y1]) << 19));
}

// One z face of a line's lattice cell: A = lerp_y(lerp_x(P_..)), B = lerp_y(lerp_x(Gz_..)) for the
// face whose z lattice byte is zb. The face depends on the z lattice index only through zb.
__device__ __forceinline__ void uw_line_face(const uw_axis& X, const uw_axis& Y, uint2 bq, uint32_t zb, const uint2* GH,
                                             float* A, float* B) {
    const unsigned char* g = reinterpret_cast<const unsigned char*>(GH);
    const uint32_t z8 = zb << 3;
    auto slot = [&](uint32_t o) { return *reinterpret_cast<const uint2*>(g + (o ^ z8)); };
    const uint2 G00 = slot(bq.x & 0xFFFFu), G10 = slot(bq.x >> 16), G01 = slot(bq.y & 0xFFFFu), G11 = slot(bq.y >> 16);
    const float P00 = uw_mix_fma_y(G00.x, Y.d, uw_mix_mul_x(G00.x, X.d));
    const float P10 = uw_mix_fma_y(G10.x, Y.d, uw_mix_mul_x(G10.x, X.dm1));
    const float P01 = uw_mix_fma_y(G01.x, Y.dm1, uw_mix_mul_x(G01.x, X.d));
    const float P11 = uw_mix_fma_y(G11.x, Y.dm1, uw_mix_mul_x(G11.x, X.dm1));
    const float a = X.fade, b = Y.fade;
    *A = uw_lerp(b, uw_lerp(a, P00, P10), uw_lerp(a, P01, P11));
    *B = uw_lerp(b, uw_mix_lerp(a, G00.y, G10.y), uw_mix_lerp(a, G01.y, G11.y));
}

// Per-line, per-octave state for the lattice cell whose low/high z bytes are packed in zbits.
__device__ __forceinline__ uw_line_oct uw_line_setup(const uw_axis& X, const uw_axis& Y, uint2 bq, uint32_t zbits,
                                                     const uint2* GH) {
    uw_line_oct s;
    uw_line_face(X, Y, bq, zbits & 255u, GH, &s.A0, &s.B0);
    uw_line_face(X, Y, bq, (zbits >> 8) & 255u, GH, &s.A1, &s.B1);
    uw_line_diff(s);
    return s;
}

// Unscaled octave value at the line sample, clamped to the unscaled image of [-1, 1]; the caller
// multiplies by the octave weight A_k (2/sqrt 3) / sum A.
// N0 + s(dz) (N1 - N0), with the face difference N1 - N0 = C + D dz formed by one FMA.
__device__ __forceinline__ float uw_line_sample(const uw_line_oct& s, float dz, float fade, float lo, float hi) {
    const float n0 = fmaf(s.B0, dz, s.A0);
    const float dn = fmaf(s.D, dz, s.C);
    return __builtin_amdgcn_fmed3f(fmaf(fade, dn, n0), lo, hi);
}

// Per-chunk LDS tables: every (axis index, octave) entry of the chunk and the z-bias split.
struct uw_chunk_tables {
    uw_axis* AX;   // [O][L], hashed
    uw_axis* AY;   // [O][L]
    uw_axis* AZ;   // [O][L]
    float* ADJ;    // [L]
    float* POST;   // [L]
};

// The x and y tables only (the density loops read the z entries from the chunk's z table in HBM,
// see uw_ztab): AX[k L + i] hashed, AY[k L + i].
// One thread per (axis, octave, sample) entry, so the short f64 chains of a chunk's entries run
// side by side; freq holds the octave frequencies (an LDS copy, indexed per lane).
__device__ __forceinline__ void uw_build_xy_tables(const uw_field& f, const double* freq, const uint8_t* perm,
                                                   int32_t cx, int32_t cy, int32_t L, float step, uw_axis* AX,
                                                   uw_axis* AY, int tid, int nthr) {
    const int32_t OL = f.octaves * L;
    const uw_divider dL = uw_make_divider(uint32_t(L));
    for (int e = tid; e < 2 * OL; e += nthr) {
        const bool is_y = e >= OL;
        const int32_t r = is_y ? e - OL : e;
        const int32_t k = int32_t(uw_div(uint32_t(r), dL)), i = r - k * L;
        const uw_axis v = uw_axis_of(uw_sample_coord(f, is_y ? 1 : 0, is_y ? cy : cx, i, step), freq[k]);
        if (is_y) AY[r] = v;
        else AX[r] = uw_hash_x(v, perm);
    }
}

// ---------------------------------------------------------------------------------------------
// Per-chunk z tables in HBM. Every lane of a wave walks its line at the same z index, so the z
// entries and the bias split of a sample are wave-uniform: kept in HBM (written by a previous
// kernel, uw_ztab_block) they are fetched with scalar loads into scalar registers, costing
// neither vector instructions nor vector registers. One record of uw_zrec_words(O) 32-bit words
// per z sample, so a sample's fetch is one wide scalar load from one address:
//   [3k] packed z lattice bytes of octave k (low face | high face << 8), [3k + 1] dz,
//   [3k + 2] fade(dz); [3O] adj, [3O + 1] post (the z-bias split); [3O + 2] face flags: bit 2k,
//   octave k enters a new lattice cell at this sample (every octave does at sample 0); bit 2k + 1,
//   that cell's low face is the previous cell's high face (z byte stepped by one), so only the new
//   high face is built.
// Records 0 .. stride: the one past the last sample is zero and only ever fetched ahead.
__host__ __device__ constexpr int32_t uw_zrec_words(int32_t octaves) { return (3 * octaves + 3 + 3) & ~3; }

struct uw_ztab {
    const uint32_t* rec;
    int32_t rw;  // words per record
};

__host__ __device__ inline size_t uw_ztab_bytes(int32_t octaves, int32_t stride) {
    return size_t(stride + 1) * size_t(uw_zrec_words(octaves)) * sizeof(uint32_t);
}

__device__ __forceinline__ uw_ztab uw_ztab_of(const unsigned char* base, int32_t chunk, int32_t octaves,
                                              int32_t stride) {
    uw_ztab t;
    t.rec = reinterpret_cast<const uint32_t*>(base + size_t(chunk) * uw_ztab_bytes(octaves, stride));
    t.rw = uw_zrec_words(octaves);
    return t;
}

// Record i of a chunk's z table (sample coordinate cz, L samples, i <= L; i == L gives the zero
// record).
__device__ __forceinline__ void uw_fill_zrec(const uw_field& f, int32_t cz, int32_t L, float step, int32_t i,
                                             uint32_t* rec) {
    const int32_t O = f.octaves;
    const int32_t rw = uw_zrec_words(O);
    if (i >= L) {
        for (int32_t w = 0; w < rw; ++w) rec[w] = 0u;
        return;
    }
    const double pz = uw_sample_coord(f, 2, cz, i, step);
    const double pp = i > 0 ? uw_sample_coord(f, 2, cz, i - 1, step) : 0.0;
    uint32_t flags = 0;
    for (int32_t k = 0; k < O; ++k) {
        const uw_axis z = uw_axis_of(pz, f.octave_freq[k]);
        rec[3 * k] = z.bits;
        rec[3 * k + 1] = __float_as_uint(z.d);
        rec[3 * k + 2] = __float_as_uint(z.fade);
        if (i == 0) {
            flags |= 1u << (2 * k);
        } else {
            const uint32_t prev = uw_axis_of(pp, f.octave_freq[k]).bits;
            if (z.bits != prev) {
                flags |= 1u << (2 * k);
                if ((z.bits & 255u) == ((prev >> 8) & 255u)) flags |= 2u << (2 * k);
            }
        }
    }
    float adj, post;
    uw_bias_terms(f, pz, &adj, &post);
    rec[3 * O] = __float_as_uint(adj);
    rec[3 * O + 1] = __float_as_uint(post);
    rec[3 * O + 2] = flags;
    for (int32_t w = 3 * O + 3; w < rw; ++w) rec[w] = 0u;
}

// The z records g0 .. g0 + THREADS - 1 of a launch (record g: chunk g / (stride + 1), sample
// g % (stride + 1)), one per thread, staged in LDS at a pitch of rw + 1 words (no bank aliasing) and
// written as one block with 16-byte stores: a thread writing its own record with 4-byte stores at a
// stride of rw words touched a separate cache line with every lane of every store. res == null:
// every chunk has n_uniform cells per axis. Records past a chunk's spare, and those of chunks whose
// resolution does not fit the stride (flagged invalid by the mesher, which never reads them), are
// written as zeros. stage: THREADS (rw + 1) words of LDS.
template <int THREADS>
__device__ __forceinline__ void uw_ztab_block(const uw_field& f, const int32_t* __restrict__ coords,
                                              const int32_t* __restrict__ res, int32_t n_uniform, int32_t nchunks,
                                              int32_t stride, unsigned char* __restrict__ out, uint64_t g0,
                                              uint32_t* stage) {
    const int tid = threadIdx.x;
    const int32_t rw = uw_zrec_words(f.octaves), pitch = rw + 1;
    const uint32_t per = uint32_t(stride) + 1u;
    const uint64_t total = uint64_t(nchunks) * per;
    const uint64_t g = g0 + uint64_t(tid);
    uint32_t* rec = stage + tid * pitch;
    bool filled = false;
    if (g < total) {
        const int32_t c = int32_t(g / per), i = int32_t(g - uint64_t(c) * per);
        const int32_t n = res ? res[c] : n_uniform;
        if (n >= 1 && n + 1 <= stride && i <= n + 1) {
            uw_fill_zrec(f, coords[3 * c + 2], n + 1, float(f.extent) / float(n), i, rec);
            filled = true;
        }
    }
    if (!filled)
        for (int32_t w = 0; w < rw; ++w) rec[w] = 0u;
    __syncthreads();
    if (g0 >= total) return;  // (block-uniform)
    const uint32_t nrec = uint32_t(min(uint64_t(THREADS), total - g0));
    const uint32_t nq = nrec * uint32_t(rw) / 4u;  // 16-byte words of the block (rw is a multiple of 4)
    uint4* dst = reinterpret_cast<uint4*>(out + g0 * uint64_t(rw) * 4u);
    for (uint32_t q = uint32_t(tid); q < nq; q += THREADS) {
        const uint32_t wd = 4u * q, r = wd / uint32_t(rw), w = wd - r * uint32_t(rw);
        const uint32_t* s = stage + r * uint32_t(pitch) + w;
        dst[q] = make_uint4(s[0], s[1], s[2], s[3]);
    }
}

// Appends the sign bit rho < iso of a line's next sample: a compare and an add with carry. Samples
// enter at bit 0, so a word of c samples is reversed with __brev(word) >> (32 - c).
__device__ __forceinline__ uint32_t uw_push_sign(uint32_t word, float rho, float iso) {
    return word + word + (rho < iso ? 1u : 0u);
}

// Scalar (constant address space) loads of wave-uniform HBM data written by an earlier kernel.
typedef const __attribute__((address_space(4))) uint32_t* uw_const_u32_ptr;

// Minimum / maximum of two finite values as single instructions (fminf / fmaxf also quiet
// signalling NaN operands first, two more instructions per call in a loop).
__device__ __forceinline__ float uw_fmin_raw(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float uw_fmax_raw(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// One z record in scalar registers (OMAX octave slots, the first O used).
template <int OMAX>
struct uw_zsample {
    uint32_t bits[OMAX];
    float d[OMAX], fade[OMAX];
    float adj, post;
    uint32_t flags;
    __device__ __forceinline__ void load(const uint32_t* rec, int32_t O) {
        const uw_const_u32_ptr q = (uw_const_u32_ptr)(rec);
#pragma unroll
        for (int k = 0; k < OMAX; ++k) {
            if (k < O) {
                bits[k] = q[3 * k];
                d[k] = __uint_as_float(q[3 * k + 1]);
                fade[k] = __uint_as_float(q[3 * k + 2]);
            }
        }
        adj = __uint_as_float(q[3 * O]);
        post = __uint_as_float(q[3 * O + 1]);
        flags = q[3 * O + 2];
    }
};

// Sign summary bits of a set of samples: some sample not above iso (so not early-blank), some
// below iso, some at or above iso (a cell can straddle iso only if both of the last two hold).
#define UW_BELOW_NOT_ABOVE 1
#define UW_BELOW_LT 2
#define UW_BELOW_GE 4

// Octave-count specialisation of the density kernels: OCT > 0 compiles for exactly OCT octaves
// (the common counts, so the octave loop unrolls with no per-octave predicates); OCT == 0 reads
// the count from the field (at most UW_MAX_OCTAVES).
template <int OCT>
struct uw_octaves {
    static constexpr int kMax = OCT > 0 ? OCT : UW_MAX_OCTAVES;
    __device__ __forceinline__ static int32_t count(const uw_field& f) { return OCT > 0 ? OCT : f.octaves; }
    __host__ __device__ static constexpr bool accepts(int32_t o) { return OCT > 0 ? o == OCT : o <= UW_MAX_OCTAVES; }
};

// Face-flag word of a z record that sets up every octave's lattice cell from scratch (bit 2k per
// octave, no "low face is the previous high face" bits): the first sample of a line that starts
// inside the z range.
__device__ __forceinline__ uint32_t uw_full_setup_flags(int32_t octaves) {
    return 0x55555555u & ((octaves >= 16) ? 0xFFFFFFFFu : ((1u << (2 * octaves)) - 1u));
}

// One z-line of samples: the line whose octave-k x / y axis entries are AX(k) / AY(k) (hashed x),
// z records from zr on (rw words each; the record after the last sample is fetched ahead and
// discarded), `count` samples. FORCE: the first sample builds every octave's lattice cell whatever
// its record's face flags say (a line that starts inside a longer z range). store(iz, rho)
// receives the densities; vmin / vmax keep the running extremes.
template <int OCT, bool FORCE, class AxisX, class AxisY, class Store>
__device__ __forceinline__ void uw_noise_zline(const uw_field& f, AxisX AX, AxisY AY, const uint8_t* P, const uint2* GH,
                                               const uint32_t* zr, int32_t rw, int32_t count,
                                               float& vmin, float& vmax, Store store) {
    constexpr int OMAX = uw_octaves<OCT>::kMax;
    const int32_t O = uw_octaves<OCT>::count(f);
    uint2 bq[OMAX];
    uw_line_oct st[OMAX];
#pragma unroll
    for (int k = 0; k < OMAX; ++k) {
        if (k < O) {
            bq[k] = uw_line_hash(AX(k).bits, AY(k).bits, P);
        }
    }
    // Sample iz, then the fetch of the record of sample iz + 1 (the fetch after the last sample
    // reads the spare record and is discarded). The fetch is issued after the face updates,
    // whose LDS reads would otherwise wait for it too, and before the sample arithmetic, which
    // covers its latency. Two records alternate, so the fetched registers are used in place.
    auto sample = [&](const uw_zsample<OMAX>& Z, uw_zsample<OMAX>& Znext, int32_t iz) {
        if (Z.flags) {  // some octave enters a new lattice cell
#pragma unroll
            for (int k = 0; k < OMAX; ++k) {
                if (k < O && (Z.flags & (1u << (2 * k)))) {
                    const uw_axis X = AX(k), Y = AY(k);
                    const uint32_t zb = Z.bits[k];
                    if (Z.flags & (2u << (2 * k))) {
                        st[k].A0 = st[k].A1;
                        st[k].B0 = st[k].B1;
                        uw_line_face(X, Y, bq[k], zb >> 8, GH, &st[k].A1, &st[k].B1);
                        uw_line_diff(st[k]);
                    } else {
                        st[k] = uw_line_setup(X, Y, bq[k], zb, GH);
                    }
                }
            }
        }
        zr += rw;
        Znext.load(zr, O);
        __builtin_amdgcn_sched_barrier(0);  // keep the fetch ahead of the arithmetic
        float total = 0.0f;
#pragma unroll
        for (int k = 0; k < OMAX; ++k)
            if (k < O) total = fmaf(f.weight[k], uw_line_sample(st[k], Z.d[k], Z.fade[k], f.clamp_lo, f.clamp_hi),
                                    total);
        const float rho = (Z.adj + total) + Z.post;
        store(iz, rho);
        vmin = uw_fmin_raw(vmin, rho);
        vmax = uw_fmax_raw(vmax, rho);
    };
    uw_zsample<OMAX> Za, Zb;
    Za.load(zr, O);
    if (FORCE) Za.flags = uw_full_setup_flags(O);
    int32_t iz = 0;
    for (; iz + 1 < count; iz += 2) {  // no exit between a fetch and its use
        sample(Za, Zb, iz);
        sample(Zb, Za, iz + 1);
    }
    if (iz < count) sample(Za, Zb, iz);
}

__device__ __forceinline__ int uw_below_bits(float vmin, float vmax, float iso) {
    return (vmin <= iso ? UW_BELOW_NOT_ABOVE : 0) | (vmin < iso ? UW_BELOW_LT : 0) | (vmax >= iso ? UW_BELOW_GE : 0);
}

// Densities of x-planes [xa, xb) of a chunk whose tables are in T, one thread per (x, y) line.
// Plane x is written to dst + slot(x) * L * L with slot(x) = x % nslot, z fastest.
// Returns, per thread, the OR of the UW_BELOW_* bits of its samples.
template <int OCT>
__device__ __forceinline__ int uw_noise_planes(const uw_field& f, const uw_chunk_tables& T, const uw_ztab& Zt,
                                               const uint8_t* P, const uint2* GH, int32_t L, int32_t xa, int32_t xb,
                                               float* dst, int32_t nslot, int tid, int nthr) {
    const int32_t lines = (xb - xa) * L;
    const uw_divider dL = uw_make_divider(uint32_t(L)), dslot = uw_make_divider(uint32_t(nslot));
    const int32_t rw = OCT > 0 ? uw_zrec_words(OCT) : Zt.rw;
    // running extremes of the thread's samples; the sign bits follow from them at the end
    float vmin = INFINITY, vmax = -INFINITY;
    for (int32_t t = tid; t < lines; t += nthr) {
        const int32_t tq = int32_t(uw_div(uint32_t(t), dL));
        const int32_t ix = xa + tq, iy = t - tq * L;
        float* out = dst + int32_t(uw_mod(uint32_t(ix), dslot)) * L * L + iy * L;
        uw_noise_zline<OCT, false>(
            f, [&](int k) { return T.AX[k * L + ix]; }, [&](int k) { return T.AY[k * L + iy]; }, P, GH, Zt.rec, rw, L,
            vmin, vmax, [&](int32_t iz, float rho) { out[iz] = rho; });
    }
    return uw_below_bits(vmin, vmax, f.iso);
}

// Octave value and gradient with respect to the octave coordinate (f32), given the per-axis lattice
// data and fade derivatives s'(d) = 30 d^2 (d - 1)^2. GH: uw_grad_half of every permutation slot, read
// as in uw_line_face: eight 8-byte LDS reads and mixed-precision FMAs on the halves (the same f32
// results) where a table of floats took 24 reads.
__device__ __forceinline__ float uw_octave_grad(const uw_axis& X, const uw_axis& Y, const uw_axis& Z, float dfx,
                                                float dfy, float dfz, const uint8_t* P, const uint2* GH, float g[3]) {
    const unsigned char* gh = reinterpret_cast<const unsigned char*>(GH);
    const uint2 bq = uw_line_hash(X.bits, Y.bits, P);
    const uint32_t z0 = (Z.bits & 255u) << 3, z1 = (Z.bits >> 8) << 3;
    auto slot = [&](uint32_t o) { return *reinterpret_cast<const uint2*>(gh + o); };
    const uint32_t b00 = bq.x & 0xFFFFu, b10 = bq.x >> 16, b01 = bq.y & 0xFFFFu, b11 = bq.y >> 16;
    const uint2 G000 = slot(b00 ^ z0), G100 = slot(b10 ^ z0), G010 = slot(b01 ^ z0), G110 = slot(b11 ^ z0);
    const uint2 G001 = slot(b00 ^ z1), G101 = slot(b10 ^ z1), G011 = slot(b01 ^ z1), G111 = slot(b11 ^ z1);
    auto dot = [](uint2 G, float x, float y, float z) {
        return uw_mix_fma_z(G.y, z, uw_mix_fma_y(G.x, y, uw_mix_mul_x(G.x, x)));
    };
    const float g000 = dot(G000, X.d, Y.d, Z.d), g100 = dot(G100, X.dm1, Y.d, Z.d);
    const float g010 = dot(G010, X.d, Y.dm1, Z.d), g110 = dot(G110, X.dm1, Y.dm1, Z.d);
    const float g001 = dot(G001, X.d, Y.d, Z.dm1), g101 = dot(G101, X.dm1, Y.d, Z.dm1);
    const float g011 = dot(G011, X.d, Y.dm1, Z.dm1), g111 = dot(G111, X.dm1, Y.dm1, Z.dm1);
    const float a = X.fade, b = Y.fade, c = Z.fade;
    const float x00 = uw_lerp(a, g000, g100), x10 = uw_lerp(a, g010, g110);
    const float x01 = uw_lerp(a, g001, g101), x11 = uw_lerp(a, g011, g111);
    const float yv0 = uw_lerp(b, x00, x10), yv1 = uw_lerp(b, x01, x11);
    const float r = uw_lerp(c, yv0, yv1) * UW_PERLIN_SCALE;
    // d/dx
    const float dx00 = fmaf(dfx, g100 - g000, uw_mix_lerp(a, G000.x, G100.x));
    const float dx10 = fmaf(dfx, g110 - g010, uw_mix_lerp(a, G010.x, G110.x));
    const float dx01 = fmaf(dfx, g101 - g001, uw_mix_lerp(a, G001.x, G101.x));
    const float dx11 = fmaf(dfx, g111 - g011, uw_mix_lerp(a, G011.x, G111.x));
    g[0] = uw_lerp(c, uw_lerp(b, dx00, dx10), uw_lerp(b, dx01, dx11)) * UW_PERLIN_SCALE;
    // d/dy
    const float dy0 = fmaf(dfy, x10 - x00, uw_lerp(b, uw_mix_lerp_hi(a, G000.x, G100.x), uw_mix_lerp_hi(a, G010.x, G110.x)));
    const float dy1 = fmaf(dfy, x11 - x01, uw_lerp(b, uw_mix_lerp_hi(a, G001.x, G101.x), uw_mix_lerp_hi(a, G011.x, G111.x)));
    g[1] = uw_lerp(c, dy0, dy1) * UW_PERLIN_SCALE;
    // d/dz
    const float ez0 = uw_lerp(b, uw_mix_lerp(a, G000.y, G100.y), uw_mix_lerp(a, G010.y, G110.y));
    const float ez1 = uw_lerp(b, uw_mix_lerp(a, G001.y, G101.y), uw_mix_lerp(a, G011.y, G111.y));
    g[2] = fmaf(dfz, yv1 - yv0, uw_lerp(c, ez0, ez1)) * UW_PERLIN_SCALE;
    if (r > 1.0f || r < -1.0f) {
        g[0] = g[1] = g[2] = 0.0f;
        return r > 1.0f ? 1.0f : -1.0f;
    }
    return r;
}

// Parameter sums of a backward. Over its endpoint samples (weight w each, f64) a kernel adds, per
// octave, N_k = sum w n_k, then G = sum w sum_k A_k f_k grad n_k (three values), W = sum w and
// T = sum w sum_k A_k n_k: one conversion and one FMA per octave. The gradients follow from the sums:
// dL/dA_k = (N_k - T / sum A) / sum A and dL/ddelta = freq (G / sum A + W bias'(p_z) e_z).
// Result q of the O + 3 from the sums S = N (O of them), G, W, T.
constexpr int kParamExtra = 5;  // G, W, T
__device__ __forceinline__ double uw_param_grad(const uw_field& f, const double* S, int32_t O, int32_t q) {
    const double inv_sum = 1.0 / double(f.amp_sum);
    if (q < O) return (S[q] - S[O + 4] * inv_sum) * inv_sum;
    const double slope = f.bias_kind == UW_BIAS_LINEAR ? double(f.bias_a) : 0.0;
    const double g = S[q] * inv_sum;
    // (no slope, no term: 0 W would be NaN where a weight is infinite)
    return f.frequency * (q == O + 2 && slope != 0.0 ? g + slope * S[O + 3] : g);
}
