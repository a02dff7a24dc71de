// Runs the tile emitter of csrc/uw_rows.h on the host (tests/test_emit_tiles.py builds and runs it): row counts,
// tilings and uw_emit_rows over whole grids, against a literal first-seen walk of the triangulation table. The
// workgroup memory ends at a page that can't be touched.
#include <sys/mman.h>
#include <unistd.h>

#include <cstdio>
#include <map>
#include <random>
#include <utility>

#include "hip/hip_runtime.h"

#include "../../underwaterworld_amd/csrc/uw_rows.h"

namespace {

#define CHECK(c, ...)                                   \
    do {                                                \
        if (!(c)) {                                     \
            std::printf("line %d: %s: ", __LINE__, #c); \
            std::printf(__VA_ARGS__);                   \
            std::printf("\n");                          \
            std::exit(1);                               \
        }                                               \
    } while (0)

uw_tables tables;

void make_tables() {
    for (int c = 0; c < 256; ++c) {
        const uint64_t row = UW_MC_TRI_PACKED[c];
        tables.tri[c] = row;
        uint32_t seen = 0;
        for (int e = 0; e < 12; ++e) tables.before[c][e] = 0xFFFF;
        for (int j = 0; j < 3 * int(row & 15u); ++j) {
            const int e = int(row >> (4 + 4 * j) & 15u);
            if (!(seen >> e & 1)) tables.before[c][e] = uint16_t(seen);
            seen |= 1u << e;
        }
        for (int e = 0; e < 12; ++e)
            if (!(seen >> e & 1)) tables.before[c][e] = uint16_t(seen);
        tables.used[c] = uint16_t(seen);
    }
    for (uint32_t i = 0; i < 256; ++i) {
        const uint32_t c = uw_case_of_index(i);
        tables.cell[i] = uint32_t(tables.used[c]) | uint32_t(tables.tri[c] & 15u) << 12 | c << 16;
    }
}

struct Mesh {
    std::vector<float> verts, normals;
    std::vector<uint32_t> inds, cells;
    std::vector<uw_vertex_tape> tape;
};

struct Grid {
    int n, L;
    float iso, step = 0.5f;
    std::vector<float> dens;  // x L^2 + y L + z
    float at(int x, int y, int z) const { return dens[size_t((x * L + y) * L + z)]; }
};

// The reference's walk: cells x -> y -> z, a vertex per ordered corner pair as it is first seen.
Mesh walk(const Grid& g) {
    Mesh m;
    std::map<std::pair<uint32_t, uint32_t>, uint32_t> ids;
    for (int x = 0; x < g.n; ++x)
        for (int y = 0; y < g.n; ++y)
            for (int z = 0; z < g.n; ++z) {
                uint32_t cs = 0, at[8];
                float r[8];
                for (uint32_t i = 0; i < 8; ++i) {
                    const uint32_t o = uw_corner_ofs(i);
                    const int cx = x + int(o & 1), cy = y + int(o >> 1 & 1), cz = z + int(o >> 2 & 1);
                    at[i] = uint32_t((cx * g.L + cy) * g.L + cz);
                    r[i] = g.dens[at[i]];
                    cs |= uint32_t(r[i] < g.iso) << i;
                }
                const uint64_t row = UW_MC_TRI_PACKED[cs];
                for (int j = 0; j < 3 * int(row & 15u); ++j) {
                    const uint32_t e = uint32_t(row >> (4 + 4 * j) & 15u), a = uw_edge_a(e), b = uw_edge_b(e);
                    const auto it = ids.emplace(std::make_pair(at[a], at[b]), uint32_t(ids.size()));
                    if (it.second) {
                        float p[3];
                        uw_edge_vertex_ab(e, x, y, z, r[a], r[b], g.iso, g.step, 3.0f, -7.0f, 11.0f, p);
                        m.verts.insert(m.verts.end(), p, p + 3);
                        m.tape.push_back({at[a], at[b], r[a], r[b]});
                    }
                    m.inds.push_back(it.first->second);
                    if (j % 3 == 2) {
                        const float* v = m.verts.data();
                        const size_t k = m.inds.size() - 3;
                        float nm[3];
                        uw_tri_normal(v + 3 * m.inds[k], v + 3 * m.inds[k + 1], v + 3 * m.inds[k + 2], nm);
                        m.normals.insert(m.normals.end(), nm, nm + 3);
                        m.cells.push_back(uint32_t((x * g.n + y) * g.n + z));
                    }
                }
            }
    return m;
}

// Workgroup memory of `bytes`, the page behind it closed.
struct Lds {
    unsigned char *base = nullptr, *p = nullptr;
    size_t pages = 0;
    explicit Lds(size_t bytes) {
        const size_t page = size_t(sysconf(_SC_PAGESIZE));
        pages = ((bytes + page - 1) / page + 1) * page;
        base = static_cast<unsigned char*>(mmap(nullptr, pages, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
        mprotect(base + pages - page, page, PROT_NONE);
        p = base + (pages - page - bytes) / 16 * 16;
        memset(base, 0xA5, pages - page);
    }
    ~Lds() { munmap(base, pages); }
};

struct Job {
    uw_emit_tile tile;
    unsigned char* smem;
    bool extra;
};
void emit_body(void* arg) {
    const Job& j = *static_cast<Job*>(arg);
    uw_emit_tables(&tables, j.smem);
    const uw_emit_row row = uw_emit_load(j.tile);
    if (j.extra) uw_emit_rows<true>(j.tile, row, j.smem);
    else uw_emit_rows<false>(j.tile, row, j.smem);
}

struct Tiles {
    int planes, xt, yt, T, cells, max_rows;
};

void check(const Grid& g, const Tiles& t, bool wire, uint32_t seed) {
    const int n = g.n, L = g.L, WL = uw_sign_words(L), T = uw_row_segs(n);
    std::vector<uint32_t> words(size_t(L) * L * WL, 0u);
    for (int x = 0; x < L; ++x)
        for (int y = 0; y < L; ++y)
            for (int z = 0; z < L; ++z)
                if (g.at(x, y, z) < g.iso) words[size_t(x * L + y) * WL + z / 32] |= 1u << (z & 31);
    std::vector<unsigned long long> rows(size_t(n) * n * T + 1, 0ull);
    unsigned long long sum = 0;
    uint32_t active = 0, want_active = 0;
    for (int x = 0; x < n; ++x)
        for (int y = 0; y < n; ++y)
            for (int tz = 0; tz < T; ++tz) {
                uw_row_bits b;
                b.load(words.data(), x, y, tz, n, L, WL);
                const uint32_t c = uw_row_counts(b, x, y, tz, tables.cell);
                rows[size_t(x * n + y) * T + tz] = sum;
                sum += (c & 0x3FFu) | (unsigned long long)(c >> 10 & 0x3FFu) << 32;
                active += c >> 20;
            }
    rows.back() = sum;
    for (int x = 0; x < n; ++x)
        for (int y = 0; y < n; ++y)
            for (int z = 0; z < n; ++z) {
                int k = 0;
                for (uint32_t i = 0; i < 8; ++i) k += g.at(x + (i & 1), y + (i >> 1 & 1), z + (i >> 2)) < g.iso;
                want_active += k > 0 && k < 8;
            }
    const Mesh want = walk(g);
    CHECK(active == want_active && uint32_t(sum) == want.verts.size() / 3 && sum >> 32 == want.inds.size() / 3,
          "n %d: %u active, %u vertices, %u triangles", n, active, uint32_t(sum), uint32_t(sum >> 32));
    const size_t nv = want.verts.size() / 3, ni = want.inds.size(), vo = 5, to = 2;  // the chunk's ranges start there
    Mesh got;
    const uint32_t vstride = wire ? 6 : 3;
    got.verts.assign((nv + vo + 4) * vstride, -1.0f);
    std::vector<uint16_t> inds16(ni + 3 * to + 8, 0xABCD);
    got.inds.assign(ni + 3 * to + 8, 0xABCDABCDu);
    got.tape.assign(nv + vo + 4, {});
    got.normals.assign(ni + 3 * to + 8, -9.0f);
    got.cells.assign(ni / 3 + to + 3, 0xABCDu);
    uw_emit_tile e;
    e.eo = {vstride, wire ? 1u : 0u, wire ? got.normals.data() : nullptr, wire ? got.cells.data() : nullptr};
    e.iso = g.iso;
    e.step = g.step;
    e.ox = 3.0f;
    e.oy = -7.0f;
    e.oz = 11.0f;
    e.extent = g.step * float(n);
    e.n = n;
    e.L = L;
    e.T = T;
    e.WL = WL;
    e.cells = t.cells;
    e.dens = g.dens.data();
    e.sx = L * L;
    e.sy = L;
    e.sz = 1;
    e.words = words.data();
    e.rows = rows.data();
    e.vo = vo;
    e.io = 3 * to;
    e.vlim = vo + nv;
    e.ilim = 3 * to + ni;
    e.verts = got.verts.data();
    e.inds = wire ? reinterpret_cast<uint32_t*>(inds16.data()) : got.inds.data();
    e.tape = got.tape.data();
    const Lds lds(uw_emit_lds_bytes(t.max_rows, t.cells));
    CHECK(uw_emit_takes(t.max_rows, t.cells + (t.yt > 1 ? 1 : 0), t.cells), "n %d planes %d: %d rows", n, t.planes, t.max_rows);
    for (int q = 0; q < t.xt * t.yt * t.T; ++q) {
        const int xt = q / (t.yt * t.T), yt = q / t.T % t.yt;
        e.X0 = xt * t.planes;
        e.X1 = min(n, e.X0 + t.planes);
        e.Y0 = yt * 32;
        e.Y1 = t.yt > 1 ? min(n, e.Y0 + 32) : n;
        e.tz = q % t.T;
        const int high = (e.X1 - e.X0 + (e.X0 > 0)) * (e.Y1 - e.Y0 + (e.Y0 > 0));
        CHECK(e.X0 < e.X1 && high <= t.max_rows, "n %d tile %d: %d rows of %d", n, q, high, t.max_rows);
        Job job = {e, lds.p, wire};
        host_block::run(emit_body, &job, seed + uint32_t(q) * 977u);
    }
    for (size_t v = 0; v < nv; ++v) {
        CHECK(!memcmp(&got.verts[(vo + v) * vstride], &want.verts[3 * v], 12), "n %d planes %d vertex %zu", n, t.planes, v);
        CHECK(!memcmp(&got.tape[vo + v], &want.tape[v], sizeof(uw_vertex_tape)), "n %d planes %d tape %zu", n, t.planes, v);
    }
    for (size_t i = 0; i < ni; ++i) {
        const uint32_t id = wire ? inds16[3 * to + i] : got.inds[3 * to + i];
        CHECK(id == (wire ? want.inds[i] & 0xFFFFu : want.inds[i]), "n %d planes %d index %zu: %u not %u", n, t.planes, i, id, want.inds[i]);
        if (wire && i % 3 == 0) {
            CHECK(got.cells[to + i / 3] == want.cells[i / 3], "n %d cell of triangle %zu", n, i / 3);
            CHECK(!memcmp(&got.normals[3 * (to + i / 3)], &want.normals[i], 12), "n %d normal of triangle %zu", n, i / 3);
        }
    }
    for (size_t i = 0; i < vo * vstride; ++i) CHECK(got.verts[i] == -1.0f, "n %d: a vertex before the range", n);
    for (size_t i = (vo + nv) * vstride; i < got.verts.size(); ++i) CHECK(got.verts[i] == -1.0f, "n %d: a vertex past the range", n);
    for (size_t i = 0; i < got.inds.size(); ++i)
        if (i < 3 * to || i >= 3 * to + ni)
            CHECK(wire ? inds16[i] == 0xABCD : got.inds[i] == 0xABCDABCDu, "n %d: an index outside the range", n);
}

// surface: 0 a smooth sheet, 1 blobs, 2 white noise (surface in nearly every cell), 3 every other sample of one
// line (a single full row among empty ones)
Grid make_grid(int n, int surface, uint32_t seed) {
    Grid g{n, n + 1, 0.0f, 0.5f, {}};
    std::mt19937 rng(seed);
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    const float ph = 3.0f * u(rng), tilt = u(rng);
    for (int x = 0; x <= n; ++x)
        for (int y = 0; y <= n; ++y)
            for (int z = 0; z <= n; ++z) {
                const float fx = float(x) / n, fy = float(y) / n, fz = float(z) / n;
                g.dens.push_back(surface == 0   ? fz - 0.5f + 0.2f * sinf(5 * fx + ph) + 0.2f * tilt * fy
                                 : surface == 1 ? sinf(9 * fx + ph) * sinf(8 * fy) + sinf(10 * fz - ph) * tilt + 0.1f * u(rng)
                                 : surface == 2 ? u(rng)
                                                : (x || y || z % 2 ? 1.0f : -1.0f) + 0.1f * u(rng));
            }
    return g;
}

Tiles chunk_tiles(int n, int rows) {
    const uw_slabs s = uw_slab_tiling(n, rows);
    return {s.planes, s.tiles, 1, 1, n, s.max_rows};
}
Tiles grid_tiles(int n, int planes) {
    const uw_tiling t = uw_tiling_for(n, planes);
    return {t.planes, t.xt, t.yt, t.T, t.cells, t.max_rows};
}

}  // namespace

int main() {
    make_tables();
    // every tiling that a launch can ask for fits the emitter
    for (int n = 1; n <= UW_VOLUME_MAX_RESOLUTION; ++n)
        for (int p = uw_tile_planes(n); p >= 1; p = p > 1 ? (p + 1) / 2 : 0) {
            const uw_tiling t = uw_tiling_for(n, p);
            CHECK(t.planes >= 1 && t.planes <= p && t.xt * t.planes >= n && (t.xt - 1) * t.planes < n && t.yt * 32 >= n && t.T * 32 >= n, "n %d", n);
            CHECK(uw_emit_takes(t.max_rows, t.cells + (t.yt > 1 ? 1 : 0), t.cells) && uw_emit_lds_bytes(t.max_rows, t.cells) <= 160 * 1024 / 5, "n %d", n);
        }
    for (int n = 1; n <= UW_BATCH_MAX_RESOLUTION; ++n)
        for (int rows = 96; rows <= kTileRows; rows += 32) {
            const uw_slabs s = uw_slab_tiling(n, rows);
            CHECK(s.tiles * s.planes >= n && (s.tiles - 1) * s.planes < n && uw_emit_takes(s.max_rows, n, n), "n %d", n);
        }
    uint32_t seed = 1;
    for (int n : {1, 2, 3, 7, 12, 15, 24, 31, 32})
        for (int surface = 0; surface < 4; ++surface) {
            const Grid g = make_grid(n, surface, seed);
            check(g, chunk_tiles(n, kTileRows), surface == 1, seed += 7919);
            if (n > 12) check(g, chunk_tiles(n, 96), surface == 0, seed += 7919);
            if (n <= 24) check(g, grid_tiles(n, 1), surface == 2, seed += 7919);
        }
    for (int n : {33, 40, 65})
        for (int surface = 0; surface < 4; ++surface)
            if (n < 65 || surface == 0) {
                const Grid g = make_grid(n, surface, seed);
                check(g, grid_tiles(n, uw_tile_planes(n)), surface == 1, seed += 7919);
            }
    std::printf("ok\n");
    return 0;
}
