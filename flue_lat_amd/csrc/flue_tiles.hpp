// flue_tiles.hpp -- how the rectangle-first kernels split the plane slices of a lattice into tiles
// of base sites, one wavefront each, and where a tile's footprint lies.
#pragma once
#include <cmath>

#include "flue_launch.hpp"

namespace flue {
namespace {

// the second direction of rectangle plane rp (0: (x, y), 1: (x, z); with TIME (x, t))
template <bool TIME = false>
__device__ __forceinline__ int rect_d2(int rp) {
    return TIME ? 0 : (rp == 0 ? 2 : 3);
}

struct Tile {
    uint32_t t1, t2, cs, ct;  // tile along x, tile along d2, spectator coordinates (z or y and t; TIME: y and z)
    uint32_t o1, o2, l1, l2;  // first site and extent along x and d2
};

template <bool TIME = false>
__device__ __forceinline__ Tile tile_at(const Lat& L, int rp, const PlaneTiles& g, uint32_t tile) {
    const uint32_t ns = (uint32_t)L.n[!TIME && rp == 0 ? 3 : 2];
    Tile t;
    t.t1 = tile % g.n1;
    uint32_t q = tile / g.n1;
    t.t2 = q % g.n2;
    q /= g.n2;
    t.cs = q % ns;
    t.ct = q / ns;
    t.o1 = t.t1 * g.q1 + min(t.t1, g.r1);
    t.o2 = t.t2 * g.q2 + min(t.t2, g.r2);
    t.l1 = g.q1 + (t.t1 < g.r1 ? 1u : 0u);
    t.l2 = g.q2 + (t.t2 < g.r2 ? 1u : 0u);
    return t;
}

// the site at x, second-direction coordinate c2 and the spectators of a tile
template <bool TIME = false>
__device__ __forceinline__ uint32_t tile_site(const Lat& L, int rp, uint32_t x, uint32_t c2, const Tile& t) {
    if (TIME) return x + L.st[2] * t.cs + L.st[3] * t.ct + L.st[0] * c2;
    return x + L.st[2] * (rp == 0 ? c2 : t.cs) + L.st[3] * (rp == 0 ? t.cs : c2) + L.st[0] * t.ct;
}

// the tile of N sites split as (q, r) that holds site c, and its first site
__device__ __forceinline__ uint32_t tile_of(uint32_t c, uint32_t q, uint32_t r, uint32_t* first) {
    const uint32_t wide = r * (q + 1);
    const uint32_t t = c < wide ? c / (q + 1) : r + (c - wide) / q;
    *first = t * q + min(t, r);
    return t;
}

// rectangle plane y of a lattice's three
__device__ __forceinline__ PlaneTiles plane_tiles(const RectTiles& g, uint32_t y = blockIdx.y) {
    return y == 0 ? g.p[0] : (y == 1 ? g.p[1] : g.p[2]);
}

// lattice whose x, y, z are the z, y, x of L: its plane (x, y) is L's plane (z, y)
Lat zy_lattice(const Lat& L) {
    const int32_t d[4] = {L.n[0], L.n[3], L.n[2], L.n[1]};
    return make_lat(d);
}

// Tiles of one plane with extents N1 x N2 and `slices` plane slices: of the splits into nearly
// equal tiles whose footprint fits the LDS, the one that keeps the chip busy shortest -- 64-site
// turns of a tile times the rounds in which the three planes' tiles run on `slots` wavefronts
// (whole rounds while there are few of them) -- then the one with the fewest footprint cells.
// The rounds are counted for kNominalNT time slices whatever the lattice has: the split sets the
// order in which a site's rectangles are added, and a field repeated along t gives the same B.
// Every tile is at least 4 sites wide (rect_fits), so a footprint's three extra rows and columns
// reach into one further tile only.  (A launch over one plane counts its own slices.)
constexpr uint32_t kNominalNT = 32, kMaxTileEdge = 32;
PlaneTiles plane_split(uint32_t N1, uint32_t N2, uint32_t N3, uint32_t NT, uint32_t max_cells, uint32_t slots,
                       double slices = 3.0 * kNominalNT) {
    PlaneTiles best{};
    double time = 0.0;
    uint64_t cells = 0;
    // tile counts along a direction of N sites, from the fewest, each with a smaller widest tile
    auto widest = [](uint32_t N, uint32_t n) { return (N + n - 1) / n; };
    auto next = [&](uint32_t N, uint32_t n) { return widest(N, widest(N, n) - 1); };
    for (uint32_t n1 = widest(N1, kMaxTileEdge); N1 / n1 >= 4; n1 = next(N1, n1))
        for (uint32_t n2 = widest(N2, kMaxTileEdge); N2 / n2 >= 4; n2 = next(N2, n2)) {
            const uint32_t l1 = widest(N1, n1), l2 = widest(N2, n2), fc = (l1 + 3) * (l2 + 3);
            if (fc > max_cells) continue;
            // (16 x 16 tiles have kernels of their own: they win ties)
            const bool sq = N1 == 16 * n1 && N2 == 16 * n2;
            const uint64_t cn = sq ? 0 : (uint64_t)n1 * n2 * fc;
            const double rounds = slices * n1 * n2 * (double)N3 / slots;
            const double tm = (double)((l1 * l2 + 63) / 64) * (rounds < 8.0 ? std::ceil(rounds) : rounds);
            if (time == 0.0 || tm < time || (tm == time && cn < cells)) {
                time = tm;
                cells = cn;
                best = PlaneTiles{n1, N1 / n1, N1 % n1, n2, N2 / n2, N2 % n2, l1 + 3, fc,
                                  n1 * n2 * N3 * NT, 0};
            }
        }
    return best;
}

// the three planes of a lattice; `slots` wavefronts are resident on the chip (1: whatever the launch
// holds besides, the chip is full)
RectTiles rect_split(const Lat& L, uint32_t max_cells, uint32_t slots) {
    const uint32_t NT = (uint32_t)L.n[0], NX = (uint32_t)L.n[1], NY = (uint32_t)L.n[2], NZ = (uint32_t)L.n[3];
    RectTiles r;
    r.p[0] = plane_split(NX, NY, NZ, NT, max_cells, slots);
    r.p[1] = plane_split(NX, NZ, NY, NT, max_cells, slots);
    r.p[2] = plane_split(NZ, NY, NX, NT, max_cells, slots);
    r.p[1].cell0 = r.p[0].cell0 + (uint64_t)r.p[0].tiles * r.p[0].fc;
    r.p[2].cell0 = r.p[1].cell0 + (uint64_t)r.p[1].tiles * r.p[1].fc;
    return r;
}

uint64_t rect_cells(const RectTiles& r) { return r.p[2].cell0 + (uint64_t)r.p[2].tiles * r.p[2].fc; }

}  // namespace
}  // namespace flue
