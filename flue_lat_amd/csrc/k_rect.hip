// k_rect.hip -- the magnetic B with rectangle-first clover sums (magnetic variant 7).
//
// Planes (x, y) and (x, z): one wavefront per tile of base sites in one plane slice, the tile's
// sites numbered x fastest and taken 64 at a time (rows of consecutive sites, so link loads
// coalesce).  Every base site forms its seven rectangles once (rect_base) and adds the AH parts
// of the leaves at the four corners of each into the tile's footprint in LDS (the tile plus the
// three rows and columns its rectangles reach beyond it).  The footprint has one wavefront, whose
// LDS additions execute in program order, so each cell's sum is formed in a fixed order.  The
// footprints go to memory; the gather adds to each site of a tile the overlapping cells of the
// tiles before it along x, along the second direction and diagonally (in that fixed order), and
// sums |F|^2.  Plane (z, y) has no x direction to coalesce along: its z and y links are first
// copied with z fastest (an LDS-tiled transpose), which makes it plane (x', y') of the lattice
// with extents (NT, NZ, NY, NX), and the same two kernels run there.  The gather can also store
// each site's AH parts instead of summing |F|^2: the clover sums of the B^2 adjoint.
#include <algorithm>

#include "flue_launch.hpp"
#include "flue_rect.hpp"
#include "flue_tiles.hpp"

namespace flue {

namespace {

constexpr int kRW = 64;  // one wavefront per tile

// LDS reals per footprint cell: 9 parts, padded to 12 in FP32 (16-byte accesses)
template <typename R>
constexpr int kCellReals = sizeof(R) == 4 ? 12 : 9;
// cells of the largest footprint: eight wavefronts (FP32, two per SIMD) or four (FP64, one per
// SIMD) share a CU's 160 KB of LDS
template <typename R>
constexpr int kMaxCells = sizeof(R) == 4 ? 420 : 560;

// Footprint accumulation.  FP64 fields: LDS atomic adds, element e of cell c at
// [e * FS + c] (a fixed stride, so the elements are offsets of one address).
// FP32 fields: the cell's 9 values padded to 12 floats at [c * 12], read, added and written
// back as three 16-byte LDS accesses, volatile so they stay in program order.  That is safe
// because the footprint belongs to one wavefront: its LDS operations execute in order and the
// lanes of one access address distinct cells.  (FP32 LDS atomic adds kept the waves waiting to
// issue LDS instructions for two thirds of their cycles; FP64 ones do not.)
template <int FS, typename R>
__device__ __forceinline__ void fp_add(R* fp, int cell, const AH<R>& p) {
    if constexpr (sizeof(R) == 4) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) volatile f4 lds_f4;
        lds_f4* q = (lds_f4*)(fp + cell * 12);
        f4 a = q[0], b = q[1], c = q[2];
        a.x += p.d[0];
        a.y += p.d[1];
        a.z += p.d[2];
        a.w += p.or_[0];
        b.x += p.or_[1];
        b.y += p.or_[2];
        b.z += p.oi[0];
        b.w += p.oi[1];
        c.x += p.oi[2];
        q[0] = a;
        q[1] = b;
        q[2] = c;
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            __hip_atomic_fetch_add(fp + k * FS + cell, p.d[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(fp + (3 + k) * FS + cell, p.or_[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(fp + (6 + k) * FS + cell, p.oi[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
}

// LDS reals of a tile's footprint, and of the stride between a cell's elements (FP64)
template <typename R, int W>
constexpr int kTileStride = W ? (W + 3) * (W + 3) : kMaxCells<R>;

// One wavefront, one tile of rectangle plane rp of f: its footprint in LDS (fp), then in memory at
// out as [e * fc + c] in both precisions.
// WPE == 1 (FP64) takes the chains with a one-link lookahead (rect_base); at two waves per
// SIMD (FP32) the other wave covers the load latency.  W > 0: every tile is W x W, so its rows and
// footprint strides are constants (48^3x96: 5.44 -> 5.35 ms in FP32, 10.2 -> 9.9 ms in FP64).
// CHECK: sets *bad where a link is not unitary, testing the one along d2 of every site, and with
// both_dirs the one along d1 (plane (x,y) tests x and y, plane (x,z) z).  The test costs 2% on 24^3x48
// (0.73 -> 0.75 ms) and nothing that shows on 48^3x96 (11.4 ms).
template <bool C2, int WPE, int W, bool CHECK, bool TIME = false, typename FV>
__device__ __forceinline__ void rect_tile(const Lat L, const FV f, int rp, const PlaneTiles g, uint32_t tile,
                                          typename FV::real* fp, typename FV::real* __restrict__ out,
                                          bool both_dirs, uint32_t* bad) {
    using R = typename FV::real;
    constexpr int CR = kCellReals<R>;
    constexpr int FS = kTileStride<R, W>;
    const int d2 = rect_d2<TIME>(rp);
    const Tile t = tile_at<TIME>(L, rp, g, tile);
    const int fc = W ? FS : (int)g.fc, f1 = W ? W + 3 : (int)g.f;
    const uint32_t w = W ? (uint32_t)W : t.l1, h = W ? (uint32_t)W : t.l2;
    bool ok = true;
    for (int k = threadIdx.x; k < (CR == 12 ? CR * fc : CR * FS); k += kRW) fp[k] = R(0);
    __syncthreads();
#pragma unroll 1
    for (uint32_t j0 = 0; j0 < w * h; j0 += kRW) {
        const uint32_t j = j0 + threadIdx.x;
        if (!W && j >= w * h) break;
        // (with W the column is the same in every turn, and its offsets are formed once)
        const int ly = W ? (int)(j0 / w + threadIdx.x / w) : (int)(j / w);
        const int lx = W ? (int)(threadIdx.x % w) : (int)(j - (uint32_t)ly * w);
        const int cx = (int)t.o1 + lx, c2 = (int)t.o2 + ly;
        const uint32_t s = tile_site<TIME>(L, rp, (uint32_t)cx, (uint32_t)c2, t);
        const PlaneGeom<FV> pg = plane_geom(L, f, s, cx, c2, 1, d2);
        const int cell = ly * f1 + lx;
        rect_base<C2, WPE == 1>(make_quad<1, 1, true>(pg), [&](int da, int db, const AH<R>& p) {
            fp_add<FS>(fp, cell + db * f1 + da, p);
        }, [&](const Mat<R>& l1, const Mat<R>& l2) {
            if constexpr (CHECK) {
                ok = ok && unitary(l2);
                if (both_dirs) ok = ok && unitary(l1);
            }
        });
    }
    if (CHECK && !ok) __hip_atomic_store(bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    for (int c = threadIdx.x; c < fc; c += kRW)
#pragma unroll
        for (int e = 0; e < 9; ++e) out[e * fc + c] = fp[CR == 12 ? c * 12 + e : e * FS + c];
}

// what an earlier tile found; read for speed alone, so a stale value is as good
template <bool CHECK>
__device__ __forceinline__ bool given_up(const uint32_t* bad) {
    return CHECK && __builtin_amdgcn_readfirstlane(__hip_atomic_load(bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}

template <typename FV, bool C2, int WPE, int W, bool CHECK>
__global__ void __launch_bounds__(kRW) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
rect_kernel(Lat L0, FV f0, Lat Lzy, FV fzy, RectTiles rt, typename FV::real* __restrict__ fpout,
            uint32_t* __restrict__ bad) {
    using R = typename FV::real;
    __shared__ __align__(16) R fp[kCellReals<R> * kTileStride<R, W>];
    // blockIdx.y: 0 plane (x,y), 1 plane (x,z), 2 plane (z,y) as plane (x,y) of the copy
    const bool zy = blockIdx.y == 2;
    const PlaneTiles g = plane_tiles(rt);
    if (blockIdx.x >= g.tiles || given_up<CHECK>(bad)) return;
    const uint32_t tile = xcd_block(blockIdx.x, g.tiles);
    rect_tile<C2, WPE, W, CHECK>(zy ? Lzy : L0, zy ? fzy : f0, zy ? 0 : (int)blockIdx.y, g, tile, fp,
                                 fpout + 9 * (g.cell0 + (uint64_t)tile * g.fc), blockIdx.y == 0, bad);
}

// the clover AH parts of tile cell (cx, cy): its own footprint's cell, then the overlapping
// cells of the tiles before it along x, along d2 and diagonally, in that order (shift1 and
// shift2 are those tiles' extents along x and d2, in cells)
template <typename R>
__device__ __forceinline__ AH<R> cell_sum(const R* own, const R* left, const R* below, const R* diag, int fc, int f,
                                          int cx, int cy, int shift1, int shift2) {
    const int c = cy * f + cx;
    R v[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        R x = own[e * fc + c];
        if (cx < 3) x += left[e * fc + c + shift1];
        if (cy < 3) x += below[e * fc + c + shift2 * f];
        if (cx < 3 && cy < 3) x += diag[e * fc + c + shift2 * f + shift1];
        v[e] = x;
    }
    AH<R> h;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h.d[k] = v[k];
        h.or_[k] = v[3 + k];
        h.oi[k] = v[6 + k];
    }
    return h;
}

// The four footprints that cover a tile's sites: its own and those of the tiles before it along x
// and d2 (periodic), and the geometry of the overlaps.  fp is the plane's first footprint.
template <typename R, int W>
struct Cover {
    const R *own, *left, *below, *diag;
    int fc, f1, shift1, shift2;
    uint32_t w, h;
    __device__ __forceinline__ Cover(const PlaneTiles& g, const Tile& t, uint32_t tile, const R* fp) {
        const uint32_t tl = t.t1 ? t.t1 - 1 : g.n1 - 1, tb = t.t2 ? t.t2 - 1 : g.n2 - 1;
        const int dl = (int)tl - (int)t.t1, db = ((int)tb - (int)t.t2) * (int)g.n1;
        shift1 = W ? W : (int)(g.q1 + (tl < g.r1 ? 1u : 0u));
        shift2 = W ? W : (int)(g.q2 + (tb < g.r2 ? 1u : 0u));
        fc = W ? (W + 3) * (W + 3) : (int)g.fc;
        f1 = W ? W + 3 : (int)g.f;
        w = W ? (uint32_t)W : t.l1;
        h = W ? (uint32_t)W : t.l2;
        own = fp + 9 * (uint64_t)tile * g.fc;
        left = own + 9 * (int64_t)fc * dl;
        below = own + 9 * (int64_t)fc * db;
        diag = own + 9 * (int64_t)fc * (dl + db);
    }
    // body(cx, cy, AH parts of the site) for this wavefront's share of the tile's sites
    template <typename Body>
    __device__ __forceinline__ void sites(Body&& body) const {
#pragma unroll
        for (uint32_t j0 = 0; j0 < w * h; j0 += kRW) {
            const uint32_t j = j0 + threadIdx.x;
            if (!W && j >= w * h) break;
            const int cy = W ? (int)(j0 / w + threadIdx.x / w) : (int)(j / w);
            const int cx = W ? (int)(threadIdx.x % w) : (int)(j - (uint32_t)cy * w);
            body(cx, cy, cell_sum(own, left, below, diag, fc, f1, cx, cy, shift1, shift2));
        }
    }
};

// Per tile (none where `bad` says that the links are not unitary): its sites' clover AH parts from the four
// footprints that cover them.  One wavefront
// (measured faster than a thread per site).  STORE = false: sum |F|^2 over the tile into one
// compensated partial per tile.  Otherwise write each site's AH parts into Abuf, 9 planes of V
// values per plane, d0 d1 d2, o01r o02r o12r, o01i o02i o12i, for a form of the B^2 adjoint:
// kTiles (k_b2tile.hip) takes the rectangle planes (x,y), (x,z), (z,y), the last with its sites
// numbered as in the copy (z fastest); kSites (k_b2grad.hip) the magnetic planes (y,x), (x,z), (z,y)
// with sites in the field's order (its plane (z,y) is written at strided sites: 1.8 ms at 48^3x96
// in FP32, against 0.6 ms for kTiles).
enum class Store { kNone, kTiles, kSites };
template <typename R, Store STORE, int W>
__global__ void __launch_bounds__(kRW) rect_gather_kernel(Lat L0, Lat Lzy, RectTiles rt, const R* __restrict__ fpin,
                                                         double* __restrict__ partials, R* __restrict__ Abuf,
                                                         const uint32_t* __restrict__ bad) {
    const bool zy = blockIdx.y == 2;
    const PlaneTiles g = plane_tiles(rt);
    if (blockIdx.x >= g.tiles || (bad && *bad)) return;
    const Lat L = zy ? Lzy : L0;
    const int rp = zy ? 0 : (int)blockIdx.y;
    const uint32_t tile = xcd_block(blockIdx.x, g.tiles);
    const Tile t = tile_at(L, rp, g, tile);
    const Cover<R, W> cover(g, t, tile, fpin + 9 * g.cell0);
    double acc = 0.0;
    cover.sites([&](int cx, int cy, const AH<R>& h) {
        if constexpr (STORE != Store::kNone) {
            const uint32_t c2 = t.o2 + (uint32_t)cy, c1 = t.o1 + (uint32_t)cx;
            uint32_t s = tile_site(L, rp, c1, c2, t);
            R sg = R(1);
            if constexpr (STORE == Store::kSites) {
                // the copy's x', y', z' are z, y, x; plane (y,x) is (x,y) reversed
                if (zy) s = t.cs + L0.st[2] * c2 + L0.st[3] * c1 + L0.st[0] * t.ct;
                if (blockIdx.y == 0) sg = R(-1);
            }
            R* o = Abuf + (size_t)blockIdx.y * 9 * L.V + s;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                o[(size_t)k * L.V] = sg * h.d[k];
                o[(size_t)(3 + k) * L.V] = sg * h.or_[k];
                o[(size_t)(6 + k) * L.V] = sg * h.oi[k];
            }
        } else {
            acc += f_norm2(h);
        }
    });
    if constexpr (STORE == Store::kNone) {
        const DD s = block_sum<kRW>(DD{acc, 0.0});
        if (threadIdx.x == 0) {
            const uint32_t i = (blockIdx.y > 0 ? rt.p[0].tiles : 0u) + (blockIdx.y > 1 ? rt.p[1].tiles : 0u) + tile;
            partials[2 * i] = s.hi;
            partials[2 * i + 1] = s.lo;
        }
    }
}

// U_mu0 and U_mu1 of the field (lattice L) into P with direction a (y or z) fastest: P holds two
// blocks of 9 complex planes, [k][e][s'] with k = 0 for U_mu0, 1 for U_mu1, and s' as in L with a and x
// exchanged.  Blocks of 256 threads take T x T (x, a) tiles at fixed other coordinates, through LDS so
// that both the reads (along x) and the writes (along a) coalesce, nine planes in flight: one 16 x 16
// tile, or four 8 x 8 ones where those cover the extents with less padding.
template <typename R, int T>
__device__ __forceinline__ void relayout(const Lat& L, int a, int mu0, int mu1, uint32_t blk, const R* __restrict__ U,
                                         R* __restrict__ P) {
    using P2 = typename Pair2<R>::type;
    constexpr int NT2 = 256 / (T * T);  // tiles per block
    __shared__ P2 tile[NT2][9][T][T + 1];
    const uint32_t NX = (uint32_t)L.n[1], NA = (uint32_t)L.n[a], NO = (uint32_t)L.n[5 - a];
    const uint32_t bxs = (NX + T - 1) / T, bas = (NA + T - 1) / T;
    const uint32_t n = threadIdx.x / (T * T), i = threadIdx.x / T % T, j = threadIdx.x % T;
    uint32_t q = blk * NT2 + n;
    const bool any = q < bxs * bas * NO * (uint32_t)L.n[0];
    const uint32_t bx = q % bxs;
    q /= bxs;
    const uint32_t ba = q % bas;
    q /= bas;
    const uint32_t o = q % NO, t = q / NO;
    const uint32_t s = bx * T + j + L.st[a] * (ba * T + i) + L.st[5 - a] * o + L.st[0] * t;
    // (with a and x exchanged: x has the stride of a, the other direction that of the exchanged extents)
    const uint32_t dx = a == 3 ? NA * NO : NA, d_o = a == 3 ? NA : NA * NX;
    const uint32_t s2 = ba * T + j + dx * (bx * T + i) + d_o * o + L.st[0] * t;
    const bool rd = any && bx * T + j < NX && ba * T + i < NA, wr = any && ba * T + j < NA && bx * T + i < NX;
    const P2* src = reinterpret_cast<const P2*>(U);
    typedef R r2 __attribute__((ext_vector_type(2)));
    r2* dst = reinterpret_cast<r2*>(P);
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
        const int mu = k == 0 ? mu0 : mu1;
        if (rd) {
            P2 v[9];
#pragma unroll
            for (int e = 0; e < 9; ++e) v[e] = src[(size_t)(mu * 9 + e) * L.V + s];
#pragma unroll
            for (int e = 0; e < 9; ++e) tile[n][e][i][j] = v[e];
        }
        __syncthreads();
        if (wr) {
#pragma unroll
            for (int e = 0; e < 9; ++e) {
                const P2 v = tile[n][e][j][i];
                r2 w;
                w.x = v.x;
                w.y = v.y;
                st_stream(dst + (size_t)(k * 9 + e) * L.V + s2, w);
            }
        }
        __syncthreads();
    }
}

// the tile edge for (x, a): 8 where its tiles cover a tenth less than those of 16
int relayout_edge(const Lat& L, int a) {
    auto covered = [&](uint64_t T) { return ((L.n[1] + T - 1) / T) * ((L.n[a] + T - 1) / T) * T * T; };
    return 10 * covered(8) <= 9 * covered(16) ? 8 : 16;
}
uint32_t relayout_blocks(const Lat& L, int a, int T) {
    const uint64_t n = (uint64_t)((L.n[1] + T - 1) / T) * (uint64_t)((L.n[a] + T - 1) / T) * (uint64_t)L.n[5 - a] *
                       (uint64_t)L.n[0];
    return (uint32_t)(T == 8 ? (n + 3) / 4 : n);
}

template <typename R, int T>
__global__ void __launch_bounds__(256) zy_relayout_kernel(Lat L, const R* __restrict__ U, R* __restrict__ P,
                                                          uint32_t* __restrict__ bad) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
    relayout<R, T>(L, 3, 3, 2, blockIdx.x, U, P);
}

// B of links that turned out not unitary, into the same `tiles` partials: the plane-major quadrants
// (k_clover.hip, variant 4), so many of whose blocks of 256 sites to a partial that no more are needed; the
// partials left over are 0.  With the tiles given up on the way (every link off) 24^3x48 takes 1.30 ms and
// 18x20x22x26 0.48 where the quadrant form alone takes 1.15 and 0.38; one bad link in the last tile, 1.49 and
// 0.53.  (64-site shares of the lattice in storage order: 3.39 and 0.93.)
constexpr int kGW = 256;
__host__ __device__ __forceinline__ uint32_t general_blocks(const Lat& L) { return 3 * ((L.V + kGW - 1) / kGW); }
__host__ __device__ __forceinline__ uint32_t general_size(const Lat& L, uint32_t tiles) {
    return (general_blocks(L) + tiles - 1) / tiles;
}
__host__ __device__ __forceinline__ uint32_t general_groups(const Lat& L, uint32_t tiles) {
    const uint32_t n = general_size(L, tiles);
    return (general_blocks(L) + n - 1) / n;
}

template <typename FV>
__device__ __forceinline__ void general_group(const Lat& L, const FV& f, const PlaneOrder& po, uint32_t grp, uint32_t tiles,
                                              double* __restrict__ partials) {
    const uint32_t n = general_size(L, tiles), nb = general_blocks(L) / 3, hi = min(3 * nb, (grp + 1) * n);
    double acc = 0.0;
#pragma unroll 1
    for (uint32_t b = grp * n; b < hi; ++b) {
        const int pl = __builtin_amdgcn_readfirstlane((int)(b / nb));  // (a division leaves the scalar registers)
        const uint32_t o = (b - (uint32_t)pl * nb) * kGW + threadIdx.x;
        if (o >= L.V) continue;
        int c[4];
        const uint32_t s = plane_site(L, po, pl, o, c);
        const int mu = plane_mu(pl), nu = plane_nu(pl);
        acc += f_norm2(plane_ah<false, true, false, true>(plane_geom(L, f, s, c[mu], c[nu], mu, nu)));
    }
    const DD r = block_sum<kGW>(DD{acc, 0.0});
    if (threadIdx.x == 0) {
        partials[2 * grp] = r.hi;
        partials[2 * grp + 1] = r.lo;
    }
    if (grp == 0)
        for (uint32_t i = 2 * general_groups(L, tiles) + threadIdx.x; i < 2 * tiles; i += kGW) partials[i] = 0.0;
    __syncthreads();  // block_sum's shared slots serve the next group
}

// workgroups that look whether there is anything to do (256 are resident at once; a multiple of the XCDs)
constexpr uint32_t kGeneralGrid = 1024;
template <typename FV>
__global__ void __launch_bounds__(kGW) __attribute__((amdgpu_waves_per_eu(1, 1)))
general_kernel(Lat L, FV f, PlaneOrder po, uint32_t tiles, const uint32_t* __restrict__ bad, double* __restrict__ partials) {
    if (!*bad) return;
    const uint32_t groups = general_groups(L, tiles);
    for (uint32_t b = blockIdx.x; b < groups; b += gridDim.x)
        general_group(L, f, po, xcd_block(b, groups), tiles, partials);
}

// the copy read as a field of Lzy whose directions 1 and 2 are its two blocks (the view's base is one
// direction block before P; directions 0 and 3 are never read)
template <typename R>
__host__ __device__ __forceinline__ const R* zy_view(const R* P, uint32_t V) {
    return (const R*)((uintptr_t)P - (uintptr_t)18 * V * sizeof(R));
}

// ---- ensembles: the same tiles, those of every configuration and plane in one launch.  16 fields of
// 16^3 with 644 time slices in all, FP32, one B of each: 3.72 ms by quadrants, 1.65 ms so.

// the configuration of a tile or of a block of the copies; table reads are uniform (scalar loads)
using CEnsRect = const __attribute__((address_space(4))) EnsRect;
using CEnsEntry = const __attribute__((address_space(4))) EnsEntry;
template <uint32_t EnsRect::*First>
__device__ __forceinline__ int rect_cfg(const EnsRect* rect, int n, uint32_t b) {
    const EnsRect* tab = (const EnsRect*)(CEnsRect*)rect;
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].*First <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// tile b of the ensemble: its plane (0 .. 2), leaving b its number in the plane
__device__ __forceinline__ uint32_t rect_plane(const EnsRect& r, uint32_t& b) {
    b -= r.tile0;
    if (b < r.rt.p[0].tiles) return 0;
    b -= r.rt.p[0].tiles;
    if (b < r.rt.p[1].tiles) return 1;
    b -= r.rt.p[1].tiles;
    return 2;
}

template <typename R, int T>
__global__ void __launch_bounds__(256) ens_relayout_kernel(const EnsEntry* __restrict__ tab,
                                                           const EnsRect* __restrict__ rect, int n,
                                                           const R* __restrict__ U, R* __restrict__ P,
                                                           uint32_t* __restrict__ bad) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
    const int c = rect_cfg<&EnsRect::copy0>(rect, n, blockIdx.x);
    const EnsEntry& e = *(const EnsEntry*)((CEnsEntry*)tab + c);
    relayout<R, T>(e.L, 3, 3, 2, blockIdx.x - rect[c].copy0, U + e.off, P + e.off);
}

template <typename R, bool C2, int WPE, int W, bool CHECK>
__global__ void __launch_bounds__(kRW) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
ens_rect_kernel(const EnsEntry* __restrict__ tab, const EnsRect* __restrict__ rect, int n, const R* __restrict__ U,
                const R* __restrict__ P, R* __restrict__ fpout, uint32_t* __restrict__ bad) {
    if (given_up<CHECK>(bad)) return;
    __shared__ __align__(16) R fp[kCellReals<R> * kTileStride<R, W>];
    uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
    const int c = rect_cfg<&EnsRect::tile0>(rect, n, tile);
    const EnsEntry& e = *(const EnsEntry*)((CEnsEntry*)tab + c);
    const EnsRect& r = *(const EnsRect*)((CEnsRect*)rect + c);
    const uint32_t y = rect_plane(r, tile);
    const PlaneTiles g = plane_tiles(r.rt, y);
    const FieldView<R, true> f{y == 2 ? zy_view(P + e.off, e.L.V) : U + e.off, e.L.V};
    rect_tile<C2, WPE, W, CHECK>(y == 2 ? r.Lzy : e.L, f, y == 1 ? 1 : 0, g, tile, fp,
                                 fpout + e.off / 72 * 48 + 9 * (g.cell0 + (uint64_t)tile * g.fc), y == 0, bad);
}

template <typename R>
__global__ void __launch_bounds__(kGW) __attribute__((amdgpu_waves_per_eu(1, 1)))
ens_general_kernel(const EnsEntry* __restrict__ tab, const EnsRect* __restrict__ rect, int n, uint32_t groups,
                   const R* __restrict__ U, const uint32_t* __restrict__ bad, double* __restrict__ partials) {
    if (!*bad) return;
    for (uint32_t b = blockIdx.x; b < groups; b += gridDim.x) {
        const uint32_t grp = xcd_block(b, groups);
        const int c = rect_cfg<&EnsRect::grp0>(rect, n, grp);
        const EnsEntry& e = *(const EnsEntry*)((CEnsEntry*)tab + c);
        const EnsRect& r = *(const EnsRect*)((CEnsRect*)rect + c);
        const FieldView<R, true> f{U + e.off, e.L.V};
        general_group(e.L, f, r.po, grp - r.grp0, r.tiles, partials + 2 * (size_t)r.tile0);
    }
}

template <typename R, int W>
__global__ void __launch_bounds__(kRW) ens_gather_kernel(const EnsEntry* __restrict__ tab,
                                                         const EnsRect* __restrict__ rect, int n,
                                                         const R* __restrict__ fpin, double* __restrict__ partials,
                                                         const uint32_t* __restrict__ bad) {
    if (bad && *bad) return;
    const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
    const int c = rect_cfg<&EnsRect::tile0>(rect, n, b);
    const EnsEntry& e = *(const EnsEntry*)((CEnsEntry*)tab + c);
    const EnsRect& r = *(const EnsRect*)((CEnsRect*)rect + c);
    uint32_t tile = b;
    const uint32_t y = rect_plane(r, tile);
    const PlaneTiles g = plane_tiles(r.rt, y);
    const Tile t = tile_at(y == 2 ? r.Lzy : e.L, y == 1 ? 1 : 0, g, tile);
    double acc = 0.0;
    Cover<R, W>(g, t, tile, fpin + e.off / 72 * 48 + 9 * g.cell0).sites([&](int, int, const AH<R>& h) {
        acc += f_norm2(h);
    });
    const DD s = block_sum<kRW>(DD{acc, 0.0});
    if (threadIdx.x == 0) {
        partials[2 * b] = s.hi;
        partials[2 * b + 1] = s.lo;
    }
}

// ---- one plane's field strength, per site.  A plane with x runs on the field; (z, y), (z, t) and
// (y, t) on a copy of their two links with z or y fastest, whose lattice has that extent as its x.  FP64
// fields: F of an FP32 field, handed out in FP64, keeps the rounding of the quadrants.  24^3x48, us by quadrants -> by tiles (tiles 255, gather 40 to 50, copy 80): (x,y) 512 -> 287,
// (x,z) 447 -> 272, (x,t) 512 -> 297, (z,y) 469 -> 355, (z,t), (y,t) 452 -> 350.  The tiles run at the
// FP64 rate of the whole form (matrix products, one wave per SIMD); one plane alone ends in a partly
// filled last round.

// the links of the copy, and the flag of links that are not unitary cleared (the copy's or, alone,
// block 0's work)
template <typename R, int T>
__global__ void __launch_bounds__(256) plane_copy_kernel(Lat L, int a, int mu0, int mu1, const R* __restrict__ U,
                                                         R* __restrict__ P, uint32_t* __restrict__ bad) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
    if (P) relayout<R, T>(L, a, mu0, mu1, blockIdx.x, U, P);
}

template <typename FV, bool TIME>
__global__ void __launch_bounds__(kRW) __attribute__((amdgpu_waves_per_eu(1, 1)))
plane_kernel(Lat L, FV f, int rp, PlaneTiles g, typename FV::real* __restrict__ fpout, uint32_t* __restrict__ bad) {
    using R = typename FV::real;
    __shared__ __align__(16) R fp[kCellReals<R> * kTileStride<R, 0>];
    if (given_up<true>(bad)) return;
    const uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
    rect_tile<false, 1, 0, true, TIME>(L, f, rp, g, tile, fp, fpout + 9 * (uint64_t)tile * g.fc, true, bad);
}

// F of every site from the footprints, in an array whose t is dense: a block has 16 x and 16 t at fixed
// y and z, reads the footprints along x and writes along t, through LDS.  sign: that of the plane's
// orientation; os: strides in the directions of L (its x may be the field's z or y).
constexpr int kFT = 16;
template <typename R, bool TIME>
__global__ void __launch_bounds__(kFT * kFT) plane_gather_kernel(Lat L, int rp, PlaneTiles g,
                                                               const R* __restrict__ fpin, R sign,
                                                               double* __restrict__ out, OutStrides os,
                                                               const uint32_t* __restrict__ bad) {
    __shared__ R parts[9][kFT][kFT + 1];
    if (*bad) return;
    const uint32_t nx = (uint32_t)L.n[1], nt = (uint32_t)L.n[0], ny = (uint32_t)L.n[2];
    const uint32_t bts = (nt + kFT - 1) / kFT, bxs = (nx + kFT - 1) / kFT;
    uint32_t q = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t t0 = (q % bts) * kFT;
    q /= bts;
    const uint32_t x0 = (q % bxs) * kFT;
    q /= bxs;
    const uint32_t y = q % ny, z = q / ny;
    const uint32_t i = threadIdx.x % kFT, j = threadIdx.x / kFT;
    if (x0 + i < nx && t0 + j < nt) {
        const uint32_t c2 = TIME ? t0 + j : (rp == 0 ? y : z);
        uint32_t o1, o2;
        Tile t;
        t.t1 = tile_of(x0 + i, g.q1, g.r1, &o1);
        t.t2 = tile_of(c2, g.q2, g.r2, &o2);
        const uint32_t cs = TIME || rp == 1 ? y : z, ct = TIME ? z : t0 + j;
        const uint32_t ns = (uint32_t)L.n[TIME || rp == 1 ? 2 : 3];
        const Cover<R, 0> cover(g, t, t.t1 + g.n1 * (t.t2 + g.n2 * (cs + ns * ct)), fpin);
        const AH<R> h = cell_sum(cover.own, cover.left, cover.below, cover.diag, cover.fc, cover.f1,
                                 (int)(x0 + i - o1), (int)(c2 - o2), cover.shift1, cover.shift2);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            parts[k][i][j] = sign * h.d[k];
            parts[3 + k][i][j] = sign * h.or_[k];
            parts[6 + k][i][j] = sign * h.oi[k];
        }
    }
    __syncthreads();
    // i along t, j along x
    if (x0 + j < nx && t0 + i < nt) {
        AH<R> h;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            h.d[k] = parts[k][j][i];
            h.or_[k] = parts[3 + k][j][i];
            h.oi[k] = parts[6 + k][j][i];
        }
        const int c[4] = {(int)(t0 + i), (int)(x0 + j), (int)y, (int)z};
        store_f(h, c, out, os);
    }
}

// How plane (mu, nu) is tiled: L and the plane of it, the field's directions along its x (d1) and its
// second direction (d2), and the directions whose links are copied (mu0 < 0: none).
struct FPlane {
    Lat L;
    int rp, d1, d2, mu0, mu1;
    PlaneTiles g;
    size_t copy_at, bytes;  // (the flag lies in front of `bytes`)
    bool first_is_zero;     // the copy's first block is its lattice's direction 0, else 1
};

}  // namespace

bool rect_by16(const Lat& L) { return L.n[1] % 16 == 0 && L.n[2] % 16 == 0 && L.n[3] % 16 == 0; }

namespace {

// (FP32 keeps 16 x 16 tiles on extents that they divide: the order of a site's FP32 sum, with it 1e-9 of B
// of few sites, goes with the tiles)
RectTiles rect_tiles_of(const Lat& L, int is_f32) {
    if (is_f32 && rect_by16(L)) return rect_split(L, 19 * 19, 1);
    return rect_split(L, is_f32 ? kMaxCells<float> : kMaxCells<double>, is_f32 ? 2048 : 1024);
}

}  // namespace

// Where the rectangle-first form runs: spatial extents of 12 or more (below, a tile is mostly
// halo), and either all multiples of 16, which tile without idle lanes, or 90000 sites.  As
// measured, quadrant form against this one, ms (FP32 / FP64 / FP64 declared SU(3)):
//   12^3x24     41,472 sites   0.051 / 0.079 / 0.070   ->   0.063 / 0.078 / 0.075
//   18x15x20x8  43,200         0.055 / 0.082 / 0.075   ->   0.063 / 0.083 / 0.080
//   18x15x20x16 86,400         0.103 / 0.162 / 0.145   ->   0.091 / 0.160 / 0.152
//   20^3x12     96,000         0.116 / 0.185 / 0.166   ->   0.087 / 0.144 / 0.137
//   24^3x48                    0.663 / 1.15  / 1.02    ->   0.433 / 0.770 / 0.734
//   33x34x32x27                0.983 / 1.75  / 1.58    ->   0.631 / 1.11  / 1.07
//   16^3x8      32,768         0.049 / 0.072 / 0.062   ->   0.036 / 0.059 / 0.057
//   48^3x96                    10.6  / 18.8  / 16.8    ->   6.26  / 11.4  / 11.0
constexpr uint32_t kRectSites = 90000;
bool rect_fits(const Lat& L) {
    if (rect_by16(L)) return true;
    return std::min({L.n[1], L.n[2], L.n[3]}) >= 12 && L.V >= kRectSites;
}

// Untuned, FP32 lattices of other extents take it from 300,000 sites on: the two forms round B apart by
// 3e-10 and 1e-7 over the root of the sites.
constexpr uint32_t kRectSitesF32 = 300000;
bool rect_untuned(const Lat& L, int is_f32) { return !is_f32 || rect_by16(L) || L.V >= kRectSitesF32; }

uint32_t rect_partials(const Lat& L, int is_f32) {
    const RectTiles r = rect_tiles_of(L, is_f32);
    return r.p[0].tiles + r.p[1].tiles + r.p[2].tiles;
}

// the three planes' footprints, then the z-fastest copy of U_z and U_y and the flag of links that are
// not unitary
static size_t rect_copy_offset(const RectTiles& r, size_t sz) { return ((size_t)rect_cells(r) * 9 * sz + 255) & ~(size_t)255; }
size_t rect_fp_bytes(const Lat& L, int is_f32) {
    const size_t sz = is_f32 ? 4 : 8;
    return rect_copy_offset(rect_tiles_of(L, is_f32), sz) + (size_t)36 * L.V * sz + 256;
}

size_t rect_footprint_bytes(const Lat& L, int is_f32) { return rect_copy_offset(rect_tiles_of(L, is_f32), is_f32 ? 4 : 8); }

// partials: rect_partials, the tiles of the planes (x, y), (x, z), (z, y) in turn.  With Abuf, the
// per-site AH parts go there instead, for the tiled B^2 adjoint or for the others (tiled == 0), and
// no partials are written.  copy_at > 0 places the z-fastest copy there in fpbuf.
hipError_t launch_magnetic_rect(const Lat& L, const void* U, int is_f32, int su3, double* partials, void* fpbuf,
                                hipStream_t st, uint32_t* npart, void* Abuf, int tiled, size_t copy_at) {
    if (!rect_fits(L) || !fits_buffer(L.V, is_f32)) return hipErrorInvalidValue;
    const RectTiles rt = rect_tiles_of(L, is_f32);
    const Lat Lzy = zy_lattice(L);
    with_view(L.V, U, is_f32, [&](auto f) {
        using F = decltype(f);
        using R = typename F::real;
        if constexpr (F::buffered) {
            R* fp = (R*)fpbuf;
            R* P = (R*)((char*)fpbuf + (copy_at ? copy_at : rect_copy_offset(rt, sizeof(R))));
            uint32_t* bad = (uint32_t*)(P + (size_t)36 * L.V);
            if (relayout_edge(L, 3) == 8)
                zy_relayout_kernel<R, 8><<<relayout_blocks(L, 3, 8), 256, 0, st>>>(L, f.p, P, bad);
            else
                zy_relayout_kernel<R, 16><<<relayout_blocks(L, 3, 16), 256, 0, st>>>(L, f.p, P, bad);
            const F fzy{zy_view<R>(P, L.V), L.V};
            const dim3 g(std::max({rt.p[0].tiles, rt.p[1].tiles, rt.p[2].tiles}), 3);
            // FP32 and declared-SU(3) FP64 links: two-row chains; plain FP64: full products, and the
            // quadrant sums for links that are not unitary
            const bool check = sizeof(R) == 8 && !su3;
            auto rect = [&](auto w) {
                constexpr int W = decltype(w)::value;
                if constexpr (sizeof(R) == 4) {
                    rect_kernel<F, true, 2, W, false><<<g, kRW, 0, st>>>(L, f, Lzy, fzy, rt, fp, bad);
                } else {
                    if (su3)
                        rect_kernel<F, true, 1, W, false><<<g, kRW, 0, st>>>(L, f, Lzy, fzy, rt, fp, bad);
                    else
                        rect_kernel<F, false, 1, W, true><<<g, kRW, 0, st>>>(L, f, Lzy, fzy, rt, fp, bad);
                }
                if (Abuf && tiled)
                    rect_gather_kernel<R, Store::kTiles, W><<<g, kRW, 0, st>>>(L, Lzy, rt, fp, nullptr, (R*)Abuf, nullptr);
                else if (Abuf)
                    rect_gather_kernel<R, Store::kSites, W><<<g, kRW, 0, st>>>(L, Lzy, rt, fp, nullptr, (R*)Abuf, nullptr);
                else
                    rect_gather_kernel<R, Store::kNone, W><<<g, kRW, 0, st>>>(L, Lzy, rt, fp, partials, nullptr, check ? bad : nullptr);
            };
            if (rt.p[0].square() && rt.p[1].square() && rt.p[2].square())
                rect(std::integral_constant<int, 16>());
            else
                rect(std::integral_constant<int, 0>());
            if constexpr (sizeof(R) == 8)
                if (check && !Abuf) {
                    const uint32_t tiles = rt.p[0].tiles + rt.p[1].tiles + rt.p[2].tiles;
                    general_kernel<<<std::min(kGeneralGrid, general_groups(L, tiles)), kGW, 0, st>>>(
                        L, f, plane_order(L, sizeof(R)), tiles, bad, partials);
                }
        }
    });
    if (npart) *npart = rect_partials(L, is_f32);
    return hipGetLastError();
}

// (FP32: each of enough sites that the forms' B differ by 6e-10 at most)
constexpr uint32_t kEnsRectSitesF32 = 49152;

// Every configuration has to suit the tiles (extents as in rect_fits) and its footprints to fit the
// plaquette parts' 48 reals a site; the sites are counted over the ensemble, since it runs as one launch,
// and the tiles are those that cost least on a full chip.  A measurement (B and the plaquettes), ms by
// quadrants -> by tiles, FP32 (of fields large enough) and FP64:
//   2 x 16^3x12         98,304 sites   0.156 -> 0.115   0.272 -> 0.194
//   5 x 12^3x13        112,320                          0.277 -> 0.241
//   8 x 12x13x14x10    174,720                          0.392 -> 0.304
//   8 x 16^4           524,288         0.665 -> 0.365   1.191 -> 0.677
bool ens_rect_plan(const EnsEntry* tab, int n, int is_f32, uint32_t maxV, EnsRect* rect, EnsRectGrid* g) {
    if (!fits_buffer(maxV, is_f32)) return false;
    uint64_t sites = 0, tiles = 0, copies = 0, groups = 0;
    g->square = true;
    g->copy_edge = 16;
    for (int c = 0; c < n; ++c)
        if (relayout_edge(tab[c].L, 3) == 8) g->copy_edge = 8;
    for (int c = 0; c < n; ++c) {
        const Lat& L = tab[c].L;
        if (std::min({L.n[1], L.n[2], L.n[3]}) < 12 || (is_f32 && L.V < kEnsRectSitesF32)) return false;
        EnsRect& r = rect[c];
        r.rt = rect_split(L, is_f32 ? kMaxCells<float> : kMaxCells<double>, 1);
        if (rect_cells(r.rt) * 9 > (uint64_t)48 * L.V) return false;
        r.Lzy = zy_lattice(L);
        r.po = plane_order(L, sizeof(double));
        r.tile0 = (uint32_t)tiles;
        r.tiles = r.rt.p[0].tiles + r.rt.p[1].tiles + r.rt.p[2].tiles;
        r.copy0 = (uint32_t)copies;
        r.grp0 = (uint32_t)groups;
        groups += general_groups(L, r.tiles);
        for (const PlaneTiles& p : r.rt.p) g->square = g->square && p.square();
        sites += L.V;
        tiles += r.tiles;
        copies += relayout_blocks(L, 3, g->copy_edge);
    }
    g->tiles = (uint32_t)tiles;
    g->copies = (uint32_t)copies;
    g->groups = (uint32_t)groups;
    return sites >= kRectSites && tiles < 0x80000000ull && copies < 0x80000000ull;
}

hipError_t launch_ens_rect(const EnsEntry* tab, const EnsRect* rect, int n, const EnsRectGrid& g, const void* fld,
                           int is_f32, void* copy, void* fp, double* partials, hipStream_t st) {
    uint32_t* bad = (uint32_t*)(partials + 2 * (size_t)g.tiles);
    auto run = [&](auto real, auto w) {
        using R = decltype(real);
        constexpr int W = decltype(w)::value;
        constexpr bool F32 = sizeof(R) == 4;  // FP32: two-row chains, two waves per SIMD
        if (g.copy_edge == 8)
            ens_relayout_kernel<R, 8><<<g.copies, 256, 0, st>>>(tab, rect, n, (const R*)fld, (R*)copy, bad);
        else
            ens_relayout_kernel<R, 16><<<g.copies, 256, 0, st>>>(tab, rect, n, (const R*)fld, (R*)copy, bad);
        ens_rect_kernel<R, F32, F32 ? 2 : 1, W, !F32>
            <<<g.tiles, kRW, 0, st>>>(tab, rect, n, (const R*)fld, (const R*)copy, (R*)fp, bad);
        ens_gather_kernel<R, W><<<g.tiles, kRW, 0, st>>>(tab, rect, n, (const R*)fp, partials, F32 ? nullptr : bad);
        if constexpr (!F32)  // links that are not unitary
            ens_general_kernel<R><<<std::min(kGeneralGrid, g.groups), kGW, 0, st>>>(tab, rect, n, g.groups,
                                                                                    (const R*)fld, bad, partials);
    };
    auto sized = [&](auto real) {
        if (g.square)
            run(real, std::integral_constant<int, 16>());
        else
            run(real, std::integral_constant<int, 0>());
    };
    if (is_f32)
        sized(float(0));
    else
        sized(double(0));
    return hipGetLastError();
}

// Planes with both extents of 12 or more on lattices of 90000 sites or more, as measured (us by quadrants
// -> by tiles): 20^3x12 82 -> 57 and, on a copy, 78 -> 73; 16^3x24 81 -> 54 and 75 -> 66.  Below, two and a half thousand tiles do not fill the
// chip's slots, and the three or four launches outweigh the products saved.
static bool f_plane(const Lat& L, int mu, int nu, FPlane* p) {
    if (mu == nu || !fits_buffer(L.V, 0) || L.V < kRectSites || std::min(L.n[mu], L.n[nu]) < 12) return false;
    auto has = [&](int d) { return mu == d || nu == d; };
    const int32_t yfast[4] = {L.n[0], L.n[2], L.n[1], L.n[3]};
    p->first_is_zero = has(0);
    p->mu0 = p->mu1 = -1;
    p->L = L;
    if (has(1)) {
        p->d1 = 1;
        p->d2 = mu + nu - 1;
    } else if (has(3)) {
        p->L = zy_lattice(L);
        p->d1 = 3;
        p->d2 = mu + nu - 3;
        p->mu0 = has(0) ? 0 : 3;
        p->mu1 = has(0) ? 3 : 2;
    } else {
        p->L = make_lat(yfast);
        p->d1 = p->mu1 = 2;
        p->d2 = p->mu0 = 0;
    }
    p->rp = p->d2 == 0 ? 2 : (p->d1 == 1 && p->d2 == 3 ? 1 : 0);
    const uint32_t NX = (uint32_t)p->L.n[1], NY = (uint32_t)p->L.n[2], NZ = (uint32_t)p->L.n[3], NT = (uint32_t)L.n[0];
    const uint32_t n2 = p->rp == 0 ? NY : (p->rp == 1 ? NZ : NT), s1 = p->rp == 0 ? NZ : NY, s2 = p->rp == 2 ? NZ : NT;
    p->g = plane_split(NX, n2, s1, s2, kMaxCells<double>, 1024, s2);
    const size_t sz = sizeof(double);
    p->copy_at = ((size_t)p->g.tiles * p->g.fc * 9 * sz + 255) & ~(size_t)255;
    p->bytes = p->copy_at + (p->mu0 >= 0 ? (size_t)36 * L.V * sz : 0) + 256;
    return true;
}

size_t fmunu_rect_bytes(const Lat& L, int mu, int nu) {
    FPlane p;
    return f_plane(L, mu, nu, &p) ? p.bytes : 0;
}

hipError_t launch_fmunu_rect(const Lat& L, const void* U, int mu, int nu, void* out, const int64_t s6[6], void* ws,
                             hipStream_t st) {
    FPlane p;
    if (!f_plane(L, mu, nu, &p) || s6[0] != 1) return hipErrorInvalidValue;
    const OutStrides os{s6[0], s6[1], s6[2], s6[3], s6[4], s6[5]};
    // the strides along the directions of p.L
    OutStrides osl = os;
    if (p.d1 != 1) {
        osl.x = p.d1 == 3 ? os.z : os.y;
        (p.d1 == 3 ? osl.z : osl.y) = os.x;
    }
    using F = FieldView<double, true>;
    const F f{(const double*)U, L.V};
    double* fp = (double*)ws;
    double* P = p.mu0 >= 0 ? (double*)((char*)ws + p.copy_at) : nullptr;
    uint32_t* bad = (uint32_t*)((char*)ws + p.bytes - 256);
    const int a = p.d1 == 1 ? 2 : p.d1;
    if (P && relayout_edge(L, a) == 16)
        plane_copy_kernel<double, 16><<<relayout_blocks(L, a, 16), 256, 0, st>>>(L, a, p.mu0, p.mu1, f.p, P, bad);
    else
        plane_copy_kernel<double, 8>
            <<<P ? relayout_blocks(L, a, 8) : 1, 256, 0, st>>>(L, a, p.mu0, p.mu1, f.p, P, bad);
    // the copy's two blocks are directions 0 and 1 of its lattice, or 1 and 2
    const F fl{P ? (p.first_is_zero ? P : zy_view<double>(P, L.V)) : f.p, L.V};
    const double sign = mu == p.d1 ? 1.0 : -1.0;
    auto run = [&](auto time) {
        constexpr bool TIME = decltype(time)::value;
        plane_kernel<F, TIME><<<p.g.tiles, kRW, 0, st>>>(p.L, fl, p.rp, p.g, fp, bad);
        const uint32_t nb = (uint32_t)((p.L.n[0] + kFT - 1) / kFT) * (uint32_t)((p.L.n[1] + kFT - 1) / kFT) *
                            (uint32_t)p.L.n[2] * (uint32_t)p.L.n[3];
        plane_gather_kernel<double, TIME><<<nb, kFT * kFT, 0, st>>>(p.L, p.rp, p.g, fp, sign, (double*)out, osl,
                                                                     bad);
    };
    if (p.rp == 2)
        run(std::true_type());
    else
        run(std::false_type());
    // by quadrants, where a link turned out not unitary
    return launch_fmunu(L, U, 0, mu, nu, 0, out, 0, s6, st, bad);
}

}  // namespace flue
