// k_wloops.hip -- all rectangular Wilson loops R x T (1 <= R <= Rmax, 1 <= T <= Tmax) of
// one plane in a single pass over the lattice.
//
// The loop at x is ReTr[CA(R,T) CB(T,R)^+] (src/wloops.F90:679-791, :567-677), with
//   CA(R,T) = Lmu(x; R) Lnu(x + R mu; T)   (R steps along mu, then T along nu),
//   CB(T,R) = Lnu(x; T) Lmu(x + T nu; R)   (T steps along nu, then R along mu),
// where L(y; n) is the product of n successive links from y.  One thread per site keeps
// the Tmax chains CB(T, .) and extends them by one link per R, and runs one CA chain per
// R: about Rmax*Tmax + 2*(Rmax + Tmax) products per site for the whole table, against
// 2(R+T)-1 products for each loop walked on its own.
//
// A loop reads links up to 6 sites away along mu and nu.  In a plane containing time those
// are up to 6 time slices apart, so there the blocks are ordered with the time slice
// fastest: a block covers kBS sites of one slice, consecutive blocks take the same sites
// of consecutive slices, and the blocks that run together on an XCD share their links in L2
// (in storage order the L2 of an XCD held no more than a slice, and 9 in 10 reads missed).
// In the (z, t) and (x, z) planes a slice is also taken with z second-fastest after x, so
// the loops' z neighbours lie in the same block or the next rather than 9 blocks on.
//
// A site's six-by-six table reads 84 links, 12 KB in FP64, and nothing of that stays in L1: the chip
// moved 25 GB from L2 for 32^3x64 (1.5 ms, three times the products' time).  Planes with x take
// tiles of up to 256 sites in the plane, whose links (the tile and six more rows and columns, up to
// 155 KB in FP64) are read into LDS once: 1.9 links of either direction per site for 16 x 16 tiles.
// Then the vector unit issues 73% of the cycles in FP64 (of 13,800 instructions a wave 9,500 are the
// products and traces; most others move the chains beyond 256 registers), and 15% wait for a tile's loads.
#include "flue_common.hpp"
#include "flue_launch.hpp"
#include "flue_tiles.hpp"

namespace flue {

namespace {

constexpr int kBS = 256;

// v of lane ^ 1 (CTRL 0xB1) or lane ^ 2 (0x4E)
template <int CTRL>
__device__ __forceinline__ double quad_swap(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// sum over the 16 lanes of a row
__device__ __forceinline__ double row_sum(double v) {
    v += quad_swap<0xB1>(v);
    v += quad_swap<0x4E>(v);
    v += quad_swap<0x141>(v);  // half row mirrored: the other four
    v += quad_swap<0x140>(v);  // row mirrored: the other eight
    return v;
}

// Grid: groups x nb logical blocks, one group per time slice for kEverySlice, else one.
// With time in the plane the slice is the fastest block index (for the whole lattice, nb
// counts the blocks of every slice, slice fastest); otherwise the block within the group is.
//
// TM = Tmax is a template argument, so a row of the table (one R) is straight code: each step's two
// products, of CA and of CB(T, .), each start the load of the link that the next step puts in place of
// the one they used.  Each four lanes write the
// sum of their traces to LDS slots of their own; the block adds those at the end, compensated like the
// final pass over the blocks.
template <typename FV, int TM>
__global__ void __launch_bounds__(kBS) __attribute__((amdgpu_waves_per_eu(sizeof(typename FV::real) == 4 ? 2 : 1)))
wloop_table_kernel(Lat L, FV f, int mu, int nu, int Rmax, int tslice, uint32_t nb, uint32_t groups,
                   double* __restrict__ partials) {
    using R_ = typename FV::real;
    __shared__ double sh[kMaxLoopRT * TM][kBS / 4];  // [(R - 1) Tmax + T - 1][four threads]
    const bool tplane = mu == 0 || nu == 0;
    const uint32_t g = xcd_block(blockIdx.x, gridDim.x);
    uint32_t grp, blk;
    if (tslice == kEverySlice && tplane) {
        grp = g % groups;
        blk = g / groups;
    } else {
        grp = g / nb;
        blk = g - grp * nb;
    }
    // tslice >= 0: that time slice; -1: every site; kEverySlice: slice grp
    const int ts = tslice == kEverySlice ? (int)grp : tslice;
    // in a time plane the slice is taken along the plane's spatial direction; in the (x, z)
    // plane along z
    const int d = tplane ? mu + nu : (mu + nu == 4 ? 3 : 1);
    bool live;
    uint32_t s;
    if (ts >= 0) {
        const uint32_t idx = blk * kBS + threadIdx.x;
        live = idx < L.Vs;
        s = (live ? slice_site_along(L, idx, d) : 0u) + L.Vs * (uint32_t)ts;
    } else if (tplane) {
        const uint32_t NT = (uint32_t)L.n[0];
        const uint32_t chunk = blk / NT, t = blk - chunk * NT;
        const uint32_t idx = chunk * kBS + threadIdx.x;
        live = idx < L.Vs;
        s = (live ? slice_site_along(L, idx, d) : 0u) + L.Vs * t;
    } else {
        const uint32_t idx = blk * kBS + threadIdx.x;
        live = idx < L.V;
        const uint32_t t = idx / L.Vs;
        s = d == 1 ? idx : slice_site_along(L, idx - t * L.Vs, d) + L.Vs * t;
    }
    // lanes past the end work on site 0 (in bounds) and contribute nothing
    if (!live) s = 0u;
    int c[4];
    site_coords(L, s, c);
    const int cmu = c[mu], cnu = c[nu];
    const int nmu = L.ext(mu), nnu = L.ext(nu);
    const uint32_t smu = L.stride(mu), snu = L.stride(nu);
    const uint32_t base = s - (uint32_t)cmu * smu - (uint32_t)cnu * snu;
    // site of x + R mu + T nu = base + a + B[T], a the offset of x + R mu
    uint32_t B[TM + 1];
#pragma unroll
    for (int k = 0; k <= TM; ++k) B[k] = (uint32_t)((cnu + k) % nnu) * snu;
    int xm = cmu;
    uint32_t a = (uint32_t)cmu * smu;
    double* mine = &sh[0][threadIdx.x >> 2];

    // CB(T, 1) for T = 1..Tmax from the nu line at x
    Mat<R_> CB[TM];
    Mat<R_> Ln = load_link(f, nu, base + a + B[0]);
#pragma unroll
    for (int T = 1; T <= TM; ++T) {
        if (T > 1) Ln = mul(Ln, load_link(f, nu, base + a + B[T - 1]));
        CB[T - 1] = mul(Ln, load_link(f, mu, base + a + B[T]));
        __builtin_amdgcn_sched_barrier(0);
    }
    Mat<R_> Lm = load_link(f, mu, base + a + B[0]);
    __builtin_amdgcn_sched_barrier(0);
    // one row: Lm = Lmu(x; R), M and N the links of its first step (EXT: the CB are extended by it too)
    auto row = [&](auto ext, uint32_t ap, Mat<R_> M, Mat<R_> N) {
        constexpr bool EXT = decltype(ext)::value;
        Mat<R_> CA;
#pragma unroll
        for (int T = 1; T <= TM; ++T) {
            CA = T == 1 ? mul(Lm, N) : mul(CA, N);
            __builtin_amdgcn_sched_barrier(0);
            if (T < TM) N = load_link(f, nu, base + a + B[T]);
            if constexpr (EXT) {
                CB[T - 1] = mul(CB[T - 1], M);
                __builtin_amdgcn_sched_barrier(0);
                if (T < TM) M = load_link(f, mu, base + ap + B[T + 1]);
            }
            double v = (double)retr_nd(CA, CB[T - 1]);
            v = live ? v : 0.0;
            v += quad_swap<0xB1>(v);
            v += quad_swap<0x4E>(v);
            mine[(T - 1) * (kBS / 4)] = v;  // (the four lanes' one value: a branch here spills the chains, 1.61 for 1.27 ms)
            __builtin_amdgcn_sched_barrier(0);
        }
        mine += TM * (kBS / 4);
    };
    auto step = [&] {
        const uint32_t ap = a;
        xm = xm + 1 == nmu ? 0 : xm + 1;
        a = (uint32_t)xm * smu;
        return ap;
    };
    {
        step();
        row(std::false_type(), 0u, Mat<R_>(), load_link(f, nu, base + a + B[0]));
    }
#pragma unroll 1
    for (int R = 2; R <= Rmax; ++R) {
        const uint32_t ap = step();
        const Mat<R_> U = load_link(f, mu, base + ap + B[0]);
        const Mat<R_> M = load_link(f, mu, base + ap + B[1]), N = load_link(f, nu, base + a + B[0]);
        Lm = mul(Lm, U);
        row(std::true_type(), ap, M, N);
    }
    __syncthreads();
    // a wave per entry sums its 64 slots, the 16 of a wave plainly, the four waves compensated (all six steps
    // compensated: 1% of a large table and 4% of a small one)
    const int lane = threadIdx.x & 63;
    for (int k = threadIdx.x >> 6; k < Rmax * TM; k += kBS / 64) {
        DD v = {row_sum(sh[k][lane]), 0.0};
        v = dd_add(v, dd_shfl_xor(v, 16));
        v = dd_add(v, dd_shfl_xor(v, 32));
        if (lane == 0) {
            double* p = partials + 2 * (((size_t)k * groups + grp) * nb + blk);
            p[0] = v.hi;
            p[1] = v.lo;
        }
    }
}

// LDS cells of a tile's links: one block of 256 threads on a CU in FP64 (one wave per SIMD, by the
// chains' registers), two in FP32
template <typename R>
constexpr uint32_t kTileCells = sizeof(R) == 4 ? 536 : 552;

// row_sum, compensated from the four sums of four lanes on
template <int CTRL>
__device__ __forceinline__ DD dd_swap_add(DD v) {
    return dd_add(v, DD{quad_swap<CTRL>(v.hi), quad_swap<CTRL>(v.lo)});
}
__device__ __forceinline__ DD row_dd_sum(double v) {
    v += quad_swap<0xB1>(v);
    v += quad_swap<0x4E>(v);
    return dd_swap_add<0x140>(dd_swap_add<0x141>(DD{v, 0.0}));
}

// The table of a plane with x, tile by tile: direction 1 of the tiles is x, direction 2 the other one,
// o.  Tile `blk` of a group: spectators y and z where o is time, else z or y and, in a group of the
// whole lattice (t0 < 0), the slice.
template <typename FV, int TM>
__global__ void __launch_bounds__(kBS) __attribute__((amdgpu_waves_per_eu(sizeof(typename FV::real) == 4 ? 2 : 1)))
wloop_tile_kernel(Lat L, FV f, int mu, int nu, int Rmax, PlaneTiles g, int tslice, uint32_t nb, uint32_t groups,
                  double* __restrict__ partials) {
    using R_ = typename FV::real;
    typedef R_ r2 __attribute__((ext_vector_type(2)));
    constexpr uint32_t KC = kTileCells<R_>;
    __shared__ r2 links[2][9][KC];  // of mu, of nu
    __shared__ double sh[kMaxLoopRT * TM][kBS / 16];
    const int o = mu + nu - 1;
    uint32_t q = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t grp = q / nb, blk = q - grp * nb;
    q = blk;
    const uint32_t t1 = q % g.n1;
    q /= g.n1;
    const uint32_t t2 = q % g.n2;
    q /= g.n2;
    uint32_t rest;  // the spectators' part of a site
    if (o == 0) {
        rest = L.st[2] * (q % (uint32_t)L.n[2]) + L.st[3] * (q / (uint32_t)L.n[2]);
    } else {
        const uint32_t no = (uint32_t)L.n[5 - o];
        const uint32_t t = tslice >= 0 ? (uint32_t)tslice : (tslice == kEverySlice ? grp : q / no);
        rest = L.st[5 - o] * (q % no) + L.st[0] * t;
    }
    const uint32_t w = g.q1 + (t1 < g.r1 ? 1u : 0u), h = g.q2 + (t2 < g.r2 ? 1u : 0u);
    const uint32_t o1 = t1 * g.q1 + min(t1, g.r1), o2 = t2 * g.q2 + min(t2, g.r2);
    const uint32_t fw = g.f, fc = fw * (h + (uint32_t)(mu == 1 ? TM : Rmax));
    for (uint32_t c = threadIdx.x; c < fc; c += kBS) {
        const uint32_t fy = c / fw, fx = c - fy * fw;
        const uint32_t s = rest + (o1 + fx) % (uint32_t)L.n[1] + L.st[o] * ((o2 + fy) % (uint32_t)L.n[o]);
        const Mat<R_> M = load_link(f, mu, s), N = load_link(f, nu, s);
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            links[0][e][c] = r2{M.r[e], M.i[e]};
            links[1][e][c] = r2{N.r[e], N.i[e]};
        }
    }
    __syncthreads();
    // lanes past the tile's end work on its first site and contribute nothing
    const bool live = threadIdx.x < w * h;
    const uint32_t j = live ? threadIdx.x : 0u;
    const uint32_t ly = j / w;
    const uint32_t c0 = ly * fw + (j - ly * w);
    const uint32_t dm = mu == 1 ? 1u : fw, dn = mu == 1 ? fw : 1u;
    auto link = [&](int d, uint32_t c) {
        Mat<R_> m;
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            const r2 v = links[d][e][c];
            m.r[e] = v.x;
            m.i[e] = v.y;
        }
        return m;
    };
    double* mine = &sh[0][threadIdx.x >> 4];
    uint32_t a = c0;  // x + R mu
    Mat<R_> CB[TM];
    Mat<R_> Ln = link(1, a);
#pragma unroll
    for (int T = 1; T <= TM; ++T) {
        if (T > 1) Ln = mul(Ln, link(1, a + (T - 1) * dn));
        CB[T - 1] = mul(Ln, link(0, a + T * dn));
        __builtin_amdgcn_sched_barrier(0);
    }
    Mat<R_> Lm = link(0, a);
    // one row, as in wloop_table_kernel
    auto row = [&](auto ext, Mat<R_> M, Mat<R_> N) {
        constexpr bool EXT = decltype(ext)::value;
        Mat<R_> CA;
#pragma unroll
        for (int T = 1; T <= TM; ++T) {
            CA = T == 1 ? mul(Lm, N) : mul(CA, N);
            __builtin_amdgcn_sched_barrier(0);
            if (T < TM) N = link(1, a + T * dn);
            if constexpr (EXT) {
                CB[T - 1] = mul(CB[T - 1], M);
                __builtin_amdgcn_sched_barrier(0);
                if (T < TM) M = link(0, a - dm + (T + 1) * dn);
            }
            double v = (double)retr_nd(CA, CB[T - 1]);
            v = row_sum(live ? v : 0.0);
            mine[(T - 1) * (kBS / 16)] = v;
            __builtin_amdgcn_sched_barrier(0);
        }
        mine += TM * (kBS / 16);
    };
    a += dm;
    row(std::false_type(), Mat<R_>(), link(1, a));
#pragma unroll 1
    for (int R = 2; R <= Rmax; ++R) {
        const Mat<R_> U = link(0, a), M = link(0, a + dn);
        a += dm;
        const Mat<R_> N = link(1, a);
        Lm = mul(Lm, U);
        row(std::true_type(), M, N);
    }
    __syncthreads();
    // 16 lanes per entry
    for (int k = threadIdx.x >> 4; k < Rmax * TM; k += kBS / 16) {
        const DD v = row_dd_sum(sh[k][threadIdx.x & 15]);
        if ((threadIdx.x & 15) == 0) {
            double* p = partials + 2 * (((size_t)k * groups + grp) * nb + blk);
            p[0] = v.hi;
            p[1] = v.lo;
        }
    }
}

// Tiles of a plane with x, n2 sites in its other direction, as the split that leaves the fewest lanes
// idle, then the one with the fewest cells; halo1 and halo2 are the loop's extents along x and o.
PlaneTiles loop_split(uint32_t n1, uint32_t n2, uint32_t halo1, uint32_t halo2, uint32_t max_cells) {
    PlaneTiles best{};
    uint64_t cells = 0;
    for (uint32_t a = (n1 + kBS - 1) / kBS; a <= n1; ++a)
        for (uint32_t b = 1; b <= n2; ++b) {
            const uint32_t w = (n1 + a - 1) / a, h = (n2 + b - 1) / b, fc = (w + halo1) * (h + halo2);
            if (w * h > kBS || fc > max_cells) continue;
            const uint64_t cn = (uint64_t)a * b * fc;
            if (best.n1 == 0 || a * b < best.n1 * best.n2 || (a * b == best.n1 * best.n2 && cn < cells)) {
                cells = cn;
                best = PlaneTiles{a, n1 / a, n1 % a, b, n2 / b, n2 % b, w + halo1, fc, 0, 0};
            }
            break;  // more tiles along o only leave more idle
        }
    return best;
}

// block (k, j) of the grid sums table entry k (of rows of `cols`) of slice
// group j (of gridDim.y) over its nb block partials in a fixed order and writes
// out[k' * gridDim.y + j] = scale * sum, k' = k or the transposed table's entry
__global__ void __launch_bounds__(kBS) wloop_finalize_kernel(const double* __restrict__ partials, uint32_t nb,
                                                             int cols, int transposed, double* __restrict__ out,
                                                             double scale) {
    const int k = blockIdx.x;
    const int to = transposed ? (k % cols) * ((int)gridDim.x / cols) + k / cols : k;
    const double* p = partials + 2 * (((size_t)k * gridDim.y + blockIdx.y) * nb);
    DD acc = {0.0, 0.0};
    for (uint32_t i = threadIdx.x; i < nb; i += kBS) acc = dd_add(acc, DD{p[2 * i], p[2 * i + 1]});
    const DD r = block_sum<kBS>(acc);
    if (threadIdx.x == 0) out[(size_t)to * gridDim.y + blockIdx.y] = (r.hi + r.lo) * scale;
}

}  // namespace

// blocks per slice group: a single slice (tslice >= 0 or kEverySlice), or the whole
// lattice (slice by slice when time is in the plane)
uint32_t wloop_blocks(const Lat& L, int tslice, int mu, int nu) {
    const uint32_t per_slice = (L.Vs + kBS - 1) / kBS;
    if (tslice != -1) return per_slice;
    return (mu == 0 || nu == 0) ? (uint32_t)L.n[0] * per_slice : (L.V + kBS - 1) / kBS;
}

// Whether n tiles beat nb blocks of 256 sites.  us by blocks -> by tiles, plane (x,t) of 32^3x64, 6 x 6:
// FP64 1270 -> 1076, FP32 755 -> 525; 6 x 3: FP64 693 -> 595, FP32 416 -> 304; 18x15x20x30, a seventh of
// the lanes idle, FP32 79 -> 68.  In FP64 a block holds a CU's LDS, so its loads are not hidden: one or two
// chains (253 -> 287 before the rows were straight) and idle lanes (24^3x48, a quarter: 504 -> 522) do
// not repay that.
static bool tiles_pay(int is_f32, int Tmax, uint64_t n, uint64_t nb) {
    return is_f32 ? n * 2 <= nb * 3 : Tmax >= 3 && n * 4 <= nb * 5;
}

// enough for every plane, and for the idle lanes that tiles_pay allows
size_t wloop_partial_bytes(const Lat& L, int tslice) {
    const size_t groups = tslice == kEverySlice ? (size_t)L.n[0] : 1;
    const size_t nb = std::max(wloop_blocks(L, tslice, 0, 1), wloop_blocks(L, tslice, 1, 2));
    return (size_t)kMaxLoopRT * kMaxLoopRT * groups * (nb + nb / 2) * 2 * sizeof(double);
}

hipError_t launch_wloop_table(const Lat& L, const void* U, int is_f32, int mu, int nu, int Rmax, int Tmax,
                              int tslice, double* partials, double* out, double scale, hipStream_t st) {
    // A loop of the plane (nu, mu) is the same loop walked the other way round, its chains and its trace the
    // same products: the longer side makes the rows, since rows are cheaper than chains (24^3x14 FP64,
    // 1 x 6 against 6 x 1: 75 and 36 us).
    const bool swapped = Tmax > Rmax;
    if (swapped) {
        std::swap(mu, nu);
        std::swap(Rmax, Tmax);
    }
    uint32_t nb = wloop_blocks(L, tslice, mu, nu);
    const uint32_t groups = tslice == kEverySlice ? (uint32_t)L.n[0] : 1u;
    PlaneTiles tiles{};
    if ((mu == 1 || nu == 1) && (tslice == -1 || (mu != 0 && nu != 0))) {
        const int o = mu + nu - 1;
        tiles = loop_split((uint32_t)L.n[1], (uint32_t)L.n[o], (uint32_t)(mu == 1 ? Rmax : Tmax),
                           (uint32_t)(mu == 1 ? Tmax : Rmax), is_f32 ? kTileCells<float> : kTileCells<double>);
        const uint64_t per = (uint64_t)tiles.n1 * tiles.n2;
        const uint64_t n = o == 0 ? per * L.n[2] * L.n[3] : per * L.n[5 - o] * (tslice == -1 ? L.n[0] : 1);
        if (tiles_pay(is_f32, Tmax, n, nb))
            nb = (uint32_t)n;
        else
            tiles.n1 = 0;
    }
    with_view(L.V, U, is_f32, [&](auto f) {
        auto run = [&](auto tm) {
            constexpr int TM = decltype(tm)::value;
            if (tiles.n1)
                wloop_tile_kernel<decltype(f), TM>
                    <<<nb * groups, kBS, 0, st>>>(L, f, mu, nu, Rmax, tiles, tslice, nb, groups, partials);
            else
                wloop_table_kernel<decltype(f), TM>
                    <<<nb * groups, kBS, 0, st>>>(L, f, mu, nu, Rmax, tslice, nb, groups, partials);
        };
        switch (Tmax) {
            case 1: run(std::integral_constant<int, 1>()); break;
            case 2: run(std::integral_constant<int, 2>()); break;
            case 3: run(std::integral_constant<int, 3>()); break;
            case 4: run(std::integral_constant<int, 4>()); break;
            case 5: run(std::integral_constant<int, 5>()); break;
            default: run(std::integral_constant<int, 6>()); break;
        }
    });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    wloop_finalize_kernel<<<dim3(Rmax * Tmax, groups), kBS, 0, st>>>(partials, nb, Tmax, swapped, out, scale);
    return hipGetLastError();
}

}  // namespace flue
