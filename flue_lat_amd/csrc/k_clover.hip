// k_clover.hip -- 5-loop improved field strength (hep-lat/0203008) and the magnetic B^2.
//
// The leaf machinery (corner chains, anti-Hermitian accumulation) is in flue_clover.hpp.
#include "flue_clover.hpp"
#include "flue_launch.hpp"

namespace flue {

namespace {

constexpr int kBS = 256;

// Two forms of the magnetic kernel, picked per precision (or by the autotuner):
//
// site-major: one thread per site does the three planes in turn, sites in storage order.
//
// plane-major: the grid is (nb, 3) and blockIdx.y is the plane, so the dispatcher runs
// the planes one after another.  The blocks of one XCD run through a contiguous range
// of a per-plane visit order; each order makes the sites in flight whole layers of
// the two plane directions, stacked along the third spatial direction (rho), so the
// +-3 reach of the leaves stays inside layers that are already in that XCD's L2:
//   plane 0 (y,x), rho = z:  x, y, z, t            (the storage order)
//   plane 1 (x,z), rho = y:  x, z, y, t
//   plane 2 (z,y), rho = x:  x mod xw, y, z, x / xw, t   (x in chunks of xw sites, at
//                            least 128 bytes of one element plane, so loads coalesce)
// This cuts the traffic behind L2 several-fold; it pays where occupancy is low (FP64).

// B = -(1/V) sum_x sum_i ReTr(F_i F_i) over the planes (y,x), (x,z), (z,y)
// (src/wloops.F90:502-506, 530-543); each block writes one compensated partial sum.
template <typename FV, int WPE, bool PLANE_MAJOR, bool C2 = sizeof(typename FV::real) == 4>
__global__ void __launch_bounds__(kBS) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
magnetic_kernel(Lat L, FV f, PlaneOrder po, uint32_t nb, double* __restrict__ partials) {
    // C2 (FP32 always; FP64 for links declared SU(3)): link chains carry two rows and row 2
    // is rebuilt where a leaf closes.  Plain FP64 keeps full products, so it makes no
    // assumption on the links.  Consecutive quadrants share their lines where the registers
    // allow it: always with C2, at one wave per SIMD otherwise.
    constexpr bool kC2 = C2;
    // FP64 at two waves per SIMD: the waiting chains are parked in LDS (quadrant_parked)
    constexpr bool kPark = sizeof(typename FV::real) == 8 && WPE == 2;
    constexpr bool kShare = !kPark && (kC2 || WPE == 1);
    // FP64 at one wave per SIMD: each group of products loads the next group's first link
    constexpr bool kLA = sizeof(typename FV::real) == 8 && WPE == 1;
    // the plane comes from blockIdx.y so that it, and every buffer descriptor derived
    // from it, stays in scalar registers (a division of blockIdx.x would not)
    const int pl = (int)blockIdx.y;
    const uint32_t blk = xcd_block(blockIdx.x, nb);
    const uint32_t o = blk * kBS + threadIdx.x;
    double acc = 0.0;
    if (o < L.V) {
        int c[4];
        if constexpr (kPark) {
            __shared__ typename FV::real park_mem[2 * 18 * kBS];
            const Park<typename FV::real, kBS> pk{park_mem + threadIdx.x};
            if constexpr (PLANE_MAJOR) {
                const uint32_t s = plane_site(L, po, pl, o, c);
                const int mu = plane_mu(pl), nu = plane_nu(pl);
                acc = f_norm2(plane_ah_parked<kC2>(plane_geom(L, f, s, c[mu], c[nu], mu, nu), pk));
            } else {
                site_coords(L, o, c);
#pragma unroll 1
                for (int p = 0; p < 3; ++p) {
                    const int mu = plane_mu(p), nu = plane_nu(p);
                    acc += f_norm2(plane_ah_parked<kC2>(plane_geom(L, f, o, c[mu], c[nu], mu, nu), pk));
                }
            }
        } else if constexpr (PLANE_MAJOR) {
            const uint32_t s = plane_site(L, po, pl, o, c);
            const int mu = plane_mu(pl), nu = plane_nu(pl);
            acc = f_norm2(plane_ah<false, kShare, kC2, kLA>(plane_geom(L, f, s, c[mu], c[nu], mu, nu)));
        } else {
            site_coords(L, o, c);
#pragma unroll 1
            for (int p = 0; p < 3; ++p) {
                const int mu = plane_mu(p), nu = plane_nu(p);
                acc += f_norm2(plane_ah<false, kShare, kC2, kLA>(plane_geom(L, f, o, c[mu], c[nu], mu, nu)));
            }
        }
    }
    DD r = block_sum<kBS>(DD{acc, 0.0});
    if (threadIdx.x == 0) {
        const uint32_t i = (uint32_t)pl * nb + blk;
        partials[2 * i] = r.hi;
        partials[2 * i + 1] = r.lo;
    }
}

// per-site F for one plane.  layout 0: complex128 at the given strides; layout 1: SoA
// planes (element e = a*3+b, re/im) in the field precision.  TESTED: only where *bad (links of an FP64 field
// that the tiles of k_rect.hip found not unitary).
template <typename FV, bool CLOVER, bool TESTED = false>
__global__ void __launch_bounds__(kBS) __attribute__((amdgpu_waves_per_eu(sizeof(typename FV::real) == 4 ? 2 : 1)))
fmunu_kernel(Lat L, FV f, int mu, int nu, void* __restrict__ out, int layout, OutStrides os, uint32_t unit,
             uint32_t tb, const uint32_t* __restrict__ bad) {
    using R = typename FV::real;
    if (TESTED && !*bad) return;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    // planes (x, z): each slice taken along z; planes containing time: along their spatial direction
    const int d = mu == 0 || nu == 0 ? mu + nu : (mu + nu == 4 ? 3 : 1);
    uint32_t s;
    if (tb) {
        // blocks or waves (units of 256 or 64 sites) take the same sites of tb consecutive slices one after
        // another, then the next sites
        const uint32_t w = unit == kBS ? blk
                                       : (uint32_t)__builtin_amdgcn_readfirstlane((int)(blk * (kBS / 64) + threadIdx.x / 64));
        const uint32_t NT = (uint32_t)L.n[0], chunks = (L.Vs + unit - 1) / unit;
        if (w >= NT * chunks) return;
        const uint32_t t0 = w / (tb * chunks) * tb, r = w - t0 * chunks;
        const uint32_t ext = min(tb, NT - t0), chunk = r / ext;
        const uint32_t idx = chunk * unit + threadIdx.x % unit;
        if (idx >= L.Vs) return;
        s = slice_site_along(L, idx, d) + L.Vs * (t0 + r - chunk * ext);
    } else {
        s = blk * kBS + threadIdx.x;
        if (s >= L.V) return;
        const uint32_t t = s / L.Vs;
        s = slice_site_along(L, s - t * L.Vs, d) + L.Vs * t;
    }
    int c[4];
    site_coords(L, s, c);
    // FP32 carries two rows, FP64 (one wave per SIMD) loads a link ahead
    const AH<R> h = plane_ah<CLOVER, true, sizeof(R) == 4, sizeof(R) == 8>(plane_geom(L, f, s, c[mu], c[nu], mu, nu));
    if (layout == 0) {
        store_f(h, c, (double*)out, os);
    } else {
        R fr[9], fi[9];
        f_entries(h, fr, fi);
        R* o = (R*)out;
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            o[(size_t)(2 * e) * L.V + s] = fr[e];
            o[(size_t)(2 * e + 1) * L.V + s] = fi[e];
        }
    }
}

}  // namespace

uint32_t magnetic_blocks(const Lat& L, int) { return 3 * ((L.V + kBS - 1) / kBS); }

// the least divisor of NX that spans 128 bytes of one element plane, else whole rows
PlaneOrder plane_order(const Lat& L, size_t real_bytes) {
    PlaneOrder po{(uint32_t)L.n[1]};
    for (int w = 1; w < L.n[1]; ++w)
        if (L.n[1] % w == 0 && (size_t)w * real_bytes >= 128) {
            po.xw = (uint32_t)w;
            break;
        }
    return po;
}

int magnetic_default_variant(int is_f32) { return is_f32 ? 5 : 4; }

// variant 1..3: site-major with an occupancy target of 1..3 waves per SIMD;
// variant 4..6: plane-major with 1..3 waves per SIMD; 7: rectangle-first (k_rect.hip, needs
// fpbuf and rect_fits); 0 picks the precision's default.
// su3 (FP64 only) selects two-row chains for the plane-major forms at 1 and 2 waves per
// SIMD; the other forms, and fields beyond the buffer-resource range, keep full products.
// *npart receives the number of partial sums written (nb or 3 nb).
hipError_t launch_magnetic(const Lat& L, const void* U, int is_f32, int su3, double* partials, hipStream_t st,
                           int variant, uint32_t* npart, void* fpbuf) {
    const uint32_t nb = magnetic_blocks(L, is_f32) / 3;
    if (variant == 0) variant = magnetic_default_variant(is_f32);
    if (variant < 1 || variant > kMagneticVariants) return hipErrorInvalidValue;
    if (variant == kMagneticRect) {
        if (!fpbuf) return hipErrorInvalidValue;
        return launch_magnetic_rect(L, U, is_f32, su3, partials, fpbuf, st, npart);
    }
    with_view(L.V, U, is_f32, [&](auto f) {
        using F = decltype(f);
        using R = typename F::real;
        const PlaneOrder po = plane_order(L, sizeof(R));
        const dim3 g1(nb, 1), g3(nb, 3);
        if constexpr (!F::buffered) {
            // fields beyond the buffer-resource range: one form only
            magnetic_kernel<F, sizeof(R) == 4 ? 2 : 1, false><<<g1, kBS, 0, st>>>(L, f, po, nb, partials);
            variant = 1;
        } else if (sizeof(R) == 8 && su3 && (variant == 4 || variant == 5)) {
            if (variant == 4)
                magnetic_kernel<F, 1, true, true><<<g3, kBS, 0, st>>>(L, f, po, nb, partials);
            else
                magnetic_kernel<F, 2, true, true><<<g3, kBS, 0, st>>>(L, f, po, nb, partials);
        } else {
            switch (variant) {
                case 1: magnetic_kernel<F, 1, false><<<g1, kBS, 0, st>>>(L, f, po, nb, partials); break;
                case 2: magnetic_kernel<F, 2, false><<<g1, kBS, 0, st>>>(L, f, po, nb, partials); break;
                case 3: magnetic_kernel<F, 3, false><<<g1, kBS, 0, st>>>(L, f, po, nb, partials); break;
                case 4: magnetic_kernel<F, 1, true><<<g3, kBS, 0, st>>>(L, f, po, nb, partials); break;
                case 5: magnetic_kernel<F, 2, true><<<g3, kBS, 0, st>>>(L, f, po, nb, partials); break;
                default: magnetic_kernel<F, 3, true><<<g3, kBS, 0, st>>>(L, f, po, nb, partials); break;
            }
        }
    });
    if (npart) *npart = variant >= 4 ? 3 * nb : nb;
    return hipGetLastError();
}

hipError_t launch_fmunu(const Lat& L, const void* U, int is_f32, int mu, int nu, int clover_only, void* out,
                        int out_layout, const int64_t s6[6], hipStream_t st, const uint32_t* bad) {
    // Order of the sites.  Planes containing time: the same sites of all slices one after another, as the
    // leaves reach 3 slices either way and the blocks running together then share those slices in L2.
    // Spatial planes: storage order, but where t is dense in the output and more than one wave per SIMD
    // runs, 8 slices, whose elements fill a line of the output, one after another: in storage order a line is
    // written 16 B at a time, long apart.  Clover sums, a third of the work, take it by waves.  48^3x96, FP32 /
    // FP64, ms: clover (x, y) 4.63 / 4.94 -> 1.59 / 2.59, (x, t) 1.88 / 3.00 -> 1.64 / 2.55; five-loop F (FP32,
    // blocks) (x, y) 4.99 -> 4.20.  Five-loop planes (y, z) lose 2% by it and those containing time 5% by
    // waves; at 10^3x43, 672 waves, every plane loses 2 to 10%.
    const bool time = mu == 0 || nu == 0;
    const bool lines = out_layout == 0 && s6 && s6[0] < s6[1] && L.V >= 65536 && L.Vs >= 2048;
    const uint32_t unit = lines && clover_only ? 64 : kBS;
    const uint32_t tb = time ? (uint32_t)L.n[0] : (lines && (clover_only || mu + nu != 5) ? 8 : 0);
    const uint32_t units = tb ? (uint32_t)L.n[0] * ((L.Vs + unit - 1) / unit) : (L.V + kBS - 1) / kBS;
    const uint32_t g = unit == 64 ? (units + kBS / 64 - 1) / (kBS / 64) : units;
    OutStrides os{0, 0, 0, 0, 0, 0};
    if (s6) os = OutStrides{s6[0], s6[1], s6[2], s6[3], s6[4], s6[5]};
    with_view(L.V, U, is_f32, [&](auto f) {
        using F = decltype(f);
        if constexpr (sizeof(typename F::real) == 8 && F::buffered) {
            if (bad) {
                fmunu_kernel<F, false, true><<<g, kBS, 0, st>>>(L, f, mu, nu, out, out_layout, os, unit, tb, bad);
                return;
            }
        }
        if (clover_only)
            fmunu_kernel<F, true><<<g, kBS, 0, st>>>(L, f, mu, nu, out, out_layout, os, unit, tb, nullptr);
        else
            fmunu_kernel<F, false><<<g, kBS, 0, st>>>(L, f, mu, nu, out, out_layout, os, unit, tb, nullptr);
    });
    return hipGetLastError();
}

}  // namespace flue
