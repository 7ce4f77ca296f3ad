// k_quad.hip -- the magnetic B of small lattices: a wave per quadrant.
//
// With a thread per site and plane (k_clover.hip) a small lattice keeps a fraction of the chip's SIMDs
// busy, each with four quadrants one after another: 8^3x16 has 384 waves for 1024 SIMDs and took 37 us.
// Here the four waves of a workgroup form the four quadrants of the same 64 sites and plane, and the
// first adds their anti-Hermitian parts from LDS in the quadrants' order.  Lines are not shared between
// quadrants (80 products for 74).
#include "flue_clover.hpp"
#include "flue_launch.hpp"

namespace flue {

namespace {

constexpr int kSites = 64;

// blockIdx.y: the plane, (y, x), (x, z) or (z, y).  C2: two-row chains, as in magnetic_kernel.
template <typename FV, bool C2>
__global__ void __launch_bounds__(4 * kSites) __attribute__((amdgpu_waves_per_eu(1)))
quad_kernel(Lat L, FV f, double* __restrict__ partials) {
    using R = typename FV::real;
    __shared__ R parts[3][9][kSites];
    const int pl = (int)blockIdx.y;
    const int mu = pl == 0 ? 2 : (pl == 1 ? 1 : 3), nu = pl == 0 ? 1 : (pl == 1 ? 3 : 2);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kSites), lane = (int)threadIdx.x % kSites;
    const uint32_t s = blockIdx.x * kSites + (uint32_t)lane;
    AH<R> h;
    ah_zero(h);
    if (s < L.V) {
        int c[4];
        site_coords(L, s, c);
        const PlaneGeom<FV> g = plane_geom(L, f, s, c[mu], c[nu], mu, nu);
        auto quad = [&](auto s1, auto s2, auto mu_first) {
            constexpr int S1 = decltype(s1)::value, S2 = decltype(s2)::value;
            quadrant_la<S1, S2, false, false, C2>(make_quad<S1, S2, decltype(mu_first)::value>(g), h);
        };
        using P = std::integral_constant<int, 1>;
        using M = std::integral_constant<int, -1>;
        switch (wave) {
            case 0: quad(P(), P(), std::true_type()); break;
            case 1: quad(P(), M(), std::false_type()); break;
            case 2: quad(M(), M(), std::true_type()); break;
            default: quad(M(), P(), std::false_type()); break;
        }
    }
    if (wave > 0)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            parts[wave - 1][k][lane] = h.d[k];
            parts[wave - 1][3 + k][lane] = h.or_[k];
            parts[wave - 1][6 + k][lane] = h.oi[k];
        }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            h.d[k] += parts[w][k][lane];
            h.or_[k] += parts[w][3 + k][lane];
            h.oi[k] += parts[w][6 + k][lane];
        }
    const DD r = block_sum<kSites>(DD{f_norm2(h), 0.0});
    if (lane == 0) {
        double* p = partials + 2 * (size_t)(blockIdx.y * gridDim.x + blockIdx.x);
        p[0] = r.hi;
        p[1] = r.lo;
    }
}

}  // namespace

// Where it runs untuned: FP64.  As measured, us with the finalize pass, the other untuned form -> this one
// (16^3 lattices take rectangle-first tiles otherwise):
//   4^4               256 sites   36 -> 16
//   8^3x16          8,192         37 -> 26
//   10^4           10,000         37 -> 28
//   8^3x24         12,288         37 -> 37
//   10^3x16        16,000         38 -> 42
//   16^3x4         16,384         49 -> 40
//   12^4           20,736         42 -> 56
// (10,922 sites are two rounds of one wave on each of the 1024 SIMDs.)  FP32 (30 -> 19 at 8^3x16) keeps a
// thread per site: with parts rounded apart B of few sites moves by up to 7e-9.
bool quad_fits(const Lat& L, int is_f32) {
    return !is_f32 && L.V <= 16384 && (L.V <= 10922 || rect_fits(L));
}

uint32_t quad_blocks(const Lat& L) { return 3 * ((L.V + kSites - 1) / kSites); }

hipError_t launch_magnetic_quad(const Lat& L, const void* U, int su3, double* partials, hipStream_t st,
                                uint32_t* npart) {
    const dim3 g((L.V + kSites - 1) / kSites, 3);
    const FieldView<double, true> f{(const double*)U, L.V};  // (within the buffer range by quad_fits)
    if (su3)
        quad_kernel<FieldView<double, true>, true><<<g, 4 * kSites, 0, st>>>(L, f, partials);
    else
        quad_kernel<FieldView<double, true>, false><<<g, 4 * kSites, 0, st>>>(L, f, partials);
    *npart = quad_blocks(L);
    return hipGetLastError();
}

}  // namespace flue
