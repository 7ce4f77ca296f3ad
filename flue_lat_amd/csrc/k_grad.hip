// k_grad.hip -- gradient of the Wilson plaquette action with respect to every link and
// the Wilson-flow (RK3) stage built on it.
//
// Convention (no reference counterpart): for a link U = U_mu(x) the Lie derivative is
// D^a f = d/ds f(exp(s T^a) U)|_0 with T^a = -i lambda_a / 2, and the gradient stored
// per link is G = sum_a T^a D^a f, traceless anti-Hermitian; D^a f = -2 Tr(T^a G).
//   Wilson action S = beta sum_p (1 - ReTr P/3):   G = (beta/6) P_TA(U Sigma)
// with Sigma the staple sum (U Sigma = the six plaquettes through U).
#include <algorithm>

#include "flue_flow.hpp"
#include "flue_launch.hpp"

namespace flue {

namespace {

constexpr int kBS = 256;

// Visit orders of the sites (the autotuner's variants of the flow and gradient stencils).
// Every order runs the same per-link code, so results are bit-identical.
//   yt = 0:  storage order (x, y, z, t), 256-site blocks.
//   yt > 0:  boxes of yt x zt rows along x, each box swept along t: the blocks of a box at t
//            are followed by its blocks at t + 1, so the lines that the z and t neighbours
//            share are read while they are still in the XCD's L2.
struct BlockOrder {
    uint32_t yt, zt;    // box extents along y and z (0 = storage order)
    uint32_t nty;       // boxes along y
    uint32_t nbt;       // 256-site blocks per box and slice
    uint32_t nb;        // blocks in all
};

// the site i of block lb of the order (0 <= i < 256), with its coordinates; false past the end
__device__ __forceinline__ bool order_site(const Lat& L, const BlockOrder& bo, uint32_t lb, uint32_t i, uint32_t& s,
                                           int c[4]) {
    if (bo.yt == 0) {
        s = lb * kBS + i;
        if (s >= L.V) return false;
        site_coords(L, s, c);
        return true;
    }
    const uint32_t q = lb / bo.nbt, k = lb - q * bo.nbt;
    const uint32_t box = q / (uint32_t)L.n[0], t = q - box * (uint32_t)L.n[0];
    const uint32_t bz = box / bo.nty, by = box - bz * bo.nty;
    const uint32_t j = k * kBS + i;
    const uint32_t r = j / (uint32_t)L.n[1], z = r / bo.yt;
    c[0] = (int)t;
    c[1] = (int)(j - r * (uint32_t)L.n[1]);
    c[2] = (int)(by * bo.yt + r - z * bo.yt);
    c[3] = (int)(bz * bo.zt + z);
    s = (uint32_t)c[1] + L.st[2] * (uint32_t)c[2] + L.st[3] * (uint32_t)c[3] + L.st[0] * t;
    return z < bo.zt && c[2] < L.n[2] && c[3] < L.n[3];
}

// One thread per link.  The direction is the fastest block index: the four blocks of the
// same 256 sites run together and read the same neighbour links, so they share them in L2
// (a thread walking the four directions of its site read them again long after).
template <typename FV>
__global__ void __launch_bounds__(kBS) wilson_grad_kernel(Lat L, FV f, BlockOrder bo, double beta,
                                                          typename FV::real* __restrict__ grad) {
    using R = typename FV::real;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int mu = (int)(blk & 3u);
    uint32_t s;
    int c[4];
    if (!order_site(L, bo, blk >> 2, threadIdx.x, s, c)) return;
    {
        const Mat<R> M = mul(load_link(f, mu, s), staple_sum(L, f, s, c, mu));
        Mat<R> G = proj_ta(M);
        const R sc = (R)(beta / 6.0);
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            G.r[e] *= sc;
            G.i[e] *= sc;
        }
        store_link_stream(grad, L.V, mu, s, G);
    }
}

template <typename FV>
__global__ void __launch_bounds__(kBS) flow_stage_kernel(Lat L, FV f, BlockOrder bo, typename FV::real* __restrict__ wout,
                                                         typename FV::real* __restrict__ acc, double eps, double ca,
                                                         double cb, int reunit) {
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int mu = (int)(blk & 3u);
    uint32_t s;
    int c[4];
    if (!order_site(L, bo, blk >> 2, threadIdx.x, s, c)) return;
    flow_link(L, f, wout, acc, s, c, mu, eps, ca, cb, reunit);
}

// Plaquette-first stencil (kFlowPF): the plaquette parts of every site, then per link, in the flow with the
// four waves of a workgroup on the four directions of 64 sites.  ROWS2: the flow.
// At 48^3x96 the first pass takes 1.15 ms (FP32) and 2.11 ms (FP64) with ROWS2, at 4.0 and 4.4
// TB/s beyond L2; taking two of the six planes per wave instead, with 21 link reads a site
// instead of 16, took 1.33 and 2.34 ms and gained nothing on a lattice of 162,000 sites.
// TEST: sets *bad where a link is not SU(3); else nothing where that was found.
template <bool ROWS2, bool TEST, typename FV>
__global__ void __launch_bounds__(kBS) plaq_ta_kernel(Lat L, FV f, BlockOrder bo, typename FV::real* __restrict__ T,
                                                      uint32_t* __restrict__ bad) {
    if (!TEST && bad && *bad) return;
    uint32_t s;
    int c[4];
    if (!order_site(L, bo, xcd_block(blockIdx.x, gridDim.x), threadIdx.x, s, c)) return;
    const bool ok = plaquette_ta_site<ROWS2, TEST>(L, f, s, c, T);
    if (TEST && !ok) __hip_atomic_store(bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void clear_word_kernel(uint32_t* w) { *w = 0; }

// a direction per workgroup, whose links are whole (with the four directions of 64 sites in one, as in the
// flow: 48^3x96, buffer loads of T: 3.61 for 3.55 ms in FP32, 6.87 for 6.69 in FP64)
template <typename FV>
__global__ void __launch_bounds__(kBS) wilson_grad_pf_kernel(Lat L, FV f, BlockOrder bo,
                                                             const typename FV::real* __restrict__ T, double beta,
                                                             typename FV::real* __restrict__ grad) {
    using R = typename FV::real;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int mu = (int)(blk & 3u);
    uint32_t s;
    int c[4];
    if (!order_site(L, bo, blk >> 2, threadIdx.x, s, c)) return;
    Mat<R> G = ta_force(L, f, T, s, c, mu);
    const R sc = (R)(beta / 6.0);
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        G.r[e] *= sc;
        G.i[e] *= sc;
    }
    store_link_stream(grad, L.V, mu, s, G);
}

// TESTED: nothing where the flow's first pass found links that are not SU(3) (flow_general_kernel's work).
// Both forms in this kernel would leave the plaquette-first one at the staple form's two waves per SIMD
// instead of four: 3.30 ms for ten steps of 18x15x20x30 instead of 3.27, and 3.26 with no test at all.
template <bool TESTED, typename FV>
__global__ void __launch_bounds__(kBS) flow_stage_pf_kernel(Lat L, FV f, BlockOrder bo,
                                                            const typename FV::real* __restrict__ T,
                                                            typename FV::real* __restrict__ wout,
                                                            typename FV::real* __restrict__ acc, double eps, double ca,
                                                            double cb, int reunit, const uint32_t* __restrict__ bad) {
    if (TESTED && *bad) return;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int mu = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint32_t s;
    int c[4];
    if (!order_site(L, bo, blk >> 2, (blk & 3u) * 64u + (threadIdx.x & 63u), s, c)) return;
    flow_link_pf(L, f, T, wout, acc, s, c, mu, eps, ca, cb, reunit);
}

// The stage by staple sums where the links turned out not SU(3): the blocks of flow_stage_kernel on more
// workgroups than are resident at once, which look first whether there is anything to do.
constexpr uint32_t kGeneralGrid = 1024;
template <typename FV>
__global__ void __launch_bounds__(kBS) flow_general_kernel(Lat L, FV f, BlockOrder bo, typename FV::real* __restrict__ wout,
                                                           typename FV::real* __restrict__ acc, double eps, double ca,
                                                           double cb, int reunit, const uint32_t* __restrict__ bad) {
    if (!*bad) return;
    for (uint32_t b = blockIdx.x; b < 4 * bo.nb; b += gridDim.x) {
        const uint32_t blk = xcd_block(b, 4 * bo.nb);
        uint32_t s;
        int c[4];
        if (!order_site(L, bo, blk >> 2, threadIdx.x, s, c)) continue;
        flow_link(L, f, wout, acc, s, c, (int)(blk & 3u), eps, ca, cb, reunit);
    }
}

}  // namespace

// Sites of a box slice for variants 1..6 (0 = storage order).  At 48^3x96 (one RK3 step, ms):
//   sites          storage   1024    2048    3072    4096    6144
//   staple  FP32     16.1    14.9    14.9    14.4    14.4    14.5
//           FP64     27.3    24.4    24.8    24.3    24.3    24.4
//   plaq.   FP32     10.9    10.7    10.7    10.5    10.5    10.5
//   first   FP64     20.9    19.8    20.0    19.6    19.6    19.7
constexpr uint32_t kBoxSites[kFlowPF - 1] = {0, 1024, 2048, 3072, 4096, 6144};

// The order of a variant: plaquette-first variant kFlowPF + k (k = 2..6) takes the boxes of
// staple variant k, kFlowPFWide the largest.  Of the boxes with at most the variant's sites, the one
// with the fewest blocks (a box's last block is padded) times lines read again by the boxes beside it.
static BlockOrder block_order(const Lat& L, int variant) {
    const uint32_t plain = (L.V + kBS - 1) / kBS, NY = (uint32_t)L.n[2], NZ = (uint32_t)L.n[3];
    const int k = variant == kFlowPFWide ? 6 : (variant > kFlowPF ? variant - kFlowPF : variant);
    const uint32_t want = k >= 1 && k < kFlowPF ? kBoxSites[k - 1] : 0;
    uint32_t yt = 0, zt = 0;
    double cost = 0.0;
    for (uint32_t y = 1; y <= NY; ++y)
        for (uint32_t z = 1; z <= NZ && (uint64_t)L.n[1] * y * z <= want; ++z) {
            const double n = (NY + y - 1) / y * (double)((NZ + z - 1) / z) * (((uint32_t)L.n[1] * y * z + kBS - 1) / kBS);
            const double c = n * (1.0 + (y < NY ? 1.0 / y : 0.0) + (z < NZ ? 1.0 / z : 0.0));
            if (yt == 0 || c < cost) {
                cost = c;
                yt = y;
                zt = z;
            }
        }
    if (yt == 0) return BlockOrder{0, 0, 1, 1, plain};  // storage order, or no row fits
    const uint32_t nty = (NY + yt - 1) / yt, nbt = ((uint32_t)L.n[1] * yt * zt + kBS - 1) / kBS;
    return BlockOrder{yt, zt, nty, nbt, nty * ((NZ + zt - 1) / zt) * nbt * (uint32_t)L.n[0]};
}

// Untuned choices, ms per RK3 step as measured (FP32 / FP64):
//                     staple sums        plaquette-first    its boxes of 3072
//   8^3x16          0.034 / 0.038       0.044 / 0.047      0.045 / 0.049
//   12^3x24         0.070 / 0.092       0.065 / 0.091      0.065 / 0.093
//   16^3x32         0.150 / 0.242       0.138 / 0.239      0.141 / 0.252
//   20^3x40         0.347 / 0.703       0.305 / 0.574      0.379 / 0.630
//   24^3x48         0.904 / 1.53        0.629 / 1.24       0.628 / 1.21
//   48^3x96         16.0  / 27.1        10.4  / 20.3       10.0  / 19.1
// The flow, whose links are SU(3), takes the plaquette-first stencil from 32768 sites (below,
// its second launch costs more than it saves).  Boxes pay once a slice's links and plaquette
// parts outgrow an XCD's 4 MB L2 several times.
constexpr uint32_t kPFSites = 32768, kBoxSlice = 32768;
int flow_default(const Lat& L) {
    if (L.V < kPFSites) return grad_default(L);
    return L.Vs >= kBoxSlice ? kFlowPF + 4 : kFlowPF;
}
int grad_default(const Lat& L) { return L.Vs >= kBoxSlice ? 4 : 1; }

size_t plaq_ta_bytes(const Lat& L, int is_f32) { return (size_t)48 * L.V * (is_f32 ? 4 : 8); }

hipError_t launch_wilson_grad(const Lat& L, const void* U, int is_f32, double beta, void* grad, hipStream_t st,
                              int variant, void* T) {
    if (flow_is_pf(variant) && !T) return hipErrorInvalidValue;
    const BlockOrder bo = block_order(L, variant);
    with_view(L.V, U, is_f32, [&](auto f) {
        using F = decltype(f);
        using R = typename F::real;
        if (flow_is_pf(variant)) {
            plaq_ta_kernel<false, false, F><<<bo.nb, kBS, 0, st>>>(L, f, bo, (R*)T, nullptr);
            wilson_grad_pf_kernel<F><<<4 * bo.nb, kBS, 0, st>>>(L, f, bo, (const R*)T, beta, (R*)grad);
        } else {
            wilson_grad_kernel<F><<<4 * bo.nb, kBS, 0, st>>>(L, f, bo, beta, (R*)grad);
        }
    });
    return hipGetLastError();
}

hipError_t launch_flow_stage(const Lat& L, const void* Win, int is_f32, void* Wout, void* acc_, double eps,
                             double ca, double cb, int reunit, hipStream_t st, int variant, void* T, uint32_t* bad) {
    if (flow_is_pf(variant) && !T) return hipErrorInvalidValue;
    const BlockOrder bo = block_order(L, variant);
    with_view(L.V, Win, is_f32, [&](auto f) {
        using F = decltype(f);
        using R = typename F::real;
        R* acc = (R*)acc_;
        if (flow_is_pf(variant)) {
            constexpr bool kF64 = sizeof(R) == 8;
            auto links = [&](auto tested) {
                flow_stage_pf_kernel<decltype(tested)::value, F>
                    <<<4 * bo.nb, kBS, 0, st>>>(L, f, bo, (const R*)T, (R*)Wout, acc, eps, ca, cb, reunit, bad);
            };
            if (kF64 && bad && ca == 0.0) {  // the step's first stage
                clear_word_kernel<<<1, 1, 0, st>>>(bad);
                plaq_ta_kernel<true, kF64, F><<<bo.nb, kBS, 0, st>>>(L, f, bo, (R*)T, bad);
            } else {
                plaq_ta_kernel<true, false, F><<<bo.nb, kBS, 0, st>>>(L, f, bo, (R*)T, bad);
            }
            if constexpr (kF64) {
                if (bad) {
                    links(std::true_type());
                    flow_general_kernel<F><<<std::min(kGeneralGrid, 4 * bo.nb), kBS, 0, st>>>(
                        L, f, bo, (R*)Wout, acc, eps, ca, cb, reunit, bad);
                    return;
                }
            }
            links(std::false_type());
        } else {
            flow_stage_kernel<F><<<4 * bo.nb, kBS, 0, st>>>(L, f, bo, (R*)Wout, acc, eps, ca, cb, reunit);
        }
    });
    return hipGetLastError();
}

}  // namespace flue
