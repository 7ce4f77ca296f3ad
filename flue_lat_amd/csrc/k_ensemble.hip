// k_ensemble.hip -- ensembles of gauge fields with different extents processed in one
// launch per operation: the RK3 flow stage, the plaquette sum and the magnetic B.
//
// The fields lie back to back, each in the SoA layout of its own lattice.  Every
// configuration owns a contiguous range of logical blocks (256 sites each).  A workgroup takes a logical
// block (or a quarter or a direction of one), finds its configuration by binary search in a table kept in
// device memory, and runs the same per-site (flow: per-link) code as the single-field kernels.  The
// logical blocks of an XCD are contiguous, so those running together share
// their links in L2, and one block per workgroup leaves the registers to the stencil: 16 fields of 16^3
// with 644 time slices, FP32, a plaquette-first flow stage 1.32 -> 0.97 ms and a plaquette sum
// 0.51 -> 0.36 ms against a persistent grid of contiguous chunks (86 registers and 5 waves per SIMD, now 72
// and 7).
// Sums are reduced per logical block and then per configuration in a fixed order.  (B takes the
// rectangle-first tiles of k_rect.hip where they apply, one launch for every tile of the ensemble.)
#include "flue_clover.hpp"
#include "flue_flow.hpp"
#include "flue_launch.hpp"

namespace flue {

namespace {

constexpr int kBS = 256;

// The table is read through the constant address space and its entries are used in
// place: uniform loads from it become scalar loads, so the lattice geometry and every
// buffer descriptor built from it stay in scalar registers.  (A local copy of an entry
// is indexed at run time by direction, lives in memory, and turns every link load into
// a loop over the distinct descriptors of the wave.)
using CEnsEntry = const __attribute__((address_space(4))) EnsEntry;

__device__ __forceinline__ const EnsEntry& entry(const EnsEntry* tab, int c) {
    return *(const EnsEntry*)((CEnsEntry*)tab + c);
}

__device__ __forceinline__ int find_cfg(const EnsEntry* __restrict__ tab, int n, uint32_t lb) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].blk0 <= lb)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Workgroups are (logical block, direction), direction fastest: one thread per link, and the four of a
// block, which read the same neighbour links, run close together.
template <typename R, bool BUF>
__global__ void __launch_bounds__(kBS) ens_flow_kernel(const EnsEntry* __restrict__ tab, int n,
                                                       const R* __restrict__ win, R* __restrict__ wout,
                                                       R* __restrict__ acc, double eps, double ca, double cb,
                                                       int reunit) {
    const uint32_t lu = xcd_block(blockIdx.x, gridDim.x), lb = lu >> 2;
    const int mu = (int)(lu & 3u);
    const EnsEntry& e = entry(tab, find_cfg(tab, n, lb));
    const uint32_t s = (lb - e.blk0) * kBS + threadIdx.x;
    if (s >= e.L.V) return;
    const FieldView<R, BUF> f{win + e.off, e.L.V};
    int c[4];
    site_coords(e.L, s, c);
    flow_link(e.L, f, wout + e.off, acc + e.acc_off, s, c, mu, eps, ca, cb, reunit);
}

// Plaquette-first stencil over the ensemble: the six plaquette parts of every site of every
// field (48 reals per site, config c's block at 2/3 of its field offset), then the links, the
// four waves of a workgroup on the four directions of 64 sites.
// TEST: sets bad[c] and bad[n] where a link of configuration c is not SU(3); else nothing for a configuration
// of which that was found.
template <typename R, bool BUF, bool TEST>
__global__ void __launch_bounds__(kBS) ens_plaq_ta_kernel(const EnsEntry* __restrict__ tab, int n,
                                                          const R* __restrict__ win, R* __restrict__ T,
                                                          uint32_t* __restrict__ bad) {
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const int cfg = find_cfg(tab, n, lb);
    if (!TEST && bad && bad[cfg]) return;
    const EnsEntry& e = entry(tab, cfg);
    const uint32_t s = (lb - e.blk0) * kBS + threadIdx.x;
    if (s >= e.L.V) return;
    const FieldView<R, BUF> f{win + e.off, e.L.V};
    int c[4];
    site_coords(e.L, s, c);
    const bool ok = plaquette_ta_site<true, TEST>(e.L, f, s, c, T + e.off / 72 * 48);
    if (TEST && !ok) {
        __hip_atomic_store(bad + cfg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(bad + n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// TESTED: nothing for a configuration with links that are not SU(3) (ens_general_flow_kernel's work)
template <typename R, bool BUF, bool TESTED>
__global__ void __launch_bounds__(kBS) ens_flow_pf_kernel(const EnsEntry* __restrict__ tab, int n,
                                                          const R* __restrict__ win, const R* __restrict__ T,
                                                          R* __restrict__ wout, R* __restrict__ acc, double eps, double ca,
                                                          double cb, int reunit, const uint32_t* __restrict__ bad) {
    const int mu = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t lu = xcd_block(blockIdx.x, gridDim.x), lb = lu >> 2;
    const int cfg = find_cfg(tab, n, lb);
    if (TESTED && bad[cfg]) return;
    const EnsEntry& e = entry(tab, cfg);
    const uint32_t s = (lb - e.blk0) * kBS + (lu & 3u) * 64u + (threadIdx.x & 63u);
    if (s >= e.L.V) return;
    const FieldView<R, BUF> f{win + e.off, e.L.V};
    int c[4];
    site_coords(e.L, s, c);
    flow_link_pf(e.L, f, T + e.off / 72 * 48, wout + e.off, acc + e.acc_off, s, c, mu, eps, ca, cb, reunit);
}

// The stage by staple sums for the configurations whose links turned out not SU(3), the (direction,
// logical block) pairs of ens_flow_kernel on as many workgroups as are resident at once, which look first
// whether there is anything to do.
constexpr uint32_t kGeneralGrid = 1024;
template <typename R, bool BUF>
__global__ void __launch_bounds__(kBS) ens_general_flow_kernel(const EnsEntry* __restrict__ tab, int n, uint32_t total,
                                                               const R* __restrict__ win, R* __restrict__ wout,
                                                               R* __restrict__ acc, double eps, double ca, double cb,
                                                               int reunit, const uint32_t* __restrict__ bad) {
    if (!bad[n]) return;
    for (uint32_t b = blockIdx.x; b < 4 * total; b += gridDim.x) {
        const uint32_t lu = xcd_block(b, 4 * total), lb = lu >> 2;
        const int cfg = find_cfg(tab, n, lb);
        if (!bad[cfg]) continue;
        const EnsEntry& e = entry(tab, cfg);
        const uint32_t s = (lb - e.blk0) * kBS + threadIdx.x;
        if (s >= e.L.V) continue;
        const FieldView<R, BUF> f{win + e.off, e.L.V};
        int c[4];
        site_coords(e.L, s, c);
        flow_link(e.L, f, wout + e.off, acc + e.acc_off, s, c, (int)(lu & 3u), eps, ca, cb, reunit);
    }
}

__global__ void clear_words_kernel(uint32_t* w, int n) {
    const int i = (int)(blockIdx.x * kBS + threadIdx.x);
    if (i < n) w[i] = 0;
}

// OBS = 0: sum of ReTr over all 6V plaquettes; OBS = 1: sum of -ReTr F_i^2 (magnetic)
template <typename R, bool BUF, int OBS>
__global__ void __launch_bounds__(kBS) ens_sum_kernel(const EnsEntry* __restrict__ tab, int n,
                                                      const R* __restrict__ fld, double* __restrict__ partials) {
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const EnsEntry& e = entry(tab, find_cfg(tab, n, lb));
    const uint32_t s = (lb - e.blk0) * kBS + threadIdx.x;
    double v = 0.0;
    if (s < e.L.V) {
        const FieldView<R, BUF> f{fld + e.off, e.L.V};
        v = OBS == 0 ? plaquette_site(e.L, f, s, 0, 3, 3) : magnetic_site(e.L, f, s);
    }
    const DD r = block_sum<kBS>(DD{v, 0.0});
    if (threadIdx.x == 0) {
        partials[2 * lb] = r.hi;
        partials[2 * lb + 1] = r.lo;
    }
}

// one workgroup per configuration: out[c * stride] = scale_c * sum of its block or tile partials
__global__ void __launch_bounds__(kBS) ens_finalize_kernel(const EnsEntry* __restrict__ tab,
                                                           const EnsRect* __restrict__ rect,
                                                           const double* __restrict__ partials,
                                                           double* __restrict__ out, int stride, int per_volume) {
    const EnsEntry e = tab[blockIdx.x];
    const uint32_t first = rect ? rect[blockIdx.x].tile0 : e.blk0, count = rect ? rect[blockIdx.x].tiles : e.nblk;
    const uint32_t lo = first + (uint32_t)(((uint64_t)count * threadIdx.x) / kBS);
    const uint32_t hi = first + (uint32_t)(((uint64_t)count * (threadIdx.x + 1)) / kBS);
    DD acc = {0.0, 0.0};
    for (uint32_t i = lo; i < hi; ++i) acc = dd_add(acc, DD{partials[2 * i], partials[2 * i + 1]});
    const DD r = block_sum<kBS>(acc);
    if (threadIdx.x == 0) {
        const double v = r.hi + r.lo;
        out[(size_t)blockIdx.x * stride] = per_volume ? v / (double)e.L.V : v;
    }
}

template <typename R>
__global__ void __launch_bounds__(kBS) copy_kernel(size_t n, const R* __restrict__ src, R* __restrict__ dst) {
    for (size_t i = (size_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (size_t)gridDim.x * kBS) dst[i] = src[i];
}

template <typename Fn>
void with_real(int is_f32, bool buf, Fn&& fn) {
    if (is_f32) {
        if (buf)
            fn(float(0), std::true_type());
        else
            fn(float(0), std::false_type());
    } else {
        if (buf)
            fn(double(0), std::true_type());
        else
            fn(double(0), std::false_type());
    }
}

}  // namespace

hipError_t launch_ens_flow_stage(const EnsEntry* tab, int n, uint32_t total, uint32_t maxV, const void* win,
                                 int is_f32, void* wout, void* acc, double eps, double ca, double cb, int reunit,
                                 void* T, hipStream_t st, uint32_t* bad) {
    with_real(is_f32, fits_buffer(maxV, is_f32), [&](auto r, auto buf) {
        using R = decltype(r);
        constexpr bool B = decltype(buf)::value;
        if (T) {
            constexpr bool kF64 = sizeof(R) == 8;
            const bool test = kF64 && bad && ca == 0.0;  // the step's first stage
            if (test) {
                clear_words_kernel<<<n / kBS + 1, kBS, 0, st>>>(bad, n + 1);
                ens_plaq_ta_kernel<R, B, kF64><<<total, kBS, 0, st>>>(tab, n, (const R*)win, (R*)T, bad);
            } else {
                ens_plaq_ta_kernel<R, B, false><<<total, kBS, 0, st>>>(tab, n, (const R*)win, (R*)T, bad);
            }
            if constexpr (kF64) {
                if (bad) {
                    ens_flow_pf_kernel<R, B, true><<<4 * total, kBS, 0, st>>>(
                        tab, n, (const R*)win, (const R*)T, (R*)wout, (R*)acc, eps, ca, cb, reunit, bad);
                    ens_general_flow_kernel<R, B><<<std::min(kGeneralGrid, 4 * total), kBS, 0, st>>>(
                        tab, n, total, (const R*)win, (R*)wout, (R*)acc, eps, ca, cb, reunit, bad);
                    return;
                }
            }
            ens_flow_pf_kernel<R, B, false><<<4 * total, kBS, 0, st>>>(tab, n, (const R*)win, (const R*)T, (R*)wout,
                                                                       (R*)acc, eps, ca, cb, reunit, nullptr);
        } else {
            ens_flow_kernel<R, B><<<4 * total, kBS, 0, st>>>(tab, n, (const R*)win, (R*)wout, (R*)acc, eps, ca, cb,
                                                             reunit);
        }
    });
    return hipGetLastError();
}

hipError_t launch_ens_sum(const EnsEntry* tab, int n, uint32_t total, uint32_t maxV, const void* fld, int is_f32,
                          int obs, double* partials, hipStream_t st) {
    with_real(is_f32, fits_buffer(maxV, is_f32), [&](auto r, auto buf) {
        using R = decltype(r);
        constexpr bool B = decltype(buf)::value;
        if (obs == 0)
            ens_sum_kernel<R, B, 0><<<total, kBS, 0, st>>>(tab, n, (const R*)fld, partials);
        else
            ens_sum_kernel<R, B, 1><<<total, kBS, 0, st>>>(tab, n, (const R*)fld, partials);
    });
    return hipGetLastError();
}

hipError_t launch_ens_finalize(const EnsEntry* tab, const EnsRect* rect, int n, const double* partials, double* out,
                               int stride, int per_volume, hipStream_t st) {
    ens_finalize_kernel<<<n, kBS, 0, st>>>(tab, rect, partials, out, stride, per_volume);
    return hipGetLastError();
}

hipError_t launch_copy(size_t n_reals, int is_f32, const void* src, void* dst, hipStream_t st) {
    const uint32_t g = (uint32_t)std::min<size_t>((n_reals + kBS - 1) / kBS, 8192);
    if (is_f32)
        copy_kernel<float><<<g, kBS, 0, st>>>(n_reals, (const float*)src, (float*)dst);
    else
        copy_kernel<double><<<g, kBS, 0, st>>>(n_reals, (const double*)src, (double*)dst);
    return hipGetLastError();
}

}  // namespace flue
