// k_field.hip -- moving gauge fields between the reference's complex layout and the
// SoA planes, precision conversion, and the on-device link generator.
#include "flue_launch.hpp"
#include "flue_su3x.hpp"

namespace flue {

namespace {

// ---------------------------------------------------------------- layout conversion
//
// A complex array has any element strides for (t, x, y, z, mu, a, b); a field's planes have x
// fastest.  Moving one into the other is a transpose whose two sides both want whole cache lines:
//   kArraySites  the 36 elements of a site are contiguous (a C-ordered array, a file's order):
//                blocks of 64 sites, read as they lie and handed over through LDS;
//   kArrayPlanes      the lattice direction f with the smallest stride is not x (a Fortran-ordered array
//                has t): 32 x 32 tiles of (f, x) through LDS, plane by plane;
//   kArrayRows        that direction is x: both sides run along x.
// 48^3x96, complex128 <-> FP64 (12.2 GB moved, 2.5 ms at the rate of a large copy): in, C order
// 7.97 -> 2.78 ms and Fortran order 8.44 -> 2.50 ms; out, Fortran order 4.37 -> 2.50 ms, against one
// thread per link running along t for every order.  24^3x48: 0.35 -> 0.19, 0.30 -> 0.17, 0.18 -> 0.17.
// Arrays whose elements are not aligned to their pair keep that form (import_kernel, export_kernel).
enum ArrayOrder { kArraySites, kArrayPlanes, kArrayRows };

struct ArrayLayout {
    int64_t st[7];   // element strides for (t, x, y, z, mu, a, b)
    int f;           // direction with the smallest stride (0 = t, 1..3 = x, y, z)
    int o1, o2;      // the directions besides x and f (kArraySites with f = x: besides x and y)
};

template <typename R>
using Pair = typename Pair2<R>::type;

template <typename Ro, typename Ri>
__device__ __forceinline__ Pair<Ro> pair_as(const Pair<Ri>& v) {
    Pair<Ro> o;
    o.x = (Ro)v.x;
    o.y = (Ro)v.y;
    return o;
}

__device__ __forceinline__ int64_t array_site(const ArrayLayout& a, const int c[4]) {
    return c[0] * a.st[0] + c[1] * a.st[1] + c[2] * a.st[2] + c[3] * a.st[3];
}
__device__ __forceinline__ uint32_t field_site(const Lat& L, const int c[4]) {
    return (uint32_t)c[1] + L.st[2] * (uint32_t)c[2] + L.st[3] * (uint32_t)c[3] + L.st[0] * (uint32_t)c[0];
}
// c[d] = v for a run-time direction (c stays in registers)
__device__ __forceinline__ void set_coord(int c[4], int d, int v) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (k == d) c[k] = v;
}

// the coordinates of a block's corner: x blocks fastest, then f blocks, o1, o2
__device__ __forceinline__ void block_corner(const Lat& L, const ArrayLayout& a, int ex, int ef, int f, int c[4]) {
    const uint32_t nbx = (uint32_t)(L.n[1] + ex - 1) / ex, nbf = (uint32_t)(L.ext(f) + ef - 1) / ef;
    uint32_t q = blockIdx.x;
    c[1] = (int)(q % nbx) * ex;
    q /= nbx;
    set_coord(c, f, (int)(q % nbf) * ef);
    q /= nbf;
    set_coord(c, a.o1, (int)(q % (uint32_t)L.ext(a.o1)));
    set_coord(c, a.o2, (int)(q / (uint32_t)L.ext(a.o1)));
}

// position of element e = mu * 9 + a * 3 + b in a site's 36, and its offset in a plane array
__device__ __forceinline__ int64_t element_offset(const ArrayLayout& l, int e) {
    return (e / 9) * l.st[4] + (e / 3 % 3) * l.st[5] + (e % 3) * l.st[6];
}

// kArraySites.  IN: array -> field, else field -> array; 64 sites, 16 x 4 along x and f, or 64 along x
// when the sites of the array follow x.  A site takes 37 pairs of LDS, which spreads the plane
// reads over the banks.
template <bool IN, typename Ra, typename Rf>
__global__ void __launch_bounds__(256) site_block_kernel(Lat L, ArrayLayout l, Pair<Ra>* __restrict__ arr,
                                                         Pair<Rf>* __restrict__ fld) {
    __shared__ Pair<Ra> sh[64 * 37];
    const int f = l.f == 1 ? 2 : l.f, bx = l.f == 1 ? 64 : 16, bf = 64 / bx;
    int c0[4];
    block_corner(L, l, bx, bf, f, c0);
    const int nx = L.n[1] - c0[1], nf = L.ext(f) - (f == 0 ? c0[0] : (f == 2 ? c0[2] : c0[3]));
    auto array_side = [&](auto&& move) {
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            // sites in the array's order: along f (or x) first
            const int k = (int)threadIdx.x + 256 * i, site = k / 36, e = k - site * 36;
            const int x = bf == 1 ? site : site / bf, g = bf == 1 ? 0 : site % bf;
            if (x < nx && g < nf) {
                int c[4] = {c0[0], c0[1] + x, c0[2], c0[3]};
                const int cf = (f == 0 ? c0[0] : (f == 2 ? c0[2] : c0[3])) + g;
                set_coord(c, f, cf);
                move(arr + array_site(l, c) + e, sh + (x * bf + g) * 37 + e);
            }
        }
    };
    auto field_side = [&](auto&& move) {
        const int lane = (int)threadIdx.x & 63, x = lane % bx, g = lane / bx;
        if (x >= nx || g >= nf) return;
        int c[4] = {c0[0], c0[1] + x, c0[2], c0[3]};
        const int cf = (f == 0 ? c0[0] : (f == 2 ? c0[2] : c0[3])) + g;
        set_coord(c, f, cf);
        const uint32_t s = field_site(L, c);
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int p = ((int)threadIdx.x >> 6) + 4 * i;
            move(fld + (size_t)p * L.V + s, sh + (x * bf + g) * 37 + (int)element_offset(l, p));
        }
    };
    if constexpr (IN) {
        array_side([](const Pair<Ra>* a, Pair<Ra>* m) { *m = *a; });
        __syncthreads();
        field_side([](Pair<Rf>* v, const Pair<Ra>* m) { *v = pair_as<Rf, Ra>(*m); });
    } else {
        field_side([](const Pair<Rf>* v, Pair<Ra>* m) { *m = pair_as<Ra, Rf>(*v); });
        __syncthreads();
        array_side([](Pair<Ra>* a, const Pair<Ra>* m) { *a = *m; });
    }
}

// out = 2 G U for a C-ordered complex128 array out (NT, NX, NY, NZ, 4, 3, 3): the gradient field G and
// the links U from their planes, the four waves on the four directions of 16 x 4 sites along x and
// z, the products handed over through LDS and written as whole sites.
template <typename R>
__global__ void __launch_bounds__(256) tangent_kernel(Lat L, ArrayLayout l, const Pair<R>* __restrict__ G,
                                                      const Pair<double>* __restrict__ U, Pair<double>* __restrict__ out) {
    __shared__ Pair<double> sh[64 * 37];
    int c0[4];
    block_corner(L, l, 16, 4, 3, c0);
    const int nx = L.n[1] - c0[1], nz = L.n[3] - c0[3];
    {
        const int lane = (int)threadIdx.x & 63, mu = (int)threadIdx.x >> 6, x = lane & 15, z = lane >> 4;
        if (x < nx && z < nz) {
            const int c[4] = {c0[0], c0[1] + x, c0[2], c0[3] + z};
            const uint32_t s = field_site(L, c);
            Mat<double> A, B;
#pragma unroll
            for (int e = 0; e < 9; ++e) {
                const Pair<R> g = G[(size_t)(mu * 9 + e) * L.V + s];
                const Pair<double> u = U[(size_t)(mu * 9 + e) * L.V + s];
                A.r[e] = 2.0 * (double)g.x;
                A.i[e] = 2.0 * (double)g.y;
                B.r[e] = u.x;
                B.i[e] = u.y;
            }
            const Mat<double> E = mul(A, B);
#pragma unroll
            for (int e = 0; e < 9; ++e) {
                Pair<double> v;
                v.x = E.r[e];
                v.y = E.i[e];
                sh[(x * 4 + z) * 37 + mu * 9 + e] = v;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int k = (int)threadIdx.x + 256 * i, site = k / 36, e = k - site * 36, x = site >> 2, z = site & 3;
        if (x < nx && z < nz) {
            const int c[4] = {c0[0], c0[1] + x, c0[2], c0[3] + z};
            out[array_site(l, c) + e] = sh[site * 37 + e];
        }
    }
}

// kArrayPlanes: a 32 x 32 tile of (f, x); blockIdx.y is a row of a link.  Bound by memory, and by the chain
// of a block's planes where the lattice is small.  FP64 import with 9 / 3 / 1 planes a block: 9x6x9x6 8.7 /
// 5.6 / 5.8 us, 16^4 19.0 / 17.3 / 21.1, 24^3x48 168 / 156 / 147, 48^3x96 2514 / 2468 / 2450; FP32 of
// complex64 there 1387 / 1380 / 1509.
template <bool IN, typename Ra, typename Rf>
__global__ void __launch_bounds__(256) plane_tile_kernel(Lat L, ArrayLayout l, Pair<Ra>* __restrict__ arr,
                                                         Pair<Rf>* __restrict__ fld) {
    __shared__ Pair<Ra> sh[32][33];
    int c0[4];
    block_corner(L, l, 32, 32, l.f, c0);
    const int f0 = l.f == 0 ? c0[0] : (l.f == 2 ? c0[2] : c0[3]);
    const int nx = L.n[1] - c0[1], nf = L.ext(l.f) - f0;
    const int j = (int)threadIdx.x & 31, i0 = (int)threadIdx.x >> 5;
#pragma unroll 1
    for (int e = (int)blockIdx.y * 3; e < (int)blockIdx.y * 3 + 3; ++e) {
        Pair<Ra>* a = arr + element_offset(l, e);
        Pair<Rf>* p = fld + (size_t)e * L.V;
        // array side: f along the lanes; field side: x along the lanes
        auto array_side = [&](auto&& move) {
#pragma unroll
            for (int i = i0; i < 32; i += 8)
                if (i < nx && j < nf) {
                    int c[4] = {c0[0], c0[1] + i, c0[2], c0[3]};
                    set_coord(c, l.f, f0 + j);
                    move(a + array_site(l, c), &sh[i][j]);
                }
        };
        auto field_side = [&](auto&& move) {
#pragma unroll
            for (int i = i0; i < 32; i += 8)
                if (j < nx && i < nf) {
                    int c[4] = {c0[0], c0[1] + j, c0[2], c0[3]};
                    set_coord(c, l.f, f0 + i);
                    move(p + field_site(L, c), &sh[j][i]);
                }
        };
        if constexpr (IN) {
            array_side([](const Pair<Ra>* q, Pair<Ra>* m) { *m = *q; });
            __syncthreads();
            field_side([](Pair<Rf>* q, const Pair<Ra>* m) { *q = pair_as<Rf, Ra>(*m); });
        } else {
            field_side([](const Pair<Rf>* q, Pair<Ra>* m) { *m = pair_as<Ra, Rf>(*q); });
            __syncthreads();
            array_side([](Pair<Ra>* q, const Pair<Ra>* m) { *q = *m; });
        }
        __syncthreads();
    }
}

// kArrayRows: one thread per link, x along the lanes
template <bool IN, typename Ra, typename Rf>
__global__ void __launch_bounds__(256) row_kernel(Lat L, ArrayLayout l, Pair<Ra>* __restrict__ arr,
                                                  Pair<Rf>* __restrict__ fld) {
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= L.V) return;
    int c[4];
    site_coords(L, s, c);
    Pair<Ra>* a = arr + array_site(l, c);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const int e = (int)blockIdx.y * 9 + k;
        Pair<Ra>* q = a + element_offset(l, e);
        Pair<Rf>* p = fld + (size_t)e * L.V + s;
        if constexpr (IN)
            *p = pair_as<Rf, Ra>(*q);
        else
            *q = pair_as<Ra, Rf>(*p);
    }
}

// Any strides and alignment: one thread per (site, mu), running along t.
template <typename Rin, typename Rout>
__global__ void __launch_bounds__(256) import_kernel(Lat L, const Rin* __restrict__ src, int64_t st_t, int64_t st_x,
                                                     int64_t st_y, int64_t st_z, int64_t st_mu, int64_t st_a,
                                                     int64_t st_b, Rout* __restrict__ dst) {
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (uint64_t)L.V * 4) return;
    const uint32_t mu = (uint32_t)(gid / L.V);
    uint32_t q = (uint32_t)(gid - (uint64_t)mu * L.V);
    const int t = (int)(q % (uint32_t)L.n[0]);
    q /= (uint32_t)L.n[0];
    const int x = (int)(q % (uint32_t)L.n[1]);
    q /= (uint32_t)L.n[1];
    const int y = (int)(q % (uint32_t)L.n[2]);
    const int z = (int)(q / (uint32_t)L.n[2]);
    const int64_t base = t * st_t + x * st_x + y * st_y + z * st_z + (int64_t)mu * st_mu;
    const uint32_t s = x + L.st[2] * y + L.st[3] * z + L.st[0] * t;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const int64_t off = 2 * (base + a * st_a + b * st_b);
            Rout* d = dst + ((size_t)(mu * 9 + a * 3 + b) * L.V + s) * 2;
            d[0] = (Rout)src[off];
            d[1] = (Rout)src[off + 1];
        }
}

template <typename Rin, typename Rout>
__global__ void __launch_bounds__(256) export_kernel(Lat L, const Rin* __restrict__ src, Rout* __restrict__ dst,
                                                     int64_t st_t, int64_t st_x, int64_t st_y, int64_t st_z,
                                                     int64_t st_mu, int64_t st_a, int64_t st_b) {
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (uint64_t)L.V * 4) return;
    const uint32_t mu = (uint32_t)(gid / L.V);
    uint32_t q = (uint32_t)(gid - (uint64_t)mu * L.V);
    const int t = (int)(q % (uint32_t)L.n[0]);
    q /= (uint32_t)L.n[0];
    const int x = (int)(q % (uint32_t)L.n[1]);
    q /= (uint32_t)L.n[1];
    const int y = (int)(q % (uint32_t)L.n[2]);
    const int z = (int)(q / (uint32_t)L.n[2]);
    const int64_t base = t * st_t + x * st_x + y * st_y + z * st_z + (int64_t)mu * st_mu;
    const uint32_t s = x + L.st[2] * y + L.st[3] * z + L.st[0] * t;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const int64_t off = 2 * (base + a * st_a + b * st_b);
            const Rin* q = src + ((size_t)(mu * 9 + a * 3 + b) * L.V + s) * 2;
            dst[off] = (Rout)q[0];
            dst[off + 1] = (Rout)q[1];
        }
}

template <typename R>
__global__ void __launch_bounds__(256) random_kernel(Lat L, uint64_t seed, double eps, R* __restrict__ dst) {
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (uint64_t)L.V * 4) return;
    const uint32_t mu = (uint32_t)(gid / L.V);
    const uint32_t s = (uint32_t)(gid - (uint64_t)mu * L.V);
    int c[4];
    site_coords(L, s, c);
    const uint64_t sref = (uint64_t)c[0] + (uint64_t)L.n[0] * (c[1] + (uint64_t)L.n[1] * (c[2] + (uint64_t)L.n[2] * c[3]));
    const Mat<double> U = random_link(seed, sref + (uint64_t)L.V * mu, eps);
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        R* d = dst + ((size_t)(mu * 9 + e) * L.V + s) * 2;
        d[0] = (R)U.r[e];
        d[1] = (R)U.i[e];
    }
}

template <typename Rin, typename Rout>
__global__ void __launch_bounds__(256) convert_kernel(size_t n, const Rin* __restrict__ src, Rout* __restrict__ dst) {
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid < n) dst[gid] = (Rout)src[gid];
}

inline uint32_t grid_for(uint64_t n) { return (uint32_t)((n + 255) / 256); }

// ---------------------------------------------------------------- SU(3) check
//
// Deviation of every link from SU(3), in FP64 whatever the storage precision.  One thread
// per site checks its four links; each block writes three values: the number of links
// with a non-finite entry, max |(U U^+ - 1)_ab| and max |det U - 1| over its finite links.
// Counts and maxima do not depend on the order of combination, so the result is the
// same on every run.

struct Dev3 {
    double bad, du, dd;
};

__device__ __forceinline__ Dev3 dev3_join(Dev3 a, Dev3 b) {
    return {a.bad + b.bad, fmax(a.du, b.du), fmax(a.dd, b.dd)};
}

// block-wide combination of Dev3 (256 threads); valid in thread 0
__device__ __forceinline__ Dev3 dev3_block(Dev3 v) {
    __shared__ double sh[3][4];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1)
        v = dev3_join(v, Dev3{__shfl_xor(v.bad, m), __shfl_xor(v.du, m), __shfl_xor(v.dd, m)});
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
        sh[0][w] = v.bad;
        sh[1][w] = v.du;
        sh[2][w] = v.dd;
    }
    __syncthreads();
    Dev3 r = {0.0, 0.0, 0.0};
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; ++k) r = dev3_join(r, Dev3{sh[0][k], sh[1][k], sh[2][k]});
    return r;
}

template <typename FV>
__global__ void __launch_bounds__(256) check_kernel(Lat L, FV f, double* __restrict__ part) {
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    Dev3 v = {0.0, 0.0, 0.0};
    if (s < L.V) {
#pragma unroll 1
        for (int mu = 0; mu < 4; ++mu) {
            const auto u = load_link(f, mu, s);
            double ur[9], ui[9];
            bool fin = true;
#pragma unroll
            for (int e = 0; e < 9; ++e) {
                ur[e] = (double)u.r[e];
                ui[e] = (double)u.i[e];
                fin = fin && isfinite(ur[e]) && isfinite(ui[e]);
            }
            if (!fin) {
                v.bad += 1.0;
                continue;
            }
            // (U U^+)_ab = sum_k U_ak conj(U_bk)
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    double mr = a == b ? -1.0 : 0.0, mi = 0.0;
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        mr += ur[a * 3 + k] * ur[b * 3 + k] + ui[a * 3 + k] * ui[b * 3 + k];
                        mi += ui[a * 3 + k] * ur[b * 3 + k] - ur[a * 3 + k] * ui[b * 3 + k];
                    }
                    v.du = fmax(v.du, sqrt(mr * mr + mi * mi));
                }
            // det U by the first row's cofactors
            double dr = 0.0, di = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int j = (c + 1) % 3, k = (c + 2) % 3;
                // cofactor C_0c = U_1j U_2k - U_1k U_2j
                const double cr = ur[3 + j] * ur[6 + k] - ui[3 + j] * ui[6 + k] - ur[3 + k] * ur[6 + j] +
                                  ui[3 + k] * ui[6 + j];
                const double ci = ur[3 + j] * ui[6 + k] + ui[3 + j] * ur[6 + k] - ur[3 + k] * ui[6 + j] -
                                  ui[3 + k] * ur[6 + j];
                dr += ur[c] * cr - ui[c] * ci;
                di += ur[c] * ci + ui[c] * cr;
            }
            v.dd = fmax(v.dd, sqrt((dr - 1.0) * (dr - 1.0) + di * di));
        }
    }
    const Dev3 r = dev3_block(v);
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = r.bad;
        part[3 * blockIdx.x + 1] = r.du;
        part[3 * blockIdx.x + 2] = r.dd;
    }
}

__global__ void __launch_bounds__(256) check_final_kernel(const double* __restrict__ part, uint32_t n,
                                                          double* __restrict__ out) {
    Dev3 v = {0.0, 0.0, 0.0};
    for (uint32_t i = threadIdx.x; i < n; i += 256u) v = dev3_join(v, Dev3{part[3 * i], part[3 * i + 1], part[3 * i + 2]});
    const Dev3 r = dev3_block(v);
    if (threadIdx.x == 0) {
        out[0] = r.bad;
        out[1] = r.du;
        out[2] = r.dd;
    }
}

}  // namespace

uint32_t check_blocks(const Lat& L) { return (L.V + 255u) / 256u; }

hipError_t launch_check_field(const Lat& L, const void* U, int is_f32, double* part, double* out3, hipStream_t st) {
    const uint32_t nb = check_blocks(L);
    with_view(L.V, U, is_f32, [&](auto f) { check_kernel<decltype(f)><<<nb, 256, 0, st>>>(L, f, part); });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    check_final_kernel<<<1, 256, 0, st>>>(part, nb, out3);
    return hipGetLastError();
}

// How an array is laid out, or -1 for the general kernels.  Reads may overlap (an expanded array),
// writes may not: an array written to with a zero stride keeps the general kernel's order.
static int array_order(const Lat& L, const int64_t s[7], bool written, ArrayLayout& l) {
    for (int k = 0; k < 7; ++k) l.st[k] = s[k];
    for (int k = 0; k < 7; ++k)
        if (s[k] < 0 || (written && s[k] == 0 && (k >= 4 || L.n[k] > 1))) return -1;
    // smallest stride of a direction with more than one site; x wins ties
    l.f = 1;
    const int dirs[4] = {1, 0, 2, 3};
    int64_t best = L.n[1] > 1 ? s[1] : INT64_MAX;
    for (int d : dirs)
        if (L.n[d] > 1 && s[d] < best) {
            best = s[d];
            l.f = d;
        }
    const int f = l.f == 1 ? 2 : l.f;
    l.o1 = l.o2 = -1;
    for (int d = 0; d < 4; ++d)
        if (d != 1 && d != f) (l.o1 < 0 ? l.o1 : l.o2) = d;
    uint64_t seen = 0;
    bool block = true;
    for (int e = 0; e < 36 && block; ++e) {
        const int64_t o = (e / 9) * s[4] + (e / 3 % 3) * s[5] + (e % 3) * s[6];
        block = o < 36 && !(seen >> o & 1);
        if (block) seen |= 1ull << o;
    }
    return block ? kArraySites : (l.f == 1 ? kArrayRows : kArrayPlanes);
}

template <bool IN, typename Ra, typename Rf>
static hipError_t convert_layout(const Lat& L, int order, const ArrayLayout& l, const void* arr, const void* fld,
                                 hipStream_t st, int ndir = 4) {
    Pair<Ra>* a = (Pair<Ra>*)arr;
    Pair<Rf>* p = (Pair<Rf>*)fld;
    const uint32_t rest = (uint32_t)L.ext(l.o1) * (uint32_t)L.ext(l.o2);
    if (order == kArraySites) {
        const int f = l.f == 1 ? 2 : l.f;
        const uint32_t bx = l.f == 1 ? 64 : 16, bf = 64 / bx;
        const uint32_t g = ((uint32_t)L.n[1] + bx - 1) / bx * (((uint32_t)L.ext(f) + bf - 1) / bf) * rest;
        site_block_kernel<IN, Ra, Rf><<<g, 256, 0, st>>>(L, l, a, p);
    } else if (order == kArrayPlanes) {
        const uint32_t g = ((uint32_t)L.n[1] + 31) / 32 * (((uint32_t)L.ext(l.f) + 31) / 32) * rest;
        plane_tile_kernel<IN, Ra, Rf><<<dim3(g, 3 * ndir), 256, 0, st>>>(L, l, a, p);
    } else {
        row_kernel<IN, Ra, Rf><<<dim3(grid_for(L.V), ndir), 256, 0, st>>>(L, l, a, p);
    }
    return hipGetLastError();
}

static bool pair_aligned(const void* p, int is_f32) { return (uintptr_t)p % (is_f32 ? 8 : 16) == 0; }

bool imports_by_direction(const Lat& L, const int64_t s[7]) {
    ArrayLayout l;
    const int order = array_order(L, s, false, l);
    return order == kArrayPlanes || order == kArrayRows;
}

hipError_t launch_import(const Lat& L, const void* src, int src_is_f32, const int64_t s[7], void* dst,
                         int dst_is_f32, hipStream_t st, int ndir) {
    ArrayLayout l;
    const int order = array_order(L, s, false, l);
    if (ndir < 4 && (!imports_by_direction(L, s) || !pair_aligned(src, src_is_f32) || !pair_aligned(dst, dst_is_f32)))
        return hipErrorInvalidValue;
    if (order >= 0 && pair_aligned(src, src_is_f32) && pair_aligned(dst, dst_is_f32)) {
        if (src_is_f32)
            return dst_is_f32 ? convert_layout<true, float, float>(L, order, l, src, dst, st, ndir)
                              : convert_layout<true, float, double>(L, order, l, src, dst, st, ndir);
        return dst_is_f32 ? convert_layout<true, double, float>(L, order, l, src, dst, st, ndir)
                          : convert_layout<true, double, double>(L, order, l, src, dst, st, ndir);
    }
    const uint32_t g = grid_for((uint64_t)L.V * 4);
    if (src_is_f32 && dst_is_f32)
        import_kernel<float, float><<<g, 256, 0, st>>>(L, (const float*)src, s[0], s[1], s[2], s[3], s[4], s[5], s[6],
                                                       (float*)dst);
    else if (src_is_f32)
        import_kernel<float, double><<<g, 256, 0, st>>>(L, (const float*)src, s[0], s[1], s[2], s[3], s[4], s[5],
                                                        s[6], (double*)dst);
    else if (dst_is_f32)
        import_kernel<double, float><<<g, 256, 0, st>>>(L, (const double*)src, s[0], s[1], s[2], s[3], s[4], s[5],
                                                        s[6], (float*)dst);
    else
        import_kernel<double, double><<<g, 256, 0, st>>>(L, (const double*)src, s[0], s[1], s[2], s[3], s[4], s[5],
                                                         s[6], (double*)dst);
    return hipGetLastError();
}

hipError_t launch_export(const Lat& L, const void* src, int src_is_f32, void* dst, int dst_is_f32,
                         const int64_t s[7], hipStream_t st) {
    ArrayLayout l;
    const int order = array_order(L, s, true, l);
    if (order >= 0 && pair_aligned(src, src_is_f32) && pair_aligned(dst, dst_is_f32)) {
        if (dst_is_f32)
            return src_is_f32 ? convert_layout<false, float, float>(L, order, l, dst, src, st)
                              : convert_layout<false, float, double>(L, order, l, dst, src, st);
        return src_is_f32 ? convert_layout<false, double, float>(L, order, l, dst, src, st)
                          : convert_layout<false, double, double>(L, order, l, dst, src, st);
    }
    const uint32_t g = grid_for((uint64_t)L.V * 4);
    if (src_is_f32 && dst_is_f32)
        export_kernel<float, float><<<g, 256, 0, st>>>(L, (const float*)src, (float*)dst, s[0], s[1], s[2], s[3], s[4],
                                                       s[5], s[6]);
    else if (src_is_f32)
        export_kernel<float, double><<<g, 256, 0, st>>>(L, (const float*)src, (double*)dst, s[0], s[1], s[2], s[3],
                                                        s[4], s[5], s[6]);
    else if (dst_is_f32)
        export_kernel<double, float><<<g, 256, 0, st>>>(L, (const double*)src, (float*)dst, s[0], s[1], s[2], s[3],
                                                        s[4], s[5], s[6]);
    else
        export_kernel<double, double><<<g, 256, 0, st>>>(L, (const double*)src, (double*)dst, s[0], s[1], s[2], s[3],
                                                         s[4], s[5], s[6]);
    return hipGetLastError();
}

hipError_t launch_tangent(const Lat& L, const void* G, int is_f32, const void* U, void* out, hipStream_t st) {
    ArrayLayout l;
    const int64_t z = 36, y = z * L.n[3], x = y * L.n[2], s[7] = {x * L.n[1], x, y, z, 9, 3, 1};
    for (int k = 0; k < 7; ++k) l.st[k] = s[k];
    l.f = 3;
    l.o1 = 2;
    l.o2 = 0;
    const uint32_t g = ((uint32_t)L.n[1] + 15) / 16 * (((uint32_t)L.n[3] + 3) / 4) * (uint32_t)L.n[2] * (uint32_t)L.n[0];
    if (is_f32)
        tangent_kernel<float><<<g, 256, 0, st>>>(L, l, (const Pair<float>*)G, (const Pair<double>*)U, (Pair<double>*)out);
    else
        tangent_kernel<double><<<g, 256, 0, st>>>(L, l, (const Pair<double>*)G, (const Pair<double>*)U, (Pair<double>*)out);
    return hipGetLastError();
}

hipError_t launch_random_field(const Lat& L, uint64_t seed, double eps, void* dst, int is_f32, hipStream_t st) {
    const uint32_t g = grid_for((uint64_t)L.V * 4);
    if (is_f32)
        random_kernel<float><<<g, 256, 0, st>>>(L, seed, eps, (float*)dst);
    else
        random_kernel<double><<<g, 256, 0, st>>>(L, seed, eps, (double*)dst);
    return hipGetLastError();
}

hipError_t launch_convert(const Lat& L, const void* src, int src_is_f32, void* dst, int dst_is_f32, hipStream_t st) {
    const size_t n = (size_t)L.V * kPlanes;
    const uint32_t g = grid_for(n);
    if (src_is_f32 == dst_is_f32)
        return hipMemcpyAsync(dst, src, n * (src_is_f32 ? 4 : 8), hipMemcpyDeviceToDevice, st);
    if (src_is_f32)
        convert_kernel<float, double><<<g, 256, 0, st>>>(n, (const float*)src, (double*)dst);
    else
        convert_kernel<double, float><<<g, 256, 0, st>>>(n, (const double*)src, (float*)dst);
    return hipGetLastError();
}

}  // namespace flue
