// k_b2tile.hip -- adjoint of the magnetic B^2 on the tiles of the rectangle-first form.
//
// Every leaf rectangle a x b of a spatial plane is walked once from its lower-left corner x, as in
// the slot form (k_b2grad.hip, whose notation this keeps): with the loop W = CA CB^+, the corner
// sums moved to x,
//   A0 = A(x), Aa = La A(x + a d1) La^+, Aab = CA A(x + a d1 + b d2) CA^+, Ah = Lb A(x + b d2) Lb^+
// (La = Line(x, d1, a), Lb = Line(x, d2, b)) and S = A0 + Aa + Aab, the links of its sides take
//   bottom  +X^+ Zb X   at x + p d1,         X = Line(x, d1, p)       p < a
//   right   +X^+ Zr X   at x + a d1 + q d2,  X = CA(a, q)             q < b
//   left    -X^+ Zl X   at x + m d2,         X = Line(x, d2, m)       m < b
//   top     -X^+ Zt X   at x + m d1 + b d2,  X = CB(b, m)             m < a
// where only anti-Hermitian parts of the sums enter (the terms are projected, X is unitary):
//   Zl = AH(S W + W Ah),   Zt = Zl + [Ah, K],   Zb = Zl - [A0, K],   Zr = Zb - [Aa, K]
// with K = AH(W) (AH(A W) - AH(W A) = [A, AH(W)] for anti-Hermitian A).
//
// The seven shapes are taken in rows of equal a.  A row shares Line(x, d1, a) and the chain CA(a, .),
// and the terms that meet at one link with one X are summed first and moved once: per row the
// bottom terms in one sum, the left and right ones in one sum per link.  Per base site and plane: 29
// chain products, 7 loops, 17 corner moves, 29 moved terms, against 38 + 38, 7, 21 and 38 in
// seven separate kernels.
//
// The terms go into the tile's footprint in LDS (8 reals for the d1 and 8 for the d2 link of a
// cell, added in FP64 in both precisions), and the footprints to memory: 2 x 16 reals a site and
// plane against 2 x 416 for the slots, whose writes and sums were half of the call.  One wavefront
// per footprint, as in the forward form, so each cell's sum is formed in a fixed order.
#include <algorithm>

#include "flue_flow.hpp"
#include "flue_launch.hpp"
#include "flue_rect.hpp"
#include "flue_tiles.hpp"

namespace flue {

namespace {

constexpr int kW = 64;  // one wavefront per tile
// cells of the largest footprint (128 bytes each): eight wavefronts (FP32, two per SIMD) or four
// (FP64, one per SIMD) share a CU's 160 KB of LDS
template <typename R>
constexpr int kAdjCells = sizeof(R) == 4 ? 160 : 320;

// parts of V^+ A V or, for the corner sums, of F A F^+
template <bool C2, typename R>
__device__ __forceinline__ AH<R> move_parts(const AH<R>& h, const Mat<R>& X) {
    return ah_conj(h, full_rows<C2>(X));
}
template <bool C2, typename R>
__device__ __forceinline__ AH<R> corner_parts(const AH<R>& h, const Mat<R>& F) {
    return ah_conj(h, dag(full_rows<C2>(F)));
}

// h += parts of AH(A M) for the anti-Hermitian A with parts a: d_i += Im (A M)_ii,
// o_ij += (A M)_ij - conj((A M)_ji)
template <typename R>
__device__ __forceinline__ void add_ah_mul(AH<R>& h, const AH<R>& a, const Mat<R>& M) {
    // off-diagonal entries of A, row-major
    R ar[9], ai[9];
    constexpr int pa[3] = {0, 0, 1}, pb[3] = {1, 2, 2};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int i = pa[q], j = pb[q];
        ar[i * 3 + j] = R(0.5) * a.or_[q];
        ai[i * 3 + j] = R(0.5) * a.oi[q];
        ar[j * 3 + i] = R(-0.5) * a.or_[q];
        ai[j * 3 + i] = R(0.5) * a.oi[q];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        h.d[i] = fmad(a.d[i], M.r[i * 4], h.d[i]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k == i) continue;
            h.d[i] = fmad(ar[i * 3 + k], M.i[k * 3 + i], h.d[i]);
            h.d[i] = fmad(ai[i * 3 + k], M.r[k * 3 + i], h.d[i]);
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int i = pa[q], j = pb[q];
        // + (A M)_ij
        h.or_[q] = fmad(-a.d[i], M.i[i * 3 + j], h.or_[q]);
        h.oi[q] = fmad(a.d[i], M.r[i * 3 + j], h.oi[q]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k == i) continue;
            h.or_[q] = fmad(ar[i * 3 + k], M.r[k * 3 + j], h.or_[q]);
            h.or_[q] = fmad(-ai[i * 3 + k], M.i[k * 3 + j], h.or_[q]);
            h.oi[q] = fmad(ar[i * 3 + k], M.i[k * 3 + j], h.oi[q]);
            h.oi[q] = fmad(ai[i * 3 + k], M.r[k * 3 + j], h.oi[q]);
        }
        // - conj((A M)_ji)
        h.or_[q] = fmad(a.d[j], M.i[j * 3 + i], h.or_[q]);
        h.oi[q] = fmad(a.d[j], M.r[j * 3 + i], h.oi[q]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k == j) continue;
            h.or_[q] = fmad(-ar[j * 3 + k], M.r[k * 3 + i], h.or_[q]);
            h.or_[q] = fmad(ai[j * 3 + k], M.i[k * 3 + i], h.or_[q]);
            h.oi[q] = fmad(ar[j * 3 + k], M.i[k * 3 + i], h.oi[q]);
            h.oi[q] = fmad(ai[j * 3 + k], M.r[k * 3 + i], h.oi[q]);
        }
    }
}

// h + s [A, K] for anti-Hermitian A, K with parts a, k (traceless-free: traces commute away).
// With A_ij = o_ij / 2 (i < j): diagonal +-(1/2) Im(k_ij conj(a_ij)); off the diagonal
//   o'_01 = i (a0 - a1) k_01 - i (k0 - k1) a_01 + (1/2) (k_02 conj(a_12) - a_02 conj(k_12))
//   o'_02 = i (a0 - a2) k_02 - i (k0 - k2) a_02 + (1/2) (a_01 k_12 - k_01 a_12)
//   o'_12 = i (a1 - a2) k_12 - i (k1 - k2) a_12 + (1/2) (conj(k_01) a_02 - conj(a_01) k_02)
template <typename R>
__device__ __forceinline__ AH<R> add_commutator(const AH<R>& h, R s, const AH<R>& a, const AH<R>& k) {
    const R g = R(0.5) * s;
    R x[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) x[q] = fmad(k.oi[q], a.or_[q], -k.or_[q] * a.oi[q]);
    AH<R> c;
    c.d[0] = fmad(g, x[0] + x[1], h.d[0]);
    c.d[1] = fmad(g, x[2] - x[0], h.d[1]);
    c.d[2] = fmad(-g, x[1] + x[2], h.d[2]);
    constexpr int pi[3] = {0, 0, 1}, pj[3] = {1, 2, 2};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const R da = s * (a.d[pi[q]] - a.d[pj[q]]), dk = s * (k.d[pi[q]] - k.d[pj[q]]);
        c.or_[q] = fmad(-da, k.oi[q], fmad(dk, a.oi[q], h.or_[q]));
        c.oi[q] = fmad(da, k.or_[q], fmad(-dk, a.or_[q], h.oi[q]));
    }
    auto term = [&](int q, R w, R ur, R ui, R vr, R vi) {  // o_q += w u v
        c.or_[q] = fmad(w * ur, vr, c.or_[q]);
        c.or_[q] = fmad(-(w * ui), vi, c.or_[q]);
        c.oi[q] = fmad(w * ur, vi, c.oi[q]);
        c.oi[q] = fmad(w * ui, vr, c.oi[q]);
    };
    term(0, g, k.or_[1], k.oi[1], a.or_[2], -a.oi[2]);
    term(0, -g, a.or_[1], a.oi[1], k.or_[2], -k.oi[2]);
    term(1, g, a.or_[0], a.oi[0], k.or_[2], k.oi[2]);
    term(1, -g, k.or_[0], k.oi[0], a.or_[2], a.oi[2]);
    term(2, g, k.or_[0], -k.oi[0], a.or_[1], a.oi[1]);
    term(2, -g, a.or_[0], -a.oi[0], k.or_[1], k.oi[1]);
    return c;
}

// anti-Hermitian parts of M: d_i = Im M_ii, o_ij = M_ij - conj(M_ji)
template <typename R>
__device__ __forceinline__ AH<R> parts_of(const Mat<R>& M) {
    AH<R> h;
    constexpr int pa[3] = {0, 0, 1}, pb[3] = {1, 2, 2};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h.d[k] = M.i[k * 4];
        h.or_[k] = M.r[pa[k] * 3 + pb[k]] - M.r[pb[k] * 3 + pa[k]];
        h.oi[k] = M.i[pa[k] * 3 + pb[k]] + M.i[pb[k] * 3 + pa[k]];
    }
    return h;
}

template <typename R>
__device__ __forceinline__ void add_scaled(AH<R>& h, R w, const AH<R>& g) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h.d[k] = fmad(w, g.d[k], h.d[k]);
        h.or_[k] = fmad(w, g.or_[k], h.or_[k]);
        h.oi[k] = fmad(w, g.oi[k], h.oi[k]);
    }
}

// the stored clover parts of a plane at site s
template <typename R, bool BUF>
__device__ __forceinline__ AH<R> load_parts(const Planes<R, BUF>& A, uint32_t s) {
    AH<R> h;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h.d[k] = A.template ld<false>(k, s);
        h.or_[k] = A.template ld<false>(3 + k, s);
        h.oi[k] = A.template ld<false>(6 + k, s);
    }
    return h;
}

template <int A, int B>
constexpr double shape_weight() {
    return A == B ? (A == 1 ? kK1 : (A == 2 ? kK2 : kK5)) : (A * B == 2 ? 0.5 * kK3 : 0.5 * kK4);
}

// One row of shapes, (A, 1), (A, 2), (A, 3) as far as they exist.  emit(dir, da, db, w, h) adds w
// times the traceless part of h to the link of direction d1 (dir = 0) or d2 (1) at x + da d1 + db d2.
template <int A, bool C2, typename FV, typename PA, typename Emit>
__device__ __forceinline__ void adjoint_row(const Quad<FV>& q, const PA& Ab, Emit&& emit) {
    using R = typename FV::real;
    constexpr int BMAX = A == 2 ? 2 : 3;
    auto site = [&](int i, int j) { return q.sp + q.T1[i] + q.T2[j]; };
    auto link = [&](int dir, int i, int j) { return load_link(q.f, dir == 0 ? q.ax1 : q.ax2, site(i, j)); };
    const AH<R> A0 = load_parts(Ab, site(0, 0));
    // Line(x, d1, p): p = 1 whole, longer ones as chains
    const Mat<R> L1 = link(0, 0, 0);
    Mat<R> L2 = L1, L = L1;
    if constexpr (A >= 2) {
        L2 = ext_by<1, C2>(L1, link(0, 1, 0));
        L = L2;
    }
    if constexpr (A >= 3) L = ext_by<1, C2>(L2, link(0, 2, 0));
    const AH<R> Aa = corner_parts<(A > 1) && C2>(load_parts(Ab, site(A, 0)), L);
    AH<R> bottom, left[BMAX], right[BMAX];
    ah_zero(bottom);
#pragma unroll
    for (int b = 0; b < BMAX; ++b) {
        ah_zero(left[b]);
        ah_zero(right[b]);
    }
    Mat<R> CA = L, Lb = L1, M1 = L1, M2 = L1;
#pragma unroll
    for (int b = 1; b <= BMAX; ++b) {
        FLUE_SCHED_FENCE();
        CA = ext_by<1, C2>(CA, link(1, A, b - 1));  // CA(A, b)
        if (b == 1) {
            Lb = M1 = link(1, 0, 0);                // Line(x, d2, 1)
        } else {
            Lb = ext_by<1, C2>(Lb, link(1, 0, b - 1));
            if (b == 2) M2 = Lb;
        }
        if (A == 3 && b == 2) continue;             // 3 x 2 is not a leaf
        const R w = b == 1 ? R(shape_weight<A, 1>()) : (b == 2 ? R(shape_weight<A, 2>()) : R(shape_weight<A, 3>()));
        Mat<R> CB[A + 1];
        CB[0] = Lb;
#pragma unroll
        for (int m = 0; m < A; ++m) CB[m + 1] = ext_by<1, C2>(CB[m], link(0, m, b));  // CB(b, m + 1)
        Mat<R> W = C2 ? mul2_nd(CA, full_rows<C2>(CB[A])) : mul_nd(CA, CB[A]);
        if constexpr (C2) fill_row2(W);
        const AH<R> Ah = b == 1 ? corner_parts<false>(load_parts(Ab, site(0, b)), Lb)
                                : corner_parts<C2>(load_parts(Ab, site(0, b)), Lb);
        AH<R> S = corner_parts<C2>(load_parts(Ab, site(A, b)), CA);
        ah_add(S, Aa);
        ah_add(S, A0);
        // AH(W Ah) = AH(Ah W^+)
        AH<R> Z;
        ah_zero(Z);
        add_ah_mul(Z, S, W);
        add_ah_mul(Z, Ah, dag(W));
        const AH<R> K = parts_of(W);
#pragma unroll
        for (int m = 0; m < b; ++m) add_scaled(left[m], w, Z);
        {
            const AH<R> Zt = add_commutator(Z, R(1), Ah, K);
#pragma unroll
            for (int m = 0; m < A; ++m)
                emit(0, m, b, -w, b == 1 && m == 0 ? move_parts<false>(Zt, CB[m]) : move_parts<C2>(Zt, CB[m]));
        }
        Z = add_commutator(Z, R(-1), A0, K);
        add_scaled(bottom, w, Z);
        Z = add_commutator(Z, R(-1), Aa, K);
#pragma unroll
        for (int m = 0; m < b; ++m) add_scaled(right[m], w, Z);
    }
    FLUE_SCHED_FENCE();
    emit(0, 0, 0, R(1), bottom);
    if constexpr (A >= 2) emit(0, 1, 0, R(1), move_parts<false>(bottom, L1));
    if constexpr (A >= 3) emit(0, 2, 0, R(1), move_parts<C2>(bottom, L2));
    FLUE_SCHED_FENCE();
    emit(1, 0, 0, R(-1), left[0]);
    emit(1, 0, 1, R(-1), move_parts<false>(left[1], M1));
    if constexpr (BMAX >= 3) emit(1, 0, 2, R(-1), move_parts<C2>(left[2], M2));
    FLUE_SCHED_FENCE();
    emit(1, A, 0, R(1), move_parts<(A > 1) && C2>(right[0], L));
    CA = ext_by<1, C2>(L, link(1, A, 0));
    emit(1, A, 1, R(1), move_parts<C2>(right[1], CA));
    if constexpr (BMAX >= 3) {
        CA = ext_by<1, C2>(CA, link(1, A, 1));
        emit(1, A, 2, R(1), move_parts<C2>(right[2], CA));
    }
    FLUE_SCHED_FENCE();
}

// The tiles of time slices [t0, t0 + nslice) of each plane, footprints from the buffer's start.  The
// adjoint admits SU(3) links only, so FP64 takes two-row chains (rms error 6.1e-16 of the gradient's
// norm).  FP32 keeps whole rows: rebuilt ones raise its error from 2.28e-7 to 2.47e-7, above the
// slot form's 2.43e-7, for 1.7% of the time.
template <typename FV, int WPE>
__global__ void __launch_bounds__(kW) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
b2_tile_kernel(Lat L0, FV f0, Lat Lzy, FV fzy, RectTiles rt, uint32_t t0, uint32_t nslice,
               const typename FV::real* __restrict__ Abuf, typename FV::real* __restrict__ fpout) {
    using R = typename FV::real;
    constexpr int FS = kAdjCells<R>;
    __shared__ double fp[16 * FS];
    const bool zy = blockIdx.y == 2;
    const PlaneTiles g = plane_tiles(rt);
    const Lat L = zy ? Lzy : L0;
    const uint32_t per_slice = g.tiles / (uint32_t)L.n[0], nt = per_slice * nslice;
    if (blockIdx.x >= nt) return;
    const FV f = zy ? fzy : f0;
    const int rp = zy ? 0 : (int)blockIdx.y;
    const int d2 = rect_d2(rp);
    const uint32_t tile = xcd_block(blockIdx.x, nt);
    const Tile t = tile_at(L, rp, g, tile + per_slice * t0);
    const int fc = (int)g.fc, f1 = (int)g.f;
    const Planes<R, FV::buffered> Ab{const_cast<R*>(Abuf) + (size_t)blockIdx.y * 9 * L.V, L.V, 9};
    for (int k = threadIdx.x; k < 16 * FS; k += kW) fp[k] = 0.0;
    __syncthreads();
    auto turn = [&](auto row) {
        constexpr int A = decltype(row)::value;
#pragma unroll 1
        for (uint32_t j = threadIdx.x; j < t.l1 * t.l2; j += kW) {
            const int ly = (int)(j / t.l1), lx = (int)(j - (uint32_t)ly * t.l1);
            const int cx = (int)t.o1 + lx, c2 = (int)t.o2 + ly;
            const int cy = rp == 0 ? c2 : (int)t.cs, cz = rp == 0 ? (int)t.cs : c2;
            const uint32_t s = (uint32_t)cx + L.st[2] * (uint32_t)cy + L.st[3] * (uint32_t)cz + L.st[0] * t.ct;
            const PlaneGeom<FV> pg = plane_geom(L, f, s, cx, c2, 1, d2);
            const int cell = ly * f1 + lx;
            adjoint_row<A, sizeof(R) == 8>(make_quad<1, 1, true>(pg), Ab, [&](int dir, int da, int db, R w, const AH<R>& h) {
                const R tr = (h.d[0] + h.d[1] + h.d[2]) * R(1.0 / 3.0);
                const R v[8] = {h.d[0] - tr, h.d[1] - tr, h.or_[0], h.oi[0], h.or_[1], h.oi[1], h.or_[2], h.oi[2]};
                double* p = fp + dir * 8 * FS + cell + db * f1 + da;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    __hip_atomic_fetch_add(p + k * FS, (double)(w * v[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            });
        }
    };
    turn(std::integral_constant<int, 1>());
    turn(std::integral_constant<int, 2>());
    turn(std::integral_constant<int, 3>());
    __syncthreads();
    // to memory as [e * fc + c]
    const uint64_t base = g.cell0 * nslice / (uint32_t)L.n[0] + (uint64_t)tile * g.fc;
    R* out = fpout + 16 * base;
    for (int c = threadIdx.x; c < fc; c += kW)
#pragma unroll
        for (int e = 0; e < 16; ++e) out[e * fc + c] = (R)fp[e * FS + c];
}

// The 8 sums of the link of direction d1 (DIR = 0) or d2 (1) at local cell (cx, cy) of a tile: its
// own footprint, then those of the tiles before it along d1, along d2 and diagonally.
template <typename R>
__device__ __forceinline__ void add_cover(double acc[8], const R* own, int64_t left, int64_t below, int fc, int f1,
                                          int dir, int cx, int cy, int shift1, int shift2) {
    const R* p = own + (size_t)dir * 8 * fc + cy * f1 + cx;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        double v = (double)ld_stream(p + k * fc);
        if (cx < 3) v += (double)ld_stream(p + k * fc + 16 * left + shift1);
        if (cy < 3) v += (double)ld_stream(p + k * fc + 16 * below + shift2 * f1);
        if (cx < 3 && cy < 3) v += (double)ld_stream(p + k * fc + 16 * (left + below) + shift2 * f1 + shift1);
        acc[k] += v;
    }
}

// the tile of plane g that holds (c1, c2) in slice ct (of the slab) and spectator slice cs, and the
// contributions of its footprint and its neighbours' to that cell's links
template <typename R>
__device__ __forceinline__ void add_site(double acc[8], const PlaneTiles& g, uint64_t cell0, uint32_t ns,
                                         const R* __restrict__ fpin, int dir, uint32_t c1, uint32_t c2, uint32_t cs,
                                         uint32_t ct) {
    uint32_t o1, o2;
    const uint32_t t1 = tile_of(c1, g.q1, g.r1, &o1), t2 = tile_of(c2, g.q2, g.r2, &o2);
    const uint32_t tl = t1 ? t1 - 1 : g.n1 - 1, tb = t2 ? t2 - 1 : g.n2 - 1;
    const uint64_t tile = (((uint64_t)ct * ns + cs) * g.n2 + t2) * g.n1 + t1;
    const R* own = fpin + 16 * (cell0 + tile * g.fc);
    add_cover(acc, own, ((int64_t)tl - t1) * (int64_t)g.fc, ((int64_t)tb - t2) * (int64_t)g.n1 * g.fc, (int)g.fc,
              (int)g.f, dir, (int)(c1 - o1), (int)(c2 - o2), (int)(g.q1 + (tl < g.r1 ? 1u : 0u)), (int)(g.q2 + (tb < g.r2 ? 1u : 0u)));
}

// Plane (z, y): the sums of the z and y links of the slab's sites, read z fastest and left x fastest
// in the first four (re, im) pairs of each link of grad, through a 16 x 16 (x, z) tile in LDS
template <typename R>
__global__ void __launch_bounds__(256) b2_zy_gather_kernel(Lat L, RectTiles rt, uint32_t t0, uint32_t nslice,
                                                           const R* __restrict__ fpin, R* __restrict__ grad) {
    typedef R r2 __attribute__((ext_vector_type(2)));
    __shared__ R sh[8][16][17];
    const uint32_t NX = (uint32_t)L.n[1], NY = (uint32_t)L.n[2], NZ = (uint32_t)L.n[3];
    const uint32_t bxs = (NX + 15) / 16, bzs = (NZ + 15) / 16;
    uint32_t q = blockIdx.x;
    const uint32_t bx = q % bxs;
    q /= bxs;
    const uint32_t bz = q % bzs;
    q /= bzs;
    const uint32_t y = q % NY, t = q / NY;
    const uint32_t i = threadIdx.x >> 4, j = threadIdx.x & 15;
    const uint64_t cell0 = rt.p[2].cell0 * nslice / (uint32_t)L.n[0];
#pragma unroll 1
    for (int dir = 0; dir < 2; ++dir) {
        // z along the lanes
        const uint32_t x = bx * 16 + i, z = bz * 16 + j;
        if (x < NX && z < NZ) {
            double acc[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = 0.0;
            add_site(acc, rt.p[2], cell0, NX, fpin, dir, z, y, x, t);
#pragma unroll
            for (int k = 0; k < 8; ++k) sh[k][i][j] = (R)acc[k];
        }
        __syncthreads();
        // x along the lanes
        const uint32_t xw = bx * 16 + j, zw = bz * 16 + i;
        if (xw < NX && zw < NZ) {
            const uint32_t s = xw + NX * (y + NY * (zw + NZ * (t + t0)));
            const int mu = dir == 0 ? 3 : 2;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                r2 v;
                v.x = sh[2 * k][j][i];
                v.y = sh[2 * k + 1][j][i];
                *(reinterpret_cast<r2*>(grad + (size_t)(mu * 9 + k) * 2 * L.V) + s) = v;
            }
        }
        __syncthreads();
    }
}

// Every link of the slab: planes (x, y) and (x, z), and for y and z links the sums of plane (z, y)
// left in grad; temporal links get 0.  blockIdx.y is the direction.
template <typename R>
__global__ void __launch_bounds__(256) b2_gather_kernel(Lat L, RectTiles rt, uint32_t t0, uint32_t nslice, double scale,
                                                        const R* __restrict__ fpin, R* __restrict__ grad) {
    typedef R r2 __attribute__((ext_vector_type(2)));
    const int mu = (int)blockIdx.y;
    const uint32_t o = xcd_block(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
    if (o >= nslice * L.Vs) return;
    const uint32_t s = o + t0 * L.Vs;
    if (mu == 0) {
        Mat<R> Z;
#pragma unroll
        for (int e = 0; e < 9; ++e) Z.r[e] = Z.i[e] = R(0);
        store_link_stream(grad, L.V, 0, s, Z);
        return;
    }
    int c[4];
    site_coords(L, o, c);  // c[0] counts within the slab
    double acc[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.0;
    const uint32_t x = (uint32_t)c[1], y = (uint32_t)c[2], z = (uint32_t)c[3], t = (uint32_t)c[0];
    if (mu != 3) add_site(acc, rt.p[0], 0, (uint32_t)L.n[3], fpin, mu - 1, x, y, z, t);
    if (mu != 2)
        add_site(acc, rt.p[1], rt.p[1].cell0 * nslice / (uint32_t)L.n[0], (uint32_t)L.n[2], fpin, mu == 1 ? 0 : 1, x, z,
                 y, t);
    if (mu != 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const r2 v = *(reinterpret_cast<const r2*>(grad + (size_t)(mu * 9 + k) * 2 * L.V) + s);
            acc[2 * k] += (double)v.x;
            acc[2 * k + 1] += (double)v.y;
        }
    }
    // the diagonal coordinates as they are, the off-diagonal parts o = 2 (entry)
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = acc[k] * (k < 2 ? scale : 0.5 * scale);
    store_link_stream(grad, L.V, mu, s, from_double<R>(su3_from8(v)));
}

RectTiles adj_tiles(const Lat& L, int is_f32) {
    return rect_split(L, is_f32 ? kAdjCells<float> : kAdjCells<double>, is_f32 ? 2048 : 1024);
}

// slices of a slab: footprints of at most kB2SlotReals reals
uint32_t adj_slab(const Lat& L, const RectTiles& rt) {
    const uint64_t per = 16 * rect_cells(rt) / (uint32_t)L.n[0];
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(kB2SlotReals / per, (uint64_t)L.n[0]));
}

}  // namespace

size_t b2_tile_bytes(const Lat& L, int is_f32) {
    const RectTiles rt = adj_tiles(L, is_f32);
    return (size_t)(16 * rect_cells(rt) / (uint32_t)L.n[0]) * adj_slab(L, rt) * (is_f32 ? 4 : 8);
}

hipError_t launch_b2_grad_tile(const Lat& L, const void* U, int is_f32, const void* zycopy, const void* Abuf, void* fpbuf,
                               void* grad, hipStream_t st) {
    if (!rect_fits(L) || !fits_buffer(L.V, is_f32)) return hipErrorInvalidValue;
    const RectTiles rt = adj_tiles(L, is_f32);
    const uint32_t S = adj_slab(L, rt), NT = (uint32_t)L.n[0];
    const Lat Lzy = zy_lattice(L);
    const double scale = 1.0 / (16.0 * (double)L.V);
    const uint32_t per = std::max({rt.p[0].tiles, rt.p[1].tiles, rt.p[2].tiles}) / NT;
    const uint32_t nxz = (uint32_t)((L.n[1] + 15) / 16) * (uint32_t)((L.n[3] + 15) / 16);
    hipError_t e = hipSuccess;
    with_view(L.V, U, is_f32, [&](auto f) {
        using F = decltype(f);
        using R = typename F::real;
        if constexpr (F::buffered) {
            const F fzy{(const R*)((uintptr_t)zycopy - (uintptr_t)18 * L.V * sizeof(R)), L.V};
            for (uint32_t t0 = 0; t0 < NT && e == hipSuccess; t0 += S) {
                const uint32_t ns = std::min(S, NT - t0);
                b2_tile_kernel<F, sizeof(R) == 4 ? 2 : 1>
                    <<<dim3(per * ns, 3), kW, 0, st>>>(L, f, Lzy, fzy, rt, t0, ns, (const R*)Abuf, (R*)fpbuf);
                b2_zy_gather_kernel<R><<<nxz * (uint32_t)L.n[2] * ns, 256, 0, st>>>(L, rt, t0, ns, (const R*)fpbuf, (R*)grad);
                b2_gather_kernel<R><<<dim3((ns * L.Vs + 255) / 256, 4), 256, 0, st>>>(L, rt, t0, ns, scale, (const R*)fpbuf,
                                                                                   (R*)grad);
                e = hipGetLastError();
            }
        }
    });
    return e;
}

}  // namespace flue
