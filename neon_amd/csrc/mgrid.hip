// mgrid.hip -- grid-refinement LBM (Neon's mGrid, depth 2 to 5, and the
// lbmMultiRes application's scheme with its BGK D3Q19 or KBC D3Q27
// collision) on a stack of block-sparse levels.
//
// Level 0 is the finest level (the domain); level l has voxels of edge 2^l,
// ceil(dim / 2^l) per axis, and a level-(l+1) voxel v covers the level-l
// voxels 2v + {0,1}^3.  Each level is a bGrid of 8^3 blocks (the library's
// builder: blocks ordered bz, by, bx, 27-entry connectivity) with AoSoA
// populations (b*Q + q)*512 + x + 8y + 64z (Q = 19 or 27), and a dense table from block
// coordinates to block index for the cross-level lookups.
//
// Everything that depends only on the geometry is resolved on the host when
// the cavity is set up: every bulk leaf voxel carries a 3-bit state per
// population (plain pull, bounce-back link, explosion link, coalescence
// link, no update), each fine-to-coarse accumulation is a gather list whose
// per-target order is the fine voxels' z, y, x order, and the coalescence
// weights are a field of every level above 0.  The kernels then do no
// searching.  One coarse step is the reference's recursion
//   step(l): collide l, store l -> l+1 | step(l-1) | stream l
//            | unless l is the top: the same once more
// (lbmMultiRes.h:141-263, baseline operation order with the fine store).
// Reference semantics restated (file:line in each kernel):
//   grid      libNeonDomain/src/domain/details/mGrid/mGrid.cpp:89-345, 466-555
//   set-up    apps/lbmMultiRes/lidDrivenCavity.h:8-78, init.h:8-86
//   collide   apps/lbmMultiRes/collide.h:8-149 (BGK), :148-284 (KBC)
//   lattice   apps/lbmMultiRes/lattice.h:14-106 (D3Q27), :108-173 (D3Q19)
//   store     apps/lbmMultiRes/store.h:98-163
//   stream    apps/lbmMultiRes/stream.h:170-225
//   helpers   apps/lbmMultiRes/util.h:19-45, mPartition_imp.h:155-235
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "block_common.hpp"

namespace nx {
namespace mres {
namespace {

// state byte of a voxel (host and device)
constexpr uint32_t kActive = 1u, kRefined = 2u;
constexpr int kClsShift = 2;
// per-population link states of a bulk leaf voxel, 3 bits each
constexpr uint64_t kPlain = 0, kWall = 1, kExpl = 2, kCoal = 3, kSkip = 4;
constexpr int kMaxDepth = 5;

__host__ __device__ inline int cls_bits(uint32_t st) { return (int)((st >> kClsShift) & 3u); }
__host__ __device__ inline bool bulk_leaf(uint32_t st)
{
    return (st & kActive) && !(st & kRefined) && cls_bits(st) == NX_CELL_BULK;
}

template <int S>
struct MS;  // storage of the refinement step: the reference's float / double fields
template <>
struct MS<NX_F64> {
    using T = double;
};
template <>
struct MS<NX_F32> {
    using T = float;
};

// ---- lattices ------------------------------------------------------------------

// D3Q27 of apps/lbmMultiRes/lattice.h:14-75 (z fastest, then y, then x, each
// over 0, -1, +1), the lattice of its default KBC collision
constexpr int K27X[27] = {0, 0, 0, 0, 0, 0, 0, 0, 0, -1, -1, -1, -1, -1, -1, -1, -1, -1, 1, 1, 1, 1, 1, 1, 1, 1, 1};
constexpr int K27Y[27] = {0, 0, 0, -1, -1, -1, 1, 1, 1, 0, 0, 0, -1, -1, -1, 1, 1, 1, 0, 0, 0, -1, -1, -1, 1, 1, 1};
constexpr int K27Z[27] = {0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1, 0, -1, 1};
constexpr int K27OPP[27] = {0,  2,  1,  6,  8,  7,  3,  5,  4,  18, 20, 19, 24, 26,
                            25, 21, 23, 22, 9,  11, 10, 15, 17, 16, 12, 14, 13};
__host__ __device__ constexpr double w27(int q)
{
    return (K27X[q] != 0) + (K27Y[q] != 0) + (K27Z[q] != 0) == 0   ? 8.0 / 27.0
           : (K27X[q] != 0) + (K27Y[q] != 0) + (K27Z[q] != 0) == 1 ? 2.0 / 27.0
           : (K27X[q] != 0) + (K27Y[q] != 0) + (K27Z[q] != 0) == 2 ? 1.0 / 54.0
                                                                    : 1.0 / 216.0;
}

// KBC D3Q27 collision (collide.h:148-284) with the reference's type
// promotions: the density and velocity sums over q in order (util.h:47-62),
// the double literals of the equilibrium, the shear split and gamma
// evaluated in binary64 and stored in T, tiny = 1e-7 in gamma's denominator.
// Two forms with the same results: kbc27_kept keeps the equilibrium and fneq
// of every population in arrays; kbc27_recomputed recomputes them in each of
// the collision's three passes -- moment flux, e0 / e1, output -- from copies
// of rho, u and usqr that the compiler may not look through, so only the 27
// populations stay live (occupancy).
//
// The pass is bound by vector instructions, so what cannot change a result is
// left out: terms times a zero velocity component or a zero shear part (0 x
// is +-0, and these sums are never -0; a non-finite x makes every output NaN
// either way), and the second half of each +-c pair's polynomial (c.u of the
// opposite is exactly -c.u).
constexpr int nonzero27(int q) { return (K27X[q] != 0) + (K27Y[q] != 0) + (K27Z[q] != 0); }

// c.v with c of population q: the reference's sum over x, y, z without its
// zero terms
template <typename T>
__device__ __forceinline__ T dot27(int q, T v0, T v1, T v2)
{
    T cu = 0;
    bool first = true;
    if (K27X[q]) cu = K27X[q] > 0 ? v0 : -v0, first = false;
    if (K27Y[q]) cu = first ? (K27Y[q] > 0 ? v1 : -v1) : (K27Y[q] > 0 ? cu + v1 : cu - v1), first = false;
    if (K27Z[q]) cu = first ? (K27Z[q] > 0 ? v2 : -v2) : (K27Z[q] > 0 ? cu + v2 : cu - v2);
    return cu;
}

template <typename T>
__device__ __forceinline__ T kbc27_feq(int q, T rho, T v0, T v1, T v2, T usqr)
{
    const T cu = (T)((double)dot27<T>(q, v0, v1, v2) * 3.0);
    return (T)((double)rho * w27(q) * (1. + (double)cu + 0.5 * (double)cu * (double)cu - (double)usqr));
}

// Six moments Pi: xx, xy, xz, yy, yz, zz
template <typename T>
__device__ __forceinline__ void kbc27_flux(int q, T fneq, T p[6])
{
    const int c[3] = {K27X[q], K27Y[q], K27Z[q]};
    int k = 0;
    for (int a = 0; a < 3; a++)
        for (int b = a; b < 3; b++, k++)
            if (c[a] * c[b] != 0) p[k] = c[a] * c[b] > 0 ? p[k] + fneq : p[k] - fneq;
}

template <typename T>
struct Shear27 {
    T face[3], xy, xz, yz;  // rho times the shear part of (x, 0, 0) .. and of (+, +)
    __device__ __forceinline__ Shear27(T rho, const T p[6])
    {
        const T Nxz = p[0] - p[5], Nyz = p[3] - p[5];
        face[0] = rho * (T)((2.0 * (double)Nxz - (double)Nyz) / 6.0);
        face[1] = rho * (T)((-(double)Nxz + 2.0 * (double)Nyz) / 6.0);
        face[2] = rho * (T)((double)(-Nxz - Nyz) / 6.0);
        xy = rho * (T)((double)p[1] / 4.0);
        xz = rho * (T)((double)p[2] / 4.0);
        yz = rho * (T)((double)p[4] / 4.0);
    }
    // populations with 1 or 2 non-zero components; the others have none
    __device__ __forceinline__ T at(int q) const
    {
        const int cx = K27X[q], cy = K27Y[q], cz = K27Z[q];
        if (nonzero27(q) == 1) return cx ? face[0] : (cy ? face[1] : face[2]);
        if (nonzero27(q) == 2)
            return !cz ? (cx * cy > 0 ? xy : -xy) : (!cy ? (cx * cz > 0 ? xz : -xz) : (cy * cz > 0 ? yz : -yz));
        return T(0);
    }
};

// Quotients by one binary32 divisor, correctly rounded, through a binary64
// reciprocal (v_rcp_f32 and one cubic step: within 2^-52) shared by them.  a /
// b of 24-bit values is never closer than 2^-49 to a rounding boundary, so
// rounding the binary64 product to binary32 is rounding the quotient; a
// division by itself is about twice the instructions.  |b| in [2^-100, 2^100];
// a quotient below the normal range may round to its neighbour.
struct Recip32 {
    double r;
    __device__ __forceinline__ explicit Recip32(float b)
    {
        const double d = (double)b, r0 = (double)__builtin_amdgcn_rcpf(b);
        const double e = __builtin_fma(-d, r0, 1.0);
        r = __builtin_fma(r0, __builtin_fma(e, e, e), r0);
    }
    __device__ __forceinline__ float operator()(float a) const { return (float)((double)a * r); }
};
__device__ __forceinline__ bool recip32_ok(float lo, float hi) { return lo >= 0x1p-100f && hi <= 0x1p100f; }

struct Relax {  // one level's relaxation: beta = omega / 2 in T, 1 / beta
    double omega, beta, inv_beta;
};

// binary32.  Measured (MI355X, 128^3 lid, coarse step): 457 us, with the
// divisions, zero terms and both halves of each pair evaluated 493 us.
__device__ __forceinline__ void kbc27_kept(const float f[27], const Relax& om, float out[27])
{
    using T = float;
    const double beta = om.beta, invBeta = om.inv_beta;
    const T tiny = (T)1e-7;
    T rho = 0;
#pragma unroll
    for (int q = 0; q < 27; q++) rho += f[q];
    T j0 = 0, j1 = 0, j2 = 0;
#pragma unroll
    for (int q = 0; q < 27; q++) {
        if (K27X[q]) j0 = K27X[q] > 0 ? j0 + f[q] : j0 - f[q];
        if (K27Y[q]) j1 = K27Y[q] > 0 ? j1 + f[q] : j1 - f[q];
        if (K27Z[q]) j2 = K27Z[q] > 0 ? j2 + f[q] : j2 - f[q];
    }
    T v0, v1, v2;
    if (recip32_ok(__builtin_fabsf(rho), __builtin_fabsf(rho))) {
        const Recip32 by(rho);
        v0 = by(j0), v1 = by(j1), v2 = by(j2);
    } else {
        v0 = j0 / rho, v1 = j1 / rho, v2 = j2 / rho;
    }
    const T usqr = (T)((3.0 / 2.0) * (double)(v0 * v0 + v1 * v1 + v2 * v2));
    const double us = (double)usqr;
    T feq[27], fneq[27];
    T p[6] = {0, 0, 0, 0, 0, 0};
    T lo, hi;
#pragma unroll
    for (int q = 0; q < 27; q++) {
        const int o = K27OPP[q];
        if (o < q) continue;
        const double rw = (double)rho * w27(q);
        if (o == q) {
            feq[q] = (T)(rw * (1. - us));
            lo = hi = __builtin_fabsf(feq[q]);
            continue;
        }
        const double cu = (double)(T)((double)dot27<T>(q, v0, v1, v2) * 3.0);
        const double sq = 0.5 * cu * cu;
        feq[q] = (T)(rw * (1. + cu + sq - us));
        feq[o] = (T)(rw * (1. - cu + sq - us));
        lo = __builtin_fminf(__builtin_fminf(lo, __builtin_fabsf(feq[q])), __builtin_fabsf(feq[o]));
        hi = __builtin_fmaxf(__builtin_fmaxf(hi, __builtin_fabsf(feq[q])), __builtin_fabsf(feq[o]));
    }
#pragma unroll
    for (int q = 0; q < 27; q++) {
        fneq[q] = f[q] - feq[q];
        kbc27_flux<T>(q, fneq[q], p);
    }
    const Shear27<T> sh(rho, p);
    T e0 = 0, e1 = 0;
    auto sums = [&](auto&& divisor) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 27; q++) {
            const auto by = divisor(feq[q]);
            const T dS = sh.at(q);
            const bool sheared = nonzero27(q) == 1 || nonzero27(q) == 2;
            const T dH = sheared ? fneq[q] - dS : fneq[q];
            if (sheared) e0 += by(dS * dH);
            e1 += by(dH * dH);
        }
    };
    if (recip32_ok(lo, hi)) {
        sums([](T b) { return Recip32(b); });
    } else {
        struct Div {
            T b;
            __device__ __forceinline__ T operator()(T a) const { return a / b; }
        };
        sums([](T b) { return Div{b}; });
    }
    const T gamma = (T)(invBeta - (2.0 - invBeta) * (double)e0 / (double)(tiny + e1));
#pragma unroll
    for (int q = 0; q < 27; q++) {
        const bool sheared = nonzero27(q) == 1 || nonzero27(q) == 2;
        const T dS = sh.at(q);
        const T dH = sheared ? fneq[q] - dS : fneq[q];
        const double g = (double)(gamma * dH);
        out[q] = (T)((double)f[q] - beta * (sheared ? 2.0 * (double)dS + g : g));
    }
}

__device__ __forceinline__ void kbc27_recomputed(const double f[27], const Relax& om, double out[27])
{
    using T = double;
    const T beta = om.beta, invBeta = om.inv_beta;
    const T tiny = (T)1e-7;
    T rho = 0;
#pragma unroll
    for (int q = 0; q < 27; q++) rho += f[q];
    T v0 = 0, v1 = 0, v2 = 0;
#pragma unroll
    for (int q = 0; q < 27; q++) {
        if (K27X[q]) v0 = K27X[q] > 0 ? v0 + f[q] : v0 - f[q];
        if (K27Y[q]) v1 = K27Y[q] > 0 ? v1 + f[q] : v1 - f[q];
        if (K27Z[q]) v2 = K27Z[q] > 0 ? v2 + f[q] : v2 - f[q];
    }
    v0 /= rho;
    v1 /= rho;
    v2 /= rho;
    const T usqr = (3.0 / 2.0) * (v0 * v0 + v1 * v1 + v2 * v2);
    T p[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 27; q++) kbc27_flux<T>(q, f[q] - kbc27_feq<T>(q, rho, v0, v1, v2, usqr), p);
    const Shear27<T> sh(rho, p);
    T e0 = 0, e1 = 0;
    {
        T r = rho, a = v0, b = v1, c = v2, us = usqr;
        nx_pin(r);
        nx_pin(a);
        nx_pin(b);
        nx_pin(c);
        nx_pin(us);
#pragma unroll
        for (int q = 0; q < 27; q++) {
            const T feq = kbc27_feq<T>(q, r, a, b, c, us);
            const bool sheared = nonzero27(q) == 1 || nonzero27(q) == 2;
            const T dS = sh.at(q);
            const T dH = sheared ? (f[q] - feq) - dS : f[q] - feq;
            if (sheared) e0 += (dS * dH / feq);
            e1 += (dH * dH / feq);
        }
    }
    const T gamma = invBeta - (2.0 - invBeta) * e0 / (tiny + e1);
    T r = rho, a = v0, b = v1, c = v2, us = usqr;
    nx_pin(r);
    nx_pin(a);
    nx_pin(b);
    nx_pin(c);
    nx_pin(us);
#pragma unroll
    for (int q = 0; q < 27; q++) {
        const T feq = kbc27_feq<T>(q, r, a, b, c, us);
        const bool sheared = nonzero27(q) == 1 || nonzero27(q) == 2;
        const T dS = sh.at(q);
        const T dH = sheared ? (f[q] - feq) - dS : f[q] - feq;
        out[q] = f[q] - beta * (sheared ? 2.0 * dS + gamma * dH : gamma * dH);
    }
}

// binary64: the recomputing form (127 instead of 221 VGPRs, 16% faster on
// the 240^3 grid); binary32: the form that keeps the values
__device__ __forceinline__ void kbc27(const double f[27], const Relax& om, double out[27]) { kbc27_recomputed(f, om, out); }
__device__ __forceinline__ void kbc27(const float f[27], const Relax& om, float out[27]) { kbc27_kept(f, om, out); }

// lattice traits: populations, velocity table, rest population, collision
struct L19 {
    static constexpr int Q = 19, REST = 9, W = 1;  // W: 64-bit link words per voxel
    static constexpr __host__ __device__ int cx(int q) { return CX[q]; }
    static constexpr __host__ __device__ int cy(int q) { return CY[q]; }
    static constexpr __host__ __device__ int cz(int q) { return CZ[q]; }
    static constexpr __host__ __device__ int opp(int q) { return OPP[q]; }
    static constexpr __host__ __device__ double w(int q) { return wq(q); }
    template <typename T>
    static __device__ __forceinline__ void collide(const T f[19], const Relax& om, T out[19])
    {
        bgk<T>(f, (T)om.omega, out);
    }
};
struct L27 {
    static constexpr int Q = 27, REST = 0, W = 2;
    static constexpr __host__ __device__ int cx(int q) { return K27X[q]; }
    static constexpr __host__ __device__ int cy(int q) { return K27Y[q]; }
    static constexpr __host__ __device__ int cz(int q) { return K27Z[q]; }
    static constexpr __host__ __device__ int opp(int q) { return K27OPP[q]; }
    static constexpr __host__ __device__ double w(int q) { return w27(q); }
    template <typename T>
    static __device__ __forceinline__ void collide(const T f[27], const Relax& om, T out[27])
    {
        kbc27(f, om, out);
    }
};

// link state of population q: 3 bits, 21 populations per 64-bit word
constexpr int kLinksPerWord = 21;

// ---- kernels ----------------------------------------------------------------

// collide.h:8-284: the lattice's collision on every bulk leaf voxel (fin ->
// fout, same voxel); a refined voxel (levels above 0) resets its fout, the
// accumulator of the fine store, to 0.
template <int S, class LT>
__global__ void __launch_bounds__(kBV)
    k_mr_collide(const typename MS<S>::T* __restrict__ fin, typename MS<S>::T* __restrict__ fout,
                 const uint32_t* __restrict__ state, Relax om)
{
    using T = typename MS<S>::T;
    constexpr int NQ = LT::Q;
    const uint32_t b = xcd_runs<4>(blockIdx.x, gridDim.x), v = threadIdx.x;
    const uint32_t st = state[(uint64_t)b * kBV + v];
    if (!(st & kActive) || cls_bits(st) != NX_CELL_BULK) return;
    const uint64_t own = (uint64_t)b * (NQ * kBV) + v;
    if (st & kRefined) {
#pragma unroll
        for (int q = 0; q < NQ; q++) __builtin_nontemporal_store(T(0), &fout[own + (uint64_t)q * kBV]);
        return;
    }
    T f[NQ], o[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) f[q] = fin[own + (uint64_t)q * kBV];
    LT::template collide<T>(f, om, o);
#pragma unroll
    for (int q = 0; q < NQ; q++) __builtin_nontemporal_store(o[q], &fout[own + (uint64_t)q * kBV]);
}

// store.h:98-163 as a gather: entry e adds its fine sources, in order, to
// the coarse accumulator target[e].
struct StoreArgs {
    void* coarse;
    const uint64_t* target;
    const uint32_t* first;
    const uint64_t* src;
    uint32_t n;
    uint32_t groups;  // workgroups of kBV entries that carry it, a multiple of the 8 XCDs
};

template <typename T>
__device__ __forceinline__ void store_entry(const T* __restrict__ fine, const StoreArgs& s, uint32_t e)
{
    if (e >= s.n) return;
    T* coarse = (T*)s.coarse;
    T acc = coarse[s.target[e]];
    for (uint32_t k = s.first[e]; k < s.first[e + 1]; k++) acc += fine[s.src[k]];
    coarse[s.target[e]] = acc;
}

template <int S>
__global__ void __launch_bounds__(kBV) k_mr_store(const typename MS<S>::T* __restrict__ fine, StoreArgs s)
{
    store_entry(fine, s, blockIdx.x * kBV + threadIdx.x);
}

struct UpLevel {  // the next coarser level, seen from this one (explosion)
    const void* fout;
    const uint32_t* table;
    int32_t nb[3];
};

// k_mr_stream's shape per lattice and type, by what it measured (coarse step
// of the 128^3 three-level lid): the wavefronts per SIMD its registers must
// allow (workgroups are 2 per SIMD each), how many links one batch of fix-up
// loads covers, and whether the neighbour offsets are formed again for the
// fix-ups (fewer registers) or kept.  KBC binary32 keeps them (414 us against
// 438 formed again; batches of 1, 3, 9: 470, 414, 431 us; the 64-bit offsets
// would spill); BGK binary32 forms
// them again (219 against 246 us, 46-74 against 85-108 registers).
template <int S, class LT>
struct StreamShape {
    static constexpr bool wide = LT::Q == 27, f64 = S == NX_F64;
    static constexpr int waves = wide || f64 ? 4 : 6;
    static constexpr int batch = wide ? 3 : f64 ? 5 : 10;
    static constexpr bool again = f64 || !wide;
};

// stream.h:170-225 (stream fused with coalescence and explosion), pull, for
// the bulk leaf voxels of one level.  The plain pull of all populations is
// issued with the state and link words, before either is known (one memory
// round trip; a slot that is no bulk leaf reads values it does not use); then
// voxels with another link state fix those links up: bounce-back (own
// opposite + the wall's opposite), explosion (the coarse post-collision
// population of the uncle, the next level's voxel holding the upstream
// position), coalescence (the refined upstream voxel's accumulated fine
// populations times its weight); links in state "none" keep the value in
// `out`.  The fix-ups' loads go out in batches of populations: on
// refined grids most wavefronts hold a wall or an interface, and a wait per
// link made the fix-ups the longest part of the pass.
// COLLIDE: the pulled populations are collided at once with omega and the
// result written to `out`, and refined voxels reset their accumulator in
// `out` -- stream followed by the next collide of the same level
// (collide.h:8-284) in one pass; the results are those of the two kernels in
// sequence, bit for bit.  KEEP = false: the level has no link in state
// "none" (checked on the host), every population is stored.  `links` holds
// LT::W words per voxel slot, word k at k * n_slots.
// The first st.groups workgroups carry the level's fine-to-coarse store (a
// launch of its own costs more than its work): it reads this level's
// post-collision field as the stream does and adds to refined voxels of the
// next level, which the explosion never reads (checked on the host).
// Measured (MI355X, coarse step of the 128^3 three-level lid; before with the
// present collision): KBC f32 414 us (457), f64 680 (737), BGK f32 219 (246),
// f64 371 (393); of the 48^3 lid 105 (144) and 67 us (90) in binary32.
template <int S, class LT, bool COLLIDE, bool KEEP, typename O>
__global__ void __launch_bounds__(kBV, (StreamShape<S, LT>::waves))
    k_mr_stream(const typename MS<S>::T* __restrict__ fout, typename MS<S>::T* __restrict__ out,
                const uint32_t* __restrict__ state, const uint64_t* __restrict__ links, uint64_t n_slots,
                const uint32_t* __restrict__ conn, const int32_t* __restrict__ origins,
                const float* __restrict__ ss, UpLevel up, Relax om, StoreArgs sa)
{
    using T = typename MS<S>::T;
    constexpr int NQ = LT::Q;
    if (blockIdx.x < sa.groups) {
        store_entry(fout, sa, blockIdx.x * kBV + threadIdx.x);
        return;
    }
    // runs of 4 blocks per XCD (240^3 lid: BGK f32 974 us a coarse step, f64
    // 1764, KBC f32 1845; one range per XCD 1043, 1830, 1896)
    const uint32_t b = xcd_runs<4>(blockIdx.x - sa.groups, gridDim.x - sa.groups), v = threadIdx.x;
    const Rows<O> rows = Rows<O>::template of<T, NQ>(load_conn(conn, b), b);
    const int x = (int)(v & 7u), y = (int)((v >> 3) & 7u), z = (int)(v >> 6);
    const O own = rows.c[13] + (O)(v * sizeof(T));
    auto ld = [](const void* p, O at) __attribute__((always_inline)) { return *(const T*)((const char*)p + at); };
    auto st = [](void* p, O at, T val) __attribute__((always_inline)) {
        __builtin_nontemporal_store(val, (T*)((char*)p + at));
    };
    uint32_t sv = state[(uint64_t)b * kBV + v];
    uint64_t lk[LT::W];
#pragma unroll
    for (int k = 0; k < LT::W; k++) lk[k] = links[(uint64_t)k * n_slots + (uint64_t)b * kBV + v];
    T f[NQ];
    for_q(std::make_integer_sequence<int, NQ>{}, [&](auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
        f[q] = ld(fout + q * kBV, rows.template at<T, -LT::cx(q), -LT::cy(q), -LT::cz(q)>(x, y, z));
    });
#pragma unroll
    for (int q = 0; q < NQ; q++) nx_pin(f[q]);
    nx_pin(sv);
#pragma unroll
    for (int k = 0; k < LT::W; k++) nx_pin(lk[k]);
    if ((sv & kActive) && (sv & kRefined) && cls_bits(sv) == NX_CELL_BULK) {
        // a refined voxel: with COLLIDE the collide's reset of its
        // accumulator (collide.h:131-141); otherwise its fin, which the
        // reference never writes after the set-up's 0, back to 0 (a fused
        // pass earlier in the call left an accumulator in this buffer)
#pragma unroll
        for (int q = 0; q < NQ; q++) st(out + q * kBV, own, T(0));
        return;
    }
    if (!bulk_leaf(sv)) return;
    uint32_t keep = 0;  // links whose value stays as it is in `out`
    // (opaque copies: the neighbour offsets are formed again where a link
    // needs them instead of staying in registers across the pass)
    int xl = x, yl = y, zl = z;
    if constexpr (StreamShape<S, LT>::again || sizeof(O) == 8) {
        nx_pin(xl);
        nx_pin(yl);
        nx_pin(zl);
    }
    constexpr int kBatch = StreamShape<S, LT>::batch;
    for_q(std::make_integer_sequence<int, (NQ + kBatch - 1) / kBatch>{}, [&](auto gc) __attribute__((always_inline)) {
        constexpr int q0 = decltype(gc)::value * kBatch, q1 = q0 + kBatch < NQ ? q0 + kBatch : NQ;
        using Batch = std::make_integer_sequence<int, q1 - q0>;
        uint32_t kind[kBatch];
        uint32_t any = 0;
        bool expl = false;
        for_q(Batch{}, [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, q = q0 + i;
            kind[i] = (uint32_t)((lk[q / kLinksPerWord] >> (3 * (q % kLinksPerWord))) & 7u);
            any |= kind[i];
            expl |= kind[i] == (uint32_t)kExpl;
        });
        if (!__any(any != 0)) return;
        uint32_t tb[kBatch], slot[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; i++) tb[i] = kInvalidBlock;
        if (__any(expl)) {
            for_q(Batch{}, [&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, q = q0 + i;
                if (kind[i] != (uint32_t)kExpl) return;
                const int ux = (origins[3 * (uint64_t)b] + xl - LT::cx(q)) >> 1;
                const int uy = (origins[3 * (uint64_t)b + 1] + yl - LT::cy(q)) >> 1;
                const int uz = (origins[3 * (uint64_t)b + 2] + zl - LT::cz(q)) >> 1;
                const int bx = ux >> 3, by = uy >> 3, bz = uz >> 3;
                slot[i] = (uint32_t)((ux & 7) + 8 * (uy & 7) + 64 * (uz & 7));
                if (up.table && !(bx < 0 || by < 0 || bz < 0 || bx >= up.nb[0] || by >= up.nb[1] || bz >= up.nb[2]))
                    tb[i] = up.table[((uint64_t)bz * up.nb[1] + by) * up.nb[0] + bx];
            });
#pragma unroll
            for (int i = 0; i < kBatch; i++) nx_pin(tb[i]);
        }
        T a[kBatch], w[kBatch];
        for_q(Batch{}, [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, q = q0 + i, o = LT::opp(q);
            a[i] = w[i] = T(0);
            if (kind[i] == (uint32_t)kPlain) return;
            const O nb = rows.template at<T, -LT::cx(q), -LT::cy(q), -LT::cz(q)>(xl, yl, zl);
            if (kind[i] == (uint32_t)kWall) {
                a[i] = ld(fout + o * kBV, own);
                w[i] = ld(fout + o * kBV, nb);
            } else if (kind[i] == (uint32_t)kCoal) {
                w[i] = (T)ss[(uint64_t)(nb / (O)sizeof(T)) + q * kBV];
            } else if (tb[i] != kInvalidBlock) {
                w[i] = ((const T*)up.fout)[((uint64_t)tb[i] * NQ + q) * kBV + slot[i]];
            } else {
                keep |= 1u << q;
                w[i] = ld(out + q * kBV, own);
            }
        });
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            nx_pin(a[i]);
            nx_pin(w[i]);
        }
        for_q(Batch{}, [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, q = q0 + i;
            const T one = kind[i] == (uint32_t)kWall ? a[i] + w[i] : w[i];
            const T scaled = kind[i] == (uint32_t)kCoal ? f[q] * w[i] : f[q];
            f[q] = kind[i] == (uint32_t)kPlain || kind[i] == (uint32_t)kCoal ? scaled : one;
        });
    });
    if constexpr (COLLIDE) {
        T o[NQ];
        LT::template collide<T>(f, om, o);
#pragma unroll
        for (int q = 0; q < NQ; q++) st(out + q * kBV, own, o[q]);
    } else if constexpr (KEEP) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
            if (!((keep >> q) & 1u)) st(out + q * kBV, own, f[q]);
    } else {
#pragma unroll
        for (int q = 0; q < NQ; q++) st(out + q * kBV, own, f[q]);
    }
}

// Elements [e0, e0 + n) of a level's dense array [q][z][y][x] (0 in inactive
// voxels), for the read-back: consecutive lanes read 8-voxel rows of a block.
template <typename T>
__global__ void __launch_bounds__(256)
    k_mr_dense(const T* __restrict__ pop, const uint32_t* __restrict__ state, const uint32_t* __restrict__ table,
               int X, int Y, uint64_t nvox, int nbx, int nby, int nq, uint64_t e0, uint32_t n, T* __restrict__ out)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint64_t e = e0 + i;
    const uint32_t q = (uint32_t)(e / nvox);
    const uint64_t v = e - q * nvox, row = v / (uint32_t)X;
    const int x = (int)(v - row * (uint32_t)X), y = (int)(row % (uint32_t)Y), z = (int)(row / (uint32_t)Y);
    const uint32_t b = table[((uint64_t)(z >> 3) * nby + (y >> 3)) * nbx + (x >> 3)];
    const uint32_t s = (uint32_t)((x & 7) + 8 * (y & 7) + 64 * (z & 7));
    T val = T(0);
    if (b != kInvalidBlock && (state[(uint64_t)b * kBV + s] & kActive)) val = pop[((uint64_t)b * nq + q) * kBV + s];
    out[i] = val;
}

// ---- host structures ------------------------------------------------------------

struct Level {
    int32_t dim[3] = {0, 0, 0};
    int32_t nb[3] = {0, 0, 0};
    uint32_t n_blocks = 0;
    std::vector<int32_t> origins;
    std::vector<uint32_t> masks, conn, table;
    std::vector<uint8_t> st;  // dense state byte per voxel
    uint32_t* d_state = nullptr;
    uint64_t* d_links = nullptr;
    uint32_t* d_conn = nullptr;
    int32_t* d_origins = nullptr;
    uint32_t* d_table = nullptr;
    float* d_ss = nullptr;  // coalescence weights (levels above 0)
    void* fin = nullptr;
    void* fout = nullptr;
    bool keep = true;      // the level has links in state "none"
    bool separate = false; // an explosion link reads a refined voxel or a store adds to a leaf: the store
                           // needs its own launch
    int nq = 19;       // populations per voxel
    // active voxels as runs (first, one past the last) of the dense order
    std::vector<std::pair<size_t, size_t>> runs;

    size_t nvox() const { return (size_t)dim[0] * dim[1] * dim[2]; }
    size_t lin(int x, int y, int z) const { return (size_t)x + (size_t)dim[0] * ((size_t)y + (size_t)dim[1] * z); }
    bool inside(int x, int y, int z) const
    {
        return x >= 0 && y >= 0 && z >= 0 && x < dim[0] && y < dim[1] && z < dim[2];
    }
    bool active(int x, int y, int z) const { return inside(x, y, z) && (st[lin(x, y, z)] & kActive); }
    // AoSoA slot (block * 512 + in-block index) of an active voxel, or -1
    int64_t slot(int x, int y, int z) const
    {
        if (!active(x, y, z)) return -1;
        const uint32_t b = table[((size_t)(z >> 3) * nb[1] + (y >> 3)) * nb[0] + (x >> 3)];
        return (int64_t)b * kBV + ((x & 7) + 8 * (y & 7) + 64 * (z & 7));
    }
    // population element of an active voxel's slot
    uint64_t elem(int64_t slot, int q) const { return ((uint64_t)(slot / kBV) * nq + q) * kBV + slot % kBV; }
    size_t slots() const { return (size_t)kBV * n_blocks; }
};

// the lattice on the host: velocities, opposites, weights, link words
struct HostLat {
    int Q = 19, rest = 9, W = 1;
    int c[27][3] = {};
    int opp[27] = {};
    double w[27] = {};
};

template <class LT>
HostLat host_lat_of()
{
    HostLat h;
    h.Q = LT::Q;
    h.rest = LT::REST;
    h.W = LT::W;
    for (int q = 0; q < LT::Q; q++) {
        h.c[q][0] = LT::cx(q);
        h.c[q][1] = LT::cy(q);
        h.c[q][2] = LT::cz(q);
        h.opp[q] = LT::opp(q);
        h.w[q] = LT::w(q);
    }
    return h;
}

struct Store {  // fine-to-coarse gather list of one level pair (l -> l + 1)
    uint32_t n = 0;
    uint64_t n_src = 0;
    uint64_t* d_target = nullptr;
    uint32_t* d_first = nullptr;
    uint64_t* d_src = nullptr;
};

}  // namespace
}  // namespace mres
}  // namespace nx

struct nx_mgrid_s {
    int storage = NX_F64;
    int lattice = NX_MGRID_BGK19;
    nx::mres::HostLat lat;
    int depth = 2;
    nx::mres::Level L[nx::mres::kMaxDepth];
    nx::mres::Store store[nx::mres::kMaxDepth];
    bool ready = false;
    int device = 0;  // the grid's memory
    // read-back: worker w's pinned and device chunk and its stream, made at the
    // first large read-back and given back with the grid
    std::mutex read_mu;
    struct Reader {
        void* host = nullptr;
        void* dev = nullptr;
        hipStream_t st = nullptr;
    } reader[8];
};

using namespace nx;
using namespace nx::mres;

namespace {

int upload(void** dst, const void* src, size_t bytes)
{
    if (*dst) {
        NX_CHECK_HIP(hipFree(*dst));
        *dst = nullptr;
    }
    NX_CHECK_HIP(hipMalloc(dst, std::max<size_t>(bytes, 8)));
    if (bytes) NX_CHECK_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return NX_OK;
}

// isRefined (mGrid.cpp:167-199): a child of level-l voxel (x, y, z) is
// active on level l - 1 (the voxel itself need not be)
bool any_child(const Level& fine, int x, int y, int z)
{
    for (int k = 0; k < 8; k++)
        if (fine.active(2 * x + (k & 1), 2 * y + ((k >> 1) & 1), 2 * z + (k >> 2))) return true;
    return false;
}

// The mGrid constructor (mGrid.cpp:89-345): activation level by level in
// 2^3 groups, each active group activating its parent; overlap culling from
// the coarsest level down (a refined voxel whose in-domain neighbours are
// all refined goes; level l - 1 is still unculled when level l is visited);
// the strong-balance pass; then the refined flags from the final masks
// (:466-555).  Returns the number of voxels the strong-balance pass added.
uint64_t activate(const int32_t dim[3], int depth, const uint8_t* const* lams, Level* L)
{
    for (int a = 0; a < 3; a++) L[0].dim[a] = dim[a];
    for (int l = 1; l < depth; l++)
        for (int a = 0; a < 3; a++) L[l].dim[a] = (L[l - 1].dim[a] + 1) / 2;
    for (int l = 0; l < depth; l++) L[l].st.assign(L[l].nvox(), 0);
    for (int l = 0; l < depth; l++) {
        Level& lv = L[l];
        const uint8_t* lam = lams[l];
        for (int gz = 0; gz < (lv.dim[2] + 1) / 2; gz++)
            for (int gy = 0; gy < (lv.dim[1] + 1) / 2; gy++)
                for (int gx = 0; gx < (lv.dim[0] + 1) / 2; gx++) {
                    bool any = false;
                    for (int k = 0; k < 8; k++) {
                        const int x = 2 * gx + (k & 1), y = 2 * gy + ((k >> 1) & 1), z = 2 * gz + (k >> 2);
                        if (lv.inside(x, y, z) && (lv.st[lv.lin(x, y, z)] || lam[lv.lin(x, y, z)])) any = true;
                    }
                    if (!any) continue;
                    for (int k = 0; k < 8; k++) {
                        const int x = 2 * gx + (k & 1), y = 2 * gy + ((k >> 1) & 1), z = 2 * gz + (k >> 2);
                        if (lv.inside(x, y, z)) lv.st[lv.lin(x, y, z)] = (uint8_t)kActive;
                    }
                    if (l + 1 < depth) L[l + 1].st[L[l + 1].lin(gx, gy, gz)] = (uint8_t)kActive;
                }
    }
    for (int l = depth - 1; l > 0; l--) {
        Level& c = L[l];
        std::vector<uint8_t> refined(c.nvox(), 0);
        for (int z = 0; z < c.dim[2]; z++)
            for (int y = 0; y < c.dim[1]; y++)
                for (int x = 0; x < c.dim[0]; x++) refined[c.lin(x, y, z)] = any_child(L[l - 1], x, y, z);
        for (int z = 0; z < c.dim[2]; z++)
            for (int y = 0; y < c.dim[1]; y++)
                for (int x = 0; x < c.dim[0]; x++) {
                    const size_t i = c.lin(x, y, z);
                    if (!c.st[i] || !refined[i]) continue;
                    bool all = true;
                    for (int d = 0; d < 27 && all; d++) {
                        if (d == 13) continue;
                        const int nx_ = x + d % 3 - 1, ny = y + (d / 3) % 3 - 1, nz = z + d / 9 - 1;
                        if (c.inside(nx_, ny, nz) && !refined[c.lin(nx_, ny, nz)]) all = false;
                    }
                    if (all) c.st[i] = 0;
                }
    }
    // strong balance: the finest active voxel covering each in-domain
    // neighbour position of an active voxel of level l lies on level l or
    // l + 1; found on l_n >= l + 2, the voxel of level l_n - 1 covering it
    // is activated alone and the search continues upwards; passes repeat
    // until one activates nothing and see their own activations
    uint64_t added = 0;
    for (bool again = true; again;) {
        again = false;
        for (int l = 0; l < depth; l++) {
            const Level& lv = L[l];
            for (int bz = 0; bz < (lv.dim[2] + 1) / 2; bz++)
                for (int by = 0; by < (lv.dim[1] + 1) / 2; by++)
                    for (int bx = 0; bx < (lv.dim[0] + 1) / 2; bx++)
                        for (int k8 = 0; k8 < 8; k8++) {
                            const int x = 2 * bx + (k8 & 1), y = 2 * by + ((k8 >> 1) & 1), z = 2 * bz + (k8 >> 2);
                            if (!lv.active(x, y, z)) continue;
                            for (int d = 0; d < 27; d++) {
                                if (d == 13) continue;
                                int p[3] = {x + d % 3 - 1, y + (d / 3) % 3 - 1, z + d / 9 - 1};
                                if (!lv.inside(p[0], p[1], p[2])) continue;
                                int prev[3] = {0, 0, 0};
                                for (int ln = l; ln < depth; ln++) {
                                    if (L[ln].active(p[0], p[1], p[2])) {
                                        if (ln <= l + 1) break;
                                        uint8_t& s = L[ln - 1].st[L[ln - 1].lin(prev[0], prev[1], prev[2])];
                                        added += (s & kActive) ? 0 : 1;
                                        s = (uint8_t)kActive;
                                        again = true;
                                    }
                                    for (int a = 0; a < 3; a++) {
                                        prev[a] = p[a];
                                        p[a] >>= 1;
                                    }
                                }
                            }
                        }
        }
    }
    for (int l = 1; l < depth; l++) {
        Level& c = L[l];
        for (int z = 0; z < c.dim[2]; z++)
            for (int y = 0; y < c.dim[1]; y++)
                for (int x = 0; x < c.dim[0]; x++) {
                    uint8_t& s = c.st[c.lin(x, y, z)];
                    if ((s & kActive) && any_child(L[l - 1], x, y, z)) s |= (uint8_t)kRefined;
                }
    }
    return added;
}

int build_level(Level& lv)
{
    std::vector<uint8_t> act(lv.nvox());
    for (size_t i = 0; i < act.size(); i++) act[i] = lv.st[i] & kActive;
    nx_bgrid g = nullptr;
    if (int e = nx_bgrid_create(lv.dim, act.data(), 0, &g)) return e;
    uint64_t n_act = 0;
    nx_bgrid_info(g, &lv.n_blocks, &n_act);
    lv.origins.resize(3 * (size_t)lv.n_blocks);
    lv.masks.resize(16 * (size_t)lv.n_blocks);
    lv.conn.resize(27 * (size_t)lv.n_blocks);
    nx_bgrid_tables(g, lv.origins.data(), lv.masks.data(), lv.conn.data());
    nx_bgrid_destroy(g);
    for (int a = 0; a < 3; a++) lv.nb[a] = (lv.dim[a] + 7) / 8;
    lv.table.assign((size_t)lv.nb[0] * lv.nb[1] * lv.nb[2], kInvalidBlock);
    for (uint32_t b = 0; b < lv.n_blocks; b++)
        lv.table[((size_t)(lv.origins[3 * b + 2] >> 3) * lv.nb[1] + (lv.origins[3 * b + 1] >> 3)) * lv.nb[0] +
                 (lv.origins[3 * b] >> 3)] = b;
    return NX_OK;
}

// uncleOffset (util.h:19-37): offset, from the parent of x, of the parent of x + d
inline int uoff(int x, int d)
{
    const int s = (x & 1) + d;
    return s <= 0 ? s : s - 1;
}

// The class of every leaf (cls[l] per level-l voxel; nullptr: the lid-driven
// cavity of lidDrivenCavity.h:8-78, leaf voxels of level 0 on the domain
// faces bounce-back, those with y = Y-1 the lid) and its populations: w_q
// (bulk), 0 (bounce-back), -6 w_q (c_q . uw) for moving-wall cells (the lid,
// or the inlet of flowOverShape.h:62-104), evaluated as the reference does in
// T with binary64 constants.
template <typename T>
void fill_cells(nx_mgrid_s& g, const uint8_t* const* cls_in, const double uw[3], std::vector<T>* pop)
{
    const HostLat& L = g.lat;
    for (int l = 0; l < g.depth; l++) {
        Level& lv = g.L[l];
        pop[l].assign((size_t)L.Q * kBV * lv.n_blocks, T(0));
        for (int z = 0; z < lv.dim[2]; z++)
            for (int y = 0; y < lv.dim[1]; y++)
                for (int x = 0; x < lv.dim[0]; x++) {
                    const size_t i = lv.lin(x, y, z);
                    if (!(lv.st[i] & kActive)) continue;
                    int cls = NX_CELL_BULK;
                    const int64_t s = lv.slot(x, y, z);
                    if (!(lv.st[i] & kRefined)) {
                        if (cls_in)
                            cls = cls_in[l][i];
                        else if (l == 0 && (x == 0 || y == 0 || z == 0 || x == lv.dim[0] - 1 ||
                                            y == lv.dim[1] - 1 || z == lv.dim[2] - 1))
                            cls = y == lv.dim[1] - 1 ? NX_CELL_MOVINGWALL : NX_CELL_BOUNCEBACK;
                        for (int q = 0; q < L.Q; q++) {
                            T p = (T)L.w[q];
                            if (cls != NX_CELL_BULK) p = 0;
                            if (cls == NX_CELL_MOVINGWALL) {
                                p = (T)((double)p + (double)L.c[q][0] * uw[0]);
                                p = (T)((double)p + (double)L.c[q][1] * uw[1]);
                                p = (T)((double)p + (double)L.c[q][2] * uw[2]);
                                p = (T)((double)p * (-6. * L.w[q]));
                            }
                            pop[l][lv.elem(s, q)] = p;
                        }
                    }
                    lv.st[i] = (uint8_t)((lv.st[i] & (kActive | kRefined)) | (cls << kClsShift));
                }
    }
}

// hasParent (mPartition_imp.h:172-208): the memory block (8^3) of level
// l + 1 holding the parent of level-l voxel (x, y, z) exists
bool has_parent(const nx_mgrid_s& g, int l, int x, int y, int z)
{
    if (l + 1 >= g.depth) return false;
    const Level& c = g.L[l + 1];
    const int bx = (x >> 1) >> 3, by = (y >> 1) >> 3, bz = (z >> 1) >> 3;
    if (bx >= c.nb[0] || by >= c.nb[1] || bz >= c.nb[2]) return false;
    return c.table[((size_t)bz * c.nb[1] + by) * c.nb[0] + bx] != kInvalidBlock;
}

// Link states of every bulk leaf voxel of level l (stream.h:170-225 decided
// per link), 3 bits per population, W words per voxel slot (word k at
// k * slots); returns the number of links in state "none".
uint64_t links_of(const nx_mgrid_s& g, int l, std::vector<uint64_t>& out, bool& refined_uncle)
{
    uint64_t n_skip = 0;
    refined_uncle = false;
    const Level& lv = g.L[l];
    const HostLat& L = g.lat;
    out.assign((size_t)L.W * lv.slots(), 0);
    for (int z = 0; z < lv.dim[2]; z++)
        for (int y = 0; y < lv.dim[1]; y++)
            for (int x = 0; x < lv.dim[0]; x++) {
                const uint8_t st = lv.st[lv.lin(x, y, z)];
                if (!bulk_leaf(st)) continue;
                const bool parent = has_parent(g, l, x, y, z);
                uint64_t lk[2] = {0, 0};
                for (int q = 0; q < L.Q; q++) {
                    if (q == L.rest) continue;  // own population: plain
                    const int nx_ = x - L.c[q][0], ny = y - L.c[q][1], nz = z - L.c[q][2];
                    uint64_t kind = kSkip;
                    if (lv.active(nx_, ny, nz)) {
                        const uint8_t ns = lv.st[lv.lin(nx_, ny, nz)];
                        if (ns & kRefined)
                            kind = kCoal;
                        else
                            kind = cls_bits(ns) == NX_CELL_BULK ? kPlain : kWall;
                    } else if (parent) {
                        const Level& c = g.L[l + 1];
                        const int ux = (x >> 1) + uoff(x, -L.c[q][0]), uy = (y >> 1) + uoff(y, -L.c[q][1]),
                                  uz = (z >> 1) + uoff(z, -L.c[q][2]);
                        if (c.active(ux, uy, uz)) {
                            kind = kExpl;
                            refined_uncle = refined_uncle || (c.st[c.lin(ux, uy, uz)] & kRefined);
                        }
                    }
                    lk[q / kLinksPerWord] |= kind << (3 * (q % kLinksPerWord));
                    n_skip += kind == kSkip;
                }
                for (int k = 0; k < L.W; k++) out[(size_t)k * lv.slots() + lv.slot(x, y, z)] = lk[k];
            }
    return n_skip;
}

int check_level(const nx_mgrid_s* g, int32_t level)
{
    if (!g) return set_error(NX_ERR_INVALID, "null mgrid");
    if (level < 0 || level >= g->depth)
        return set_error(NX_ERR_INVALID, "mgrid: level " + std::to_string(level) + " outside [0, " +
                                             std::to_string(g->depth) + ")");
    return NX_OK;
}

}  // namespace

extern "C" int nx_mgrid_create_levels(const int32_t dim[3], int32_t depth, const uint8_t* const* lams,
                                      int32_t storage, int32_t lattice, nx_mgrid* out)
{
    if (!dim || !lams || !out) return set_error(NX_ERR_INVALID, "nx_mgrid_create_levels: null argument");
    if (depth < 2 || depth > kMaxDepth)
        return set_error(NX_ERR_INVALID, "nx_mgrid_create_levels: depth in [2, " + std::to_string(kMaxDepth) + "]");
    for (int l = 0; l < depth; l++)
        if (!lams[l]) return set_error(NX_ERR_INVALID, "nx_mgrid_create_levels: null lambda array");
    for (int a = 0; a < 3; a++)
        if (dim[a] < 2 || dim[a] > (1 << 14))
            return set_error(NX_ERR_INVALID, "nx_mgrid_create_levels: dimensions in [2, 16384]");
    if (storage != NX_F64 && storage != NX_F32)
        return set_error(NX_ERR_UNSUPPORTED, "nx_mgrid_create: storage NX_F64 or NX_F32 (the reference's types)");
    if (lattice != NX_MGRID_BGK19 && lattice != NX_MGRID_KBC27)
        return set_error(NX_ERR_INVALID, "nx_mgrid_create_levels: lattice NX_MGRID_BGK19 or NX_MGRID_KBC27");
    auto* g = new nx_mgrid_s;
    g->storage = storage;
    g->lattice = lattice;
    g->lat = lattice == NX_MGRID_KBC27 ? host_lat_of<L27>() : host_lat_of<L19>();
    g->depth = depth;
    for (int l = 0; l < depth; l++) g->L[l].nq = g->lat.Q;
    activate(dim, depth, lams, g->L);
    for (int l = 0; l < depth; l++)
        if (int e = build_level(g->L[l])) {
            nx_mgrid_destroy(g);
            return e;
        }
    *out = g;
    return NX_OK;
}

extern "C" int nx_mgrid_create(const int32_t dim[3], const uint8_t* lam0, const uint8_t* lam1, int32_t storage,
                               nx_mgrid* out)
{
    if (!lam0 || !lam1) return set_error(NX_ERR_INVALID, "nx_mgrid_create: null argument");
    const uint8_t* lams[2] = {lam0, lam1};
    return nx_mgrid_create_levels(dim, 2, lams, storage, NX_MGRID_BGK19, out);
}

extern "C" int nx_mgrid_depth(nx_mgrid g, int32_t* depth, int32_t* dims)
{
    if (!g) return set_error(NX_ERR_INVALID, "null mgrid");
    if (depth) *depth = g->depth;
    if (dims)
        for (int l = 0; l < g->depth; l++)
            for (int a = 0; a < 3; a++) dims[3 * l + a] = g->L[l].dim[a];
    return NX_OK;
}

extern "C" int nx_mgrid_populations(nx_mgrid g, int32_t* q)
{
    if (!g || !q) return set_error(NX_ERR_INVALID, "nx_mgrid_populations: null argument");
    *q = g->lat.Q;
    return NX_OK;
}

extern "C" int nx_mgrid_info(nx_mgrid g, uint32_t* n_blocks, uint64_t* n_active, uint64_t* n_leaf,
                             uint64_t* n_store, int32_t* fine_fused)
{
    if (!g) return set_error(NX_ERR_INVALID, "null mgrid");
    if (fine_fused) {  // bit l: level l's stream runs fused with its next collide
        *fine_fused = 0;
        for (int l = 0; l < g->depth; l++)
            if (g->ready && !g->L[l].keep) *fine_fused |= 1 << l;
    }
    uint64_t ns = 0;
    for (int l = 0; l < g->depth; l++) {
        uint64_t a = 0, lf = 0;
        for (uint8_t s : g->L[l].st) {
            a += (s & kActive) ? 1 : 0;
            lf += ((s & kActive) && !(s & kRefined)) ? 1 : 0;
        }
        if (n_blocks) n_blocks[l] = g->L[l].n_blocks;
        if (n_active) n_active[l] = a;
        if (n_leaf) n_leaf[l] = lf;
        ns += g->store[l].n_src;
    }
    if (n_store) *n_store = ns;
    return NX_OK;
}

extern "C" int nx_mgrid_state_level(nx_mgrid g, int32_t level, uint8_t* st)
{
    if (int e = check_level(g, level)) return e;
    if (!st) return set_error(NX_ERR_INVALID, "nx_mgrid_state_level: null output");
    std::copy(g->L[level].st.begin(), g->L[level].st.end(), st);
    return NX_OK;
}

extern "C" int nx_mgrid_state(nx_mgrid g, uint8_t* st0, uint8_t* st1)
{
    if (!g) return set_error(NX_ERR_INVALID, "null mgrid");
    if (st0) std::copy(g->L[0].st.begin(), g->L[0].st.end(), st0);
    if (st1) std::copy(g->L[1].st.begin(), g->L[1].st.end(), st1);
    return NX_OK;
}

namespace {

int setup_cells(nx_mgrid g, const uint8_t* const* cls, const double uw[3])
{
    NX_CHECK_HIP(hipGetDevice(&g->device));
    const int D = g->depth;
    const size_t es = g->storage == NX_F64 ? 8 : 4;
    // populations
    std::vector<double> p64[kMaxDepth];
    std::vector<float> p32[kMaxDepth];
    if (g->storage == NX_F64)
        fill_cells<double>(*g, cls, uw, p64);
    else
        fill_cells<float>(*g, cls, uw, p32);
    for (int l = 0; l < D; l++) {
        Level& lv = g->L[l];
        const size_t elems = (size_t)g->lat.Q * kBV * lv.n_blocks;
        if (int e = upload((void**)&lv.d_conn, lv.conn.data(), lv.conn.size() * 4)) return e;
        if (int e = upload((void**)&lv.d_origins, lv.origins.data(), lv.origins.size() * 4)) return e;
        if (int e = upload((void**)&lv.d_table, lv.table.data(), lv.table.size() * 4)) return e;
        const void* src = g->storage == NX_F64 ? (const void*)p64[l].data() : (const void*)p32[l].data();
        if (int e = upload(&lv.fin, src, elems * es)) return e;
        if (int e = upload(&lv.fout, src, elems * es)) return e;
        std::vector<uint32_t> st((size_t)kBV * lv.n_blocks, 0);
        for (int z = 0; z < lv.dim[2]; z++)
            for (int y = 0; y < lv.dim[1]; y++)
                for (int x = 0; x < lv.dim[0]; x++) {
                    const int64_t s = lv.slot(x, y, z);
                    if (s >= 0) st[s] = lv.st[lv.lin(x, y, z)];
                }
        if (int e = upload((void**)&lv.d_state, st.data(), st.size() * 4)) return e;
        lv.runs.clear();
        for (size_t i = 0; i < lv.nvox(); i++)
            if (lv.st[i] & kActive) {
                if (lv.runs.empty() || lv.runs.back().second != i) lv.runs.emplace_back(i, i);
                lv.runs.back().second = i + 1;
            }
        std::vector<uint64_t> lk;
        const uint64_t n_skip = links_of(*g, l, lk, lv.separate);
        lv.keep = n_skip != 0;
        if (int e = upload((void**)&lv.d_links, lk.data(), lk.size() * 8)) return e;
    }
    // fine store gather lists (store.h:98-163) and sumStore counts
    // (init.h:8-55) of every level pair: fine voxels in z, y, x order, q
    // ascending.  The counts take every active fine voxel with a parent,
    // the store only those without children whose csChild is active.
    for (int l = 0; l + 1 < D; l++) {
        const Level& f = g->L[l];
        const Level& c = g->L[l + 1];
        std::vector<float> cnt((size_t)g->lat.Q * kBV * c.n_blocks, 0.f);
        std::vector<std::pair<uint64_t, uint64_t>> tl;  // (target element, source element)
        for (int z = 0; z < f.dim[2]; z++)
            for (int y = 0; y < f.dim[1]; y++)
                for (int x = 0; x < f.dim[0]; x++) {
                    if (!f.active(x, y, z) || !has_parent(*g, l, x, y, z)) continue;
                    const bool leaf = !(f.st[f.lin(x, y, z)] & kRefined);
                    const int px = x >> 1, py = y >> 1, pz = z >> 1;
                    for (int q = 0; q < g->lat.Q; q++) {
                        if (q == g->lat.rest) continue;
                        const int* cq = g->lat.c[q];
                        const int ux = uoff(x, cq[0]), uy = uoff(y, cq[1]), uz = uoff(z, cq[2]);
                        if (f.active(x + ux, y + uy, z + uz)) continue;
                        if (!c.active(px + ux, py + uy, pz + uz)) continue;
                        const int sx = ux - cq[0], sy = uy - cq[1], sz = uz - cq[2];
                        const int64_t cs = c.slot(px + sx, py + sy, pz + sz);
                        if (cs < 0) continue;
                        cnt[c.elem(cs, q)] += 1.f;
                        if (!leaf || !f.active(x + sx, y + sy, z + sz)) continue;
                        // a target that is a leaf: the streams of both levels read it
                        if (!(c.st[c.lin(px + sx, py + sy, pz + sz)] & kRefined))
                            g->L[l].separate = g->L[l + 1].separate = true;
                        tl.emplace_back(c.elem(cs, q), f.elem(f.slot(x, y, z), q));
                    }
                }
        for (float& v : cnt)
            if ((double)v > 0.001) v = g->storage == NX_F64 ? (float)(1.0 / (2.0 * (double)v)) : 1.f / (2.f * v);
        if (int e = upload((void**)&g->L[l + 1].d_ss, cnt.data(), cnt.size() * 4)) return e;
        std::stable_sort(tl.begin(), tl.end(),
                         [](const std::pair<uint64_t, uint64_t>& a, const std::pair<uint64_t, uint64_t>& b) {
                             return a.first < b.first;
                         });
        std::vector<uint64_t> target, src;
        std::vector<uint32_t> first;
        for (size_t k = 0; k < tl.size(); k++) {
            if (k == 0 || tl[k].first != tl[k - 1].first) {
                target.push_back(tl[k].first);
                first.push_back((uint32_t)k);
            }
            src.push_back(tl[k].second);
        }
        first.push_back((uint32_t)tl.size());
        Store& sl = g->store[l];
        sl.n = (uint32_t)target.size();
        sl.n_src = src.size();
        if (int e = upload((void**)&sl.d_target, target.data(), target.size() * 8)) return e;
        if (int e = upload((void**)&sl.d_first, first.data(), first.size() * 4)) return e;
        if (int e = upload((void**)&sl.d_src, src.data(), src.size() * 8)) return e;
    }
    g->ready = true;
    return NX_OK;
}

}  // namespace

extern "C" int nx_mgrid_cavity(nx_mgrid g, double ulb)
{
    if (!g) return set_error(NX_ERR_INVALID, "null mgrid");
    if (!std::isfinite(ulb)) return set_error(NX_ERR_INVALID, "nx_mgrid_cavity: non-finite lid speed");
    const double uw[3] = {ulb, 0., 0.};
    return setup_cells(g, nullptr, uw);
}

extern "C" int nx_mgrid_setup_cells(nx_mgrid g, const uint8_t* const* cls, const double u_wall[3])
{
    if (!g || !cls || !u_wall) return set_error(NX_ERR_INVALID, "nx_mgrid_setup_cells: null argument");
    for (int l = 0; l < g->depth; l++) {
        if (!cls[l]) return set_error(NX_ERR_INVALID, "nx_mgrid_setup_cells: null class array");
        const Level& lv = g->L[l];
        for (size_t i = 0; i < lv.nvox(); i++)
            if ((lv.st[i] & kActive) && !(lv.st[i] & kRefined) && cls[l][i] != NX_CELL_BULK &&
                cls[l][i] != NX_CELL_BOUNCEBACK && cls[l][i] != NX_CELL_MOVINGWALL)
                return set_error(NX_ERR_INVALID, "nx_mgrid_setup_cells: classes NX_CELL_BULK, NX_CELL_BOUNCEBACK or "
                                                 "NX_CELL_MOVINGWALL");
    }
    for (int a = 0; a < 3; a++)
        if (!std::isfinite(u_wall[a])) return set_error(NX_ERR_INVALID, "nx_mgrid_setup_cells: non-finite velocity");
    return setup_cells(g, cls, u_wall);
}

namespace {

// One coarse step as the sequence of the reference's recursion
// (lbmMultiRes.h:141-263): per level l from the top, collide l and store
// l -> l+1, the step of level l-1, stream l, and below the top level the
// same once more.
struct Op {
    uint8_t kind;   // 0 collide, 1 store, 2 stream
    uint8_t level;
    bool last;      // the level's last stream of the coarse step
};

void expand(int l, int depth, std::vector<Op>& ops)
{
    for (int half = 0; half < 2; half++) {
        ops.push_back({0, (uint8_t)l, false});
        if (l + 1 < depth) ops.push_back({1, (uint8_t)l, false});
        if (l != 0) expand(l - 1, depth, ops);
        ops.push_back({2, (uint8_t)l, false});
        if (l == depth - 1) break;
    }
}

template <int S, class LT>
struct Stepper {
    using T = typename MS<S>::T;
    nx_mgrid_s& g;
    double omega0;
    hipStream_t st;

    // computeOmega (util.h:40-45): omega0 is the coarsest level's
    double omega(int l) const
    {
        const int il = g.depth - l - 1;
        return 2 * omega0 / (std::scalbln(1.0, il + 1) + (1. - std::scalbln(1.0, il)) * omega0);
    }
    // beta and 1 / beta in T, as the reference's collision evaluates them
    Relax relax(int l) const
    {
        const T om = (T)omega(l), beta = (T)((double)om * 0.5);
        return Relax{(double)om, (double)beta, (double)(T)(1.0 / (double)beta)};
    }
    UpLevel up(int l) const
    {
        if (l + 1 >= g.depth) return UpLevel{nullptr, nullptr, {0, 0, 0}};
        const Level& c = g.L[l + 1];
        return UpLevel{c.fout, c.d_table, {c.nb[0], c.nb[1], c.nb[2]}};
    }
    void collide(int l) const
    {
        const Level& lv = g.L[l];
        if (lv.n_blocks)
            hipLaunchKernelGGL((k_mr_collide<S, LT>), dim3(lv.n_blocks), dim3(kBV), 0, st, (const T*)lv.fin,
                               (T*)lv.fout, lv.d_state, relax(l));
    }
    StoreArgs store_args(int l) const
    {
        const Store& sl = g.store[l];
        if (l + 1 >= g.depth || !sl.n) return StoreArgs{nullptr, nullptr, nullptr, nullptr, 0, 0};
        return StoreArgs{g.L[l + 1].fout, sl.d_target, sl.d_first, sl.d_src, sl.n, ((sl.n + kBV - 1) / kBV + 7u) & ~7u};
    }
    void store(int l) const
    {
        const StoreArgs a = store_args(l);
        if (a.n)
            hipLaunchKernelGGL((k_mr_store<S>), dim3(a.groups), dim3(kBV), 0, st, (const T*)g.L[l].fout, a);
    }
    // with_store: the level's store, due since its collide, rides along
    template <bool COLLIDE, bool KEEP>
    void stream(int l, bool with_store) const
    {
        const Level& lv = g.L[l];
        if (!lv.n_blocks) return;
        const StoreArgs a = with_store ? store_args(l) : StoreArgs{nullptr, nullptr, nullptr, nullptr, 0, 0};
        auto go = [&](auto off) {
            hipLaunchKernelGGL((k_mr_stream<S, LT, COLLIDE, KEEP, decltype(off)>), dim3(lv.n_blocks + a.groups), dim3(kBV),
                               0, st, (const T*)lv.fout, (T*)lv.fin, lv.d_state, lv.d_links, (uint64_t)lv.slots(),
                               lv.d_conn, lv.d_origins, (const float*)lv.d_ss, up(l),
                               COLLIDE ? relax(l) : Relax{0.0, 0.0, 0.0}, a);
        };
        // byte offsets in 32 bits where the level's populations allow it
        if (!wide_offsets() && (uint64_t)lv.slots() * LT::Q * sizeof(T) < (1ull << 32)) go(uint32_t{});
        else go(uint64_t{});
    }

    // n coarse steps.  A level's stream and its next collide touch no other
    // level and nothing of the level runs between them (the operations in
    // between are the coarser levels' stream, collide and store), so on a
    // level without links in state "none" they run as one pass (fout -> fin
    // buffer, then the two buffers trade roles) and the collide is skipped
    // when its turn comes; the store after it then reads the fused pass's
    // output.  The last stream of each level in the call is not fused, so
    // the fields between calls are those of the unfused sequence.
    //
    // The store after a collide runs in the launch of the level's next
    // stream: between the two only finer levels run, whose streams read
    // unrefined voxels of this level and whose stores add to its refined
    // ones, while this store reads its unrefined voxels and adds to the next
    // level's refined ones, first used by that level's own stream.
    void run(const std::vector<Op>& ops, int n) const
    {
        bool done[kMaxDepth] = {};  // the level's next collide already ran in a fused pass
        for (int k = 0; k < n; k++)
            for (const Op& op : ops) {
                const int l = op.level;
                Level& lv = g.L[l];
                if (op.kind == 0) {
                    if (done[l])
                        done[l] = false;
                    else
                        collide(l);
                } else if (op.kind == 1) {
                    if (lv.separate) store(l);
                } else if (!lv.keep && !(op.last && k == n - 1)) {
                    stream<true, false>(l, !lv.separate);
                    std::swap(lv.fin, lv.fout);
                    done[l] = true;
                } else if (lv.keep) {
                    stream<false, true>(l, !lv.separate);
                } else {
                    stream<false, false>(l, !lv.separate);
                }
            }
    }
};

}  // namespace

extern "C" int nx_mgrid_step(nx_mgrid g, double omega0, int32_t n_steps, nx_stream s)
{
    if (!g || n_steps < 0) return set_error(NX_ERR_INVALID, "nx_mgrid_step: bad arguments");
    if (!g->ready) return set_error(NX_ERR_NOT_INIT, "nx_mgrid_step: call nx_mgrid_cavity first");
    if (!(omega0 > 0.0 && omega0 < 2.0)) return set_error(NX_ERR_INVALID, "nx_mgrid_step: omega0 in (0, 2)");
    std::vector<Op> ops;
    expand(g->depth - 1, g->depth, ops);
    for (int l = 0; l < g->depth; l++)
        for (size_t i = ops.size(); i-- > 0;)
            if (ops[i].kind == 2 && ops[i].level == l) {
                ops[i].last = true;
                break;
            }
    const hipStream_t st = (hipStream_t)s;
    if (g->lattice == NX_MGRID_KBC27) {
        if (g->storage == NX_F64)
            Stepper<NX_F64, L27>{*g, omega0, st}.run(ops, n_steps);
        else
            Stepper<NX_F32, L27>{*g, omega0, st}.run(ops, n_steps);
    } else {
        if (g->storage == NX_F64)
            Stepper<NX_F64, L19>{*g, omega0, st}.run(ops, n_steps);
        else
            Stepper<NX_F32, L19>{*g, omega0, st}.run(ops, n_steps);
    }
    NX_CHECK_LAUNCH("mgrid step");
    return NX_OK;
}

namespace {

// Read-back in chunks: gathered on the device, copied to pinned memory, its
// active voxels copied to the caller's array (the others keep what they hold
// there).  128^3, 27 populations, float: one host copy per voxel took 155 ms,
// this about 6 ms with 8 workers (bound by the page faults of a fresh array).
// Levels up to kPlainBytes, and any level where the chunks' memory cannot be
// had, take the host copies: the first chunked read of a grid pays 0.2 to 0.3 ms
// for that memory and a stream (17 x 13 x 9, 19 populations, float: 312 us, with
// host copies 146; 24^3, 1 MB: 313 and 522).
constexpr size_t kReadBytes = 4u << 20, kPlainBytes = 256u << 10;

bool make_reader(nx_mgrid_s::Reader& r)
{
    const bool ok = (r.st || hipStreamCreateWithFlags(&r.st, hipStreamNonBlocking) == hipSuccess) &&
                    (r.dev || hipMalloc(&r.dev, kReadBytes) == hipSuccess) &&
                    (r.host || hipHostMalloc(&r.host, kReadBytes, hipHostMallocDefault) == hipSuccess);
    if (!ok) (void)hipGetLastError();
    return ok;
}

template <typename T>
int read_chunk(const nx_mgrid_s& g, const Level& lv, int which, size_t e0, size_t e1, nx_mgrid_s::Reader& r, void* dense)
{
    const uint32_t n = (uint32_t)(e1 - e0);
    hipLaunchKernelGGL(k_mr_dense<T>, dim3((n + 255) / 256), dim3(256), 0, r.st, (const T*)(which ? lv.fout : lv.fin),
                       lv.d_state, lv.d_table, lv.dim[0], lv.dim[1], (uint64_t)lv.nvox(), lv.nb[0], lv.nb[1], lv.nq,
                       (uint64_t)e0, n, (T*)r.dev);
    NX_CHECK_LAUNCH("k_mr_dense");
    NX_CHECK_HIP(hipMemcpyAsync(r.host, r.dev, (size_t)n * sizeof(T), hipMemcpyDeviceToHost, r.st));
    NX_CHECK_HIP(hipStreamSynchronize(r.st));
    for (size_t e = e0; e < e1;) {
        const size_t base = e / lv.nvox() * lv.nvox(), v0 = e - base, v1 = std::min(lv.nvox(), e1 - base);
        auto it = std::upper_bound(lv.runs.begin(), lv.runs.end(), v0,
                                   [](size_t v, const std::pair<size_t, size_t>& q) { return v < q.second; });
        for (; it != lv.runs.end() && it->first < v1; ++it) {
            const size_t a = std::max(it->first, v0), b = std::min(it->second, v1);
            std::memcpy((T*)dense + base + a, (const T*)r.host + (base + a - e0), (b - a) * sizeof(T));
        }
        e = base + v1;
    }
    return NX_OK;
}

int read_plain(const Level& lv, int which, size_t es, void* dense)
{
    std::vector<uint8_t> buf((size_t)lv.nq * kBV * lv.n_blocks * es);
    if (!buf.empty()) NX_CHECK_HIP(hipMemcpy(buf.data(), which ? lv.fout : lv.fin, buf.size(), hipMemcpyDeviceToHost));
    for (int z = 0; z < lv.dim[2]; z++)
        for (int y = 0; y < lv.dim[1]; y++)
            for (int x = 0; x < lv.dim[0]; x++) {
                const int64_t s = lv.slot(x, y, z);
                if (s < 0) continue;
                for (int q = 0; q < lv.nq; q++)
                    std::memcpy((uint8_t*)dense + ((size_t)q * lv.nvox() + lv.lin(x, y, z)) * es, buf.data() + lv.elem(s, q) * es,
                                es);
            }
    return NX_OK;
}

int read_chunks(nx_mgrid_s& g, const Level& lv, int which, size_t total, size_t es, void* dense)
{
    const size_t chunk = kReadBytes / es, chunks = (total + chunk - 1) / chunk;
    std::atomic<size_t> next{0};
    std::atomic<int> code{NX_OK};
    std::mutex err_mu;
    std::string err;
    auto work = [&](size_t w) {
        int e = NX_OK;
        try {
            // (a worker that cannot have its chunk leaves the work to the others)
            if (w > 0 && (hipSetDevice(g.device) != hipSuccess || !make_reader(g.reader[w]))) return;
            for (size_t c; e == NX_OK && code == NX_OK && (c = next++) < chunks;) {
                const size_t e0 = c * chunk, e1 = std::min(total, e0 + chunk);
                e = es == 8 ? read_chunk<double>(g, lv, which, e0, e1, g.reader[w], dense)
                            : read_chunk<float>(g, lv, which, e0, e1, g.reader[w], dense);
            }
            if (e != NX_OK) {
                std::lock_guard<std::mutex> el(err_mu);
                if (code == NX_OK) err = nx_last_error();  // (per thread)
                code = e;
            }
        } catch (...) {
            code = NX_ERR_HIP;  // no memory for a message
        }
    };
    // one worker per 2 chunks, the calling thread among them
    const size_t workers = std::min<size_t>(8, (chunks + 1) / 2);
    std::vector<std::thread> th;
    try {
        for (size_t w = 1; w < workers; w++) th.emplace_back(work, w);
    } catch (...) {
        // fewer threads than wished for: the others take the chunks
    }
    work(0);
    for (auto& x : th) x.join();
    return code == NX_OK ? NX_OK : set_error(code, err);
}

}  // namespace

extern "C" int nx_mgrid_fields(nx_mgrid g, int32_t level, int32_t which, void* dense)
{
    if (int e = check_level(g, level)) return e;
    if ((which != 0 && which != 1) || !dense) return set_error(NX_ERR_INVALID, "nx_mgrid_fields: bad arguments");
    if (!g->ready) return set_error(NX_ERR_NOT_INIT, "nx_mgrid_fields: call nx_mgrid_cavity first");
    NX_CHECK_HIP(hipDeviceSynchronize());
    const Level& lv = g->L[level];
    const size_t total = lv.nvox() * (size_t)lv.nq, es = g->storage == NX_F64 ? 8 : 4;
    if (lv.runs.empty()) return NX_OK;
    if (total * es <= kPlainBytes) return read_plain(lv, which, es, dense);
    std::lock_guard<std::mutex> lk(g->read_mu);
    int dev = 0;
    NX_CHECK_HIP(hipGetDevice(&dev));
    if (dev != g->device) {
        NX_CHECK_HIP(hipSetDevice(g->device));
        NX_CHECK_HIP(hipDeviceSynchronize());
    }
    const int e = make_reader(g->reader[0]) ? read_chunks(*g, lv, which, total, es, dense) : read_plain(lv, which, es, dense);
    if (dev != g->device) NX_CHECK_HIP(hipSetDevice(dev));
    return e;
}

extern "C" int nx_mgrid_destroy(nx_mgrid g)
{
    if (!g) return NX_OK;
    for (auto& lv : g->L)
        for (void* p : {(void*)lv.d_state, (void*)lv.d_links, (void*)lv.d_conn, (void*)lv.d_origins,
                        (void*)lv.d_table, (void*)lv.d_ss, lv.fin, lv.fout})
            if (p) hipFree(p);
    for (auto& r : g->reader) {
        if (r.dev) hipFree(r.dev);
        if (r.host) hipHostFree(r.host);
        if (r.st) hipStreamDestroy(r.st);
    }
    for (auto& sl : g->store)
        for (void* p : {(void*)sl.d_target, (void*)sl.d_first, (void*)sl.d_src})
            if (p) hipFree(p);
    delete g;
    return NX_OK;
}
