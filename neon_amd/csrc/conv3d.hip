// BF16 3D convolution forward, backward-data and backward-weight on the gfx950
// matrix cores, FP32 accumulation (the learned warm start's network).  No
// counterpart in the reference.
//
// All three are implicit GEMMs:
//   forward      M = cout, N = voxels, K = taps*cin (A: 8 weights, B: 8 channels
//                of one tap, 16 bytes each); the input with its halo is staged
//                in LDS (k_fwd_z16, k_fwd_blk, k_fwd_tap); thin grids read their
//                fragments from global memory (k_fwd), 1^3 kernels need no halo
//                (k_pw)
//   bwd-data     the forward on the flipped, transposed weights
//   bwd-weight   M = cout, N = cin, K = voxels (split over workgroups, FP32
//                partials, fixed-order reduction): all 27 taps at once on rows
//                of >= 32 voxels (k_bwd_wr, k_bwd_w27), the 9 of a z shift on
//                rows of 4 to 16 (k_bwd_wc), else one tap per workgroup
//                (k_bwd_w)
// MFMA 16x16x32 bf16 operand layout: lane l holds row (A) / column (B) l%16
// and the 8 K values of group l/16; D register r of lane l is row 4*(l/16)+r,
// column l%16.
//
// Order of the sums.  The matrix core adds the four 8-value K groups of an
// instruction one after another to the accumulator, each rounded (measured:
// the order inside a group, the roles of A and B and groups of zeros change no
// bit, the order of the groups does).  Every kernel here visits the groups of
// an output in one order fixed by the shape, so that which kernel computes a
// layer never shows in the bits: a network multiplies a changed bf16 rounding
// some 20 times per layer (one training step of the 64^3 network computed in
// another order is off by up to 0.1 in its gradients after three more steps).
//   forward      rows of >= 32 voxels, >= 4 rows and planes: slices of 16
//                channels, in each the taps (z, y, x ascending); other grids:
//                the taps, in each the channels
//   bwd-weight   a split's voxels ascending (plan_w); partials as k_reduce_w
//                adds them
#include "conv3d.hpp"
#include "nx_common.hpp"

#include <algorithm>

namespace nx::conv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Geo {
    uint32_t V;          // voxels = n*d*h*w
    int D, H, W;         // powers of two
    int lw, lh;          // log2 W, log2 H
};

__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
    u += 0x7fffu + ((u >> 16) & 1u);                                            // nearest even
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ bf16x8 ld8(const uint16_t* p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// a bf16 value > 0 (or NaN without sign): ReLU passes its gradient
__device__ __forceinline__ bool positive(uint16_t h) { return (h & 0x8000u) == 0 && (h & 0x7fffu) != 0; }

// Four consecutive channels of a voxel at element i + o of y (i the same for
// the whole wavefront); mask as in k_fwd_blk.
__device__ __forceinline__ void put4(void* y, const uint16_t* mask, size_t i, uint32_t o, f32x4 v, bool f32out)
{
    if (f32out) {
        float* p = static_cast<float*>(y) + i + o;
#pragma unroll
        for (int r = 0; r < 4; r++) p[r] = v[r];
        return;
    }
    typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
    u16x4 h = __builtin_bit_cast(u16x4, __builtin_convertvector(v, bf16x4));
    if (mask) {
        const u16x4 m = *reinterpret_cast<const u16x4*>(mask + i + o);
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (!positive(m[r])) h[r] = 0;
    }
    __builtin_memcpy(static_cast<uint16_t*>(y) + i + o, &h, 8);
}

template <int KS>
__device__ __forceinline__ void tap_offset(int tap, int& dz, int& dy, int& dx)
{
    if constexpr (KS == 3) {
        dz = tap / 9 - 1;
        dy = (tap / 3) % 3 - 1;
        dx = tap % 3 - 1;
    } else {
        dz = dy = dx = 0;
    }
}

// 1^3 convolution: out[v][co] = sum_ci x[v][ci] w[co][ci] (and backward-data on
// the flipped weights).  A wavefront takes 64 voxels x 16 NCO output channels;
// M = channels (A: weights), N = voxels (B: 16 bytes of a voxel straight from
// memory), so a lane ends with 4 consecutive channels of a voxel.  Bound by
// HBM.  Stores the first `keep` channels, `keep` apart, where that is not cout.
// Measured (MI355X, 64^3, batch 8, 16 -> 16): 23 us (float, 4 of 16 channels
// kept), 32 us backward (before, one 2- or 4-byte store per channel and all 16
// floats of a voxel: 36 and 36 us).
template <int NCO>
__global__ void __launch_bounds__(256)
    k_pw(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
         const uint16_t* __restrict__ mask, void* __restrict__ y, uint32_t V, int cin, int cout, int flags, int keep)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const uint32_t v0 = (blockIdx.x * 4u + (uint32_t)wave) * 64u;
    if (v0 >= V) return;  // whole wave
    const int co0 = (int)blockIdx.y * 16 * NCO;
    f32x4 acc[4][NCO];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int n = 0; n < NCO; n++) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < cin; c0 += 32) {
        const bool in = c0 + 8 * grp < cin;
        bf16x8 a[NCO], b[4];
#pragma unroll
        for (int t = 0; t < 4; t++)
            b[t] = in && v0 + 16 * t + r16 < V ? ld8(x + (size_t)v0 * cin + (uint32_t)((16 * t + r16) * cin + c0 + 8 * grp))
                                               : bf16x8{};
#pragma unroll
        for (int n = 0; n < NCO; n++)
            a[n] = in ? ld8(w + (size_t)(co0 + 16 * n) * cin + (uint32_t)(r16 * cin + c0 + 8 * grp)) : bf16x8{};
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int n = 0; n < NCO; n++) acc[t][n] = mfma(a[n], b[t], acc[t][n]);
    }
    const bool relu = flags & kRelu, f32out = flags & kOutF32;
#pragma unroll
    for (int n = 0; n < NCO; n++) {
        const int co = co0 + 16 * n + 4 * grp;
        f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias)
#pragma unroll
            for (int r = 0; r < 4; r++) bv[r] = bias[co + r];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (v0 + 16 * t + r16 >= V) continue;
            f32x4 o = acc[t][n] + bv;
            if (relu)
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = o[r] > 0.f ? o[r] : 0.f;
            if (keep == cout) {
                put4(y, mask, (size_t)v0 * cout + co0 + 16 * n, (uint32_t)((16 * t + r16) * cout + 4 * grp), o, f32out);
            } else if (co < keep) {
                float* p = static_cast<float*>(y) + (size_t)(v0 + 16 * t + r16) * keep + co;
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (co + r < keep) p[r] = o[r];
            }
        }
    }
}

// 3^3 on thin grids and on rows of 1 or 2 voxels.  One wave: 32 voxels x (16*NT) output
// channels; 4 waves per workgroup.  grid.y selects the block of 16*NT output channels.
template <int NT>
__global__ void __launch_bounds__(256)
    k_fwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
          const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cin, int cout, int flags)
{
    constexpr int T = 27;
    const int K = T * cin, KC = (K + 31) / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, grp = lane >> 4;
    const uint32_t vbase = (blockIdx.x * 4u + (uint32_t)wave) * 32u;
    if (vbase >= g.V) return;  // whole wave
    const int co0 = (int)blockIdx.y * NT * 16;

    int px[2], py[2], pz[2];
    uint32_t pv[2];
    bool pok[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint32_t v = vbase + 16u * t + (uint32_t)r16;
        pok[t] = v < g.V;
        pv[t] = v;
        px[t] = (int)(v & (uint32_t)(g.W - 1));
        py[t] = (int)((v >> g.lw) & (uint32_t)(g.H - 1));
        pz[t] = (int)((v >> (g.lw + g.lh)) & (uint32_t)(g.D - 1));
    }
    const uint16_t* wrow[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) wrow[n] = w + (size_t)(co0 + n * 16 + r16) * K;

    f32x4 acc[2][NT];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    // K position of this lane group: kk = 32*kc + 8*grp = tap*cin + ci.
    // Fragments are double-buffered: the loads of chunk kc+1 are issued
    // before the MFMAs of chunk kc.
    int tap = 0, ci = 8 * grp;
    while (ci >= cin) { ci -= cin; ++tap; }
    auto fetch = [&](int kc, bf16x8* a, bf16x8* b) {
        const int kk = kc * 32 + 8 * grp;
        if (kk < K) {
            int dz, dy, dx;
            tap_offset<3>(tap, dz, dy, dx);
            const int off = (dz * g.H + dy) * g.W + dx;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const bool ok = pok[t] && (unsigned)(px[t] + dx) < (unsigned)g.W &&
                                (unsigned)(py[t] + dy) < (unsigned)g.H &&
                                (unsigned)(pz[t] + dz) < (unsigned)g.D;
                a[t] = ok ? ld8(x + (size_t)(int64_t)((int64_t)pv[t] + off) * cin + ci) : bf16x8{};
            }
#pragma unroll
            for (int n = 0; n < NT; n++) b[n] = ld8(wrow[n] + kk);
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++) a[t] = bf16x8{};
#pragma unroll
            for (int n = 0; n < NT; n++) b[n] = bf16x8{};
        }
        ci += 32;
        while (ci >= cin) { ci -= cin; ++tap; }
    };
    auto mma = [&](const bf16x8* a, const bf16x8* b) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int n = 0; n < NT; n++) acc[t][n] = mfma(a[t], b[n], acc[t][n]);
    };
    bf16x8 a0[2], b0[NT], a1[2], b1[NT];
    fetch(0, a0, b0);
    for (int kc = 0; kc < KC; kc += 2) {
        if (kc + 1 < KC) fetch(kc + 1, a1, b1);
        mma(a0, b0);
        if (kc + 1 < KC) {
            if (kc + 2 < KC) fetch(kc + 2, a0, b0);
            mma(a1, b1);
        }
    }

    const bool relu = flags & kRelu, f32out = flags & kOutF32;
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int co = co0 + n * 16 + r16;
        const float bv = bias ? bias[co] : 0.f;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t v = vbase + 16u * t + 4u * grp + (uint32_t)r;
                if (v >= g.V) continue;
                float s = acc[t][n][r] + bv;
                if (relu) s = s > 0.f ? s : 0.f;
                if (f32out)
                    static_cast<float*>(y)[(size_t)v * cout + co] = s;
                else
                    static_cast<uint16_t*>(y)[(size_t)v * cout + co] =
                        mask && !positive(mask[(size_t)v * cout + co]) ? (uint16_t)0 : f2bf(s);
            }
    }
}

// 3^3 forward (and backward-data) with the input block in LDS, rows of at
// least 32 voxels, more than 16 input channels.  M = output channels (A:
// weights, one 16-byte load per lane), N = 16 voxels (B: 8 channels of a voxel,
// one ds_read_b128), K = 16 channels of the taps (dx = -1, dx = 0) of a voxel
// pair, then of dx = 1 alone.  A wavefront computes 4 x 2 tiles of 16 voxels
// along x in y and z for NCO blocks of 16 output channels; 2 x 2 wavefronts in
// x and z share one staged block of 32 x 4 x 4 voxels with its halo, 32
// channels at a time in two planes of 16.  A B fragment serves every output
// row of the wavefront that a tap reaches from it and all NCO channel blocks
// (3 or 4 MFMAs): with one LDS read per MFMA the LDS takes twice the MFMA's
// time.  The second workgroup of the CU hides the staging.  A lane ends with 4 consecutive channels of a voxel: 8- or
// 16-byte stores.
// Measured (MI355X): 64^3 x 8, 48 -> 16 164 us, 32^3 x 8, 96 -> 32 72 us, 32^3
// x 16, 64 -> 64 184 us (with one LDS read per MFMA, 16 channels staged at a
// time, 226, 103 and 243 us).
// mask: null, or the activations whose ReLU the result passes back through
// (0 where the activation is not positive).
template <int NCO>
__global__ void __launch_bounds__(256, 2)
    k_fwd_blk(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
              const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cin, int cout, int flags)
{
    constexpr int RY = 4, RZ = 2, SY = RY + 2;                   // rows, planes, source rows of a wavefront
    constexpr int BX = 32, BY = RY, BZ = 2 * RZ, HX = BX + 2, HY = BY + 2, HZ = BZ + 2, HV = HX * HY * HZ;
    constexpr int ROWS = HY * HZ;
    constexpr int PLANE = HV * 16 + 64;                          // halves of 16 channels (+ 64: the two on other banks)
    constexpr int ZG = NCO == 1 ? 1 : 3, NDZ = 3 / ZG;           // weight groups: all dz, or one each
    constexpr int WB = ZG == 1 ? 1 : 2;                          // weight groups held
    constexpr bool PIPE = NCO == 1;                              // fragments of the next plane read ahead
    __shared__ __attribute__((aligned(16))) uint16_t tile[2 * PLANE];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const bool half = grp >= 2;                                  // the second tap of a pair
    const uint32_t ncb = (uint32_t)(cout / (16 * NCO));
    const uint32_t nbx = (uint32_t)(g.W / BX), nby = (uint32_t)(g.H / BY), nbz = (uint32_t)(g.D / BZ);
    const int wx = wave & 1, wz = wave >> 1;
    // halo-block voxel of this lane at offset (-1, -1, -1) of its first tile
    const int hv0 = wz * RZ * HY * HX + wx * 16 + r16;

    // blocks of one XCD in order: channel blocks of a position, then x, y, z, sample
    uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const int co0 = (int)(id % ncb) * 16 * NCO;
    id /= ncb;
    const int x0 = (int)(id % nbx) * BX;
    id /= nbx;
    const int y0 = (int)(id % nby) * BY;
    id /= nby;
    const int z0 = (int)(id % nbz) * BZ;
    const uint32_t smp = id / nbz;
    // Staging by whole rows (BX x PV 16-byte pieces fill one or two loads of a
    // wavefront: address and test are scalar), then the two halo columns.  A
    // slice is 32 channels (PV = 4 pieces a voxel) or the last 16 (PV = 2).
    auto row_base = [&](int row, bool& in) {
        const int gy = y0 - 1 + row % HY, gz = z0 - 1 + row / HY;
        in = row < ROWS && (unsigned)gy < (unsigned)g.H && (unsigned)gz < (unsigned)g.D;
        return (uint32_t)((gz * g.H + gy) * g.W + x0);
    };
    auto spot = [&](int hv, int pc) { return tile + (pc >> 1) * PLANE + hv * 16 + (pc & 1) * 8; };
    auto stage = [&](auto pvc, int c0) __attribute__((always_inline)) {
        constexpr int PV = decltype(pvc)::value, RP = BX * PV, KM = (ROWS * RP + 255) / 256, NB = 9;
        constexpr int NH = (ROWS * 2 * PV + 255) / 256;
        const uint16_t* xs = x + (size_t)smp * (uint32_t)(g.D * g.H * g.W) * (uint32_t)cin + c0;
        auto row_of = [&](int k, int& row, int& q) {
            const int at = (k * 4 + wave) * 64;
            row = at / RP;
            q = at % RP + lane;
        };
        uint4 h[NH];
#pragma unroll
        for (int k = 0; k < NH; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            bool in;
            const uint32_t v = row_base(row, in) + (side ? (uint32_t)BX : ~0u);
            in = in && (side ? x0 + BX < g.W : x0 > 0);
            h[k] = in ? *reinterpret_cast<const uint4*>(xs + (uint32_t)(v * (uint32_t)cin + 8 * pc)) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll 1
        for (int k0 = 0; k0 < KM; k0 += NB) {
            uint4 v[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) {
                int row, q;
                row_of(k0 + k, row, q);
                bool in;
                const uint16_t* p = xs + (size_t)(row_base(row, in) * (uint32_t)cin);
                v[k] = in ? *reinterpret_cast<const uint4*>(p + (uint32_t)((q / PV) * cin + 8 * (q % PV))) : uint4{0u, 0u, 0u, 0u};
            }
#pragma unroll
            for (int k = 0; k < NB; k++) {
                int row, q;
                row_of(k0 + k, row, q);
                if (row < ROWS) *reinterpret_cast<uint4*>(spot(row * HX + 1 + q / PV, q % PV)) = v[k];
            }
        }
#pragma unroll
        for (int k = 0; k < NH; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            if (row < ROWS) *reinterpret_cast<uint4*>(spot(row * HX + (side ? HX - 1 : 0), pc)) = h[k];
        }
    };

    f32x4 acc[RZ][RY][NCO];
#pragma unroll
    for (int i = 0; i < RZ; i++)
#pragma unroll
        for (int j = 0; j < RY; j++)
#pragma unroll
            for (int n = 0; n < NCO; n++) acc[i][j][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint16_t* wb = w + (size_t)co0 * 27 * cin;
    const uint32_t wo = (uint32_t)(r16 * 27 * cin + 8 * (grp & 1) + (grp >> 1) * cin);
    bf16x8 a[WB][NDZ][3][2][NCO];
    // weights of 16 channels from c, dz group zg; past dx = 1 a pair has no second tap
    auto load_w = [&](int c, int zg, bf16x8 (*d)[3][2][NCO]) {
#pragma unroll
        for (int i = 0; i < NDZ; i++)
#pragma unroll
            for (int dyo = 0; dyo < 3; dyo++)
#pragma unroll
                for (int kx = 0; kx < 2; kx++)
#pragma unroll
                    for (int n = 0; n < NCO; n++) {
                        const int tap = ((zg + i) * 3 + dyo) * 3 + 2 * kx;
                        d[i][dyo][kx][n] = kx == 1 && half ? bf16x8{} : ld8(wb + (size_t)((n * 16 * 27 + tap) * cin + c) + wo);
                    }
    };
    // the 16 channels in LDS plane h: taps in order (dz, dy, dx)
    auto slice = [&](int c, int h) __attribute__((always_inline)) {
        const uint16_t* tl = tile + h * PLANE + hv0 * 16 + 8 * grp;  // groups 2, 3 read the next voxel
        constexpr int NZR = RZ + NDZ - 1;                    // source planes of a weight group
        bf16x8 v[PIPE ? 2 : 1][SY][2];
        auto plane = [&](int st) {
#pragma unroll
            for (int s = 0; s < SY; s++)
#pragma unroll
                for (int kx = 0; kx < 2; kx++) {
                    bf16x8 q = ld8(tl + (((st % NZR + st / NZR) * HY + s) * HX + 2 * kx) * 16);
                    if (kx == 1 && half) q = bf16x8{};
                    v[PIPE ? st & 1 : 0][s][kx] = q;
                }
        };
        if (PIPE) plane(0);
#pragma unroll
        for (int st = 0; st < ZG * NZR; st++) {
            const int zg = st / NZR, zr = st % NZR;
            if (ZG > 1 && zr == 0 && zg + 1 < ZG) load_w(c, zg + 1, a[(zg + 1) % WB]);
            if (PIPE && st + 1 < ZG * NZR) plane(st + 1);
            if (PIPE || zr == 0) __builtin_amdgcn_sched_barrier(0);
            if (!PIPE) plane(st);
#pragma unroll
            for (int s = 0; s < SY; s++)
#pragma unroll
                for (int kx = 0; kx < 2; kx++)
#pragma unroll
                    for (int i = 0; i < NDZ; i++)
#pragma unroll
                        for (int dyo = 0; dyo < 3; dyo++) {
                            const int jz = zr - i, jy = s - dyo;
                            if (jz < 0 || jz >= RZ || jy < 0 || jy >= RY) continue;
#pragma unroll
                            for (int n = 0; n < NCO; n++)
                                acc[jz][jy][n] = mfma(a[zg % WB][i][dyo][kx][n], v[PIPE ? st & 1 : 0][s][kx], acc[jz][jy][n]);
                        }
        }
    };
    for (int c0 = 0; c0 < cin; c0 += 32) {
        load_w(c0, 0, a[0]);
        __syncthreads();                                     // the previous slice's reads are done
        if (cin - c0 >= 32) stage(std::integral_constant<int, 4>{}, c0);
        else stage(std::integral_constant<int, 2>{}, c0);
        __syncthreads();
        slice(c0, 0);
        if (cin - c0 >= 32) {
            load_w(c0 + 16, 0, a[0]);
            slice(c0 + 16, 1);
        }
    }
    const bool relu = flags & kRelu, f32out = flags & kOutF32;
    f32x4 bv[NCO];
#pragma unroll
    for (int n = 0; n < NCO; n++) {
        bv[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias)
#pragma unroll
            for (int r = 0; r < 4; r++) bv[n][r] = bias[co0 + n * 16 + 4 * grp + r];
    }
#pragma unroll
    for (int jz = 0; jz < RZ; jz++)
#pragma unroll
        for (int jy = 0; jy < RY; jy++) {
            const size_t v = (((size_t)smp * g.D + z0 + wz * RZ + jz) * g.H + y0 + jy) * g.W + x0 + wx * 16;
#pragma unroll
            for (int n = 0; n < NCO; n++) {
                f32x4 o = acc[jz][jy][n] + bv[n];
                if (relu)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[r] = o[r] > 0.f ? o[r] : 0.f;
                put4(y, mask, v * cout + co0 + n * 16, (uint32_t)(r16 * cout + 4 * grp), o, f32out);
            }
        }
}

// 3^3 forward (and backward-data) of a 16-channel input, rows of >= 32 voxels:
// the multiply-adds per voxel are too few there to hide a block's staging, so
// 8 wavefronts march along z over 8 rows of 32 voxels instead.  The weights
// of a 16-channel output block stay in registers (18 K steps: per (dz, dy)
// the taps dx = -1, 0 of a voxel pair, then dx = 1), each plane of rows is
// staged once, two planes ahead, and adds to the three output planes it
// reaches, whose accumulators turn with it.  The columns (x segment, 8 rows,
// sample) times D planes are cut evenly into `splits` runs, one workgroup a CU.
// Bound: HBM (16 -> 16 reads and writes each voxel once) and the stores.
// Measured (MI355X, 64^3, batch 8): 16 -> 16 51 us, 16 -> 48 146 us (block by
// block 68 and 224 us).
__global__ void __launch_bounds__(512)
    k_fwd_z16(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
              const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cout, int flags, uint32_t planes,
              uint32_t planes_per_split)
{
    constexpr int TY = 8, XV = 34, PIECES = (TY + 2) * XV * 2, NJ = (PIECES + 511) / 512, BUF = PIECES * 8 + 16;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    // the channel blocks of one run side by side on one XCD
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x), ncb = (uint32_t)cout / 16u;
    const int co0 = (int)(id % ncb) * 16;
    const uint32_t split = id / ncb;
    const int nxs = g.W / 32, nyb = (g.H + TY - 1) / TY;
    const bool relu = flags & kRelu, f32out = flags & kOutF32, half = grp >= 2;
    bf16x8 a[3][3][2];
    f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dz = 0; dz < 3; dz++)
#pragma unroll
        for (int dyo = 0; dyo < 3; dyo++)
#pragma unroll
            for (int kx = 0; kx < 2; kx++)
                a[dz][dyo][kx] = kx == 1 && half ? bf16x8{}
                                                 : ld8(w + (size_t)(co0 * 27 + (dz * 3 + dyo) * 3 + 2 * kx) * 16 +
                                                       (uint32_t)(r16 * 27 * 16 + 8 * grp));
    if (bias)
#pragma unroll
        for (int r = 0; r < 4; r++) bv[r] = bias[co0 + 4 * grp + r];

    const uint32_t r1 = min(planes, (split + 1) * planes_per_split);
    for (uint32_t r = split * planes_per_split; r < r1;) {
        const uint32_t colm = r / (uint32_t)g.D;
        const int za = (int)(r % (uint32_t)g.D);
        const int zb = min(g.D, za + (int)(r1 - r));
        r += (uint32_t)(zb - za);
        const int x0 = (int)(colm % (uint32_t)nxs) * 32, y0 = (int)((colm / (uint32_t)nxs) % (uint32_t)nyb) * TY;
        const uint32_t smp = colm / (uint32_t)(nxs * nyb);
        const uint32_t plane = (uint32_t)(g.H * g.W);
        const uint16_t* xs = x + (size_t)(smp * (uint32_t)g.D) * plane * 16u;
        uint32_t off[NJ];
        bool ok[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int p = tid + 512 * j, hv = p >> 1, gx = x0 - 1 + hv % XV, gy = y0 - 1 + hv / XV;
            ok[j] = p < PIECES && (unsigned)gx < (unsigned)g.W && (unsigned)gy < (unsigned)g.H;
            off[j] = ((uint32_t)gy * (uint32_t)g.W + (uint32_t)gx) * 16u + 8u * (uint32_t)(p & 1);
        }
        uint4 R[3][NJ];
        auto fetch = [&](int s, uint4* q) __attribute__((always_inline)) {
            const bool in = s <= zb && (unsigned)s < (unsigned)g.D;
#pragma unroll
            for (int j = 0; j < NJ; j++)
                q[j] = in && ok[j] ? *reinterpret_cast<const uint4*>(xs + (size_t)((uint32_t)s * plane * 16u) + off[j])
                                   : uint4{0u, 0u, 0u, 0u};
        };
        auto put = [&](int buf, const uint4* q) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (tid + 512 * j < PIECES) *reinterpret_cast<uint4*>(lds + buf * BUF + (tid + 512 * j) * 8) = q[j];
        };
        const int yw = y0 + wave;
        f32x4 acc[3][2];                                      // [output plane slot][x tile]
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k][0] = acc[k][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        // x plane s; slots: output plane s + 1 in ph, s in ph + 2, s - 1 in ph + 1 (mod 3)
        auto step = [&](auto phase, int s, int buf) __attribute__((always_inline)) {
            constexpr int ph = decltype(phase)::value;
            fetch(s + 3, R[ph]);
            acc[ph][0] = acc[ph][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (yw < g.H) {
                const uint16_t* L = lds + buf * BUF + (wave * XV + r16) * 16 + 8 * grp;
#pragma unroll
                for (int dyo = 0; dyo < 3; dyo++)
#pragma unroll
                    for (int xt = 0; xt < 2; xt++)
#pragma unroll
                        for (int kx = 0; kx < 2; kx++) {
                            bf16x8 v = ld8(L + (dyo * XV + xt * 16 + 2 * kx) * 16);
                            if (kx == 1 && half) v = bf16x8{};
#pragma unroll
                            for (int dz = 0; dz < 3; dz++) {
                                f32x4& c = acc[dz == 0 ? ph : dz == 1 ? (ph + 2) % 3 : (ph + 1) % 3][xt];
                                c = mfma(a[dz][dyo][kx], v, c);
                            }
                        }
                if (s > za) {                                 // output plane s - 1 is complete
                    const size_t v = ((size_t)(smp * (uint32_t)g.D + (uint32_t)(s - 1)) * g.H + yw) * g.W + x0;
#pragma unroll
                    for (int xt = 0; xt < 2; xt++) {
                        f32x4 o = acc[(ph + 1) % 3][xt] + bv;
                        if (relu)
#pragma unroll
                            for (int q = 0; q < 4; q++) o[q] = o[q] > 0.f ? o[q] : 0.f;
                        put4(y, mask, (v + 16 * xt) * cout + co0, (uint32_t)(r16 * cout + 4 * grp), o, f32out);
                    }
                }
            }
            put(buf ^ 1, R[(ph + 1) % 3]);
            __syncthreads();
        };
        const int s0 = za - 1;
        fetch(s0, R[0]);
        fetch(s0 + 1, R[1]);
        fetch(s0 + 2, R[2]);
        put(0, R[0]);
        __syncthreads();
        int buf = 0;
        for (int s = s0; s <= zb;) {
            step(std::integral_constant<int, 0>{}, s, buf);
            buf ^= 1;
            if (++s > zb) break;
            step(std::integral_constant<int, 1>{}, s, buf);
            buf ^= 1;
            if (++s > zb) break;
            step(std::integral_constant<int, 2>{}, s, buf);
            buf ^= 1;
            ++s;
        }
        __syncthreads();
    }
}

// 3^3 forward (and backward-data) on rows of 4, 8 or 16 voxels: the taps in
// order, in each all the channels (k_fwd's K order), which takes every channel
// of a source row at once.  A workgroup computes WX x 4 x BZ voxels for 16 NCO
// NCW output channels; it marches over the three dz, the BZ source planes of
// one in LDS (a plane makes way for the next, loaded during the one before).
// LDS holds 16-byte pieces [8 channels][voxel], so that 16 lanes read 256
// bytes in a row, at most CMAX channels.  A tile is 16 voxels, WX along x times
// YT rows; 4 wavefronts, NCW beside each other in channels.  The weights come
// from L2, four K steps ahead.
// Measured (MI355X): 16^3 x 8, 64 -> 64 26 us; 16^3 x 16, 256 -> 128 257 us; 8^3
// x 8, 64 -> 64 22 us (fragments from global memory, k_fwd: 43, 475 and 41 us).
template <int WX, int CMAX, int NCO, int NCW>
__global__ void __launch_bounds__(256)
    k_fwd_tap(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
              const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cin, int cout, int flags)
{
    constexpr int YT = 16 / WX, BY = 4, BZ = WX == 16 ? 2 : 4, HX = WX + 2, HY = BY + 2, PV = HX * HY;
    constexpr int TP = BY / YT, NT = BZ * TP;                    // tiles of a plane, of the block
    constexpr int TW = NT * NCW / 4;                             // tiles of a wavefront
    constexpr int PITCH = BZ * PV + (BZ * PV % 2 == 0);          // odd: neighbouring pieces of a voxel on other banks
    constexpr int NP = (PV * (CMAX / 8) + 255) / 256;            // 16-byte pieces of a plane per thread
    constexpr int U = 4;                                         // K steps of a weight batch
    __shared__ __attribute__((aligned(16))) uint16_t tile[CMAX / 8 * PITCH * 8];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const int lx = r16 % WX, ly = r16 / WX;
    uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t ncb = (uint32_t)(cout / (16 * NCO * NCW)), nby = (uint32_t)(g.H / BY), nbz = (uint32_t)(g.D / BZ);
    const int co0 = ((int)(id % ncb) * NCW + wave % NCW) * 16 * NCO;
    id /= ncb;
    const int y0 = (int)(id % nby) * BY;
    id /= nby;
    const int z0 = (int)(id % nbz) * BZ;
    const uint32_t smp = id / nbz;
    const int t0 = (wave / NCW) * TW;                            // the wavefront's first tile

    // a source plane (z0 - 1 + sp): through registers into its slot sp % BZ
    const uint32_t c8 = (uint32_t)cin / 8u, pieces = (uint32_t)PV * c8;
    const uint16_t* xs = x + (size_t)smp * (uint32_t)(g.D * g.H * g.W) * (uint32_t)cin;
    uint4 pre[NP];
    auto fetch = [&](int sp) {
        const int gz = z0 - 1 + sp;
#pragma unroll
        for (int k = 0; k < NP; k++) {
            const uint32_t it = (uint32_t)tid + 256u * k, hv = it / c8, pc = it % c8;
            const int gx = (int)(hv % HX) - 1, gy = y0 - 1 + (int)(hv / HX);
            const bool in = it < pieces && (unsigned)gx < (unsigned)g.W && (unsigned)gy < (unsigned)g.H && (unsigned)gz < (unsigned)g.D;
            pre[k] = in ? *reinterpret_cast<const uint4*>(xs + (uint32_t)(((gz * g.H + gy) * g.W + gx) * cin) + 8u * pc)
                        : uint4{0u, 0u, 0u, 0u};
        }
    };
    auto put = [&](int sp) {
#pragma unroll
        for (int k = 0; k < NP; k++) {
            const uint32_t it = (uint32_t)tid + 256u * k, hv = it / c8, pc = it % c8;
            if (it < pieces) *reinterpret_cast<uint4*>(tile + (pc * PITCH + (sp % BZ) * PV + hv) * 8) = pre[k];
        }
    };

    f32x4 acc[TW][NCO];
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
        for (int n = 0; n < NCO; n++) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int K9 = 9 * cin, KC = (K9 + 31) / 32;                 // of one dz
#pragma unroll
    for (int sp = 0; sp < BZ; sp++) {
        fetch(sp);
        put(sp);
    }
    for (int dz = 0; dz < 3; dz++) {
        const uint16_t* wd = w + (size_t)co0 * 27 * cin + (uint32_t)((r16 * 27 + 9 * dz) * cin + 8 * grp);
        bf16x8 a[2][U][NCO];
        auto load_w = [&](int kc, bf16x8 (*d)[NCO]) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int n = 0; n < NCO; n++)
                    d[u][n] = 32 * (kc + u) + 8 * grp < K9 ? ld8(wd + (uint32_t)(n * 16 * 27 * cin) + 32 * (kc + u)) : bf16x8{};
        };
        load_w(0, a[0]);
        __syncthreads();                                         // the planes are there
        if (dz < 2) fetch(BZ + dz);
        int vox[TW];                                             // LDS voxel of this lane per tile, at tap (-1, -1)
#pragma unroll
        for (int t = 0; t < TW; t++)
            vox[t] = (((t0 + t) / TP + dz) % BZ) * PV + ((t0 + t) % TP * YT + ly) * HX + lx;
        int tap = 0, ci = 8 * grp;
        while (ci >= cin) { ci -= cin; ++tap; }
        auto run = [&](int kc, bf16x8 (*d)[NCO]) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (kc + u >= KC) break;
                const bool ok = tap < 9;                         // past it: weights 0, and no value of the next plane
                const int off = (ci >> 3) * PITCH + tap / 3 * HX + tap % 3;
                bf16x8 v[TW];
#pragma unroll
                for (int t = 0; t < TW; t++) v[t] = ok ? ld8(tile + (vox[t] + off) * 8) : bf16x8{};
#pragma unroll
                for (int t = 0; t < TW; t++)
#pragma unroll
                    for (int n = 0; n < NCO; n++) acc[t][n] = mfma(d[u][n], v[t], acc[t][n]);
                ci += 32;
                while (ci >= cin) { ci -= cin; ++tap; }
            }
        };
        for (int kc = 0; kc < KC; kc += 2 * U) {
            load_w(kc + U, a[1]);
            run(kc, a[0]);
            load_w(kc + 2 * U, a[0]);
            run(kc + U, a[1]);
        }
        __syncthreads();                                         // its reads are done
        if (dz < 2) put(BZ + dz);
    }
    const bool relu = flags & kRelu, f32out = flags & kOutF32;
#pragma unroll
    for (int n = 0; n < NCO; n++) {
        f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias)
#pragma unroll
            for (int r = 0; r < 4; r++) bv[r] = bias[co0 + n * 16 + 4 * grp + r];
#pragma unroll
        for (int t = 0; t < TW; t++) {
            const int gz = z0 + (t0 + t) / TP, gy = y0 + (t0 + t) % TP * YT;
            const size_t v = (((size_t)smp * g.D + gz) * g.H + gy) * g.W;
            f32x4 o = acc[t][n] + bv;
            if (relu)
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = o[r] > 0.f ? o[r] : 0.f;
            put4(y, mask, v * cout + co0 + n * 16, (uint32_t)((ly * g.W + lx) * cout + 4 * grp), o, f32out);
        }
    }
}

// Weight gradient of one tap for a (16*NM) x (16*NN) block of (co, ci): the
// 1^3 kernel, and 3^3 on rows of 1 or 2 voxels, planes of less than 32 and
// the least work (plan_w).
// grid.x = T * splits (tap fastest), grid.y = channel blocks.  Each wave
// takes every 4th 32-voxel chunk of its split and writes its own partial:
// part[(split*4 + wave)][tap][co][ci].
// The GEMM's K index is the voxel, but channels are contiguous in memory:
// each wave loads its chunk of dy (32 voxels x 16*NM channels) and of the
// shifted input (32 voxels x 16*NN channels) with 16-byte loads and writes
// it transposed into its own LDS tile [channel][voxel], from which every
// MFMA fragment (8 consecutive voxels of one channel) is one ds_read_b128.
// The next chunk's global loads are issued before the current chunk's MFMAs.
template <int NM, int NN, int KS>
__global__ void __launch_bounds__(256)
    k_bwd_w(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
            float* __restrict__ part, Geo g, int cin, int cout, uint32_t chunks_per_split)
{
    constexpr int T = KS * KS * KS;
    constexpr int CM = 16 * NM, CN = 16 * NN;       // channels of the two operands
    constexpr int PITCH = 40;                        // halves per LDS row (32 voxels + pad)
    __shared__ __attribute__((aligned(16))) uint16_t lds[4][(CM + CN) * PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, grp = lane >> 4;
    const int tap = (int)(blockIdx.x % T);
    const uint32_t split = blockIdx.x / T;
    const int mblocks = cout / CM;
    const int co0 = (int)(blockIdx.y % mblocks) * CM;
    const int ci0 = (int)(blockIdx.y / mblocks) * CN;
    int dz, dyo, dx;
    tap_offset<KS>(tap, dz, dyo, dx);
    const int off = (dz * g.H + dyo) * g.W + dx;
    uint16_t* la = lds[wave];
    uint16_t* lb = lds[wave] + CM * PITCH;

    f32x4 acc[NM][NN];
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int n = 0; n < NN; n++) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    // element e = lane + 64 k of a chunk: voxel quad e / (C/8) (4 consecutive
    // voxels), channel group e % (C/8) (8 channels): four 16-byte loads, then
    // eight 8-byte LDS writes (4 voxels of one channel each)
    constexpr int GA = CM / 8, GB = CN / 8;
    constexpr int EA = 8 * GA, EB = 8 * GB;
    constexpr int NA = (EA + 63) / 64, NB = (EB + 63) / 64;
    auto fetch = [&](uint32_t c, uint4 (*va)[4], uint4 (*vb)[4]) {
#pragma unroll
        for (int k = 0; k < NA; k++) {
            const int e = lane + 64 * k;
            const uint32_t v0 = c * 32u + 4u * (uint32_t)(e / GA);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const uint32_t v = v0 + (uint32_t)t;
                const bool ok = e < EA && v < g.V;
                va[k][t] = ok ? *reinterpret_cast<const uint4*>(dy + (size_t)v * cout + co0 + 8 * (e % GA))
                              : uint4{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int e = lane + 64 * k;
            const uint32_t v0 = c * 32u + 4u * (uint32_t)(e / GB);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const uint32_t v = v0 + (uint32_t)t;
                const int px = (int)(v & (uint32_t)(g.W - 1));
                const int py = (int)((v >> g.lw) & (uint32_t)(g.H - 1));
                const int pz = (int)((v >> (g.lw + g.lh)) & (uint32_t)(g.D - 1));
                const bool ok = e < EB && v < g.V && (unsigned)(px + dx) < (unsigned)g.W &&
                                (unsigned)(py + dyo) < (unsigned)g.H && (unsigned)(pz + dz) < (unsigned)g.D;
                vb[k][t] = ok ? *reinterpret_cast<const uint4*>(x + (size_t)(int64_t)((int64_t)v + off) * cin +
                                                                ci0 + 8 * (e % GB))
                              : uint4{0u, 0u, 0u, 0u};
            }
        }
    };
    // channel j of two voxels' 8-channel words -> one 32-bit word (voxel a low)
    auto pair = [](const uint4& a, const uint4& b, int j) {
        const uint32_t wa = (j >> 1) == 0 ? a.x : (j >> 1) == 1 ? a.y : (j >> 1) == 2 ? a.z : a.w;
        const uint32_t wb = (j >> 1) == 0 ? b.x : (j >> 1) == 1 ? b.y : (j >> 1) == 2 ? b.z : b.w;
        return (j & 1) ? ((wa >> 16) | (wb & 0xffff0000u)) : ((wa & 0xffffu) | (wb << 16));
    };
    auto put = [&](uint16_t* tile, int e, int G, const uint4* q4) {
        const int quad = e / G, ch = 8 * (e % G);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t w2[2] = {pair(q4[0], q4[1], j), pair(q4[2], q4[3], j)};
            __builtin_memcpy(__builtin_assume_aligned(tile + (ch + j) * PITCH + 4 * quad, 8), w2, 8);
        }
    };
    auto stage = [&](uint4 (*va)[4], uint4 (*vb)[4]) {
#pragma unroll
        for (int k = 0; k < NA; k++)
            if (lane + 64 * k < EA) put(la, lane + 64 * k, GA, va[k]);
#pragma unroll
        for (int k = 0; k < NB; k++)
            if (lane + 64 * k < EB) put(lb, lane + 64 * k, GB, vb[k]);
    };
    // 16-byte fragment from the LDS tile (byte copy: the tile is written as
    // 16-bit values, so the read must not be reordered by type-based aliasing)
    auto frag = [&](const uint16_t* row) {
        uint4 t;
        __builtin_memcpy(&t, __builtin_assume_aligned(row, 16), 16);
        return __builtin_bit_cast(bf16x8, t);
    };
    auto mma = [&]() {
        bf16x8 a[NM], b[NN];
#pragma unroll
        for (int m = 0; m < NM; m++) a[m] = frag(la + (m * 16 + r16) * PITCH + 8 * grp);
#pragma unroll
        for (int n = 0; n < NN; n++) b[n] = frag(lb + (n * 16 + r16) * PITCH + 8 * grp);
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int n = 0; n < NN; n++) acc[m][n] = mfma(a[m], b[n], acc[m][n]);
    };

    const uint32_t n_chunks = (g.V + 31u) / 32u;
    const uint32_t c0 = split * chunks_per_split;
    const uint32_t c1 = min(n_chunks, c0 + chunks_per_split);
    uint4 va[NA][4], vb[NB][4], wa[NA][4], wb[NB][4];
    uint32_t c = c0 + (uint32_t)wave;
    if (c < c1) fetch(c, va, vb);
    for (; c < c1; c += 8u) {
        const uint32_t cn = c + 4u;
        if (cn < c1) fetch(cn, wa, wb);
        stage(va, vb);
        __builtin_amdgcn_wave_barrier();
        mma();
        __builtin_amdgcn_wave_barrier();
        if (cn < c1) {
            if (cn + 4u < c1) fetch(cn + 4u, va, vb);
            stage(wa, wb);
            __builtin_amdgcn_wave_barrier();
            mma();
            __builtin_amdgcn_wave_barrier();
        }
    }

    float* out = part + ((size_t)(split * 4u + (uint32_t)wave) * T + tap) * (size_t)cout * cin;
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int n = 0; n < NN; n++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                out[(size_t)(co0 + m * 16 + 4 * grp + r) * cin + ci0 + n * 16 + r16] = acc[m][n][r];
}

// Weight gradient of the 9 taps of one z shift of a 3^3 convolution for one
// 16 x 16 block of (co, ci), rows of 32 NS voxels (NS = 1, 2): one wavefront a
// split, whose chunks (32 voxels of a row) it takes in order.  It marches along
// the rows of a plane: per row it stages the row of x that comes into reach and
// the row of dy ahead in LDS, two rows ahead through registers, holds the dy
// fragments of the 3 rows that an x row meets and shifts the x fragment in
// registers, so 2 fragment reads feed 9 MFMAs.  (All 27 taps in one wavefront
// leave one per SIMD and its latencies open.)  Both operands lie channels-last
// in LDS, 32 bytes a voxel; ds_read_b64_tr_b16 hands each lane 4 voxels of one
// channel.  Each 8 voxels start 384 bytes after the last (those of two lane
// groups lie on different banks).
// part[split][tap][co][ci]; from the middle z shift's wavefronts of the first
// ci block the bias sums part_b[split][co], voxel by voxel: lane group g adds
// its 8 voxels and hands the sum on to the next.  (Wavefronts of their own for
// them read dy once more: 64^3 x 8, 16 -> 48 243 us.)
// Bound: at 16 -> 16 channels the partials and the reads of x and dy, with more
// output channels the lines of dy that several channel blocks read.  Measured
// (MI355X, whole call): 64^3 x 8, 16 -> 16 78 us, 48 -> 16 149 us, 32^3 x 16, 64
// -> 64 232 us (27 shifted copies of a row staged per chunk, k_bwd_w27: 187, 644
// and 584 us).
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 tr_frag(const uint16_t* lo, const uint16_t* hi)
{
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)hi);
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
}

// the value of the lanes 16 below (lane groups 0 -> 1 -> 2 -> 3 -> 0)
template <int FROM>
__device__ __forceinline__ float hand_on(float v)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    // 32_swap: first result (own 0-31, other's 0-31), second (own 32-63, other's 32-63);
    // 16_swap: first (own row 0, other's 0, own 2, other's 2), second (own 1, other's 1, own 3, other's 3)
    if constexpr (FROM % 2 == 0) {
        const u32x2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return __builtin_bit_cast(float, (uint32_t)r[0]);                  // rows 0 0 2 2
    } else {
        const u32x2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        const uint32_t o = r[1];                                           // rows 1 1 3 3
        const u32x2 q = __builtin_amdgcn_permlane32_swap(o, o, false, false);
        return __builtin_bit_cast(float, FROM == 1 ? (uint32_t)q[0] : (uint32_t)q[1]);  // 1 1 1 1 or 3 3 3 3
    }
}

// The fragments of x at x - 1 and x + 1 from the one at x (8 voxels of a row
// per lane; the words before and after them, 0 past the row's ends).  Three
// reads of LDS in their place were what bound the weight gradients.
struct Shifts {
    bf16x8 at[3];
};
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t join(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_alignbit(hi, lo, 16); }

// ROW4: the 8 voxels are two rows of 4
template <bool ROW4>
__device__ __forceinline__ Shifts shifts_of(bf16x8 f, uint32_t before, uint32_t after)
{
    const u32x4 e = __builtin_bit_cast(u32x4, f);
    const uint32_t m1 = join(e[0], e[1]), m2 = join(e[1], e[2]), m3 = join(e[2], e[3]);
    u32x4 l, r;
    if constexpr (ROW4) {
        l = u32x4{e[0] << 16, m1, m2 & 0xffff0000u, m3};
        r = u32x4{m1, m2 & 0xffffu, m3, e[3] >> 16};
    } else {
        l = u32x4{join(before, e[0]), m1, m2, m3};
        r = u32x4{m1, m2, m3, join(e[3], after)};
    }
    return Shifts{{__builtin_bit_cast(bf16x8, l), f, __builtin_bit_cast(bf16x8, r)}};
}

// a word of the lane group before / after (cyclic)
__device__ __forceinline__ uint32_t group_before(uint32_t u, int grp)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 a = __builtin_amdgcn_permlane16_swap(u, u, false, false);        // rows 0 0 2 2, 1 1 3 3
    const u32x2 q = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);  // rows 1 1 1 1, 3 3 3 3
    return grp & 1 ? (uint32_t)a[0] : grp ? (uint32_t)q[0] : (uint32_t)q[1];
}
__device__ __forceinline__ uint32_t group_after(uint32_t u, int grp)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const u32x2 q = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);  // rows 0 0 0 0, 2 2 2 2
    return grp & 1 ? (grp == 1 ? (uint32_t)q[1] : (uint32_t)q[0]) : (uint32_t)a[1];
}

template <int NS>
__global__ void __launch_bounds__(64)
    k_bwd_wr(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, float* __restrict__ part,
             float* __restrict__ part_b, Geo g, int cin, int cout, uint32_t chunks, uint32_t chunks_per_split,
             uint32_t pairs)
{
    constexpr int W = 32 * NS, OCT = 192;                      // halves of an octet's pitch
    constexpr int XR = W / 8 * OCT;                            // halves of a row
    constexpr int BUF = 2 * XR, NJ = 2 * NS;                  // 16-byte pieces per lane: NS of x, NS of dy
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];
    const int lane = (int)threadIdx.x;
    const int r16 = lane & 15, grp = lane >> 4;
    // consecutive workgroups of one XCD: the channel blocks and z shifts of one
    // split (they share its lines), then the next split
    const int mblocks = cout / 16;
    auto at = [](int v) { return (v >> 3) * OCT + (v & 7) * 16; };  // LDS halves of voxel v of a row
    // this lane's part of a fragment's first 4 voxels (8 grp .. + 3; the others 64 on)
    const int k0 = grp * OCT + (r16 >> 2) * 16 + 4 * (r16 & 3);
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t pair = id % pairs, split = id / pairs / 3u;
    const int dz = (int)(id / pairs % 3u);
    const int co0 = (int)(pair % (uint32_t)mblocks) * 16, ci0 = (int)(pair / (uint32_t)mblocks) * 16;
    const bool bias = part_b != nullptr && ci0 == 0 && dz == 1;
    if (bias) __builtin_amdgcn_s_setprio(3);  // its additions make it the longest

    f32x4 acc[9];
#pragma unroll
    for (int t = 0; t < 9; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float sb = 0.f;
    int to[NJ];
    uint32_t fx[NS], fd[NS];                                   // element offsets inside a row
#pragma unroll
    for (int j = 0; j < NS; j++) {
        const int p = lane + 64 * j, v = p >> 1, h = 8 * (p & 1);
        to[j] = at(v) + h;
        to[NS + j] = XR + at(v) + h;
        fx[j] = (uint32_t)(v * cin + ci0 + h);
        fd[j] = (uint32_t)(v * cout + co0 + h);
    }

    const uint32_t c1 = min(chunks, (split + 1) * chunks_per_split);
    for (uint32_t c = split * chunks_per_split; c < c1;) {
        // the part of one plane: rows ya .. yb - 1, in the first and the last
        // perhaps not both segments
        const uint32_t row0 = c / NS, P = row0 / (uint32_t)g.H;
        const uint32_t ce = min(c1, (P + 1) * (uint32_t)g.H * NS);
        const int ya = (int)(row0 - P * (uint32_t)g.H), yb = (int)((ce - 1) / NS - P * (uint32_t)g.H) + 1;
        const int sa = (int)(c % NS), se = (int)((ce - 1) % NS);
        const bool zin = (unsigned)((int)(P % (uint32_t)g.D) + dz - 1) < (unsigned)g.D;
        c = ce;
        uint4 R[3][NJ];
        // step s: the x row y = s of plane z + dz - 1, the dy row y = s + 1
        auto fetch = [&](int s, uint4* q) __attribute__((always_inline)) {
            const bool inx = zin && s <= yb && (unsigned)s < (unsigned)g.H, ind = s + 1 >= ya && s + 1 < yb;
            const uint16_t* px = x + (size_t)((P + (uint32_t)(dz - 1)) * (uint32_t)g.H + (uint32_t)s) * (uint32_t)(W * cin);
            const uint16_t* pd = dy + (size_t)(P * (uint32_t)g.H + (uint32_t)(s + 1)) * (uint32_t)(W * cout);
#pragma unroll
            for (int j = 0; j < NS; j++) {
                q[j] = inx ? *reinterpret_cast<const uint4*>(px + fx[j]) : uint4{0u, 0u, 0u, 0u};
                q[NS + j] = ind ? *reinterpret_cast<const uint4*>(pd + fd[j]) : uint4{0u, 0u, 0u, 0u};
            }
        };
        auto put = [&](int buf, const uint4* q) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NJ; j++) *reinterpret_cast<uint4*>(lds + buf * BUF + to[j]) = q[j];
        };
        bf16x8 A[3][NS];                                      // dy rows [y slot][segment]
        auto step = [&](auto phase, int s, int buf) __attribute__((always_inline)) {
            constexpr int ph = decltype(phase)::value;
            const uint16_t* L = lds + buf * BUF;
            put(buf ^ 1, R[(ph + 1) % 3]);
            fetch(s + 3, R[ph]);
            bf16x8 X[NS];
            uint32_t before[NS], after[NS];
#pragma unroll
            for (int sg = 0; sg < NS; sg++) {
                A[ph][sg] = tr_frag(L + XR + sg * 4 * OCT + k0, L + XR + sg * 4 * OCT + k0 + 64);
                X[sg] = tr_frag(L + sg * 4 * OCT + k0, L + sg * 4 * OCT + k0 + 64);
                const u32x4 e = __builtin_bit_cast(u32x4, X[sg]);
                before[sg] = group_before(e[3], grp);
                after[sg] = group_after(e[0], grp);
            }
            // past a row's ends 0; between its two segments the other one's (cyclic) word
            if constexpr (NS == 2) {
                before[1] = grp == 0 ? before[0] : before[1];
                after[0] = grp == 3 ? after[1] : after[0];
            }
            before[0] = grp == 0 ? 0u : before[0];
            after[NS - 1] = grp == 3 ? 0u : after[NS - 1];
#pragma unroll
            for (int sg = 0; sg < NS; sg++) {
                const Shifts B = shifts_of<false>(X[sg], before[sg], after[sg]);
                auto mine = [&](int d) { return d >= ya && d < yb && (NS == 1 || ((d > ya || sg >= sa) && (d < yb - 1 || sg <= se))); };
#pragma unroll
                for (int dyo = 0; dyo < 3; dyo++)             // dy row s + 1 - dyo
                    if (mine(s + 1 - dyo))
#pragma unroll
                        for (int dx = 0; dx < 3; dx++)
                            acc[3 * dyo + dx] = mfma(A[(ph + 3 - dyo) % 3][sg], B.at[dx], acc[3 * dyo + dx]);
                if (bias && mine(s + 1)) {
                    const u16x8 q = __builtin_bit_cast(u16x8, A[ph][sg]);
                    auto add = [&]() __attribute__((always_inline)) {
#pragma unroll
                        for (int i = 0; i < 8; i++) sb += __builtin_bit_cast(float, (uint32_t)q[i] << 16);
                    };
                    add();
                    sb = hand_on<0>(sb);
                    add();
                    sb = hand_on<1>(sb);
                    add();
                    sb = hand_on<2>(sb);
                    add();
                    sb = hand_on<3>(sb);
                }
            }
        };
        const int s0 = ya - 1;
        fetch(s0, R[0]);
        fetch(s0 + 1, R[1]);
        fetch(s0 + 2, R[2]);
        put(0, R[0]);
        int buf = 0;
        // three steps a turn (those past yb add nothing): with a way out after
        // each the accumulators do not stay in their registers
        for (int s = s0; s <= yb; s += 3) {
            step(std::integral_constant<int, 0>{}, s, buf);
            step(std::integral_constant<int, 1>{}, s + 1, buf ^ 1);
            step(std::integral_constant<int, 2>{}, s + 2, buf);
            buf ^= 1;
        }
    }
    float* out = part + ((size_t)split * 27 + 9 * dz) * cout * cin;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) out[((size_t)t * cout + co0 + 4 * grp + q) * cin + ci0 + r16] = acc[t][q];
    if (bias && grp == 0) part_b[(size_t)split * cout + co0 + r16] = sb;
}

// Weight gradient of the 9 taps of one z shift for one 16 x 16 block of (co,
// ci), rows of W = 4, 8 or 16 voxels, planes of at least 32.  Partial
// 4 s + v of k_bwd_w is the sum over every 4th chunk (32 voxels: 32 / W rows of
// a plane) from chunk v of split s; one wavefront adds the partials v, v + 4,
// .. of a slice of S in registers (the first of k_reduce_w's sums, in its order):
// written out one by one the partials' way through memory can take most of the
// time.  With S = 4 a wavefront has one partial (plan_w).  Per chunk it stages
// the rows of x that the taps reach and the chunk of dy in LDS, a chunk ahead,
// two more in registers on their way; fragments as in k_bwd_wr.
// part[4 slice + v][tap][co][ci].
// Measured (MI355X, whole call): 16^3 x 8, 64 -> 64 55 us; 16^3 x 16, 256 -> 128
// 353 us; 8^3 x 8, 64 -> 64 26 us (k_bwd_w: 88, 600 and 43 us).
template <int W>
__global__ void __launch_bounds__(64)
    k_bwd_wc(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, float* __restrict__ part, Geo g, int cin,
             int cout, uint32_t chunks_per_split, uint32_t partials, uint32_t S, uint32_t pairs)
{
    constexpr int RY = 32 / W, XRY = RY + 2;                     // rows of a chunk, source rows
    // LDS halves: a voxel 16; the pitches put the 4-voxel groups of two lane groups on different banks
    constexpr int XP = W == 16 ? 2 * 192 : W == 8 ? 192 : 96;    // a row of x (each 8 voxels 192)
    constexpr int XN = XRY * XP, BUF = XN + 4 * 192;         // x rows, then dy (8 voxels 192)
    constexpr int NV = XRY * W * 2, NX = (NV + 63) / 64;     // 16-byte pieces of x, per lane
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];
    const int lane = (int)threadIdx.x;
    const int r16 = lane & 15, grp = lane >> 4;
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t pair = id % pairs, slice = id / pairs / 12u, v4 = id / pairs / 3u & 3u;
    const int dz = (int)(id / pairs % 3u) - 1;
    const int mblocks = cout / 16;
    const int co0 = (int)(pair % (uint32_t)mblocks) * 16, ci0 = (int)(pair / (uint32_t)mblocks) * 16;
    // this lane's pieces of x: source row (from -1) and offsets
    int to[NX], rel[NX], row[NX];
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int p = lane + 64 * j, v = p >> 1, xv = v % W, ry = v / W;
        to[j] = ry * XP + (xv >> 3) * 192 + (xv & 7) * 16 + 8 * (p & 1);
        rel[j] = ((dz * g.H + ry - 1) * g.W + xv) * cin + ci0 + 8 * (p & 1);
        row[j] = p < NV ? ry : -1;
    }
    const uint32_t fd = (uint32_t)((lane >> 1) * cout + co0 + 8 * (lane & 1));
    const int dto = XN + (lane >> 4) * 192 + (lane >> 1 & 7) * 16 + 8 * (lane & 1);
    // this lane's part of a fragment's first and last 4 voxels
    const int lo = (r16 >> 2) * 16 + 4 * (r16 & 3);
    const int x0 = (W == 16 ? (grp >> 1) * XP + (grp & 1) * 192 : W == 8 ? grp * XP : 2 * grp * XP) + lo;
    const int x1 = x0 + (W == 4 ? XP : 64), do0 = XN + grp * 192 + lo, do1 = do0 + 64;

    const uint32_t n_chunks = g.V / 32u, k1 = min(partials, (slice + 1) * S);
    struct At {  // chunk c of partial k; past the partial's last one, the next partial's first
        uint32_t k, c;
    };
    auto settle = [&](At a) {
        while (a.k < k1 && a.c >= min(n_chunks, ((a.k >> 2) + 1) * chunks_per_split)) {
            a.k += 4;
            a.c = (a.k >> 2) * chunks_per_split + (a.k & 3u);
        }
        return a;
    };
    auto next = [&](At a) { return settle(At{a.k, a.c + 4}); };
    uint4 R[2][NX + 1];
    auto fetch = [&](At a, uint4* q) __attribute__((always_inline)) {
        const uint32_t v0 = a.c * 32u;
        const int y0 = (int)((v0 >> g.lw) & (uint32_t)(g.H - 1)), z0 = (int)((v0 >> (g.lw + g.lh)) & (uint32_t)(g.D - 1));
        const bool any = a.k < k1, zin = any && (unsigned)(z0 + dz) < (unsigned)g.D;
        const uint16_t* xs = x + (size_t)v0 * (uint32_t)cin;
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const bool in = zin && row[j] >= 0 && (unsigned)(y0 + row[j] - 1) < (unsigned)g.H;
            q[j] = in ? *reinterpret_cast<const uint4*>(xs + rel[j]) : uint4{0u, 0u, 0u, 0u};
        }
        q[NX] = any ? *reinterpret_cast<const uint4*>(dy + (size_t)v0 * (uint32_t)cout + fd) : uint4{0u, 0u, 0u, 0u};
    };
    auto put = [&](int buf, const uint4* q) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NX; j++)
            if (64 * (j + 1) <= NV || row[j] >= 0) *reinterpret_cast<uint4*>(lds + buf * BUF + to[j]) = q[j];
        *reinterpret_cast<uint4*>(lds + buf * BUF + dto) = q[NX];
    };
    f32x4 acc[9], sum[9];
#pragma unroll
    for (int t = 0; t < 9; t++) acc[t] = sum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // chunk a in buffer buf (and R[buf ^ 1]: the one after, R[buf]: the one after that)
    auto step = [&](auto bufc, const At& a, const At& b, const At& d) __attribute__((always_inline)) {
        constexpr int buf = decltype(bufc)::value;
        const uint16_t* L = lds + buf * BUF;
        put(buf ^ 1, R[buf ^ 1]);
        fetch(d, R[buf ^ 1]);
        const bf16x8 A = tr_frag(L + do0, L + do1);
#pragma unroll
        for (int dyo = 0; dyo < 3; dyo++) {
            const bf16x8 X = tr_frag(L + dyo * XP + x0, L + dyo * XP + x1);
            uint32_t before = 0u, after = 0u;                    // (rows of 16: the other half's word)
            if constexpr (W == 16) {
                const u32x4 e = __builtin_bit_cast(u32x4, X);
                // (the swaps run in all lanes, then the choice)
                const uint32_t eb = group_before(e[3], grp), ea = group_after(e[0], grp);
                before = grp & 1 ? eb : 0u;
                after = grp & 1 ? 0u : ea;
            }
            const Shifts B = shifts_of<W == 4>(X, before, after);
#pragma unroll
            for (int dx = 0; dx < 3; dx++) acc[3 * dyo + dx] = mfma(A, B.at[dx], acc[3 * dyo + dx]);
        }
        if (a.k != b.k)
#pragma unroll
            for (int t = 0; t < 9; t++) {
                sum[t] += acc[t];
                acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
    };
    const uint32_t k0 = slice * S + v4;
    At a = settle(At{k0, (k0 >> 2) * chunks_per_split + (k0 & 3u)});
    At b = next(a), d = next(b);
    fetch(a, R[0]);
    fetch(b, R[1]);
    put(0, R[0]);
    fetch(d, R[0]);
    // two chunks a turn (one past the last adds zeros)
    while (a.k < k1) {
        At e = next(d), f = next(e);
        step(std::integral_constant<int, 0>{}, a, b, e);
        step(std::integral_constant<int, 1>{}, b, d, f);
        a = d;
        b = e;
        d = f;
    }
    float* out = part + ((size_t)(4 * slice + v4) * 27 + 9 * (dz + 1)) * cout * cin;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) out[((size_t)t * cout + co0 + 4 * grp + q) * cin + ci0 + r16] = sum[t][q];
}

// Weight gradient of all 27 taps of a 3^3 convolution for a (16*NM) x 16
// block of (co, ci), rows of 128 voxels and more.  grid.x = splits,
// grid.y = channel blocks.  The workgroup walks 32-voxel chunks (one row
// segment each): it stages the chunk's dy (32 voxels x 16*NM channels) and,
// for every tap, the input the tap reads (the 9 neighbour row segments, each
// in the 3 x shifts: 27 tiles of 16 channels x 32 voxels) transposed into
// LDS [channel][voxel], so every MFMA fragment is one 16-byte LDS read and
// each input element is fetched from memory once per chunk instead of once
// per tap.  Wave w accumulates taps w, w+4, ..., w+24; one partial per split:
// part[split][tap][co][ci].
// With part_b, the workgroups of the first input-channel block also sum the
// staged dy over their voxels (bias gradient): part_b[split][co].
template <int NM>
__global__ void __launch_bounds__(256)
    k_bwd_w27(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
              float* __restrict__ part, float* __restrict__ part_b, Geo g, int cin, int cout,
              uint32_t chunks_per_split)
{
    constexpr int CM = 16 * NM, CN = 16, T = 27, TW = 7;
    constexpr int PITCH = 40;                            // halves per LDS row (32 voxels + pad)
    constexpr int XITEMS = T * 8 * 2;                    // (tile, voxel quad, 8-channel group)
    constexpr int DITEMS = 8 * (CM / 8);                 // (voxel quad, 8-channel group)
    __shared__ __attribute__((aligned(16))) uint16_t lx[T * CN * PITCH];
    __shared__ __attribute__((aligned(16))) uint16_t ld[CM * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, grp = lane >> 4;
    const int mblocks = cout / CM;
    const int co0 = (int)(blockIdx.y % mblocks) * CM;
    const int ci0 = (int)(blockIdx.y / mblocks) * CN;

    f32x4 acc[TW][NM];
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
        for (int m = 0; m < NM; m++) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

    // this thread's staging items: x items tid, tid + 256 (< XITEMS), dy item tid (< DITEMS)
    uint4 qx[2][4], qd[4];
    auto fetch = [&](uint32_t c) {
        const uint32_t v0 = c * 32u;
        const int x0 = (int)(v0 & (uint32_t)(g.W - 1));
        const int y0 = (int)((v0 >> g.lw) & (uint32_t)(g.H - 1));
        const int z0 = (int)((v0 >> (g.lw + g.lh)) & (uint32_t)(g.D - 1));
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int it = tid + 256 * k;
            const int tile = it >> 4, quad = (it >> 1) & 7, cg = it & 1;
            int dz, dyo, dx;
            tap_offset<3>(tile, dz, dyo, dx);
            const bool row = it < XITEMS && (unsigned)(z0 + dz) < (unsigned)g.D &&
                             (unsigned)(y0 + dyo) < (unsigned)g.H;
            const int64_t base = (int64_t)v0 + (int64_t)(dz * g.H + dyo) * g.W + dx;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int pos = 4 * quad + t;
                const bool ok = row && (unsigned)(x0 + pos + dx) < (unsigned)g.W;
                qx[k][t] = ok ? *reinterpret_cast<const uint4*>(x + (size_t)(base + pos) * cin + ci0 + 8 * cg)
                              : uint4{0u, 0u, 0u, 0u};
            }
        }
        {
            const int quad = tid / (CM / 8), cg = tid % (CM / 8);
#pragma unroll
            for (int t = 0; t < 4; t++)
                qd[t] = tid < DITEMS ? *reinterpret_cast<const uint4*>(dy + (size_t)(v0 + 4u * quad + t) * cout +
                                                                      co0 + 8 * cg)
                                     : uint4{0u, 0u, 0u, 0u};
        }
    };
    // channel j of two voxels' 8-channel words -> one 32-bit word (voxel a low)
    auto pair = [](const uint4& a, const uint4& b, int j) {
        const uint32_t wa = (j >> 1) == 0 ? a.x : (j >> 1) == 1 ? a.y : (j >> 1) == 2 ? a.z : a.w;
        const uint32_t wb = (j >> 1) == 0 ? b.x : (j >> 1) == 1 ? b.y : (j >> 1) == 2 ? b.z : b.w;
        return (j & 1) ? ((wa >> 16) | (wb & 0xffff0000u)) : ((wa & 0xffffu) | (wb << 16));
    };
    // 4 voxels x 8 channels -> eight 8-byte LDS writes (4 voxels of one channel each)
    auto put = [&](uint16_t* tile, int ch, int quad, const uint4* q4) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t w2[2] = {pair(q4[0], q4[1], j), pair(q4[2], q4[3], j)};
            __builtin_memcpy(__builtin_assume_aligned(tile + (ch + j) * PITCH + 4 * quad, 8), w2, 8);
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int it = tid + 256 * k;
            if (it < XITEMS) put(lx + (it >> 4) * CN * PITCH, 8 * (it & 1), (it >> 1) & 7, qx[k]);
        }
        if (tid < DITEMS) put(ld, 8 * (tid % (CM / 8)), tid / (CM / 8), qd);
    };
    auto frag = [&](const uint16_t* row) {
        uint4 t;
        __builtin_memcpy(&t, __builtin_assume_aligned(row, 16), 16);
        return __builtin_bit_cast(bf16x8, t);
    };

    const uint32_t n_chunks = g.V / 32u;
    const uint32_t c0 = blockIdx.x * chunks_per_split;
    const uint32_t c1 = min(n_chunks, c0 + chunks_per_split);
    const bool bias = part_b != nullptr && ci0 == 0 && tid < CM;
    float sb = 0.f;
    if (c0 < c1) fetch(c0);
    for (uint32_t c = c0; c < c1; c++) {
        stage();
        __syncthreads();
        if (c + 1 < c1) fetch(c + 1);
        if (bias)
            for (int v = 0; v < 32; v++) sb += __builtin_bit_cast(float, (uint32_t)ld[tid * PITCH + v] << 16);
        bf16x8 a[NM];
#pragma unroll
        for (int m = 0; m < NM; m++) a[m] = frag(ld + (m * 16 + r16) * PITCH + 8 * grp);
#pragma unroll
        for (int t = 0; t < TW; t++) {
            const int tap = wave + 4 * t;
            if (tap < T) {
                const bf16x8 b = frag(lx + (tap * CN + r16) * PITCH + 8 * grp);
#pragma unroll
                for (int m = 0; m < NM; m++) acc[t][m] = mfma(a[m], b, acc[t][m]);
            }
        }
        __syncthreads();
    }

    if (bias) part_b[(size_t)blockIdx.x * cout + co0 + tid] = sb;
#pragma unroll
    for (int t = 0; t < TW; t++) {
        const int tap = wave + 4 * t;
        if (tap >= T) continue;
        float* out = part + ((size_t)blockIdx.x * T + tap) * (size_t)cout * cin;
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                out[(size_t)(co0 + m * 16 + 4 * grp + r) * cin + ci0 + r16] = acc[t][m][r];
    }
}

// dw[co][tap][ci] = sum_p part[p][tap][co][ci] in two fixed-order levels
// (deterministic, coalesced over the outputs, 64 outputs per workgroup with
// 4 threads per output adding every 4th partial, the four sums combined in
// a fixed order):
//   level 1 (grid.y = G slices of S partials): the sum of slice y replaces
//            its first partial, part[y*S] (only this workgroup touches it)
//   level 2: dw = sum over y of part[y*S]
__global__ void __launch_bounds__(256)
    k_reduce_w(float* __restrict__ part, int P, int S, int T, int cin, int cout, float* __restrict__ dw,
               int level)
{
    __shared__ float lds[4][64];
    const size_t n = (size_t)cout * T * cin;
    const int e = threadIdx.x & 63, k0 = threadIdx.x >> 6;
    const size_t i = (size_t)blockIdx.x * 64 + e;
    const size_t stride = (size_t)T * cout * cin;
    size_t at = 0;
    float s = 0.f;
    if (i < n) {
        const int ci = (int)(i % cin);
        const int tap = (int)((i / cin) % T);
        const int co = (int)(i / ((size_t)cin * T));
        at = ((size_t)tap * cout + co) * cin + ci;
        if (level == 1) {
            const int k1 = min(P, (int)(blockIdx.y + 1) * S);
            for (int k = (int)blockIdx.y * S + k0; k < k1; k += 4) s += part[(size_t)k * stride + at];
        } else {
            for (int y = k0; y * S < P; y += 4) s += part[(size_t)y * S * stride + at];
        }
    }
    lds[k0][e] = s;
    __syncthreads();
    if (k0 == 0 && i < n) {
        const float t = ((lds[0][e] + lds[1][e]) + lds[2][e]) + lds[3][e];
        if (level == 1)
            part[(size_t)blockIdx.y * S * stride + at] = t;
        else
            dw[i] = t;
    }
}

// Per-channel sums of dy over voxel ranges: part[blockIdx.x][c].  Thread (j, c)
// adds every rows-th voxel from the j-th, then the threads of a channel are
// added in order.  The range goes through LDS, 16 bytes a lane and 16 voxels a
// thread at a time, the next ones on their way: read 2 bytes a lane and one
// voxel after another it was bound by the latency of its loads.  Ranges of one
// or two voxels a thread are read directly, without the barriers (8^3, 64
// channels 2.8 us, through LDS 3.5; 12 voxels a thread 6.2 against 3.7).
// Measured (MI355X, 64^3, batch 8, with the sum of the partials): 16 channels 22
// us, 48 channels 56 us (before 73 and 240 us).
__global__ void __launch_bounds__(256)
    k_colsum(const uint16_t* __restrict__ dy, uint32_t V, int C, uint32_t per_block,
             float* __restrict__ part)
{
    __shared__ __attribute__((aligned(16))) uint16_t tile[16 * 256];
    __shared__ float lds[256];
    const int rows = 256 / C;  // C <= 256; threads past rows*C idle
    const int c = threadIdx.x % C, j = threadIdx.x / C;
    const uint32_t v0 = blockIdx.x * per_block, v1 = min(V, v0 + per_block);
    const uint32_t step = 16u * (uint32_t)rows, pieces = step * (uint32_t)C / 8u;  // voxels and 16-byte pieces a turn
    uint4 q[2];
    auto fetch = [&](uint32_t v) __attribute__((always_inline)) {
        const uint32_t n = v < v1 ? min(pieces, (v1 - v) * (uint32_t)C / 8u) : 0u;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t p = threadIdx.x + 256u * k;
            q[k] = p < n ? *reinterpret_cast<const uint4*>(dy + (size_t)v * C + 8u * p) : uint4{0u, 0u, 0u, 0u};
        }
    };
    float s = 0.f;
    if (per_block <= 2u * (uint32_t)rows) {
        if (j < rows)
            for (uint32_t v = v0 + (uint32_t)j; v < v1; v += (uint32_t)rows)
                s += __builtin_bit_cast(float, (uint32_t)dy[(size_t)v * C + c] << 16);
    } else {
        fetch(v0);
        for (uint32_t v = v0; v < v1; v += step) {
            __syncthreads();                                  // the last turn's reads are done
#pragma unroll
            for (int k = 0; k < 2; k++)
                if (threadIdx.x + 256u * k < pieces) *reinterpret_cast<uint4*>(tile + 8u * (threadIdx.x + 256u * k)) = q[k];
            __syncthreads();
            fetch(v + step);
            if (j < rows)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int at = j + i * rows;
                    if (v + (uint32_t)at < v1) s += __builtin_bit_cast(float, (uint32_t)tile[at * C + c] << 16);
                }
        }
    }
    lds[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < C) {
        float t = 0.f;
        for (int k = 0; k < rows; k++) t += lds[k * C + threadIdx.x];
        part[(size_t)blockIdx.x * C + threadIdx.x] = t;
    }
}

// out[c] = sum_k part[k][c]: one workgroup per channel, fixed-order tree
__global__ void __launch_bounds__(256)
    k_reduce_cols(const float* __restrict__ part, int P, int C, float* __restrict__ out)
{
    __shared__ float lds[256];
    const int c = (int)blockIdx.x;
    float s = 0.f;
    for (int k = threadIdx.x; k < P; k += 256) s += part[(size_t)k * C + c];
    lds[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) lds[threadIdx.x] += lds[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[c] = lds[0];
}

// grid.y selects the convolution of the table
__global__ void __launch_bounds__(256)
    k_flip(const uint16_t* __restrict__ w_all, uint16_t* __restrict__ wt_all, FlipTable tab)
{
    const FlipEntry f = tab.e[blockIdx.y];
    const uint16_t* w = w_all + f.off;
    uint16_t* wt = wt_all + f.off;
    const uint32_t n = (uint32_t)(f.cout * f.taps * f.cin);
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        // i indexes wt[ci][tap][co]
        const int co = (int)(i % (uint32_t)f.cout);
        const int tap = (int)((i / (uint32_t)f.cout) % (uint32_t)f.taps);
        const int ci = (int)(i / (uint32_t)(f.cout * f.taps));
        wt[i] = w[((uint32_t)co * f.taps + (f.taps - 1 - tap)) * f.cin + ci];
    }
}

Geo geo_of(const Shape& s)
{
    Geo g;
    g.V = (uint32_t)((uint64_t)s.n * s.d * s.h * s.w);
    g.D = s.d;
    g.H = s.h;
    g.W = s.w;
    g.lw = __builtin_ctz((unsigned)s.w);
    g.lh = __builtin_ctz((unsigned)s.h);
    return g;
}

bool pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

template <typename F>
int by_ks(int ks, F&& f)
{
    if (ks == 3) { f(std::integral_constant<int, 3>{}); return NX_OK; }
    if (ks == 1) { f(std::integral_constant<int, 1>{}); return NX_OK; }
    return set_error(NX_ERR_INVALID, "conv3d: kernel size must be 1 or 3");
}

// largest supported tile count (8, 6, 4, 3, 2, 1) dividing c16 = channels/16,
// at most `cap`
int tiles_of(int c16, int cap)
{
    for (int t : {8, 6, 4, 3, 2})
        if (t <= cap && c16 % t == 0) return t;
    return 1;
}

// The kernel of a shape.  Beside the order of the sums (above) it follows the
// row length; grids of less than the staged blocks' 4 rows and planes and rows of
// 1 or 2 voxels take their fragments from global memory (k_fwd).
int launch_fwd(const Shape& s, const uint16_t* x, const uint16_t* w, const float* bias, const uint16_t* mask,
               void* y, int flags, int keep, hipStream_t st)
{
    const Geo g = geo_of(s);
    if (g.V == 0) return NX_OK;
    using std::integral_constant;
    const integral_constant<int, 1> i1{};
    const integral_constant<int, 2> i2{};
    if (s.ks == 1) {
        const int nco = tiles_of(s.cout / 16, 4);
        const dim3 grid((g.V + 255u) / 256u, (unsigned)(s.cout / (16 * nco)));
        auto go = [&](auto NCO) {
            hipLaunchKernelGGL((k_pw<decltype(NCO)::value>), grid, dim3(256), 0, st, x, w, bias, mask, y, g.V, s.cin,
                               s.cout, flags, keep);
        };
        switch (nco) {
            case 4: go(integral_constant<int, 4>{}); break;
            case 3: go(integral_constant<int, 3>{}); break;
            case 2: go(i2); break;
            default: go(i1); break;
        }
        return NX_OK;
    }
    const bool flat = s.h < 4 || s.d < 4;
    if (s.w >= 32 && !flat && s.cin == 16) {
        const uint32_t cb = (uint32_t)s.cout / 16u;
        const uint32_t planes = (uint32_t)((s.w / 32) * ((s.h + 7) / 8)) * (uint32_t)s.n * (uint32_t)s.d;
        const uint32_t splits = std::max(1u, std::min(256u / cb, planes)), per = (planes + splits - 1) / splits;
        hipLaunchKernelGGL(k_fwd_z16, dim3((planes + per - 1) / per * cb), dim3(512), 0, st, x, w, bias, mask, y, g,
                           s.cout, flags, planes, per);
        return NX_OK;
    }
    if (s.w >= 32 && !flat) {
        // two channel blocks a wavefront where cout allows it (three or four
        // leave no registers for the loads)
        auto go = [&](auto NCO) {
            constexpr int nc = decltype(NCO)::value;
            const unsigned n = (unsigned)(s.n * (s.w / 32) * (s.h / 4) * (s.d / 4)) * (unsigned)(s.cout / (16 * nc));
            hipLaunchKernelGGL((k_fwd_blk<nc>), dim3(n), dim3(256), 0, st, x, w, bias, mask, y, g, s.cin, s.cout, flags);
        };
        if (s.cout % 32 == 0) go(i2);
        else go(i1);
        return NX_OK;
    }
    if (s.w >= 4 && s.w < 32 && !flat) {
        auto go = [&](auto WX, auto CMAX, auto NCO, auto NCW) {
            constexpr int wx = decltype(WX)::value, cm = decltype(CMAX)::value, nco = decltype(NCO)::value,
                          ncw = decltype(NCW)::value, bz = wx == 16 ? 2 : 4;
            const unsigned n = (unsigned)(s.n * (s.h / 4) * (s.d / bz)) * (unsigned)(s.cout / (16 * nco * ncw));
            hipLaunchKernelGGL((k_fwd_tap<wx, cm, nco, ncw>), dim3(n), dim3(256), 0, st, x, w, bias, mask, y, g, s.cin,
                               s.cout, flags);
        };
        auto by_cout = [&](auto WX, auto CMAX) {
            // 64 output channels a workgroup where that still gives one per CU
            const unsigned blocks = (unsigned)(s.n * (s.h / 4) * (s.d / (s.w == 16 ? 2 : 4)));
            if (s.cout % 64 == 0 && blocks * (unsigned)(s.cout / 64) >= 256u) go(WX, CMAX, i2, i2);
            else if (s.cout % 32 == 0) go(WX, CMAX, i2, i1);
            else go(WX, CMAX, i1, i1);
        };
        auto by_cin = [&](auto WX) {
            if (s.cin <= 64) by_cout(WX, integral_constant<int, 64>{});
            else if (s.cin <= 128) by_cout(WX, integral_constant<int, 128>{});
            else by_cout(WX, integral_constant<int, 256>{});
        };
        switch (s.w) {
            case 16: by_cin(integral_constant<int, 16>{}); break;
            case 8: by_cin(integral_constant<int, 8>{}); break;
            default: by_cin(integral_constant<int, 4>{}); break;
        }
        return NX_OK;
    }
    const int nt = tiles_of(s.cout / 16, 8);
    const dim3 grid((g.V + 127u) / 128u, (unsigned)(s.cout / (16 * nt)));
    auto go = [&](auto NT) {
        hipLaunchKernelGGL((k_fwd<decltype(NT)::value>), grid, dim3(256), 0, st, x, w, bias, mask, y, g, s.cin, s.cout,
                           flags);
    };
    switch (nt) {
        case 8: go(integral_constant<int, 8>{}); break;
        case 6: go(integral_constant<int, 6>{}); break;
        case 4: go(integral_constant<int, 4>{}); break;
        case 3: go(integral_constant<int, 3>{}); break;
        case 2: go(i2); break;
        default: go(i1); break;
    }
    return NX_OK;
}

constexpr uint32_t kColBlocks = 512;

// How a weight gradient is cut up; the cut decides the order of the sums, so
// it follows the shape alone.  Rows of >= 32 voxels: 768 splits (three
// workgroups of k_bwd_w27 per CU) over its channel blocks, at most 16 M partial
// floats; k_bwd_wr takes one wavefront per split and 16 x 16 channel block.
// part_splits bounds the splits of every smaller batch too (a network's
// workspace is sized once for its largest).
struct WPlan {
    int nm, nn, T;
    bool all_taps;
    uint32_t chunks, per, splits, part_splits;
    uint32_t partials, slices, S;   // partials per output element, added slice by slice (S each)
    bool staged, classes;           // k_bwd_wc; it adds every 4th partial of a slice itself
};

WPlan plan_w(const Shape& s)
{
    WPlan p{};
    p.T = s.ks * s.ks * s.ks;
    p.all_taps = s.ks == 3 && s.w >= 32;
    p.nm = tiles_of(s.cout / 16, 4);
    p.chunks = (uint32_t)(((uint64_t)s.n * s.d * s.h * s.w + 31) / 32);
    if (p.all_taps) {
        p.nn = 1;
        const uint32_t blocks = (uint32_t)((s.cout / (16 * p.nm)) * (s.cin / 16));
        const uint32_t cap = (uint32_t)std::max<uint64_t>(1, (16ull << 20) / ((uint64_t)27 * s.cout * s.cin));
        p.part_splits = std::max(1u, std::min({(768u + blocks - 1) / blocks, cap, p.chunks}));
    } else {
        p.nn = tiles_of(s.cin / 16, 4);
        const uint32_t blocks = (uint32_t)(p.T * (s.cout / (16 * p.nm)) * (s.cin / (16 * p.nn)));
        p.part_splits = std::max(1u, std::min({(2048u + blocks - 1) / blocks, 512u, (p.chunks + 3u) / 4u}));
    }
    p.per = (p.chunks + p.part_splits - 1) / p.part_splits;
    p.splits = (p.chunks + p.per - 1) / p.per;
    p.partials = p.all_taps ? p.splits : 4 * p.splits;
    const uint32_t G = std::max(1u, std::min(64u, p.partials / 32));
    p.S = (p.partials + G - 1) / G;
    p.slices = (p.partials + p.S - 1) / p.S;
    // k_bwd_wc, except where there is little to do (chunks x channel blocks: its
    // start costs 3 us; 16 -> 16 at 8^3 x 3 16.7 against 12.5 us, 64 -> 64 at 4 x 8 x 4
    // 13.6 and 11.9, from 256 on even or faster).  A wavefront per class of partials
    // has chunks / (4 slices) chunks to take one after another, one per partial
    // writes nm nn x 8.4 MB; even at 8 chunks per nm nn (16 -> 16 at 16^3 x 3, 10
    // chunks: 18.5 and 16.5 us; 32 -> 32 x 8, 28: 31.3 and 30.0; 128 -> 128 x 8, 128:
    // 109.8 and 110.0; 112 -> 16 x 8, 256: 139 and 28; 64 -> 64 x 8, 28: 46 and 65).
    p.staged = s.ks == 3 && s.w >= 4 && s.w < 32 && s.w * s.h >= 32 &&
               (uint64_t)p.chunks * (uint32_t)(s.cout / 16) * (uint32_t)(s.cin / 16) > 256;
    p.classes = p.staged && p.chunks <= 32u * p.slices * (uint32_t)(p.nm * p.nn);
    return p;
}

}  // namespace

int check(const Shape& s)
{
    if (s.n < 1 || !pow2(s.d) || !pow2(s.h) || !pow2(s.w))
        return set_error(NX_ERR_INVALID, "conv3d: batch >= 1 and power-of-two depth/height/width required");
    if (s.cin < 16 || s.cin % 16 || s.cout < 16 || s.cout % 16 || s.cin > 256 || s.cout > 256)
        return set_error(NX_ERR_INVALID, "conv3d: channel counts must be multiples of 16 in [16, 256]");
    if (s.ks != 1 && s.ks != 3) return set_error(NX_ERR_INVALID, "conv3d: kernel size must be 1 or 3");
    if ((uint64_t)s.n * s.d * s.h * s.w * std::max(s.cin, s.cout) >= (1ull << 31))
        return set_error(NX_ERR_INVALID, "conv3d: tensor too large (2^31 elements)");
    return NX_OK;
}

int fwd(const Shape& s, const uint16_t* x, const uint16_t* w, const float* bias, void* y, int flags,
        hipStream_t st, int keep)
{
    if (int e = launch_fwd(s, x, w, bias, nullptr, y, flags, keep ? keep : s.cout, st)) return e;
    NX_CHECK_LAUNCH("k_fwd");
    return NX_OK;
}

int flip(const FlipTable& tab, const uint16_t* w, uint16_t* wt, hipStream_t st)
{
    uint32_t most = 1;
    for (int k = 0; k < tab.n; k++)
        most = std::max(most, (uint32_t)(tab.e[k].cout * tab.e[k].taps * tab.e[k].cin));
    hipLaunchKernelGGL(k_flip, dim3(std::min((most + 255u) / 256u, 4096u), (unsigned)tab.n), dim3(256), 0, st, w, wt, tab);
    NX_CHECK_LAUNCH("k_flip");
    return NX_OK;
}

int bwd_data(const Shape& s, const uint16_t* dy, const uint16_t* wt, const uint16_t* mask, void* dx, int flags,
             hipStream_t st)
{
    Shape t = s;
    t.cin = s.cout;
    t.cout = s.cin;
    if (int e = launch_fwd(t, dy, wt, nullptr, mask, dx, flags & kOutF32, s.cin, st)) return e;
    NX_CHECK_LAUNCH("k_fwd (bwd-data)");
    return NX_OK;
}

// weight partials (k_bwd_w's column sums take their place afterwards), then
// the bias partials of the all-taps kernels
size_t bwd_weight_ws(const Shape& s)
{
    const WPlan p = plan_w(s);
    const size_t nw = (size_t)p.T * s.cout * s.cin, cols = (size_t)kColBlocks * s.cout;
    if (p.all_taps) return (size_t)p.part_splits * (nw + s.cout) * sizeof(float);
    return std::max(4 * p.part_splits * nw, cols) * sizeof(float);
}

int bwd_weight(const Shape& s, const uint16_t* x, const uint16_t* dy, float* dw, float* db, void* ws,
               hipStream_t st)
{
    const Geo g = geo_of(s);
    const WPlan p = plan_w(s);
    const size_t nw = (size_t)s.cout * p.T * s.cin;
    float* part = static_cast<float*>(ws);
    float* part_b = db && p.all_taps ? part + (size_t)p.splits * nw : nullptr;
    if (p.all_taps && s.w <= 64) {
        const uint32_t pairs = (uint32_t)((s.cout / 16) * (s.cin / 16));
        const dim3 grid(3 * p.splits * pairs);
        if (s.w == 64)
            hipLaunchKernelGGL((k_bwd_wr<2>), grid, dim3(64), 0, st, x, dy, part, part_b, g, s.cin, s.cout, p.chunks, p.per,
                               pairs);
        else
            hipLaunchKernelGGL((k_bwd_wr<1>), grid, dim3(64), 0, st, x, dy, part, part_b, g, s.cin, s.cout, p.chunks, p.per,
                               pairs);
        NX_CHECK_LAUNCH("k_bwd_wr");
    } else if (p.all_taps) {
        const dim3 grid(p.splits, (unsigned)((s.cout / (16 * p.nm)) * (s.cin / 16)));
        auto go27 = [&](auto NM) {
            hipLaunchKernelGGL((k_bwd_w27<decltype(NM)::value>), grid, dim3(256), 0, st, x, dy, part, part_b, g, s.cin,
                               s.cout, p.per);
        };
        switch (p.nm) {
            case 4: go27(std::integral_constant<int, 4>{}); break;
            case 3: go27(std::integral_constant<int, 3>{}); break;
            case 2: go27(std::integral_constant<int, 2>{}); break;
            default: go27(std::integral_constant<int, 1>{}); break;
        }
        NX_CHECK_LAUNCH("k_bwd_w27");
    } else if (p.staged) {
        const uint32_t pairs = (uint32_t)((s.cout / 16) * (s.cin / 16));
        auto go = [&](auto W) {
            hipLaunchKernelGGL((k_bwd_wc<decltype(W)::value>), dim3(12 * (p.classes ? p.slices : p.splits) * pairs), dim3(64),
                               0, st, x, dy, part, g, s.cin, s.cout, p.per, p.partials, p.classes ? p.S : 4u, pairs);
        };
        switch (s.w) {
            case 16: go(std::integral_constant<int, 16>{}); break;
            case 8: go(std::integral_constant<int, 8>{}); break;
            default: go(std::integral_constant<int, 4>{}); break;
        }
        NX_CHECK_LAUNCH("k_bwd_wc");
    } else {
        const dim3 grid(p.T * p.splits, (unsigned)((s.cout / (16 * p.nm)) * (s.cin / (16 * p.nn))));
        const int err = by_ks(s.ks, [&](auto KS) {
            auto go = [&](auto NM, auto NN) {
                hipLaunchKernelGGL((k_bwd_w<decltype(NM)::value, decltype(NN)::value, KS>), grid, dim3(256), 0, st, x, dy,
                                   part, g, s.cin, s.cout, p.per);
            };
            auto by_nn = [&](auto NM) {
                switch (p.nn) {
                    case 4: go(NM, std::integral_constant<int, 4>{}); break;
                    case 3: go(NM, std::integral_constant<int, 3>{}); break;
                    case 2: go(NM, std::integral_constant<int, 2>{}); break;
                    default: go(NM, std::integral_constant<int, 1>{}); break;
                }
            };
            switch (p.nm) {
                case 4: by_nn(std::integral_constant<int, 4>{}); break;
                case 3: by_nn(std::integral_constant<int, 3>{}); break;
                case 2: by_nn(std::integral_constant<int, 2>{}); break;
                default: by_nn(std::integral_constant<int, 1>{}); break;
            }
        });
        if (err) return err;
        NX_CHECK_LAUNCH("k_bwd_w");
    }
    // level 1 in slices of S partials (k_bwd_wc leaves 4 of each slice), then the slice sums
    const int P = (int)(p.classes ? 4 * p.slices : p.partials), S = p.classes ? 4 : (int)p.S;
    const unsigned gx = (unsigned)((nw + 63) / 64);
    hipLaunchKernelGGL(k_reduce_w, dim3(gx, p.slices), dim3(256), 0, st, part, P, S, p.T, s.cin, s.cout, dw, 1);
    hipLaunchKernelGGL(k_reduce_w, dim3(gx), dim3(256), 0, st, part, P, S, p.T, s.cin, s.cout, dw, 2);
    NX_CHECK_LAUNCH("k_reduce_w");
    if (part_b) {
        hipLaunchKernelGGL(k_reduce_cols, dim3(s.cout), dim3(256), 0, st, part_b, (int)p.splits, s.cout, db);
        NX_CHECK_LAUNCH("k_reduce_cols");
    } else if (db) {
        // the column partials reuse the workspace after the weight reduction
        const uint32_t per = (g.V + kColBlocks - 1) / kColBlocks;
        hipLaunchKernelGGL(k_colsum, dim3(kColBlocks), dim3(256), 0, st, dy, g.V, s.cout, per, part);
        NX_CHECK_LAUNCH("k_colsum");
        hipLaunchKernelGGL(k_reduce_cols, dim3(s.cout), dim3(256), 0, st, part, (int)kColBlocks, s.cout, db);
        NX_CHECK_LAUNCH("k_reduce_cols");
    }
    return NX_OK;
}

}  // namespace nx::conv

using namespace nx;

namespace {

int shape_of(const int32_t shape[4], int cin, int cout, int ks, conv::Shape& s)
{
    if (!shape) return set_error(NX_ERR_INVALID, "conv3d: null shape");
    s = conv::Shape{shape[0], shape[1], shape[2], shape[3], cin, cout, ks};
    return conv::check(s);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

extern "C" {

int nx_conv3d_fwd_bf16(const uint16_t* x, const uint16_t* w, const float* bias, void* y,
                       const int32_t shape[4], int32_t cin, int32_t cout, int32_t ksize, int32_t flags,
                       nx_stream s)
{
    conv::Shape sh;
    if (int e = shape_of(shape, cin, cout, ksize, sh)) return e;
    if (!x || !w || !y) return set_error(NX_ERR_INVALID, "nx_conv3d_fwd_bf16: null pointer");
    if (!aligned16(x) || !aligned16(w))
        return set_error(NX_ERR_INVALID, "nx_conv3d_fwd_bf16: x and w must be 16-byte aligned");
    return conv::fwd(sh, x, w, bias, y, flags & (conv::kRelu | conv::kOutF32), (hipStream_t)s);
}

int nx_conv3d_bwd_data_bf16(const uint16_t* dy, const uint16_t* w, void* dx, const int32_t shape[4],
                            int32_t cin, int32_t cout, int32_t ksize, int32_t flags, nx_stream s)
{
    conv::Shape sh;
    if (int e = shape_of(shape, cin, cout, ksize, sh)) return e;
    if (!dy || !w || !dx) return set_error(NX_ERR_INVALID, "nx_conv3d_bwd_data_bf16: null pointer");
    if (!aligned16(dy)) return set_error(NX_ERR_INVALID, "nx_conv3d_bwd_data_bf16: dy must be 16-byte aligned");
    void* ws = nullptr;
    const size_t nw = (size_t)cout * ksize * ksize * ksize * cin;
    if (int e = scratch(nw * sizeof(uint16_t), &ws)) return e;
    const conv::FlipTable tab{1, {{0, cin, cout, ksize * ksize * ksize}}};
    if (int e = conv::flip(tab, w, static_cast<uint16_t*>(ws), (hipStream_t)s)) return e;
    return conv::bwd_data(sh, dy, static_cast<uint16_t*>(ws), nullptr, dx, flags & conv::kOutF32, (hipStream_t)s);
}

int nx_conv3d_bwd_weight_bf16(const uint16_t* x, const uint16_t* dy, float* dw, float* db,
                              const int32_t shape[4], int32_t cin, int32_t cout, int32_t ksize,
                              nx_stream s)
{
    conv::Shape sh;
    if (int e = shape_of(shape, cin, cout, ksize, sh)) return e;
    if (!x || !dy || !dw) return set_error(NX_ERR_INVALID, "nx_conv3d_bwd_weight_bf16: null pointer");
    void* ws = nullptr;
    if (int e = scratch(conv::bwd_weight_ws(sh), &ws)) return e;
    return conv::bwd_weight(sh, x, dy, dw, db, ws, (hipStream_t)s);
}

}  // extern "C"
