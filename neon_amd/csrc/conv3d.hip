// BF16 3D convolution forward, backward-data and backward-weight on the gfx950
// matrix cores, FP32 accumulation (the learned warm start's network).  No
// counterpart in the reference.
//
// All three are implicit GEMMs:
//   forward      M = voxels, N = cout, K = taps*cin      (A: 8 channels of one
//                tap per lane = one 16-byte load; B: 8 weights, 16 bytes);
//                the input block with its halo is staged in LDS (k_fwd_blk, and
//                k_fwd_y16 for 16 channels); rows of 1 or 2 voxels read their
//                fragments from global memory (k_fwd), 1^3 kernels need no
//                halo (k_pw)
//   bwd-data     the forward on the flipped, transposed weights
//   bwd-weight   M = cout, N = cin, K = voxels (split over workgroups,
//                FP32 partials, fixed-order reduction): all 27 taps from one
//                staging of each row (k_bwd_wy, 3^3 on rows of >= 4 voxels),
//                else one tap per workgroup (k_bwd_w)
// MFMA 16x16x32 bf16 operand layout: lane l holds row (A) / column (B) l%16
// and the 8 K values of group l/16; D register r of lane l is row 4*(l/16)+r,
// column l%16.
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
            f32x4 o = acc[t][n];
            if (bias) o += bv;
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

// 3^3 on rows of 1 or 2 voxels.  One wave: 32 voxels x (16*NT) output
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

// 3^3 forward (and backward-data) with the input block in LDS, for rows of at
// least 4 voxels.  M = output channels (A: weights, one 16-byte load per
// lane), N = 16 voxels (B: 8 channels of a voxel, one ds_read_b128), K = 32
// channels of one tap, or for the last 16 channels of an odd count the taps
// (dx = -1, dx = 0) of a voxel pair, then dx = 1 alone.  A tile is 16 voxels:
// WX along x times YT = 16 / WX rows.  A wavefront computes RY x RZ tiles in y
// and z for NCO blocks of 16 output channels; NXW x NYW x NZW wavefronts share
// one staged block with its halo, CM channels (32, or 16 where the input has
// no more) at a time.  A B fragment serves every output row of the wavefront
// that a tap reaches from it and all NCO channel blocks (3 or 9 NCO MFMAs):
// with one LDS read per MFMA the LDS takes twice the MFMA's time.  A
// workgroup takes a run of blocks; the next slice of channels, or of the next
// block, is loaded into registers while the matrix cores work on this one,
// and the next weights likewise.  A lane ends with 4 consecutive channels of
// a voxel: 8- or 16-byte stores.
// Measured (MI355X): 64^3 x 8, 48 -> 16 157 us (225 us with one LDS read per
// MFMA, 16 channels at a time); 32^3 x 8, 96 -> 32 55 us (101); 32^3 x 16,
// 64 -> 64 165 us (250); 16^3 x 8, 64 -> 64 22 us (43, fragments from memory).
// mask: null, or the activations whose ReLU the result passes back through
// (0 where the activation is not positive).
template <int WX, int NXW, int NYW, int NZW, int RY, int RZ, int NCO, bool AHEAD>
__global__ void __launch_bounds__(256, 2)
    k_fwd_blk(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
              const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cin, int cout, int flags,
              uint32_t blocks, uint32_t per_wg)
{
    static_assert(NXW * NYW * NZW == 4, "four wavefronts");
    constexpr int CM = 32;                                       // channels of a full slice
    constexpr int YT = 16 / WX, SY = (RY - 1) * YT + 3;          // SY: source row offsets of a wavefront
    constexpr int BX = NXW * WX, BY = NYW * YT * RY, BZ = NZW * RZ;
    constexpr int HX = BX + 2, HY = BY + 2, HZ = BZ + 2, HV = HX * HY * HZ;
    constexpr int ROWS = HY * HZ;
    // 16-byte pieces of a slice per thread: own voxels, halo columns
    constexpr int NM = (ROWS * BX * (CM / 8) + 255) / 256, NH = (ROWS * 2 * (CM / 8) + 255) / 256;
    constexpr int ZG = NCO == 1 || (!AHEAD && NCO == 2) ? 1 : 3; // weight groups per K step: all dz, or one each
    constexpr int NDZ = 3 / ZG;
    __shared__ __attribute__((aligned(16))) uint16_t tile[HV * CM];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const uint32_t ncb = (uint32_t)(cout / (16 * NCO));
    const uint32_t nbx = (uint32_t)(g.W / BX), nby = (uint32_t)((g.H + BY - 1) / BY), nbz = (uint32_t)((g.D + BZ - 1) / BZ);
    const int wx = wave % NXW, wy = (wave / NXW) % NYW, wz = wave / (NXW * NYW);
    const int lx = r16 % WX, ly = r16 / WX;
    // halo-block voxel of this lane at offset (-1, -1, -1) of its first tile
    const int hv0 = (wz * RZ * HY + wy * YT * RY + ly) * HX + wx * WX + lx;

    // blocks of one XCD in order: channel blocks of a position, then x, y, z, sample
    struct Block {
        int co0, x0, y0, z0;
        uint32_t smp;
    };
    auto block_of = [&](uint32_t id) {
        Block b;
        b.co0 = (int)(id % ncb) * 16 * NCO;
        id /= ncb;
        b.x0 = (int)(id % nbx) * BX;
        id /= nbx;
        b.y0 = (int)(id % nby) * BY;
        id /= nby;
        b.z0 = (int)(id % nbz) * BZ;
        b.smp = id / nbz;
        return b;
    };
    // Staging: the block's own voxels by whole rows (BX x PV pieces, a power of
    // two; where a row fills a wavefront's load its address and its test are
    // scalar), then the two halo columns.  A slice is 32 channels (PV = 4
    // 16-byte pieces a voxel) or the last 16 (PV = 2).
    uint4 pre[NM], pre_h[NH];
    auto row_of = [&](auto pvc, int k, int& row, int& q) {
        constexpr int RP = BX * decltype(pvc)::value;
        const int at = (k * 4 + wave) * 64;
        if constexpr (RP >= 64) {
            row = at / RP;
            q = at % RP + lane;
        } else {
            row = at / RP + lane / RP;
            q = lane % RP;
        }
    };
    auto row_base = [&](const Block& b, int row, bool& in) {
        const int gy = b.y0 - 1 + row % HY, gz = b.z0 - 1 + row / HY;
        in = row < ROWS && (unsigned)gy < (unsigned)g.H && (unsigned)gz < (unsigned)g.D;
        return (uint32_t)((gz * g.H + gy) * g.W + b.x0);
    };
    auto fetch_pv = [&](auto pvc, const Block& b, int c0) __attribute__((always_inline)) {
        constexpr int PV = decltype(pvc)::value;
        const uint16_t* xs = x + (size_t)b.smp * (uint32_t)(g.D * g.H * g.W) * (uint32_t)cin + c0;
#pragma unroll
        for (int k = 0; k < (ROWS * BX * PV + 255) / 256; k++) {
            int row, q;
            row_of(pvc, k, row, q);
            bool in;
            const uint16_t* p = xs + (size_t)(row_base(b, row, in) * (uint32_t)cin);
            pre[k] = in ? *reinterpret_cast<const uint4*>(p + (uint32_t)((q / PV) * cin + 8 * (q % PV))) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int k = 0; k < (ROWS * 2 * PV + 255) / 256; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            bool in;
            const uint32_t v = row_base(b, row, in) + (side ? (uint32_t)BX : ~0u);
            in = in && (side ? b.x0 + BX < g.W : b.x0 > 0);
            pre_h[k] = in ? *reinterpret_cast<const uint4*>(xs + (uint32_t)(v * (uint32_t)cin + 8 * pc)) : uint4{0u, 0u, 0u, 0u};
        }
    };
    auto fetch = [&](const Block& b, int c0) __attribute__((always_inline)) {
        if (cin - c0 >= 32) fetch_pv(std::integral_constant<int, CM / 8>{}, b, c0);
        else fetch_pv(std::integral_constant<int, 2>{}, b, c0);
    };
    // the same without registers held: a batch of loads, then their LDS writes
    auto stage = [&](auto pvc, const Block& b, int c0) __attribute__((always_inline)) {
        constexpr int PV = decltype(pvc)::value, KM = (ROWS * BX * PV + 255) / 256, NB = 9;
        const uint16_t* xs = x + (size_t)b.smp * (uint32_t)(g.D * g.H * g.W) * (uint32_t)cin + c0;
        uint4 h[NH];
#pragma unroll
        for (int k = 0; k < (ROWS * 2 * PV + 255) / 256; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            bool in;
            const uint32_t v = row_base(b, row, in) + (side ? (uint32_t)BX : ~0u);
            in = in && (side ? b.x0 + BX < g.W : b.x0 > 0);
            h[k] = in ? *reinterpret_cast<const uint4*>(xs + (uint32_t)(v * (uint32_t)cin + 8 * pc)) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll 1
        for (int k0 = 0; k0 < KM; k0 += NB) {
            uint4 v[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) {
                int row, q;
                row_of(pvc, k0 + k, row, q);
                bool in;
                const uint16_t* p = xs + (size_t)(row_base(b, row, in) * (uint32_t)cin);
                v[k] = in ? *reinterpret_cast<const uint4*>(p + (uint32_t)((q / PV) * cin + 8 * (q % PV))) : uint4{0u, 0u, 0u, 0u};
            }
#pragma unroll
            for (int k = 0; k < NB; k++) {
                int row, q;
                row_of(pvc, k0 + k, row, q);
                if (row < ROWS) *reinterpret_cast<uint4*>(tile + (row * HX + 1) * PV * 8 + q * 8) = v[k];
            }
        }
#pragma unroll
        for (int k = 0; k < (ROWS * 2 * PV + 255) / 256; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            if (row < ROWS) *reinterpret_cast<uint4*>(tile + ((row * HX + (side ? HX - 1 : 0)) * PV + pc) * 8) = h[k];
        }
    };
    auto put = [&](auto pvc) {
        constexpr int PV = decltype(pvc)::value;
#pragma unroll
        for (int k = 0; k < (ROWS * BX * PV + 255) / 256; k++) {
            int row, q;
            row_of(pvc, k, row, q);
            if (row < ROWS) *reinterpret_cast<uint4*>(tile + (row * HX + 1) * PV * 8 + q * 8) = pre[k];
        }
#pragma unroll
        for (int k = 0; k < (ROWS * 2 * PV + 255) / 256; k++) {
            const int it = tid + 256 * k, row = it / (2 * PV), side = (it / PV) & 1, pc = it % PV;
            if (row < ROWS) *reinterpret_cast<uint4*>(tile + ((row * HX + (side ? HX - 1 : 0)) * PV + pc) * 8) = pre_h[k];
        }
    };

    const uint32_t first = xcd_remap(blockIdx.x, gridDim.x) * per_wg, last = min(blocks, first + per_wg);
    if (first >= last) return;
    f32x4 acc[RZ][RY][NCO];
    auto slice = [&](auto csc, const Block& b, int c0, const Block& nb, int nc0, bool more) __attribute__((always_inline)) {
        constexpr int CS = decltype(csc)::value, PV = CS / 8;
        constexpr int NK = CS == 32 ? 3 : 2;                     // K steps per (dz, dy): dx, or dx pairs
        const bool half = CS == 16 && grp >= 2;                  // the second tap of a pair
        const uint16_t* wb = w + (size_t)b.co0 * 27 * cin + c0;
        const uint32_t wo = (uint32_t)(r16 * 27 * cin + (CS == 32 ? 8 * grp : 8 * (grp & 1) + (grp >> 1) * cin));
        const uint16_t* tl = tile + hv0 * CS + 8 * grp;          // CS = 16: groups 2, 3 read the next voxel
        bf16x8 a[AHEAD ? 2 : 1][NDZ][3][NCO];
        // weight group wg = (K step, last first) * ZG + dz group; past dx = 1 a
        // pair has no second tap
        auto load_w = [&](int wg, bf16x8 (*d)[3][NCO]) {
            const int kx = NK - 1 - wg / ZG;
            const bool none = CS == 16 && kx == 1 && half;
#pragma unroll
            for (int i = 0; i < NDZ; i++)
#pragma unroll
                for (int dyo = 0; dyo < 3; dyo++)
#pragma unroll
                    for (int n = 0; n < NCO; n++) {
                        const int tap = ((wg % ZG + i) * 3 + dyo) * 3 + (CS == 32 ? kx : 2 * kx);
                        d[i][dyo][n] = none ? bf16x8{} : ld8(wb + (size_t)((n * 16 * 27 + tap) * cin) + wo);
                    }
        };
        auto load_x = [&](int kx, int zr, int s) {
            bf16x8 v = ld8(tl + ((zr * HY + s) * HX + (CS == 32 ? kx : 2 * kx)) * CS);
            if (CS == 16 && kx == 1 && half) v = bf16x8{};
            return v;
        };
        // Loads return in order, so a wait for weights would also wait for
        // the next slice if that was asked for first: it goes after the last
        // weights, which are never far ahead.
        constexpr int NG = NK * ZG;
        load_w(0, a[0]);
        if (AHEAD && NG == 2) load_w(1, a[1]);
        __syncthreads();                                         // the previous slice's reads are done
        if (AHEAD) put(std::integral_constant<int, PV>{});
        else stage(std::integral_constant<int, PV>{}, b, c0);
        __syncthreads();
        if (AHEAD && NG == 2 && more) fetch(nb, nc0);
        // steps of one source plane; its fragments are read while the matrix
        // cores work on the plane before where the registers allow it (NCO = 1)
        constexpr int NZR = RZ + NDZ - 1;
        constexpr bool PIPE = NCO == 1 && !AHEAD;
        bf16x8 v[PIPE ? 2 : 1][SY];
        auto plane = [&](int st) {
#pragma unroll
            for (int s = 0; s < SY; s++) v[PIPE ? st & 1 : 0][s] = load_x(NK - 1 - st / NZR / ZG, st % NZR + st / NZR % ZG, s);
        };
        if (PIPE) plane(0);
#pragma unroll
        for (int st = 0; st < NG * NZR; st++) {
            const int wg = st / NZR, zr = st % NZR;
            if (zr == 0) {
                if (AHEAD && NG > 2 && wg + 1 < NG) {
                    load_w(wg + 1, a[(wg + 1) & 1]);
                    if (wg + 2 == NG && more) fetch(nb, nc0);
                }
                if (!AHEAD && wg > 0) load_w(wg, a[0]);
            }
            if (PIPE && st + 1 < NG * NZR) plane(st + 1);
            if (PIPE || zr == 0) __builtin_amdgcn_sched_barrier(0);
            if (!PIPE) plane(st);
#pragma unroll
            for (int s = 0; s < SY; s++)
#pragma unroll
                for (int i = 0; i < NDZ; i++)
#pragma unroll
                    for (int dyo = 0; dyo < 3; dyo++) {
                        const int jz = zr - i, jt = s - dyo;
                        if (jz < 0 || jz >= RZ || jt < 0 || jt % YT || jt / YT >= RY) continue;
#pragma unroll
                        for (int n = 0; n < NCO; n++)
                            acc[jz][jt / YT][n] = mfma(a[AHEAD ? wg & 1 : 0][i][dyo][n], v[PIPE ? st & 1 : 0][s], acc[jz][jt / YT][n]);
                    }
        }
    };

    Block b = block_of(first);
    if (AHEAD) fetch(b, 0);
    for (uint32_t id = first; id < last; id++) {
#pragma unroll
        for (int i = 0; i < RZ; i++)
#pragma unroll
            for (int j = 0; j < RY; j++)
#pragma unroll
                for (int n = 0; n < NCO; n++) acc[i][j][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        const Block next = block_of(min(id + 1, last - 1));
        f32x4 bv[NCO];
#pragma unroll
        for (int n = 0; n < NCO; n++) {
            bv[n] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (bias)
#pragma unroll
                for (int r = 0; r < 4; r++) bv[n][r] = bias[b.co0 + n * 16 + 4 * grp + r];
        }
        for (int c0 = 0; c0 < cin;) {
            const int cn = c0 + (cin - c0 >= 32 ? 32 : 16);
            const bool end = cn >= cin, more = !end || id + 1 < last;
            if (cn - c0 == 32)
                slice(std::integral_constant<int, CM>{}, b, c0, end ? next : b, end ? 0 : cn, more);
            else
                slice(std::integral_constant<int, 16>{}, b, c0, end ? next : b, end ? 0 : cn, more);
            c0 = cn;
        }
        const bool relu = flags & kRelu, f32out = flags & kOutF32;
#pragma unroll
        for (int jz = 0; jz < RZ; jz++)
#pragma unroll
            for (int jy = 0; jy < RY; jy++) {
                const int gz = b.z0 + wz * RZ + jz, gy = b.y0 + (wy * RY + jy) * YT;
                if (gz >= g.D || gy + ly >= g.H) continue;
                const size_t v = (((size_t)b.smp * g.D + gz) * g.H + gy) * g.W + b.x0 + wx * WX;
#pragma unroll
                for (int n = 0; n < NCO; n++) {
                    f32x4 o = acc[jz][jy][n];
                    if (bias) o += bv[n];
                    if (relu)
#pragma unroll
                        for (int r = 0; r < 4; r++) o[r] = o[r] > 0.f ? o[r] : 0.f;
                    put4(y, mask, v * cout + b.co0 + n * 16, (uint32_t)((ly * g.W + lx) * cout + 4 * grp), o, f32out);
                }
            }
        b = next;
    }
}

// 3^3 forward (and backward-data) of a 16-channel input, rows of >= 32 voxels:
// the multiply-adds per voxel are too few there to hide a block's staging, so
// 8 wavefronts march along y over 8 z rows of 32 voxels instead.  The weights
// of a 16-channel output block stay in registers (18 K steps: per (dz, dy)
// the taps dx = -1, 0 of a voxel pair, then dx = 1), each x row is staged
// once, two rows ahead, and adds to the three output rows it reaches, whose
// accumulators turn with it.  The columns (x segment, 8 z rows, sample) times
// H rows are cut evenly into `splits` runs, one workgroup a CU.
// Bound: HBM (16 -> 16 reads and writes each voxel once) and the stores.
// Measured (MI355X, 64^3, batch 8): 16 -> 16 52 us, 16 -> 48 134 us (before,
// block by block: 67 and 227 us; k_fwd_blk's form: 75 and 172 us).
__global__ void __launch_bounds__(512)
    k_fwd_y16(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
              const uint16_t* __restrict__ mask, void* __restrict__ y, Geo g, int cout, int flags, uint32_t rows,
              uint32_t rows_per_split)
{
    constexpr int TZ = 8, XV = 34, PIECES = (TZ + 2) * XV * 2, NJ = (PIECES + 511) / 512, BUF = PIECES * 8 + 16;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    // the channel blocks of one run side by side on one XCD
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x), ncb = (uint32_t)cout / 16u;
    const int co0 = (int)(id % ncb) * 16;
    const uint32_t split = id / ncb;
    const int nxs = g.W / 32, nzb = (g.D + TZ - 1) / TZ;
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

    const uint32_t r1 = min(rows, (split + 1) * rows_per_split);
    for (uint32_t r = split * rows_per_split; r < r1;) {
        const uint32_t colm = r / (uint32_t)g.H;
        const int ya = (int)(r % (uint32_t)g.H);
        const int yb = min(g.H, ya + (int)(r1 - r));
        r += (uint32_t)(yb - ya);
        const int x0 = (int)(colm % (uint32_t)nxs) * 32, z0 = (int)((colm / (uint32_t)nxs) % (uint32_t)nzb) * TZ;
        const uint32_t smp = colm / (uint32_t)(nxs * nzb);
        const uint32_t sv = smp * (uint32_t)g.D;
        uint32_t off[NJ];
        bool ok[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int p = tid + 512 * j, hv = p >> 1, gx = x0 - 1 + hv % XV, gz = z0 - 1 + hv / XV;
            ok[j] = p < PIECES && (unsigned)gx < (unsigned)g.W && (unsigned)gz < (unsigned)g.D;
            off[j] = ((sv + (uint32_t)gz) * (uint32_t)(g.H * g.W) + (uint32_t)gx) * 16u + 8u * (uint32_t)(p & 1);
        }
        uint4 R[3][NJ];
        auto fetch = [&](int s, uint4* q) __attribute__((always_inline)) {
            const bool in = s <= yb && (unsigned)s < (unsigned)g.H;
#pragma unroll
            for (int j = 0; j < NJ; j++)
                q[j] = in && ok[j] ? *reinterpret_cast<const uint4*>(x + (size_t)(s * g.W * 16) + off[j])
                                   : uint4{0u, 0u, 0u, 0u};
        };
        auto put = [&](int buf, const uint4* q) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (tid + 512 * j < PIECES) *reinterpret_cast<uint4*>(lds + buf * BUF + (tid + 512 * j) * 8) = q[j];
        };
        const int zw = z0 + wave;
        f32x4 acc[3][2];                                      // [output row slot][x tile]
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k][0] = acc[k][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        // x row s; slots: output row s + 1 in ph, s in ph + 2, s - 1 in ph + 1 (mod 3)
        auto step = [&](auto phase, int s, int buf) __attribute__((always_inline)) {
            constexpr int ph = decltype(phase)::value;
            fetch(s + 3, R[ph]);
            acc[ph][0] = acc[ph][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (zw < g.D) {
                if ((unsigned)s < (unsigned)g.H) {
                    const uint16_t* L = lds + buf * BUF + (wave * XV + r16) * 16 + 8 * grp;
#pragma unroll
                    for (int dz = 2; dz >= 0; dz--)
#pragma unroll
                        for (int xt = 0; xt < 2; xt++)
#pragma unroll
                            for (int kx = 0; kx < 2; kx++) {
                                bf16x8 v = ld8(L + (dz * XV + xt * 16 + 2 * kx) * 16);
                                if (kx == 1 && half) v = bf16x8{};
#pragma unroll
                                for (int dyo = 0; dyo < 3; dyo++) {
                                    f32x4& c = acc[dyo == 0 ? ph : dyo == 1 ? (ph + 2) % 3 : (ph + 1) % 3][xt];
                                    c = mfma(a[dz][dyo][kx], v, c);
                                }
                            }
                }
                if (s > ya) {                                 // output row s - 1 is complete
                    const size_t v = ((size_t)(sv + (uint32_t)zw) * g.H + (s - 1)) * g.W + x0;
#pragma unroll
                    for (int xt = 0; xt < 2; xt++) {
                        f32x4 o = acc[(ph + 1) % 3][xt];
                        if (bias) o += bv;
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
        const int s0 = ya - 1;
        fetch(s0, R[0]);
        fetch(s0 + 1, R[1]);
        fetch(s0 + 2, R[2]);
        put(0, R[0]);
        __syncthreads();
        int buf = 0;
        for (int s = s0; s <= yb;) {
            step(std::integral_constant<int, 0>{}, s, buf);
            buf ^= 1;
            if (++s > yb) break;
            step(std::integral_constant<int, 1>{}, s, buf);
            buf ^= 1;
            if (++s > yb) break;
            step(std::integral_constant<int, 2>{}, s, buf);
            buf ^= 1;
            ++s;
        }
        __syncthreads();
    }
}

// Weight gradient of one tap for a (16*NM) x (16*NN) block of (co, ci): the
// 1^3 kernel, and 3^3 on rows of 1 or 2 voxels.
// grid.x = T * splits (tap fastest), grid.y = channel blocks.  Each wave
// takes every 4th 32-voxel chunk of its split; the four waves' sums are
// added in wave order: part[split][tap][co][ci], and part_b[split][co] (the
// bias sums) from the middle tap's workgroups of the first ci block.
// The GEMM's K index is the voxel, but channels are contiguous in memory:
// each wave loads its chunk of dy (32 voxels x 16*NM channels) and of the
// shifted input (32 voxels x 16*NN channels) with 16-byte loads and writes
// it transposed into its own LDS tile [channel][voxel], from which every
// MFMA fragment (8 consecutive voxels of one channel) is one ds_read_b128.
// The next chunk's global loads are issued before the current chunk's MFMAs.
template <int NM, int NN, int KS>
__global__ void __launch_bounds__(256)
    k_bwd_w(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
            float* __restrict__ part, float* __restrict__ part_b, Geo g, int cin, int cout,
            uint32_t chunks_per_split)
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
    const bool bias = part_b != nullptr && ci0 == 0 && tap == T / 2;
    f32x4 accb[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const u16x8 one8 = {0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80};
    const bf16x8 ones = __builtin_bit_cast(bf16x8, one8);

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
        if (bias)
#pragma unroll
            for (int m = 0; m < NM; m++) accb[m] = mfma(a[m], ones, accb[m]);
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

    // the four waves' sums, one 16 x 16 block at a time
    float* sum = reinterpret_cast<float*>(&lds[0][0]);
    float* out = part + ((size_t)split * T + tap) * (size_t)cout * cin;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int n = 0; n < NN; n++) {
#pragma unroll
            for (int r = 0; r < 4; r++) sum[wave * 256 + (4 * grp + r) * 16 + r16] = acc[m][n][r];
            __syncthreads();
            const int t = threadIdx.x;
            out[(size_t)(co0 + m * 16 + (t >> 4)) * cin + ci0 + n * 16 + (t & 15)] =
                ((sum[t] + sum[256 + t]) + sum[512 + t]) + sum[768 + t];
            __syncthreads();
        }
    if (bias) {
        if (r16 == 0)
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int r = 0; r < 4; r++) sum[wave * CM + m * 16 + 4 * grp + r] = accb[m][r];
        __syncthreads();
        const int t = threadIdx.x;
        if (t < CM) part_b[(size_t)split * cout + co0 + t] = ((sum[t] + sum[CM + t]) + sum[2 * CM + t]) + sum[3 * CM + t];
    }
}

// Weight gradient of all 27 taps of a 3^3 convolution for one 16 x 16 block
// of (co, ci), rows of at least 4 voxels.  512 threads (8 wavefronts).
// A wavefront takes K = 32 voxels of x at a time -- WS = min(W, 32) voxels
// of NZ = 32 / WS consecutive z rows -- and marches along y.  Per row it
// reads 3 fragments of x (the x shifts) and 3 of dy (the row just ahead, at
// the three z shifts) from LDS and holds the dy fragments of the 3 x 3
// neighbouring rows in registers, so 6 fragment reads feed 27 MFMAs: the
// LDS would otherwise bound it (one fragment read per MFMA takes the LDS
// twice the MFMA's time).  Both operands lie channels-last in LDS, 32 bytes
// per voxel; ds_read_b64_tr_b16 hands each lane 4 voxels of one channel, so
// a tap's shift is a row offset and nothing is transposed or staged twice.
// Rows reach LDS through registers, two rows ahead of the row in use.
// Bound: at 16 -> 16 channels the HBM reads and the MFMAs alike.
// Measured (MI355X, 64^3, batch 8): 16 -> 16 50 us, 48 -> 16 123 us (before,
// staging 27 shifted copies of x per row: 203 and 648 us); 16^3, 64 -> 64
// 24 us (one tap per workgroup: 90 us).
// Pairs of rows outside the grid are left out (a zero row would turn an
// infinite partner into NaN).  Work: the columns (x segment, 8 NZ z rows,
// sample) times H rows are one sequence of row steps, cut evenly into
// `splits` runs; part[split][tap][co][ci], and from the workgroups of the
// first ci block the bias sums part_b[split][co].
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

template <int WS>
__global__ void __launch_bounds__(512)
    k_bwd_wy(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, float* __restrict__ part,
             float* __restrict__ part_b, Geo g, int cin, int cout, uint32_t rows, uint32_t rows_per_split,
             uint32_t pairs)
{
    constexpr int NZ = 32 / WS, TZ = 8 * NZ, XV = WS + 2, T = 27;
    constexpr int XP = TZ * XV * 2, DP = (TZ + 2) * WS * 2;   // 16-byte pieces of an x and a dy row set
    constexpr int NJ = (XP + DP + 511) / 512;
    constexpr int RT = 4;                                     // taps per round of the final sum
    constexpr int BUF = (XP + DP) * 8;                        // halves per buffer
    constexpr int SUMH = 8 * RT * 256 * 2;                    // halves of the final sum's floats
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF > SUMH ? 2 * BUF : SUMH];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    // consecutive workgroups of one XCD: the channel blocks of one run (they
    // share its lines), then the next run
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t pair = id % pairs, split = id / pairs;
    const int mblocks = cout / 16;
    const int co0 = (int)(pair % (uint32_t)mblocks) * 16, ci0 = (int)(pair / (uint32_t)mblocks) * 16;
    const bool bias = part_b != nullptr && ci0 == 0;
    const int nxs = g.W / WS, nzb = (g.D + TZ - 1) / TZ;

    f32x4 acc[T], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const s16x4 one4 = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
    const bf16x8 ones = __builtin_bit_cast(bf16x8, __builtin_shufflevector(one4, one4, 0, 1, 2, 3, 4, 5, 6, 7));

    // this lane's two 4-voxel groups of a fragment: voxels 4 grp + r16 / 4 and 16 more
    const int k0 = 4 * grp + (r16 >> 2), k1 = k0 + 16, col = 4 * (r16 & 3);
    const int xo0 = ((wave * NZ + k0 / WS) * XV + k0 % WS) * 16 + col;
    const int xo1 = ((wave * NZ + k1 / WS) * XV + k1 % WS) * 16 + col;
    const int do0 = XP * 8 + ((wave * NZ + k0 / WS) * WS + k0 % WS) * 16 + col;
    const int do1 = XP * 8 + ((wave * NZ + k1 / WS) * WS + k1 % WS) * 16 + col;
    // z of the voxel groups this lane's 8 K values belong to (K value order:
    // voxels 4 grp .. 4 grp + 3, then the same 16 on)
    const int zk0 = (4 * grp) / WS, zk1 = (16 + 4 * grp) / WS;

    const uint32_t r1 = min(rows, (split + 1) * rows_per_split);
    for (uint32_t r = split * rows_per_split; r < r1;) {
        const uint32_t colm = r / (uint32_t)g.H;
        const int ya = (int)(r % (uint32_t)g.H);
        const int yb = min(g.H, ya + (int)(r1 - r));
        r += (uint32_t)(yb - ya);
        const int xs = (int)(colm % (uint32_t)nxs), zb = (int)((colm / (uint32_t)nxs) % (uint32_t)nzb);
        const int x0 = xs * WS, z0 = zb * TZ;
        const uint32_t smp = colm / (uint32_t)(nxs * nzb);

        // this thread's pieces of a step: where from (the row y = 0) and whether inside
        uint32_t off[NJ];
        bool ok[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int p = tid + 512 * j;
            const bool isx = p < XP;
            const int hv = (isx ? p : p - XP) >> 1, zr = isx ? hv / XV : hv / WS;
            const int gx = isx ? x0 - 1 + hv % XV : x0 + hv % WS, gz = isx ? z0 + zr : z0 - 1 + zr;
            ok[j] = p < XP + DP && (unsigned)gx < (unsigned)g.W && (unsigned)gz < (unsigned)g.D;
            const uint32_t v = ((smp * (uint32_t)g.D + (uint32_t)gz) * (uint32_t)g.H) * (uint32_t)g.W + (uint32_t)gx;
            off[j] = v * (uint32_t)(isx ? cin : cout) + (uint32_t)((isx ? ci0 : co0) + 8 * (p & 1));
        }
        uint4 R[3][NJ];
        // step s: the x rows y = s (from s = ya on) and the dy rows y = s + 1
        auto fetch = [&](int s, uint4* q) {
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const bool isx = tid + 512 * j < XP;
                const int yy = isx ? s : s + 1;
                const bool in = ok[j] && s < yb && (isx ? s >= ya : (unsigned)yy < (unsigned)g.H);
                const uint16_t* base = isx ? x : dy;
                q[j] = in ? *reinterpret_cast<const uint4*>(base + off[j] + (uint32_t)(yy * g.W) * (uint32_t)(isx ? cin : cout))
                          : uint4{0u, 0u, 0u, 0u};
            }
        };
        auto put = [&](int buf, const uint4* q) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (tid + 512 * j < XP + DP) *reinterpret_cast<uint4*>(lds + buf * BUF + (tid + 512 * j) * 8) = q[j];
        };
        const int zw = z0 + wave * NZ;                        // the wavefront's first z row
        bf16x8 A[3][3];                                       // [y slot][dz + 1]
        auto step = [&](auto phase, int s, int buf) {
            constexpr int ph = decltype(phase)::value;
            fetch(s + 3, R[ph]);
            const uint16_t* L = lds + buf * BUF;
            if (zw < g.D) {
#pragma unroll
                for (int dz = 0; dz < 3; dz++) A[ph][dz] = tr_frag(L + do0 + dz * WS * 16, L + do1 + dz * WS * 16);
                if (s >= ya) {
                    bf16x8 B[3];
#pragma unroll
                    for (int dx = 0; dx < 3; dx++) B[dx] = tr_frag(L + xo0 + dx * 16, L + xo1 + dx * 16);
#pragma unroll
                    for (int dz = 0; dz < 3; dz++) {          // dy row z + dz - 1
                        if (NZ == 1 && (unsigned)(zw + dz - 1) >= (unsigned)g.D) continue;
                        bf16x8 Bz[3];
#pragma unroll
                        for (int dx = 0; dx < 3; dx++) {
                            Bz[dx] = B[dx];
                            if (NZ > 1 && dz != 1) {
                                // K values whose dy row lies outside the grid
                                uint4 u = __builtin_bit_cast(uint4, B[dx]);
                                if ((unsigned)(zw + zk0 + dz - 1) >= (unsigned)g.D) u.x = u.y = 0u;
                                if ((unsigned)(zw + zk1 + dz - 1) >= (unsigned)g.D) u.z = u.w = 0u;
                                Bz[dx] = __builtin_bit_cast(bf16x8, u);
                            }
                        }
#pragma unroll
                        for (int dyo = 0; dyo < 3; dyo++) {   // dy row s + dyo - 1
                            if ((unsigned)(s + dyo - 1) >= (unsigned)g.H) continue;
                            const bf16x8 a = A[dyo == 2 ? ph : dyo == 1 ? (ph + 2) % 3 : (ph + 1) % 3][dz];
#pragma unroll
                            for (int dx = 0; dx < 3; dx++) {
                                const int tap = ((2 - dz) * 3 + (2 - dyo)) * 3 + dx;
                                acc[tap] = mfma(a, Bz[dx], acc[tap]);
                            }
                            if (dz == 1 && dyo == 1 && bias) accb = mfma(a, ones, accb);
                        }
                    }
                }
            }
            put(buf ^ 1, R[(ph + 1) % 3]);
            __syncthreads();
        };
        const int s0 = ya - 2;
        fetch(s0, R[0]);
        fetch(s0 + 1, R[1]);
        fetch(s0 + 2, R[2]);
        put(0, R[0]);
        __syncthreads();
        int buf = 0;
        for (int s = s0; s < yb;) {
            step(std::integral_constant<int, 0>{}, s, buf);
            buf ^= 1;
            if (++s >= yb) break;
            step(std::integral_constant<int, 1>{}, s, buf);
            buf ^= 1;
            if (++s >= yb) break;
            step(std::integral_constant<int, 2>{}, s, buf);
            buf ^= 1;
            ++s;
        }
        __syncthreads();
    }

    // the 8 wavefronts' sums, RT taps at a time, in wavefront order
    float* sum = reinterpret_cast<float*>(lds);
    float* out = part + (size_t)split * T * cout * cin;
#pragma unroll
    for (int t0 = 0; t0 < T; t0 += RT) {
#pragma unroll
        for (int t = 0; t < RT; t++)
            if (t0 + t < T) {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    sum[(wave * RT + t) * 256 + (4 * grp + q) * 16 + r16] = acc[t0 + t < T ? t0 + t : 0][q];
            }
        __syncthreads();
        for (int e = tid; e < RT * 256; e += 512) {
            const int t = t0 + e / 256, m = (e >> 4) & 15, n = e & 15;
            if (t < T) {
                float s = 0.f;
#pragma unroll
                for (int w = 0; w < 8; w++) s += sum[w * RT * 256 + e];
                out[((size_t)t * cout + co0 + m) * cin + ci0 + n] = s;
            }
        }
        __syncthreads();
    }
    if (bias) {
        if (r16 == 0)
#pragma unroll
            for (int q = 0; q < 4; q++) sum[wave * 16 + 4 * grp + q] = accb[q];
        __syncthreads();
        if (tid < 16) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < 8; w++) s += sum[w * 16 + tid];
            part_b[(size_t)split * cout + co0 + tid] = s;
        }
    }
}

// dw[co][tap][ci] = sum_p part[p][tap][co][ci] (and db[co] = sum_p
// part_b[p][co], the last workgroups), in a fixed order: 16 groups of
// threads each add every 16th partial, then the 16 sums are added in order.
// A thread holds 4 consecutive ci (one 16-byte load per partial).
__global__ void __launch_bounds__(256)
    k_reduce_w(const float* __restrict__ part, const float* __restrict__ part_b, int P, int T, int cin, int cout,
               float* __restrict__ dw, float* __restrict__ db)
{
    __shared__ float4 lds[256];
    const int e = threadIdx.x & 15, k0 = threadIdx.x >> 4;
    const size_t n = (size_t)cout * T * cin, nq = n / 4;
    const size_t i = (size_t)blockIdx.x * 16 + e;
    const bool isb = i >= nq;                          // the bias rows follow the weights
    const size_t ib = i - nq;
    const bool ok = !isb || (db != nullptr && ib < (size_t)cout / 4);
    const float* src = isb ? part_b + 4 * ib : part + 4 * i;
    const size_t stride = isb ? (size_t)cout : n;
    float4 s = float4{0.f, 0.f, 0.f, 0.f};
    if (ok)
        for (int k = k0; k < P; k += 16) {
            const float4 v = *reinterpret_cast<const float4*>(src + (size_t)k * stride);
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
    lds[threadIdx.x] = s;
    __syncthreads();
    if (k0 != 0 || !ok) return;
    float4 t = lds[e];
    for (int k = 1; k < 16; k++) {
        const float4 v = lds[16 * k + e];
        t.x += v.x;
        t.y += v.y;
        t.z += v.z;
        t.w += v.w;
    }
    if (isb) {
        float* o = db + 4 * ib;                        // (the caller's arrays: 4-byte aligned)
        o[0] = t.x, o[1] = t.y, o[2] = t.z, o[3] = t.w;
    } else {
        // part order [tap][co][ci] -> dw order [co][tap][ci]
        const int c4 = cin / 4;
        const int ci = (int)(i % c4) * 4, co = (int)((i / c4) % cout), tap = (int)(i / ((size_t)c4 * cout));
        float* o = dw + ((size_t)co * T + tap) * cin + ci;
        o[0] = t.x, o[1] = t.y, o[2] = t.z, o[3] = t.w;
    }
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

int launch_fwd(const Shape& s, const uint16_t* x, const uint16_t* w, const float* bias, const uint16_t* mask,
               void* y, int flags, int keep, hipStream_t st)
{
    const Geo g = geo_of(s);
    if (g.V == 0) return NX_OK;
    if (s.ks == 1) {
        const int nco = tiles_of(s.cout / 16, 4);
        const dim3 grid((g.V + 255u) / 256u, (unsigned)(s.cout / (16 * nco)));
        auto go = [&](auto NCO) {
            hipLaunchKernelGGL((k_pw<decltype(NCO)::value>), grid, dim3(256), 0, st, x, w, bias, mask, y, g.V, s.cin,
                               s.cout, flags, keep);
        };
        switch (nco) {
            case 4: go(std::integral_constant<int, 4>{}); break;
            case 3: go(std::integral_constant<int, 3>{}); break;
            case 2: go(std::integral_constant<int, 2>{}); break;
            default: go(std::integral_constant<int, 1>{}); break;
        }
        return NX_OK;
    }
    if (s.w >= 32 && s.cin == 16) {
        const uint32_t cb = (uint32_t)s.cout / 16u;
        const uint32_t rows = (uint32_t)((s.w / 32) * ((s.d + 7) / 8)) * (uint32_t)s.n * (uint32_t)s.h;
        const uint32_t splits = std::max(1u, std::min(256u / cb, rows)), per = (rows + splits - 1) / splits;
        hipLaunchKernelGGL(k_fwd_y16, dim3((rows + per - 1) / per * cb), dim3(512), 0, st, x, w, bias, mask, y, g,
                           s.cout, flags, rows, per);
        return NX_OK;
    }
    // rows of >= 4 voxels: the block kernel.  Its block follows the row's
    // length, smaller per wavefront on small grids (which would leave CUs
    // idle); two channel blocks a wavefront where cout allows it (three or
    // four leave no registers for the loads).  Blocks of small grids load the
    // next slice ahead; the large block's slice would not fit the registers,
    // there the second workgroup of the CU hides the staging.
    if (s.w >= 4) {
        auto go = [&](auto WX, auto NXW, auto NYW, auto NZW, auto RY, auto RZ, auto NCO, auto AHEAD) {
            constexpr int wx = decltype(WX)::value, nx_ = decltype(NXW)::value, ny = decltype(NYW)::value,
                          nz = decltype(NZW)::value, ry = decltype(RY)::value, rz = decltype(RZ)::value,
                          nc = decltype(NCO)::value;
            constexpr bool ahead = decltype(AHEAD)::value;
            constexpr int bx = nx_ * wx, by = ny * (16 / wx) * ry, bz = nz * rz;
            const unsigned n = (unsigned)(s.n * (s.w / bx) * ((s.h + by - 1) / by) * ((s.d + bz - 1) / bz)) *
                               (unsigned)(s.cout / (16 * nc));
            const unsigned per = (n + 511u) / 512u;  // two workgroups per CU
            hipLaunchKernelGGL((k_fwd_blk<wx, nx_, ny, nz, ry, rz, nc, ahead>), dim3((n + per - 1) / per), dim3(256), 0,
                               st, x, w, bias, mask, y, g, s.cin, s.cout, flags, n, per);
        };
        using std::integral_constant;
        const integral_constant<int, 1> i1{};
        const integral_constant<int, 2> i2{};
        const integral_constant<int, 4> i4{};
        const integral_constant<int, 8> i8{};
        const integral_constant<int, 16> i16{};
        const std::true_type yes{};
        const std::false_type no{};
        const bool even = s.cout % 32 == 0;
        if (s.w >= 32) {
            if (even) go(i16, i2, i1, i2, i4, i2, i2, no);
            else go(i16, i2, i1, i2, i4, i2, i1, no);
        } else if (s.w == 16) {
            if (even) go(i16, i1, i2, i2, i2, i2, i2, yes);
            else go(i16, i1, i2, i2, i2, i2, i1, yes);
        } else if (s.w == 8) {
            go(i8, i1, i2, i2, i1, i2, i1, yes);
        } else {
            go(i4, i1, i1, i4, i1, i1, i1, yes);
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
        case 8: go(std::integral_constant<int, 8>{}); break;
        case 6: go(std::integral_constant<int, 6>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        default: go(std::integral_constant<int, 1>{}); break;
    }
    return NX_OK;
}

// How a weight gradient is cut up.  k_bwd_wy (3^3, rows of >= 4 voxels: its
// LDS row sets fit two buffers down to 4-voxel rows) takes one workgroup per
// CU and 16 x 16 channel block; fewer, longer runs would leave CUs idle, more
// would only add partials.  part_splits bounds the splits of every smaller
// batch too (the workspace is sized once for the largest).
struct WPlan {
    int T;
    bool rows_kernel;
    int nm, nn;                     // k_bwd_w
    uint32_t pairs, rows, per;      // k_bwd_wy: channel blocks, row steps, row steps per split
    uint32_t splits, part_splits;
};

WPlan plan_w(const Shape& s)
{
    WPlan p{};
    p.T = s.ks * s.ks * s.ks;
    p.rows_kernel = s.ks == 3 && s.w >= 4;
    uint32_t units;
    if (p.rows_kernel) {
        const int ws = std::min(s.w, 32), tz = 8 * (32 / ws);
        p.pairs = (uint32_t)((s.cout / 16) * (s.cin / 16));
        units = p.rows = (uint32_t)((s.w / ws) * ((s.d + tz - 1) / tz)) * (uint32_t)s.n * (uint32_t)s.h;
        p.part_splits = std::max(1u, std::min(256u / p.pairs, units));
    } else {
        p.nm = tiles_of(s.cout / 16, 4);
        p.nn = tiles_of(s.cin / 16, 4);
        units = (uint32_t)(((uint64_t)s.n * s.d * s.h * s.w + 31) / 32);
        const uint32_t blocks = (uint32_t)(p.T * (s.cout / (16 * p.nm)) * (s.cin / (16 * p.nn)));
        p.part_splits = std::max(1u, std::min({(2048u + blocks - 1) / blocks, 512u, (units + 3u) / 4u}));
    }
    p.per = (units + p.part_splits - 1) / p.part_splits;
    p.splits = (units + p.per - 1) / p.per;
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

// weight partials, then bias partials
size_t bwd_weight_ws(const Shape& s)
{
    const WPlan p = plan_w(s);
    return (size_t)p.part_splits * ((size_t)p.T * s.cout * s.cin + s.cout) * sizeof(float);
}

int bwd_weight(const Shape& s, const uint16_t* x, const uint16_t* dy, float* dw, float* db, void* ws,
               hipStream_t st)
{
    const Geo g = geo_of(s);
    const WPlan p = plan_w(s);
    const size_t nw = (size_t)s.cout * p.T * s.cin;
    float* part = static_cast<float*>(ws);
    float* part_b = db ? part + (size_t)p.splits * nw : nullptr;
    if (p.rows_kernel) {
        auto go = [&](auto WS) {
            hipLaunchKernelGGL((k_bwd_wy<decltype(WS)::value>), dim3(p.splits * p.pairs), dim3(512), 0, st, x, dy,
                               part, part_b, g, s.cin, s.cout, p.rows, p.per, p.pairs);
        };
        switch (std::min(s.w, 32)) {
            case 32: go(std::integral_constant<int, 32>{}); break;
            case 16: go(std::integral_constant<int, 16>{}); break;
            case 8: go(std::integral_constant<int, 8>{}); break;
            default: go(std::integral_constant<int, 4>{}); break;
        }
        NX_CHECK_LAUNCH("k_bwd_wy");
    } else {
        const dim3 grid(p.T * p.splits, (unsigned)((s.cout / (16 * p.nm)) * (s.cin / (16 * p.nn))));
        const int err = by_ks(s.ks, [&](auto KS) {
            auto go = [&](auto NM, auto NN) {
                hipLaunchKernelGGL((k_bwd_w<decltype(NM)::value, decltype(NN)::value, KS>), grid, dim3(256), 0, st,
                                   x, dy, part, part_b, g, s.cin, s.cout, p.per);
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
    const size_t quads = nw / 4 + (db ? (size_t)s.cout / 4 : 0);
    hipLaunchKernelGGL(k_reduce_w, dim3((unsigned)((quads + 15) / 16)), dim3(256), 0, st, part, part_b, (int)p.splits,
                       p.T, s.cin, s.cout, dw, db);
    NX_CHECK_LAUNCH("k_reduce_w");
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
