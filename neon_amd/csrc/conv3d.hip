// BF16 3D convolution forward, backward-data and backward-weight on the gfx950
// matrix cores, FP32 accumulation (the learned warm start's network).  No
// counterpart in the reference.
//
// All three are implicit GEMMs.  On grids whose rows hold >= 32 voxels the
// operands are staged in LDS (the input block with its halo for the forward); smaller grids
// read their fragments straight from global memory (the 27-fold reuse of
// every input voxel served by L1/L2):
//   forward      M = voxels, N = cout, K = taps*cin      (A: 8 channels of one
//                tap per lane = one 16-byte load; B: 8 weights, 16 bytes);
//                for rows of >= 32 voxels the input block with its halo is
//                staged in LDS, 16 channels at a time (k_fwd_tile)
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

// One wave: 32 voxels x (16*NT) output channels; 4 waves per workgroup.
// grid.y selects the block of 16*NT output channels.
template <int NT, int KS>
__global__ void __launch_bounds__(256)
    k_fwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
          const float* __restrict__ bias, void* __restrict__ y, Geo g, int cin, int cout, int flags)
{
    constexpr int T = KS * KS * KS;
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
            tap_offset<KS>(tap, dz, dy, dx);
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
                    static_cast<uint16_t*>(y)[(size_t)v * cout + co] = f2bf(s);
            }
    }
}

// 3^3 forward (and backward-data) with the input tile in LDS, for rows of
// >= 32 voxels.  A workgroup computes a 32 x 4 x 4 block of output voxels
// (x, y, z).  For each slice of 16 input channels it stages the block's input
// with its one-voxel halo, 34 x 6 x 6 voxels x 16 channels (39 KB), in
// channels-last order (one 16-byte LDS write per load); each wave then
// takes 4 rows of 32 voxels, reads every A fragment (8 channels of one tap
// for one voxel) with one ds_read_b128, and uses each weight fragment for
// all of its rows.  Each input voxel is read from memory ~2x instead of 27x.
// CINC = 16 fixes the channel count (one slice, fewer registers); 0 reads it
// from the argument.
template <int NT, int CINC>
__global__ void __launch_bounds__(256)
    k_fwd_tile(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
               const float* __restrict__ bias, void* __restrict__ y, Geo g, int cin_arg, int cout, int flags)
{
    const int cin = CINC ? CINC : cin_arg;           // CINC: channel count fixed at compile time
    constexpr int TX = 32, TY = 4, TZ = 4, HX = TX + 2, HY = TY + 2, HZ = TZ + 2, CS = 16;
    constexpr int RW = TY * TZ / 4;                  // rows per wave
    constexpr int KS_ = 27 * CS, KC = (KS_ + 31) / 32;
    constexpr int ITEMS = HX * HY * HZ * (CS / 8);   // 16-byte pieces of one slice's halo tile
    __shared__ __attribute__((aligned(16))) uint16_t tile[HX * HY * HZ * CS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, grp = lane >> 4;
    const int co0 = (int)blockIdx.y * NT * 16;
    const int K = 27 * cin;
    // tile origin: blocks x fastest, then y, then z (z spans batch * depth)
    const int nbx = g.W / TX, nby = g.H / TY, nbz = g.D / TZ;
    const int bx = (int)(blockIdx.x % (uint32_t)nbx);
    const int by = (int)((blockIdx.x / (uint32_t)nbx) % (uint32_t)nby);
    const int bzall = (int)(blockIdx.x / (uint32_t)(nbx * nby));   // (sample, z block)
    const int sample = bzall / nbz, z0 = (bzall % nbz) * TZ, y0 = by * TY, x0 = bx * TX;
    const size_t sample_base = (size_t)sample * g.D * g.H * g.W;

    const uint16_t* wrow[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) wrow[n] = w + (size_t)(co0 + n * 16 + r16) * K;
    f32x4 acc[RW][2][NT];
#pragma unroll
    for (int j = 0; j < RW; j++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int n = 0; n < NT; n++) acc[j][t][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int c0 = 0; c0 < cin; c0 += CS) {
        if (c0) __syncthreads();                     // the previous slice's reads are done
        for (int it = tid; it < ITEMS; it += 256) {
            const int piece = it & 1, hv = it >> 1;
            const int hx = hv % HX, hy = (hv / HX) % HY, hz = hv / (HX * HY);
            const int gx = x0 - 1 + hx, gy = y0 - 1 + hy, gz = z0 - 1 + hz;
            uint4 v = uint4{0u, 0u, 0u, 0u};
            if ((unsigned)gx < (unsigned)g.W && (unsigned)gy < (unsigned)g.H && (unsigned)gz < (unsigned)g.D)
                v = *reinterpret_cast<const uint4*>(
                    x + (sample_base + ((size_t)gz * g.H + gy) * g.W + gx) * cin + c0 + 8 * piece);
            *reinterpret_cast<uint4*>(tile + (size_t)hv * CS + 8 * piece) = v;
        }
        __syncthreads();

        // K step kc of the slice: lane group grp holds tap (32 kc + 8 grp) / 16,
        // channels c0 + (8 grp) % 16 ..+7; past the last tap it contributes
        // zeros -- the MFMAs run for every lane (a lane left out of one would
        // not receive its accumulator rows)
        auto fetch_b = [&](int kc, bf16x8* b) {
            const int kk = kc * 32 + 8 * grp;
            const int tap = kk / CS, ci = kk % CS;
#pragma unroll
            for (int n = 0; n < NT; n++)
                b[n] = kk < KS_ ? ld8(wrow[n] + tap * cin + c0 + ci) : bf16x8{};
        };
        bf16x8 b0[NT], b1[NT];
        fetch_b(0, b0);
        for (int kc = 0; kc < KC; kc++) {
            if (kc + 1 < KC) fetch_b(kc + 1, b1);
            const int kk = kc * 32 + 8 * grp;
            const bool kok = kk < KS_;
            const int tap = kok ? kk / CS : 26, ci = kok ? kk % CS : 0;
            int dz, dyo, dx;
            tap_offset<3>(tap, dz, dyo, dx);
#pragma unroll
            for (int j = 0; j < RW; j++) {
                const int row = wave * RW + j;
                const int ly = row % TY, lz = row / TY;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const int hv = ((lz + dz + 1) * HY + (ly + dyo + 1)) * HX + (16 * t + r16 + dx + 1);
                    const bf16x8 a = kok ? ld8(tile + (size_t)hv * CS + ci) : bf16x8{};
#pragma unroll
                    for (int n = 0; n < NT; n++) acc[j][t][n] = mfma(a, b0[n], acc[j][t][n]);
                }
            }
#pragma unroll
            for (int n = 0; n < NT; n++) b0[n] = b1[n];
        }
    }

    const bool relu = flags & kRelu, f32out = flags & kOutF32;
#pragma unroll
    for (int j = 0; j < RW; j++) {
        const int row = wave * RW + j;
        const int ly = row % TY, lz = row / TY;
        const size_t vrow = sample_base + ((size_t)(z0 + lz) * g.H + (y0 + ly)) * g.W + x0;
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const int co = co0 + n * 16 + r16;
            const float bv = bias ? bias[co] : 0.f;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const size_t v = vrow + 16 * t + 4 * grp + r;
                    float sv = acc[j][t][n][r] + bv;
                    if (relu) sv = sv > 0.f ? sv : 0.f;
                    if (f32out)
                        static_cast<float*>(y)[v * cout + co] = sv;
                    else
                        static_cast<uint16_t*>(y)[v * cout + co] = f2bf(sv);
                }
        }
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

__global__ void __launch_bounds__(256)
    k_flip(const uint16_t* __restrict__ w, uint16_t* __restrict__ wt, int T, int cin, int cout)
{
    const size_t n = (size_t)cout * T * cin;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        // i indexes wt[ci][tap][co]
        const int co = (int)(i % cout);
        const int tap = (int)((i / cout) % T);
        const int ci = (int)(i / ((size_t)cout * T));
        wt[i] = w[((size_t)co * T + (T - 1 - tap)) * cin + ci];
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

int launch_fwd(const Shape& s, const uint16_t* x, const uint16_t* w, const float* bias, void* y,
               int flags, hipStream_t st)
{
    const Geo g = geo_of(s);
    if (g.V == 0) return NX_OK;
    // LDS-tiled kernel: 3^3, rows of >= 32 voxels, blocks of 32 x 4 x 4
    if (s.ks == 3 && s.w >= 32 && s.h >= 4 && s.d >= 4) {
        const int nt = tiles_of(s.cout / 16, 4);
        const dim3 grid((unsigned)((size_t)s.n * (s.d / 4) * (s.h / 4) * (s.w / 32)),
                        (unsigned)(s.cout / (16 * nt)));
        auto go = [&](auto NTc) {
            constexpr int NT = decltype(NTc)::value;
            if (s.cin == 16)
                hipLaunchKernelGGL((k_fwd_tile<NT, 16>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout,
                                   flags);
            else
                hipLaunchKernelGGL((k_fwd_tile<NT, 0>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout,
                                   flags);
        };
        switch (nt) {
            case 4: go(std::integral_constant<int, 4>{}); break;
            case 3: go(std::integral_constant<int, 3>{}); break;
            case 2: go(std::integral_constant<int, 2>{}); break;
            default: go(std::integral_constant<int, 1>{}); break;
        }
        return NX_OK;
    }
    const int nt = tiles_of(s.cout / 16, 8);
    const dim3 grid((g.V + 127u) / 128u, (unsigned)(s.cout / (16 * nt)));
    return by_ks(s.ks, [&](auto KS) {
        switch (nt) {
            case 8: hipLaunchKernelGGL((k_fwd<8, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
            case 6: hipLaunchKernelGGL((k_fwd<6, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
            case 4: hipLaunchKernelGGL((k_fwd<4, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
            case 3: hipLaunchKernelGGL((k_fwd<3, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
            case 2: hipLaunchKernelGGL((k_fwd<2, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
            default: hipLaunchKernelGGL((k_fwd<1, KS>), grid, dim3(256), 0, st, x, w, bias, y, g, s.cin, s.cout, flags); break;
        }
    });
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
        hipStream_t st)
{
    if (int e = launch_fwd(s, x, w, bias, y, flags, st)) return e;
    NX_CHECK_LAUNCH("k_fwd");
    return NX_OK;
}

int flip(const Shape& s, const uint16_t* w, uint16_t* wt, hipStream_t st)
{
    const int T = s.ks * s.ks * s.ks;
    const size_t n = (size_t)s.cout * T * s.cin;
    hipLaunchKernelGGL(k_flip, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0,
                       st, w, wt, T, s.cin, s.cout);
    NX_CHECK_LAUNCH("k_flip");
    return NX_OK;
}

int bwd_data(const Shape& s, const uint16_t* dy, const uint16_t* wt, void* dx, int flags,
             hipStream_t st)
{
    Shape t = s;
    t.cin = s.cout;
    t.cout = s.cin;
    if (int e = launch_fwd(t, dy, wt, nullptr, dx, flags & kOutF32, st)) return e;
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
    if (int e = conv::flip(sh, w, static_cast<uint16_t*>(ws), (hipStream_t)s)) return e;
    return conv::bwd_data(sh, dy, static_cast<uint16_t*>(ws), dx, flags & conv::kOutF32, (hipStream_t)s);
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
