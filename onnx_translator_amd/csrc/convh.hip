// convh.hip — float16 Conv2d on the f16 matrix cores of gfx950.
//
// tensor_ops/tensor_ops.c:1036-1114 with f16 X and W: every product of two halves is
// exact in f32 and the sums are f32 (v_mfma_f32_32x32x16_f16), the tolerance class of
// the f32 convolution; the result is rounded once to the output type.  The implicit
// GEMM of conv.hip, which took these layers before, decodes both operands to f32 one
// element at a time and multiplies on the f32 matrix cores, at 1/16 of the f16 rate.
//
// A half MFMA wants 8 consecutive k per lane, and k can only be contiguous along the
// channels, which NCHW keeps H * W apart.  So a first kernel writes X as [N, H, W,
// group, C8] and W as [M, KH, KW, C8] in chunks of 8 channels (16 bytes, the last one
// zero-padded), and the GEMM fetches whole chunks straight into LDS:
//   A = weights [Mg, KHW * C8 * 8], B = im2col of the chunks, k = (kh, kw, channel).
// The copy costs one read and one write of X (2 bytes an element), which the GEMM's
// 16-byte loads earn back: gathering halves one at a time needs 8 loads and 4 packs
// for what is one load here, again for every tile of output channels.
// Measured on MI355X, [32, 128, 28, 28] * [128, 128, 3, 3] (7.4 GFLOP): 643 -> 24.6 us
// with both kernels (300 TFLOP/s), [32, 512, 7, 7] 3x3 2330 -> 31 us, one image of
// [64, 56, 56] 316 -> 12.6 us.  What bounds the GEMM is LDS traffic (each k-tile is
// written once and read by two or four waves) and the work per k-tile around 16 MFMAs.
#include <algorithm>

#include "conv.h"

namespace tohip {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(1))) uint16_t gu16;
typedef __attribute__((address_space(1))) float gfloat;

constexpr int kHBK = 64;             // k per tile: 8 chunks
constexpr int kHThreads = 256;

struct ConvH {
    int C, H, W, M, KW, OHW, OW, P;          // P = N * OHW
    int pt, pl, sh, sw, dh, dw, group;
    int Cg, Mg, KHW, C8, KC;                 // C8 chunks per tap, KC = KHW * C8 chunks per output
    int HW, NHW;
    uint32_t rb;                             // bytes of a pixel's chunks: group * C8 * 16
    uint32_t xbytes, wbytes;
    FastDiv fd_hw, fd_ohw, fd_ow, fd_c8, fd_kw, fd_khw;
};

// ---- layout: X -> [N * H * W][group][C8] chunks, W -> [M][KHW][C8] chunks --------------
// X: a block takes 64 consecutive pixels and eight chunks (64 channels): its loads run
// along the pixels (PAIR, planes of an even size: two halves at a time), LDS turns the
// tile, and the stores run along the chunks, 128 bytes of a pixel from eight threads
// (16-byte stores straight from the loads' lanes, one per pixel, took 14.7 us where
// this takes 9.7, [32, 64, 56, 56]).  W: one chunk per thread, taps fastest, so neighbouring threads
// read neighbouring halves.
template <bool PAIR>
__global__ __launch_bounds__(kHThreads) void k_convh_pack(const uint16_t* __restrict__ X, const uint16_t* __restrict__ Wt,
                                                          uint4* __restrict__ Xp, uint4* __restrict__ Wp, ConvH g,
                                                          int xblocks, int qblocks) {
    __shared__ uint4 turn[64][8];
    auto pack = [](const uint16_t (&h)[8]) {
        uint4 v;
        v.x = h[0] | (uint32_t)h[1] << 16;
        v.y = h[2] | (uint32_t)h[3] << 16;
        v.z = h[4] | (uint32_t)h[5] << 16;
        v.w = h[6] | (uint32_t)h[7] << 16;
        return v;
    };
    const int b = blockIdx.x;
    if (b < xblocks) {
        const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
        const int pb = b / qblocks, qb = b - pb * qblocks;
        const int G8 = g.group * g.C8;
        // PAIR: lanes 0-31 pixel pairs of one chunk, lanes 32-63 of the next; else a
        // pixel per lane, two chunks in turn
#pragma unroll
        for (int u = 0; u < (PAIR ? 1 : 2); u++) {
            const int ql = wave * 2 + (PAIR ? lane >> 5 : u), q = qb * 8 + ql;
            const int pl = PAIR ? 2 * (lane & 31) : lane, p = pb * 64 + pl;
            const int n = (int)g.fd_hw.div((uint32_t)p);
            const int grp = (int)g.fd_c8.div((uint32_t)q), c0 = (q - grp * g.C8) * 8;
            const bool live = p < g.NHW && q < G8;
            const int64_t at = ((int64_t)n * g.C + grp * g.Cg + c0) * g.HW + (p - n * g.HW);
            uint32_t v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                v[e] = 0;
                if (live && c0 + e < g.Cg) {
                    const uint16_t* src = X + at + (int64_t)e * g.HW;
                    if constexpr (PAIR) v[e] = *reinterpret_cast<const uint32_t*>(src);
                    else v[e] = *src;
                }
            }
            uint16_t h[8];
#pragma unroll
            for (int e = 0; e < 8; e++) h[e] = (uint16_t)v[e];
            turn[pl][ql ^ (pl & 7)] = pack(h);
            if constexpr (PAIR) {
#pragma unroll
                for (int e = 0; e < 8; e++) h[e] = (uint16_t)(v[e] >> 16);
                turn[pl + 1][ql ^ ((pl + 1) & 7)] = pack(h);
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int pl = (t >> 3) + 32 * u, p = pb * 64 + pl, ql = t & 7, q = qb * 8 + ql;
            if (p < g.NHW && q < G8) Xp[(int64_t)p * G8 + q] = turn[pl][ql ^ (pl & 7)];
        }
        return;
    }
    const uint32_t i = (uint32_t)(b - xblocks) * kHThreads + threadIdx.x;       // (m, c8, tap), taps fastest
    if (i >= (uint32_t)(g.M * g.KC)) return;
    const uint32_t mc = g.fd_khw.div(i), tap = i - mc * (uint32_t)g.KHW;
    const uint32_t m = g.fd_c8.div(mc), c8 = mc - m * (uint32_t)g.C8;
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int c = (int)c8 * 8 + e;
        h[e] = c < g.Cg ? Wt[((int64_t)m * g.Cg + c) * g.KHW + tap] : (uint16_t)0;
    }
    Wp[((int64_t)m * g.KHW + tap) * g.C8 + c8] = pack(h);
}

// 16 bytes per lane from r + off into LDS, lane l to the l-th 16 bytes of `to` (1 KB).
// (Called out: the builtin in a lambda of a kernel template leaves the host without
// the kernel's launch stub.)
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, _Float16* to, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, off, 0, 0, 0);
}

// What is added to a sum: a convolution's bias (one value per channel), or a Gemm's
// alpha * acc + beta * c in double, rounded once (c f32: cmode 0 none, 1 one
// value, 2 per column, 3 per row).
struct EpiH {
    const void* b;
    int dtb;
    int cmode;
    double alpha, beta;
    __device__ __forceinline__ float bias(int m) const {
        return b ? (dtb == kF16 ? (float)((const _Float16*)b)[m] : ((const float*)b)[m]) : 0.0f;
    }
    __device__ __forceinline__ float gemm(float acc, int m, int n) const {
        double r = alpha * (double)acc;
        if (cmode) r += beta * (double)((const float*)b)[cmode == 1 ? 0 : cmode == 2 ? n : m];
        return (float)r;
    }
};

// Waits until at most N of this wave's memory loads are outstanding (they complete in
// order; N <= 63) and its LDS reads have returned (the barrier after it tells the other
// waves that a slot may be filled again).
template <int N> __device__ __forceinline__ void wait_loads() {
    static_assert(N <= 63, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// ---- GEMM ---------------------------------------------------------------------------
// BM channels x BP pixels per block of four waves (two by two), two LDS buffers filled
// by loads that write LDS directly.  LDS rows are 128 bytes (8 chunks); chunk c of row r
// sits in slot c ^ ((r >> 1) & 7), so the 16 rows of a fragment read cover the banks
// once.  One load of a wave fills 8 rows: lane l writes slot l & 7 of row l >> 3, and
// since a wave's loads are 32 rows apart its chunk index q is the same in all of them:
// the tap, the channel chunk and their offset are worked out once per k-tile and lane.
// Padding taps, rows past M and chunks past KC lie past the buffer's range: zeros.
// SPLIT: slice z covers k-tiles [z * kt_per, ...) and stores f32 sums to Y + z * total.
template <int BM, int BP, int R, int ODT, bool SPLIT, bool GEMM>
__global__ __launch_bounds__(kHThreads, 2) void k_convh(const uint4* __restrict__ Xp, const uint4* __restrict__ Wp,
                                                     EpiH epi, void* __restrict__ Y, ConvH g, int ntm, int ntp, int kt_per, int64_t total, int ywidth) {
    constexpr int TI = BM / 64, TJ = BP / 64, NA = BM / 32, NB = BP / 32;
    // the ring's slots: distinct arrays, so that a read of one does not wait for the
    // loads in flight to the others
    __shared__ __attribute__((aligned(1024))) _Float16 lds0[(BM + BP) * kHBK];
    __shared__ __attribute__((aligned(1024))) _Float16 lds1[(BM + BP) * kHBK];
    __shared__ __attribute__((aligned(1024))) _Float16 lds2[R > 2 ? (BM + BP) * kHBK : 8];
    __shared__ __attribute__((aligned(1024))) _Float16 lds3[R > 3 ? (BM + BP) * kHBK : 8];
    // XCD-aware order: workgroups are dealt to the 8 XCDs in turn; each gets a
    // contiguous run of tiles, the channel tile fastest (one input tile, one L2)
    const int nb = ntm * ntp;
    int bid = blockIdx.x;
    if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    const int tp = bid / ntm, tm = bid - tp * ntm;
    const int m0 = tm * BM, p0 = tp * BP, grp = blockIdx.y;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const __amdgpu_buffer_rsrc_t ar = buffer_rsrc(Wp, g.wbytes), br = buffer_rsrc(Xp, g.xbytes);
    const int q = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));
    uint32_t arow[NA], prow[NB];
    int ih0[NB], iw0[NB];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int m = m0 + (wave + 4 * i) * 8 + (lane >> 3);
        arow[i] = m < g.Mg ? (uint32_t)((grp * g.Mg + m) * g.KC) * 16u : kOOB;
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int p = p0 + (wave + 4 * i) * 8 + (lane >> 3);
        const uint32_t n = g.fd_ohw.div((uint32_t)p), r = (uint32_t)p - n * (uint32_t)g.OHW;
        const uint32_t oh = g.fd_ow.div(r), ow = r - oh * (uint32_t)g.OW;
        ih0[i] = p < g.P ? (int)oh * g.sh - g.pt : -0x40000000;
        iw0[i] = (int)ow * g.sw - g.pl;
        prow[i] = (uint32_t)(((int)n * g.H + (int)oh * g.sh - g.pt) * g.W + iw0[i]) * g.rb;
    }
    auto load = [&](_Float16* lds, int kt) {
        const uint32_t kc = (uint32_t)(kt * 8 + q);
        const uint32_t tap = g.fd_c8.div(kc), c8 = kc - tap * (uint32_t)g.C8;
        const uint32_t kh = g.fd_kw.div(tap), kw = tap - kh * (uint32_t)g.KW;
        const int dy = (int)kh * g.dh, dx = (int)kw * g.dw;
        const bool in = kc < (uint32_t)g.KC;
        const uint32_t toff = (uint32_t)(dy * g.W + dx) * g.rb + (uint32_t)(grp * g.C8 + (int)c8) * 16u;
        const uint32_t koff = in ? kc * 16u : kOOB;
#pragma unroll
        for (int i = 0; i < NA; i++)
            load_lds16(ar, lds + (wave + 4 * i) * 512, arow[i] + koff);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const bool ok = in & ((unsigned)(ih0[i] + dy) < (unsigned)g.H) & ((unsigned)(iw0[i] + dx) < (unsigned)g.W);
            load_lds16(br, lds + BM * kHBK + (wave + 4 * i) * 512, ok ? prow[i] + toff : kOOB);
        }
        __builtin_amdgcn_sched_barrier(0);      // all of them before the multiply
    };
    const int lr = lane & 31, h = lane >> 5;
    int aoff[4], boff[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int slot = (2 * s + h) ^ ((lr >> 1) & 7);
        aoff[s] = (wm * (BM / 2) + lr) * kHBK + slot * 8;
        boff[s] = (BM + wn * (BP / 2) + lr) * kHBK + slot * 8;
    }
    floatx16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    auto multiply = [&](const _Float16* lds) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            halfx8 a[TI], b[TJ];
#pragma unroll
            for (int i = 0; i < TI; i++) a[i] = *reinterpret_cast<const halfx8*>(lds + aoff[s] + i * 32 * kHBK);
#pragma unroll
            for (int j = 0; j < TJ; j++) b[j] = *reinterpret_cast<const halfx8*>(lds + boff[s] + j * 32 * kHBK);
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    const int nk = (g.KC + 7) / 8;
    const int k0 = SPLIT ? (int)blockIdx.z * kt_per : 0, k1 = SPLIT ? min(nk, k0 + kt_per) : nk;
    // Step kt: this wave's loads of tile kt have landed (those of the R - 2 tiles after it
    // may still be in flight), every wave's have after the barrier, and every wave is done
    // with the slot that tile kt + R - 1 goes to.  (Loads past the last tile read zeros, or
    // a tile of the next slice, and are not multiplied.)
    auto step = [&](int kt, _Float16* cur, _Float16* into) {
        wait_loads<(R - 2) * (NA + NB)>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load(into, kt + R - 1);
        if (kt < k1) multiply(cur);
    };
    load(lds0, k0);
    if constexpr (R > 2) load(lds1, k0 + 1);
    if constexpr (R > 3) load(lds2, k0 + 2);
    for (int kt = k0; kt < k1; kt += R) {
        if constexpr (R == 2) {
            step(kt, lds0, lds1);
            step(kt + 1, lds1, lds0);
        } else if constexpr (R == 3) {
            step(kt, lds0, lds2);
            step(kt + 1, lds1, lds0);
            step(kt + 2, lds2, lds1);
        } else {
            step(kt, lds0, lds3);
            step(kt + 1, lds1, lds0);
            step(kt + 2, lds2, lds1);
            step(kt + 3, lds3, lds2);
        }
    }
    wait_loads<0>();        // nothing may land in LDS after the block ends or reuses it
    if constexpr (ODT == kF16 && !SPLIT) {
        // Halves leave through LDS, V pixels (V the power of two up to 8 that divides
        // OHW, so they share an image and an aligned address) of one channel per thread
        // and store ([32, 64, 56, 56] -> 256 1x1: 63.8 us with 2-byte stores from the
        // accumulators' lanes, 38.3 so)
        __syncthreads();
        uint16_t* out = reinterpret_cast<uint16_t*>(lds0);      // [BM][BP]
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = wm * (BM / 2) + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                const int m = grp * g.Mg + min(m0 + row, g.Mg - 1);
                const float bias = GEMM ? 0.0f : epi.bias(m);
#pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const int c = wn * (BP / 2) + j * 32 + lr;
                    const float v = GEMM ? epi.gemm(acc[i][j][r], m, min(p0 + c, g.P - 1)) : acc[i][j][r] + bias;
                    out[row * BP + c] = enc_f16(v);
                }
            }
        __syncthreads();
        auto store = [&](auto tag) {
            using T = decltype(tag);
            constexpr int V = sizeof(T) / 2, CH = BP / V, ROWS = kHThreads / CH;
            const int c = t % CH, p = p0 + c * V;
            const uint32_t n = g.fd_ohw.div((uint32_t)p);
            uint16_t* y = (uint16_t*)Y + ((int64_t)n * g.M + grp * g.Mg + m0) * g.OHW + ((uint32_t)p - n * (uint32_t)g.OHW);
            const int rows = p < g.P ? min(BM, g.Mg - m0) : 0;
            for (int row = t / CH; row < rows; row += ROWS)
                *reinterpret_cast<T*>(y + (int64_t)row * g.OHW) = *reinterpret_cast<const T*>(out + row * BP + c * V);
        };
        if (ywidth == 8) store(uint4{});
        else if (ywidth == 4) store(uint2{});
        else if (ywidth == 2) store(uint32_t{});
        else store(uint16_t{});
        return;
    }
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        const int p = p0 + wn * (BP / 2) + j * 32 + lr;
        const uint32_t n = g.fd_ohw.div((uint32_t)p), r0 = (uint32_t)p - n * (uint32_t)g.OHW;
        const bool live = p < g.P;
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int ml = m0 + wm * (BM / 2) + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                if (!live || ml >= g.Mg) continue;
                const int m = grp * g.Mg + ml;
                const int64_t yi = ((int64_t)n * g.M + m) * g.OHW + r0;
                if constexpr (SPLIT) ((gfloat*)Y)[(int64_t)blockIdx.z * total + yi] = acc[i][j][r];
                else ((gfloat*)Y)[yi] = GEMM ? epi.gemm(acc[i][j][r], m, p) : acc[i][j][r] + epi.bias(m);
            }
    }
}

// The slices' sum in slice order (double) and the bias, rounded once to the output type.
template <int ODT>
__global__ __launch_bounds__(256) void k_convh_reduce(const float* __restrict__ part, const void* __restrict__ Bv, int dtb,
                                                      void* __restrict__ Y, int total, FastDiv fd_ohw, FastDiv fd_m,
                                                      int nsplit) {
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i >= total) return;
    double acc = 0.0;
    for (int s = 0; s < nsplit; s++) acc += (double)part[(int64_t)s * total + i];
    if (Bv) {
        const uint32_t r = fd_ohw.div((uint32_t)i), m = r - fd_m.div(r) * fd_m.d;
        acc += dtb == kF16 ? (double)(float)((const _Float16*)Bv)[m] : (double)((const float*)Bv)[m];
    }
    st_d<ODT>(Y, i, acc);
}

template <int BM, int BP, int R, bool GEMM>
void launch_tiles(const uint4* xp, const uint4* wp, const EpiH& epi, void* y, int dty, float* part,
                  const ConvH& g, int split, int64_t total, hipStream_t s) {
    const int ntm = (g.Mg + BM - 1) / BM, ntp = (g.P + BP - 1) / BP, nk = (g.KC + 7) / 8;
    const int kt_per = (nk + split - 1) / split;
    int yw = 8;
    while (yw > 1 && (g.OHW % yw || (uintptr_t)y % (2 * yw))) yw /= 2;
    const dim3 grid((unsigned)(ntm * ntp), (unsigned)g.group, (unsigned)split), blk(kHThreads);
    if (split > 1)
        hipLaunchKernelGGL((k_convh<BM, BP, R, kF32, true, false>), grid, blk, 0, s, xp, wp, epi, (void*)part, g, ntm, ntp,
                           kt_per, total, yw);
    else if (dty == kF16)
        hipLaunchKernelGGL((k_convh<BM, BP, R, kF16, false, GEMM>), grid, blk, 0, s, xp, wp, epi, y, g, ntm, ntp, kt_per,
                           total, yw);
    else
        hipLaunchKernelGGL((k_convh<BM, BP, R, kF32, false, GEMM>), grid, blk, 0, s, xp, wp, epi, y, g, ntm, ntp, kt_per,
                           total, yw);
}

// Ring slots per tile shape: more loads in flight against more blocks per CU.  128x128
// with three or four slots (one block per CU) takes [32, 64, 56, 56] -> 256 1x1 from 46.5
// to 76 us; 64x128 with two 35.4 against 34.9 us at [32, 64, 56, 56] 3x3; 64x64 with four
// 31.7 against 26.0 us at [32, 128, 28, 28] 3x3 (its LDS reads, two per MFMA, need the
// blocks more than the prefetch).
constexpr int kRing128x128 = 2, kRing64x128 = 3, kRing64x64 = 2;

// Tile shape and k slices of a GEMM of Mg rows per group, P columns and KC chunks of k.
struct TilesH {
    int bm, bp, split;
};

TilesH tiles_h(int64_t P, int64_t Mg, int64_t group, int64_t KC) {
    // Tiles: 128x128 from two blocks per CU on ([32, 128, 28, 28] 3x3, 196 of them: 40
    // against 24.6 us with 392 of 64x128), 64x128 from one and a half on, else 64x64; then,
    // with less than one block per CU, slices of k (each at least four k-tiles deep).
    const int cus = num_cus();
    auto tiles = [&](int bm, int bp) { return ((P + bp - 1) / bp) * ((Mg + bm - 1) / bm) * group; };
    int bm = Mg > 64 ? 128 : 64, bp = 128;
    if (bm == 128 && tiles(128, 128) < 2 * cus) bm = 64;
    if (2 * tiles(bm, bp) < 3 * cus) bp = 64;
    const int nk = (int)((KC + 7) / 8);
    int split = 1;
    const int64_t nt = tiles(bm, bp);
    if (nt < cus) split = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>((2 * cus + nt - 1) / nt, 16), nk / 4));
    if (split > 1) split = (nk + (nk + split - 1) / split - 1) / ((nk + split - 1) / split);     // no empty slice
    return TilesH{bm, bp, split};
}

template <bool GEMM>
void launch_tiles_h(const TilesH& t, const uint4* xp, const uint4* wp, const EpiH& epi, void* y, int dty, float* part,
                   const ConvH& g, int64_t total, hipStream_t s) {
    if (t.bm == 128) launch_tiles<128, 128, kRing128x128, GEMM>(xp, wp, epi, y, dty, part, g, t.split, total, s);
    else if (t.bp == 128) launch_tiles<64, 128, kRing64x128, GEMM>(xp, wp, epi, y, dty, part, g, t.split, total, s);
    else launch_tiles<64, 64, kRing64x64, GEMM>(xp, wp, epi, y, dty, part, g, t.split, total, s);
}

// Layers that the general kernel (k_conv_mfma_f32, which gathers halves one by one) does
// faster: so few products per output and so few channels out that the chunk copies of X
// and 64-channel tiles are most of the work here, over enough pixels to fill the chip; with
// few pixels its one pass over k per block is the slower one.  1x1 windows with a stride
// copy pixels that no output uses, so more layers are among them, as are the depthwise
// ones whose stride is past the window (seven of a chunk's eight channels are padding).
// Measured, general kernel -> this: [8, C, 256, 256] 1x1, C = 8 to one channel 35 -> 61 us, to
// eight 46 -> 61, to 16 61 -> 63; C = 16 to eight 54 -> 65, 3x3 C = 2 to eight 68 -> 62; at
// [16, 8, 64, 64] to eight channels 14.2 -> 11.5; eight groups [8, 8, 128, 128] to eight
// channels each 87 -> 102, 16 channels to eight 125 -> 102.  Stride 2: C = 16 to 16 24 -> 31,
// C = 32 to eight 29 -> 33, C = 32 to 32 43 -> 34; stride 4 C = 16 to 16 21 -> 20.  Planes too
// wide for the depthwise kernel, [1, 2, 2000, 2000] 3x3: 495 -> 753; [32, 16, 112, 112] to 64 by
// groups of one, 5x5 stride 8: 26 -> 71.
bool few_products(const ConvGeom& g) {
    const int64_t K = (int64_t)g.Cg * g.KH * g.KW, pixels = (int64_t)g.N * g.OH * g.OW * g.group;
    const bool point = g.KH == 1 && g.KW == 1 && (g.sh > 1 || g.sw > 1);
    // (a stride's copies count as a quarter of the work that their pixels would be)
    const int64_t work = point ? std::max(pixels, (int64_t)g.N * g.H * g.W / 4 * g.group) : pixels;
    const bool skips = point || (g.Cg == 1 && (g.sh > g.KH || g.sw > g.KW));
    const int64_t most = skips && g.Mg <= 8 ? 32 : g.group == 1 || g.Cg == 1 ? 16 : 8;
    if (g.Mg <= 8) return K <= most && work > 65536;
    return g.Mg <= 16 && K <= most && (point || g.Cg == 1) && pixels > 65536;
}

}  // namespace

bool launch_conv_f16(const void* x, const void* w, const void* b, int dtb, void* y, int dty, const ConvGeom& cg,
                     hipStream_t s) {
    if ((dty != kF16 && dty != kF32) || (b && dtb != kF32 && dtb != kF16)) return false;
    // (an image without pixels, whose outputs are all padding, has no copy to index: H * W is divided by)
    if (cg.N < 1 || cg.Cg < 1 || cg.H < 1 || cg.W < 1 || cg.KH < 1 || cg.KW < 1 || cg.group > 65535) return false;
    // the layout copies live in a workspace, which a captured call may not take
    if (stream_capturing(s)) return false;
    if (few_products(cg)) return false;
    ConvH g;
    const int64_t C8 = (cg.Cg + 7) / 8, KHW = (int64_t)cg.KH * cg.KW, KC = KHW * C8;
    const int64_t NHW = (int64_t)cg.N * cg.H * cg.W, P = (int64_t)cg.N * cg.OH * cg.OW;
    const int64_t xb = NHW * cg.group * C8 * 16, wb = (int64_t)cg.M * KC * 16, total = P * cg.M;
    const int64_t reach = (int64_t)1 << 31;
    // byte offsets of the loads and the pixel and output indices stay below 2^31
    if (xb >= reach || wb >= reach || total >= reach / 4 || NHW >= reach / 4 ||
        (int64_t)(cg.H + (int64_t)cg.KH * cg.dh) * (cg.W + (int64_t)cg.KW * cg.dw) >= reach / 4)
        return false;
    g.C = cg.C; g.H = cg.H; g.W = cg.W; g.M = cg.M; g.KW = cg.KW; g.OHW = cg.OH * cg.OW; g.OW = cg.OW; g.P = (int)P;
    g.pt = cg.pt; g.pl = cg.pl; g.sh = cg.sh; g.sw = cg.sw; g.dh = cg.dh; g.dw = cg.dw; g.group = cg.group;
    g.Cg = cg.Cg; g.Mg = cg.Mg; g.KHW = (int)KHW; g.C8 = (int)C8; g.KC = (int)KC;
    g.HW = cg.H * cg.W; g.NHW = (int)NHW;
    g.rb = (uint32_t)(cg.group * C8 * 16);
    g.xbytes = (uint32_t)xb; g.wbytes = (uint32_t)wb;
    g.fd_hw = make_fastdiv((uint32_t)g.HW);
    g.fd_ohw = make_fastdiv((uint32_t)g.OHW);
    g.fd_ow = make_fastdiv((uint32_t)g.OW);
    g.fd_c8 = make_fastdiv((uint32_t)C8);
    g.fd_kw = make_fastdiv((uint32_t)g.KW);
    g.fd_khw = make_fastdiv((uint32_t)KHW);
    const TilesH t = tiles_h(P, cg.Mg, cg.group, KC);
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int split = t.split;
    const int64_t pb = split > 1 ? (int64_t)split * total * 4 : 0;
    char* ws = (char*)pool_alloc((size_t)(up(xb) + up(wb) + pb), true);
    if (!ws) return false;
    uint4 *xp = (uint4*)ws, *wp = (uint4*)(ws + up(xb));
    float* part = (float*)(ws + up(xb) + up(wb));
    const int qblocks = (int)((cg.group * C8 + 7) / 8);
    const int64_t xblocks = (NHW + 63) / 64 * qblocks, wblocks = ((int64_t)cg.M * KC + kHThreads - 1) / kHThreads;
    const dim3 pg((unsigned)(xblocks + wblocks)), pblk(kHThreads);
    if (g.HW % 2 == 0 && ((uintptr_t)x & 3) == 0)
        hipLaunchKernelGGL(k_convh_pack<true>, pg, pblk, 0, s, (const uint16_t*)x, (const uint16_t*)w, xp, wp, g,
                           (int)xblocks, qblocks);
    else
        hipLaunchKernelGGL(k_convh_pack<false>, pg, pblk, 0, s, (const uint16_t*)x, (const uint16_t*)w, xp, wp, g,
                           (int)xblocks, qblocks);
    launch_tiles_h<false>(t, xp, wp, EpiH{b, dtb, 0, 0.0, 0.0}, y, dty, part, g, total, s);
    if (split > 1) {
        const dim3 rg((unsigned)((total + 255) / 256));
        const FastDiv fo = g.fd_ohw, fm = make_fastdiv((uint32_t)g.M);
        if (dty == kF16) hipLaunchKernelGGL(k_convh_reduce<kF16>, rg, dim3(256), 0, s, part, b, dtb, y, (int)total, fo, fm, split);
        else hipLaunchKernelGGL(k_convh_reduce<kF32>, rg, dim3(256), 0, s, part, b, dtb, y, (int)total, fo, fm, split);
    }
    pool_free(ws);   // stream-ordered reuse: later work on this stream runs after the kernels
    return true;
}

// Y[M, N] = alpha A' B' + beta C of halves as the GEMM above: A's rows are the output
// channels, B's columns the pixels of one image, K the channels.  An operand with k along its
// rows (A [M, K], B [N, K]) in whole, aligned chunks is read where it lies; any other is
// copied into rows of chunks first, by the weights' part of k_convh_pack where k runs along
// its rows, else by the images' part.  Against the
// 128x128x32 kernel without a k split that took these layouts: [512, 1024] x [1024, 4096]
// 85 -> 23 us, [87, 1728] x [1728, 421] 177 -> 17.6, [300, 1003] x [1001, 1003]^T 93 -> 18;
// short k is left to it, as three launches cost 12.5 us ([20, 80] x [80, 64] 12.0, [7, 65] x
// [64, 65]^T 9.0).
constexpr int kGemmHMinK = 128;

int launch_gemm_f16_packed(const GemmH& q, hipStream_t s, float** part, int* nsplit, void** ws) {
    if ((q.dty != kF16 && q.dty != kF32) || q.M < 1 || q.N < 1 || q.K < kGemmHMinK) return 0;
    const int64_t KC = ((int64_t)q.K + 7) / 8, reach = (int64_t)1 << 31;
    const int64_t ab = (int64_t)q.M * KC * 16, bb = (int64_t)q.N * KC * 16, total = (int64_t)q.M * q.N;
    if (ab >= reach || bb >= reach || total >= reach / 4) return 0;
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    const TilesH t = tiles_h(q.N, q.M, 1, KC);
    const int64_t pb = t.split > 1 ? (int64_t)t.split * total * 4 : 0;
    // k along the rows, whole chunks and an aligned base: the operand is its own copy
    const bool a_own = !q.ta && q.K % 8 == 0 && ((uintptr_t)q.A & 15) == 0;
    const bool b_own = q.tb && q.K % 8 == 0 && ((uintptr_t)q.B & 15) == 0;
    const int64_t ac = a_own ? 0 : up(ab), bc = b_own ? 0 : up(bb);
    char* w = nullptr;      // (none to be had under graph capture: only calls without copies and slices then)
    if (ac + bc + pb && !(w = (char*)pool_alloc((size_t)(ac + bc + pb), true))) return 0;
    const uint4 *ap = a_own ? (const uint4*)q.A : (const uint4*)w, *bp = b_own ? (const uint4*)q.B : (const uint4*)(w + ac);
    ConvH g;
    g.H = 1; g.KW = 1; g.pt = g.pl = 0; g.sh = g.sw = g.dh = g.dw = 1; g.group = 1;
    g.C = g.Cg = q.K; g.KHW = 1; g.C8 = g.KC = (int)KC;
    g.rb = (uint32_t)(KC * 16);
    g.fd_c8 = make_fastdiv((uint32_t)KC);
    g.fd_kw = g.fd_khw = make_fastdiv(1);
    // n rows of chunks from src into dst; along: k runs along src's rows
    auto pack = [&](const void* src, int n, bool along, uint4* dst) {
        g.HW = g.NHW = g.M = n;
        g.fd_hw = make_fastdiv((uint32_t)n);
        const int qblocks = (int)((KC + 7) / 8);
        const uint16_t* h = (const uint16_t*)src;
        const dim3 blk(kHThreads);
        if (along) {
            const dim3 grid((unsigned)(((int64_t)n * KC + kHThreads - 1) / kHThreads));
            hipLaunchKernelGGL(k_convh_pack<false>, grid, blk, 0, s, h, h, dst, dst, g, 0, qblocks);
        } else {
            const int xblocks = (n + 63) / 64 * qblocks;
            if (n % 2 == 0 && ((uintptr_t)src & 3) == 0)
                hipLaunchKernelGGL(k_convh_pack<true>, dim3((unsigned)xblocks), blk, 0, s, h, h, dst, dst, g, xblocks, qblocks);
            else
                hipLaunchKernelGGL(k_convh_pack<false>, dim3((unsigned)xblocks), blk, 0, s, h, h, dst, dst, g, xblocks, qblocks);
        }
    };
    if (!a_own) pack(q.A, q.M, !q.ta, (uint4*)w);
    if (!b_own) pack(q.B, q.N, q.tb != 0, (uint4*)(w + ac));
    g.W = g.OW = g.OHW = g.P = g.HW = g.NHW = q.N;
    g.M = g.Mg = q.M;
    g.xbytes = (uint32_t)bb; g.wbytes = (uint32_t)ab;
    g.fd_hw = g.fd_ohw = g.fd_ow = make_fastdiv((uint32_t)q.N);
    const EpiH epi{q.c, kF32, q.c ? q.cmode : 0, q.alpha, q.beta};
    float* ps = t.split > 1 ? (float*)(w + ac + bc) : nullptr;
    launch_tiles_h<true>(t, bp, ap, epi, q.Y, q.dty, ps, g, total, s);
    if (t.split == 1) {
        if (w) pool_free(w);    // stream-ordered reuse
        return 1;
    }
    const int nk = (int)((KC + 7) / 8), per = (nk + t.split - 1) / t.split;
    *part = ps;
    *nsplit = (nk + per - 1) / per;
    *ws = w;
    return 2;
}

}  // namespace tohip
