// convdw.hip — depthwise Conv2d (one input channel per group) for gfx950.
//
// tensor_ops/tensor_ops.c:1036-1114 with C / group == 1: each output plane is a
// KH x KW stencil over one input plane, plus a bias.  There is no reduction over
// channels, so nothing for the matrix cores: the operator is bound by reading each
// input plane and writing each output plane once.  The implicit GEMM, which took
// these layers before, gave a group's one channel a 64-channel tile.
//
// A block stages one tile of rows of a plane (or several small planes) in LDS as
// f32, zero padding included (planes.h); then a thread computes a strip of R output rows of one column, reading
// each input row of the strip once (K values) and adding it to the up to K outputs
// that use it: (R - 1) S + K rows of K reads for R outputs instead of K K each.
// The sum runs over (kh, kw) in the reference's order, in f32 with fused
// multiply-adds: the convolution's tolerance class.  Padded taps contribute
// 0 * w, as the reference's do.
// [32, 96, 56, 56] 3x3 (77 MB f32): 320 -> 17.2 us (4.5 TB/s), f16 594 -> 14.2 us,
// stride 2 84 -> 11.7 us; the vector instructions and LDS reads of about 9 M
// outputs, not only the traffic, bound the f16 form.  Output rows are stored plain:
// nontemporal stores of rows that are no whole cache lines took 47 us.
#include "conv.h"
#include "planes.h"

namespace tohip {
namespace {

// dec_f16's value (v_cvt_f32_f16 keeps f16 denormals; a NaN comes back quiet).
__device__ __forceinline__ float f16_value(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// An input value as f32; off == kOOB (padding) gives 0.  Codes are dequantised.
template <int DT> __device__ __forceinline__ float dw_ld(__amdgpu_buffer_rsrc_t r, uint32_t off, float xs, int xz) {
    if constexpr (DT == kU8 || DT == kI8) {
        const float v = xq_value<DT == kU8 ? 1 : 2>(__builtin_amdgcn_raw_buffer_load_b8(r, off, 0, 0), xs, xz);
        return off == kOOB ? 0.0f : v;
    } else if constexpr (DT == kF16) return f16_value((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
    else return u2f(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// A weight: of the input's dtype, f32 with codes.
template <int DT> __device__ __forceinline__ float dw_wt(const void* w, int i) {
    if constexpr (DT == kF16) return f16_value(((const uint16_t*)w)[i]);
    else return ((const float*)w)[i];
}

// K x K window at stride S, no dilation, R output rows per strip; K == 0: any
// window, stride and dilation, R == 1.  MULTI: several planes per block.
// FQ: the epilogue fake-quantizes (its fp64 fallback costs the other layers 10%).
template <int DT, int ODT, int K, int S, int R, bool MULTI, bool FQ>
__global__ __launch_bounds__(kPlaneThreads) void k_conv_dw(const void* __restrict__ X, const void* __restrict__ Wt,
                                                        const void* __restrict__ Bv, int dtb, void* __restrict__ Y,
                                                        PlaneTiles g, ConvEpi epi, ConvXQ xq) {
    extern __shared__ float tile[];
    constexpr int EB = DT == kF32 ? 4 : DT == kF16 ? 2 : 1;
    constexpr int KK = K > 0 ? K * K : 1;
    const int t = threadIdx.x;
    const int kk = K > 0 ? KK : g.KH * g.KW;
    const int bp = (int)g.fd_tiles.div(blockIdx.x), tl = (int)blockIdx.x - bp * g.tiles;
    const int p0 = bp * g.np;
    const int np = MULTI ? min(g.np, g.planes - p0) : 1;
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(X, g.xbytes);
    float* wlds = tile + g.np * g.PR * g.PW;            // MULTI: the planes' weights
    float xs = 0.0f;
    int xz = 0;
    if constexpr (DT == kU8 || DT == kI8) {
        xs = xq.s[0];
        if (xq.z) xz = DT == kU8 ? (int)*(const uint8_t*)xq.z : (int)*(const int8_t*)xq.z;
    }
    // rows and columns outside the plane read zero
    stage_planes<EB, MULTI>(tile, g, tl, p0, np, [&](uint32_t off) { return dw_ld<DT>(xr, off, xs, xz); });
    if constexpr (MULTI) {
        for (int i = t; i < np * kk; i += kPlaneThreads) {
            const int q = i / kk;
            wlds[i] = dw_wt<DT>(Wt, g.channel(p0 + q) * kk + (i - q * kk));
        }
    }
    __syncthreads();
    // ---- strips of R output rows of one column
    const int tx = t & ((1 << g.lxo) - 1), ty = t >> g.lxo, step = kPlaneThreads >> g.lxo;
    FQParm fqp;
    if constexpr (FQ) fqp = fq_parm(epi.fq);
    float w[KK];
    if constexpr (!MULTI && K > 0) {
        const int m = g.channel(p0);
#pragma unroll
        for (int i = 0; i < KK; i++) w[i] = dw_wt<DT>(Wt, m * KK + i);
    }
    for (int st = ty; st < np * g.ns; st += step) {
        const int q = MULTI ? (int)g.fd_ns.div((uint32_t)st) : 0;
        const int strip = st - q * g.ns, p = p0 + q, m = g.channel(p);
        if constexpr (MULTI && K > 0) {
#pragma unroll
            for (int i = 0; i < KK; i++) w[i] = wlds[q * KK + i];
        }
        const float bias = Bv ? (dtb == kF16 ? dec_f16(((const uint16_t*)Bv)[m]) : ((const float*)Bv)[m]) : 0.0f;
        const int oh0 = tl * g.TR + strip * R;
        for (int ow = tx; ow < g.OW; ow += 1 << g.lxo) {
            float acc[R];
#pragma unroll
            for (int o = 0; o < R; o++) acc[o] = 0.0f;
            if constexpr (K > 0) {
                const float* tp = tile + (q * g.PR + strip * R * S) * g.PW + ow * S;
#pragma unroll
                for (int j = 0; j < (R - 1) * S + K; j++) {
                    float x[K > 0 ? K : 1];
#pragma unroll
                    for (int kw = 0; kw < K; kw++) x[kw] = tp[kw];
                    tp += g.PW;
#pragma unroll
                    for (int o = 0; o < R; o++) {
                        const int kh = j - o * S;
                        if (kh < 0 || kh >= K) continue;
#pragma unroll
                        for (int kw = 0; kw < K; kw++) acc[o] = __builtin_fmaf(x[kw], w[kh * K + kw], acc[o]);
                    }
                }
            } else {
                const float* tp = tile + (q * g.PR + strip * g.sh) * g.PW + ow * g.sw;
                for (int kh = 0; kh < g.KH; kh++)
                    for (int kw = 0; kw < g.KW; kw++) {
                        const int i = kh * g.KW + kw;
                        const float wv = MULTI ? wlds[q * kk + i] : dw_wt<DT>(Wt, m * kk + i);
                        acc[0] = __builtin_fmaf(tp[kh * g.dh * g.PW + kw * g.dw], wv, acc[0]);
                    }
            }
#pragma unroll
            for (int o = 0; o < R; o++) {
                const int oh = oh0 + o;
                if (oh >= g.OH) break;
                const int yi = (p * g.OH + oh) * g.OW + ow;
                float v = acc[o] + bias;     // + 0.0f without one, as the reference adds it
                if constexpr (ODT == kF16) {
                    ((uint16_t*)Y)[yi] = enc_f16(v);
                } else {
                    if (epi.relu) v = relu_f(v);
                    if (epi.skip) v += epi.skip[yi];
                    if constexpr (FQ) v = fq_apply(v, fqp);
                    ((float*)Y)[yi] = v;
                }
            }
        }
    }
}

template <int DT, int ODT, int K, int S, int R>
void launch_dw(const void* x, const void* w, const void* b, int dtb, void* y, const PlaneTiles& p, const ConvEpi& epi,
               const ConvXQ& xq, hipStream_t s) {
    const dim3 grid((unsigned)((p.planes + p.np - 1) / p.np * p.tiles)), blk(kPlaneThreads);
    const size_t lds = ((size_t)p.np * p.PR * p.PW + (p.np > 1 ? (size_t)p.np * p.KH * p.KW : 0)) * sizeof(float);
#define DW_LAUNCH(MULTI, FQ) \
    hipLaunchKernelGGL((k_conv_dw<DT, ODT, K, S, R, MULTI, FQ>), grid, blk, lds, s, x, w, b, dtb, y, p, epi, xq)
    if (ODT == kF32 && epi.fq.kind) {
        if (p.np > 1) DW_LAUNCH(true, ODT == kF32);
        else DW_LAUNCH(false, ODT == kF32);
    } else if (p.np > 1) DW_LAUNCH(true, false);
    else DW_LAUNCH(false, false);
#undef DW_LAUNCH
}

// Strip length: seven rows for 3x3 (27 LDS reads a strip; planes of 7, 14, 28, ...
// rows divide evenly), four for 5x5.  3x3 with four: 17.8 against 17.2 us at
// [32, 96, 56, 56], 18.3 against 15.2 at [16, 64, 112, 112] stride 2; 5x5 with
// seven: 12.9 against 7.8 us at [2, 40, 100, 100] stride 2.
constexpr int kDwR3 = 7, kDwR5 = 4;

// Up to 16 output channels per input channel: more fill the implicit GEMM's
// 64-channel tile better than they pay for reading the plane again (one input
// channel, 3x3: 16 outputs 7.6 -> 4.6 us, 32 6.9 against 7.6, 64 10.9 against 11.4).
constexpr int kDwMaxMult = 16;

// Strides past the window stage rows and columns that no output uses (a plane's tiles
// whole, once per output channel), where the implicit GEMM gathers what it needs.  A pixel
// of one group costs that about as much as 28 + 1.75 KH KW staged values (2.5 times as many
// with f16 operands, which it decodes); here a plane's second and further reads, from L2, count
// 0.6, and a tap of the general form (R == 1) about 1 / 4.
// Measured on both sides of the line, GEMM -> this, [32, 64, 112, 112] f32: 1x1 stride 5
// 27 -> 23 us, stride 6 20 -> 24, stride 8 12.4 -> 20.5; 3x3 stride 6 29 -> 23, stride 8
// 19 -> 23; four output channels per input channel, 16 -> 64: 1x1 stride 3 24 -> 21, stride
// 4 15 -> 25, stride 8 6.4 -> 20.8, 7x7 stride 2 146 -> 105; eight, 8 -> 64, 7x7 stride 4
// 28 -> 39; sixteen, 4 -> 64: 3x3 stride 2 25 -> 22; int8 codes 5x5 stride 8 29 -> 22.  f16: 1x1 stride 8 23 -> 18; four, 1x1
// stride 4 33 -> 23, stride 6 14.6 -> 21.8; eight, 3x3 stride 4 28 -> 21; sixteen, 3x3 stride
// 3 24 -> 30.
bool dw_pays(const ConvGeom& g, const PlaneTiles& p, int R, bool half) {
    const double staged = (double)p.PR * p.PW * p.tiles / ((double)g.OH * g.OW), taps = (double)g.KH * g.KW;
    return (0.4 + 0.6 * g.Mg) * staged + (R == 1 ? 0.26 * g.Mg * taps : 0.0) <= (28.0 + 1.75 * taps) * (half ? 2.5 : 1.0);
}

bool dw_plan(const ConvGeom& g, bool half, PlaneTiles& p) {
    if (g.Cg != 1 || g.Mg > kDwMaxMult || g.KH < 1 || g.KW < 1 || g.sh < 1 || g.sw < 1 || g.dh < 1 || g.dw < 1) return false;
    const int64_t reach = (int64_t)1 << 29;              // elements: byte offsets stay below 2^31
    const int64_t planes = (int64_t)g.N * g.M;
    if ((int64_t)g.N * g.C * g.H * g.W >= reach || planes * g.OH * g.OW >= reach || planes >= reach) return false;
    if ((int64_t)g.KH * g.KW > 1024 || (int64_t)g.M * g.KH * g.KW >= ((int64_t)1 << 31) || (int64_t)g.H + g.W > (1 << 20) || (int64_t)g.OH + g.OW > (1 << 20)) return false;
    const bool strip = g.KH == g.KW && (g.KH == 3 || g.KH == 5) && g.sh == g.sw && (g.sh == 1 || g.sh == 2) &&
                       g.dh == 1 && g.dw == 1;
    const int R = strip ? (g.KH == 3 ? kDwR3 : kDwR5) : 1;
    p.C = g.C; p.H = g.H; p.W = g.W; p.OH = g.OH; p.OW = g.OW; p.M = g.M; p.KH = g.KH; p.KW = g.KW;
    p.pt = g.pt; p.pl = g.pl; p.sh = g.sh; p.sw = g.sw; p.dh = g.dh; p.dw = g.dw;
    p.planes = (int)planes;
    return plan_planes(p, R, g.KH * g.KW) && dw_pays(g, p, R, half);
}

template <int DT, int ODT>
void launch_dw_window(const void* x, const void* w, const void* b, int dtb, void* y, const PlaneTiles& p, const ConvEpi& epi,
                      const ConvXQ& xq, hipStream_t s) {
    const bool strip = p.KH == p.KW && p.sh == p.sw && p.sh <= 2 && p.dh == 1 && p.dw == 1;
    if (strip && p.KH == 3 && p.sh == 1) launch_dw<DT, ODT, 3, 1, kDwR3>(x, w, b, dtb, y, p, epi, xq, s);
    else if (strip && p.KH == 3) launch_dw<DT, ODT, 3, 2, kDwR3>(x, w, b, dtb, y, p, epi, xq, s);
    else if (strip && p.KH == 5 && p.sh == 1) launch_dw<DT, ODT, 5, 1, kDwR5>(x, w, b, dtb, y, p, epi, xq, s);
    else if (strip && p.KH == 5) launch_dw<DT, ODT, 5, 2, kDwR5>(x, w, b, dtb, y, p, epi, xq, s);
    else launch_dw<DT, ODT, 0, 1, 1>(x, w, b, dtb, y, p, epi, xq, s);
}

}  // namespace

bool conv_depthwise_shape(const ConvGeom& g, bool half) {
    PlaneTiles p;
    return dw_plan(g, half, p);
}

bool launch_conv_depthwise(const void* x, int dtx, const void* w, const void* b, int dtb, void* y, int dty,
                           const ConvGeom& g, const ConvEpi& epi, const ConvXQ& xq, hipStream_t s) {
    const bool codes = dtx == kU8 || dtx == kI8;
    if ((dtx != kF32 && dtx != kF16 && !codes) || (codes && dty != kF32) || (dty != kF32 && dty != kF16) || (b && dtb != kF32 && dtb != kF16)) return false;
    PlaneTiles p;
    if (!dw_plan(g, dtx == kF16, p)) return false;
    p.xbytes = (uint32_t)((int64_t)g.N * g.C * g.H * g.W * (codes ? 1 : dtx == kF16 ? 2 : 4));
    if (dtx == kU8) launch_dw_window<kU8, kF32>(x, w, b, dtb, y, p, epi, xq, s);
    else if (dtx == kI8) launch_dw_window<kI8, kF32>(x, w, b, dtb, y, p, epi, xq, s);
    else if (dtx == kF32 && dty == kF32) launch_dw_window<kF32, kF32>(x, w, b, dtb, y, p, epi, xq, s);
    else if (dtx == kF32) launch_dw_window<kF32, kF16>(x, w, b, dtb, y, p, epi, xq, s);
    else if (dty == kF32) launch_dw_window<kF16, kF32>(x, w, b, dtb, y, p, epi, xq, s);
    else launch_dw_window<kF16, kF16>(x, w, b, dtb, y, p, epi, xq, s);
    return true;
}

}  // namespace tohip
