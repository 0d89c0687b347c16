// conv.h — what the convolution sources share: the layer's geometry, the fused
// epilogue, and the plans that live outside conv.hip.
#pragma once

#include "quant.h"
#include "runtime.h"

namespace tohip {

struct ConvGeom {
    int N, C, H, W;      // input
    int M, KH, KW;       // weights [M, C/g, KH, KW]
    int OH, OW;          // output (from Y)
    int pt, pl, sh, sw, dh, dw, group;
    int Cg, Mg, Kg;      // per-group channels in / out, Cg * KH * KW
};

// Fused epilogue of conv2d_fused_forward (f32 output): y = conv + bias, then
// Relu (v > 0 ? v : 0, as relu_forward), then + skip (an f32 tensor of Y's
// shape, as add_forward).  Each step rounds to f32 exactly as the standalone
// operator does, so the result equals the three calls bit for bit.
struct ConvEpi {
    const float* skip;
    int relu;
    FakeQuant fq;   // applied last (kind 0: none)
};
__device__ __forceinline__ float relu_f(float v) { return v > 0.0f ? v : 0.0f; }

// Quantized input of dequantize_conv2d_fused_forward: X holds uint8 (XQ = 1) or
// int8 (XQ = 2) codes with a per-tensor scale and zero point; the gather forms
// (float)(q - z) * s, which is the value DequantizeLinear writes (q - z has at
// most 9 bits, so the fp32 product is the correctly rounded exact product, as
// the reference's double product rounded once).  Padding taps stay 0.
struct ConvXQ {
    const float* s;      // scale (one element)
    const void* z;       // zero point of the codes' dtype (one element), or null for 0
};
template <int XQ> __device__ __forceinline__ float xq_value(uint32_t code, float s, int z) {
    const int c = XQ == 2 ? (int)(int8_t)(uint8_t)code : (int)(code & 0xFFu);
    return (float)(c - z) * s;
}

// Convolutions of one input channel per group (depthwise, convdw.hip): f32 or f16
// input and weights of one dtype, f32 / f16 output, f32 / f16 or no bias; epi (f32
// output and f32 or no bias only) is applied whole.  dtx kU8 / kI8: codes with xq's
// scale and zero point, f32 weights and output.  False (nothing launched) when the
// layer is outside the plan.
bool launch_conv_depthwise(const void* x, int dtx, const void* w, const void* b, int dtb, void* y, int dty,
                           const ConvGeom& g, const ConvEpi& epi, const ConvXQ& xq, hipStream_t s);
// The layers launch_conv_depthwise takes, by their shape and whether X is f16 alone.
bool conv_depthwise_shape(const ConvGeom& g, bool half);
// float16 X and W on the f16 matrix cores (convh.hip): f16 / f32 output, f32 / f16 or
// no bias, any groups.  False, with nothing launched and no error, when the layer is outside
// the plan or there is no memory for the copies.
bool launch_conv_f16(const void* x, const void* w, const void* b, int dtb, void* y, int dty, const ConvGeom& g,
                     hipStream_t s);

// A Gemm of halves in the layouts and sizes that gemm.hip's f16 kernels do not fetch
// directly (convh.hip): c f32, cmode 0 none, 1 one value, 2 per column, 3 per row.
// 0: not taken (no memory for the copies included); 1: done; 2: *nsplit slices of M x N
// f32 sums at *part, which the caller reduces (with the epilogue) and then frees *ws.
struct GemmH {
    const void* A;
    const void* B;
    void* Y;
    int ta, tb, dty, M, N, K;
    double alpha, beta;
    const float* c;
    int cmode;
};
int launch_gemm_f16_packed(const GemmH& q, hipStream_t s, float** part, int* nsplit, void** ws);

}  // namespace tohip
