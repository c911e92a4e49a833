// Shared by the bf16 / fp32 Linear kernels of libi64hip_dense.so: conversions, activations, the epilogue.
#ifndef I64H_DENSE_DEV_H
#define I64H_DENSE_DEV_H
#include "i64h_common.h"
#include "i64h_dense.h"

typedef float dn_v4f __attribute__((ext_vector_type(4)));
typedef __bf16 dn_v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t dn_bf16_rne(float f) {  // round to nearest even, NaN stays NaN: the hardware conversion of this chip
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}
// two of them in one instruction, the first in the low half
__device__ __forceinline__ uint32_t dn_bf16_pair(float a, float b) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2bf));
}
__device__ __forceinline__ float dn_bf16_to_f32(uint32_t h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ float dn_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float dn_gelu_tanh(float z) {
    const float inner = 0.7978845608028654f * (z + 0.044715f * z * z * z);
    return 0.5f * z * (1.0f + tanhf(inner));
}

__device__ __forceinline__ float dn_gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

// log(1 + e^z) with one logarithm: with u = 1 + x rounded, log(u) x / (u - 1) is log(1 + x) to a few units in the last place (Kahan's
// correction of the rounding of u)
__device__ __forceinline__ float dn_softplus(float z) {
    const float x = expf(z), u = 1.0f + x, d = u - 1.0f;
    const float l = d > 0.0f ? logf(u) * (x * __builtin_amdgcn_rcpf(d)) : x;
    return z > 20.0f ? z : l;
}

__device__ __forceinline__ float dn_xielu(float z, float a, float b) {
    return z > 0.0f ? a * z * z + 0.5f * z : b * (expm1f(z) - z) + 0.5f * z;
}
constexpr bool dn_dual(int epi) { return epi == I64H_EPI_GELU_MUL || epi == I64H_EPI_SILU_MUL || epi == I64H_EPI_CLAMP_GLU; }  // two accumulators: gate rows and up rows

template <int EPI>
__device__ __forceinline__ float dn_epilogue(const i64h_linear& p, float acc, float acc2, int64_t b, int64_t r, int c) {
    if (dn_dual(EPI) && p.row_scale) {      // a factor on the input row
        const float s = p.row_scale[r];
        acc *= s, acc2 *= s;
    }
    if (EPI == I64H_EPI_GELU_MUL) return dn_gelu_tanh(acc) * acc2;
    if (EPI == I64H_EPI_SILU_MUL) return acc * dn_sigmoid(acc) * acc2;
    if (EPI == I64H_EPI_CLAMP_GLU) {
        const float u = fminf(acc, p.act_b), w = fminf(fmaxf(acc2, -p.act_b), p.act_b);
        return u * dn_sigmoid(p.act_a * u) * (w + 1.0f);
    }
    if (p.bias) acc += p.bias[b * p.bias_batch + c];
    if (EPI == I64H_EPI_XIELU) return dn_xielu(acc, p.act_a, p.act_b);
    if (EPI == I64H_EPI_RELU_SQ) return acc > 0.0f ? acc * acc : 0.0f;
    if (EPI == I64H_EPI_GELU_ERF) return dn_gelu_erf(acc);
    if (EPI == I64H_EPI_SCALE) return acc * p.scale;
    if (EPI == I64H_EPI_MUL_SIGMOID) return acc * dn_sigmoid(p.E[b * p.e_batch + r * p.lde + c]);
    if (EPI == I64H_EPI_ROW_SIGMOID) return acc * dn_sigmoid(p.E[b * p.e_batch + r * p.lde]);
    if (EPI == I64H_EPI_SOFTCAP) return p.softcap * tanhf(acc / p.softcap);
    if (EPI == I64H_EPI_ADD) return acc + p.E[b * p.e_batch + r * p.lde + c];
    if (EPI == I64H_EPI_DECAY) return expf(-p.E[b * p.e_batch + r * p.lde + c] * dn_softplus(acc));
    return acc;
}

// the matrix-core tile forms of i64h_linear_run (i64h_linear_block.hip): operands readable 16 bytes at a time.
// form: -1 chosen by size, else the number of a tile form (tests, measurements).  False: the launch does not fit this form.
bool dn_linear_block(const i64h_linear& d, int form, hipStream_t s);

#endif
