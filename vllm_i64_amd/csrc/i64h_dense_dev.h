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
// x sigmoid(z) = x / (1 + e^-z), z a multiple of x (so a NaN is in x already): e^-z = 2^n 2^f with f at most half, log2(e) in two parts, from the native base-2
// exponential; the quotient from a native reciprocal and its own remainder, one rounding less than by way of 1 / (1 + e^-z).  The reciprocal is that of a sixteenth: by itself
// it is zero where it would lie below the smallest normal number, which 1 / (1 + e^-z) does for z from -87.4 on, down to -88.7, where e^-z ends (as with expf, the result is
// zero from there on).  No remainder of an infinite x, or of no quotient, is let in.
// Against 64 bits, times another factor, of the result at most and on average: 2.16e-7 and 4.6e-8 over z of +- 20, 1.7e-7 and 4.5e-8 from -88.7 to -20; with expf and a division
// 2.20e-7 and 5.0e-8, 1.95e-7 and 5.1e-8 down to -87.2, 3.3e-7 and 8.8e-8 below.  17 instructions for 27.
__device__ __forceinline__ float dn_gated(float x, float z) {
    const float c = __builtin_amdgcn_fmed3f(z, -100.0f, 88.0f), n = __builtin_rintf(c * -1.44269504f);
    const float f = __builtin_fmaf(c, -1.92596299e-8f, __builtin_fmaf(c, -1.44269504f, -n));
    const float d = 1.0f + __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n), y = __builtin_amdgcn_rcpf(d * 0.0625f) * 0.0625f, q = x * y;
    return __builtin_fmaf(fmaxf(__builtin_fmaf(-d, q, x), -3.4e38f), y, q);
}
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
    if (EPI == I64H_EPI_SILU_MUL) return dn_gated(acc, acc) * acc2;
    if (EPI == I64H_EPI_CLAMP_GLU) {
        const float u = fminf(acc, p.act_b), w = fminf(fmaxf(acc2, -p.act_b), p.act_b);
        return dn_gated(u, p.act_a * u) * (w + 1.0f);
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

// 16-byte loads through a buffer descriptor: a 32-bit offset per lane, the step's offset in a scalar register, and offsets past the end read
// as zeros - a ragged end needs no branch and nothing is done to the registers behind the load
typedef uint32_t dn_v4u __attribute__((ext_vector_type(4)));
typedef uint32_t dn_v2u __attribute__((ext_vector_type(2)));
constexpr uint32_t DN_BUF_END = 0xfffffff0u;       // from here on: zeros
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dn_buffer(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)DN_BUF_END, 0x00020000);
}
__device__ __forceinline__ dn_v4u dn_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_bytes, uint32_t step_bytes) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, lane_bytes, step_bytes, 0);
}

// The tile of a workgroup.  Workgroups go to the 8 XCDs in turn, so that every XCD gets a run of neighbouring tiles (its L2 then serves their common
// rows and columns); within the run, columns of eight row tiles.
struct dn_tile {
    int64_t b, g0, rows;      // batch, its first row, its rows
    int mt, nt;
    bool any;
};
template <int BM>
__device__ __forceinline__ dn_tile dn_find_tile(const i64h_linear& p, int n_tiles, int m_tiles, int lane) {
    dn_tile o{(int64_t)blockIdx.z, 0, p.M, 0, 0, true};
    int R = m_tiles;
    // rows dealt to batches: lane l counts the tiles of batch 64 c + l, the lanes up to it their sum (one round of loads, not a chain of them)
    const int batches = p.group_off ? p.batch : 0;
    auto count = [&](int c) {
        const int e = c + lane;
        int t = e < batches ? (min(p.group_off[e + 1] - p.group_off[e], (int)p.M) + BM - 1) / BM : 0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(t, d);
            t += lane >= d ? up : 0;
        }
        return t;
    };
    if (p.group_off) {
        R = 0;
        for (int c = 0; c < batches; c += 64) R += __builtin_amdgcn_readlane(count(c), 63);
    }
    const int T = R * n_tiles, id = blockIdx.x;
    if (id >= T) {
        o.any = false;
        return o;
    }
    const int q = T >> 3, r = T & 7, x = id & 7;
    const int t = x * q + min(x, r) + (id >> 3);
    const int per = 8 * n_tiles, g = t / per, first = g * 8, width = min(8, R - first), in = t - g * per;
    o.mt = first + in % width;
    o.nt = in / width;
    for (int c = 0; c < batches; c += 64) {
        const int upto = count(c), all = __builtin_amdgcn_readlane(upto, 63);
        if (o.mt >= all) {
            o.mt -= all;
            continue;
        }
        const int e = __ffsll((unsigned long long)__ballot(upto > o.mt)) - 1;
        if (e > 0) o.mt -= __builtin_amdgcn_readlane(upto, e - 1);
        o.b = c + e;
        o.g0 = p.group_off[o.b];
        o.rows = min(p.M, p.group_off[o.b + 1] - o.g0);
        break;
    }
    return o;
}

// the matrix-core tile forms of i64h_linear_run (i64h_linear_block.hip): operands readable 16 bytes at a time.
// form: -1 chosen by size, else the number of a tile form (tests, measurements).  False: the launch does not fit this form.
bool dn_linear_block(const i64h_linear& d, int form, hipStream_t s);

// launches whose input rows come in bf16 (i64h_linear_wide.hip).  form as above.  False: the launch does not fit.
bool dn_linear_wide(const i64h_linear& d, int form, hipStream_t s);
int dn_linear_wide_form(const i64h_linear& d);

#endif
