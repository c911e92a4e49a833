// A token's step of the recurrences of i64h_gdn_scan (delta rule) and i64h_gla_scan, shared by the scans token by token.
#ifndef I64H_SCAN_DEV_H
#define I64H_SCAN_DEV_H
#include "i64h_common.h"

enum { GD_DELTA = 0, GD_KEYS = 1, GD_FORGET = 2 };
// A lane's KPT channels: four neighbours in every stripe of 64 (so that 16 lanes read 256 consecutive bytes at a time).
template <int KPT>
__device__ __forceinline__ int gd_channel(int nlane, int k) {
    return KPT >= 4 ? 4 * (nlane + 16 * (k >> 2)) + (k & 3) : nlane * KPT + k;
}
// A token's part in a column's state and what it reads, shared by both kernels: a lane's sums run in two chains (even and odd channels), whose
// instructions follow each other without waiting.
template <int KPT, bool CHD>
__device__ __forceinline__ float gd_delta(float (&S)[KPT], const float* f, const float* k, const float* q, float v, float beta) {
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        S[i] *= f[CHD ? i : 0];
        if (i & 1) s1 = fmaf(S[i], k[i], s1);
        else s0 = fmaf(S[i], k[i], s0);
    }
    const float d = beta * (v - group_sum(s0 + s1, 16));
    float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        S[i] = fmaf(k[i], d, S[i]);
        if (i & 1) o1 = fmaf(S[i], q[i], o1);
        else o0 = fmaf(S[i], q[i], o0);
    }
    return group_sum(o0 + o1, 16);
}
template <int KPT, bool CHD, bool FORGET>
__device__ __forceinline__ float gd_linear(float (&S)[KPT], const float* f, const float* k, const float* q, float v) {
    float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const float fi = f[CHD ? i : 0];
        S[i] = fmaf(fi, S[i], (FORGET ? 1.0f - fi : k[FORGET ? 0 : i]) * v);
        if (i & 1) o1 = fmaf(S[i], q[i], o1);
        else o0 = fmaf(S[i], q[i], o0);
    }
    return group_sum(o0 + o1, 16);
}

#endif
