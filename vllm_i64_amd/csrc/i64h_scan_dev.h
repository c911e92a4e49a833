// A token's step of the recurrences of i64h_gdn_scan (delta rule) and i64h_gla_scan, shared by the scans token by token.
#ifndef I64H_SCAN_DEV_H
#define I64H_SCAN_DEV_H
#include "i64h_common.h"

enum { GD_DELTA = 0, GD_KEYS = 1, GD_FORGET = 2 };
// The y-th run to be started (the same for the whole workgroup), those of more than 16 rows before the others: workgroups start in their order, and a launch that came to
// its long runs behind many single rows would wait for them alone.  Delta rule, 16 heads of 128, token by token: 27 single rows in front of 229 and 256
// 67 -> 50 us, 40 in front of 100 39 -> 27, 8 heads, 20 in front of 128 26.4 -> 24.6; 64 runs of 17 in any order 39.4 -> 40.7.
// (Beyond 256 runs finding out would cost more than it gives: as they lie.)
__device__ __forceinline__ int gd_run(const int32_t* __restrict__ seg_start, int nseg, int y) {
    if (nseg == 1 || nseg > 256) return y;
    const int lane = threadIdx.x & 63;
    unsigned long long is[4];
    int longs = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int s = min(64 * b + lane, nseg - 1);
        is[b] = 64 * b < nseg ? __ballot(seg_start[s + 1] - seg_start[s] > 16 && 64 * b + lane < nseg) : 0;
        longs += __popcll(is[b]);
    }
    int k = y < longs ? y : y - longs, run = y;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int have = min(64, max(0, nseg - 64 * b));
        const unsigned long long all = have == 64 ? ~0ull : (1ull << have) - 1, m = y < longs ? is[b] : ~is[b] & all;
        const int c = __popcll(m);
        if (k >= 0 && k < c)      // the k-th of these
            run = 64 * b + __ffsll(__ballot(((m >> lane) & 1) && __popcll(m & ((1ull << lane) - 1)) == k)) - 1;
        k -= c;
    }
    return __builtin_amdgcn_readfirstlane(run);
}
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
