// The choice of a row's experts and the plan of a step's (token, choice) pairs (i64h_route_topk, i64h_moe_plan), shared by their own launches and the residual's.
#ifndef I64H_ROUTE_DEV_H
#define I64H_ROUTE_DEV_H
#include <type_traits>

#include "i64h_common.h"
#include "i64h_dense.h"

#define RT_MAX_TOP 32
__device__ __forceinline__ float rt_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// Eight values' sums over a wave in the order of wave_sum: lane j of eight (lane >> 3) ends with the sum of a[j].  Seven exchanges in the place of 48.
__device__ __forceinline__ float rt_sum8(const float* a) {
    auto swapped = [](float x, float y, auto half) {      // half: {x.lo, y.lo} + {x.hi, y.hi}, else the same over neighbouring rows of 16
        unsigned u = __builtin_bit_cast(unsigned, x), v = __builtin_bit_cast(unsigned, y);
        if constexpr (decltype(half)::value) asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(u), "+v"(v));
        else asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(u), "+v"(v));
        return __builtin_bit_cast(float, u) + __builtin_bit_cast(float, v);
    };
    float b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = swapped(a[j], a[j + 4], std::true_type());
    const float c0 = swapped(b[0], b[2], std::false_type()), c1 = swapped(b[1], b[3], std::false_type());
    const bool up = threadIdx.x & 8;
    const float give = up ? c0 : c1;
    float v = (up ? c1 : c0) + I64H_DPPF(give, 0x128);      // row_ror:8
    const int w = __builtin_bit_cast(int, v);
    int x = __builtin_amdgcn_update_dpp(w, w, 0x104, 0xf, 0x5, false);      // lane ^ 4: row_shl:4 in the even quads, row_shr:4 in the odd ones
    x = __builtin_amdgcn_update_dpp(x, w, 0x114, 0xf, 0xa, false);
    v += __builtin_bit_cast(float, x);
    v += I64H_DPPF(v, 0x4E);
    v += I64H_DPPF(v, 0xB1);
    return v;
}

// What a wave's lanes make of the choices: lane k has the k-th (weight, index); PUBLISH: for a workgroup of the same launch
template <bool PUBLISH>
__device__ __forceinline__ void rt_store(const i64h_route_args& p, int64_t t, int lane, float w, int i, float wsum) {
    if (p.chosen_softmax) {     // the weights are the softmax over the chosen ones
        const float top1 = wave_max(lane < p.top ? w : -INFINITY);
        w = lane < p.top ? expf(w - top1) : 0.0f;
        wsum = wave_sum(w);
    }
    if (lane < p.top) {
        const float v = (p.raw_weights ? w : w / (wsum + 1e-20f)) * p.scale;
        if (PUBLISH) {
            st_agent((float*)p.idx + t * p.top + lane, __builtin_bit_cast(float, i));
            st_agent(p.wgt + t * p.top + lane, v);
        } else {
            p.idx[t * p.top + lane] = i;
            p.wgt[t * p.top + lane] = v;
        }
    }
}

// At most 64 entries in one group, an entry's logit z in its lane: all of it in registers, a choice one maximum and one ballot (through LDS, with a second maximum over the indexes, a
// launch of 7 rows of 1024 took 7.6 us, 4.4 so; 64 rows of 2048 8.0 and 5.6)
template <bool PUBLISH>
__device__ __forceinline__ void rt_choose_few(const i64h_route_args& p, int64_t t, int lane, float z) {
    const bool mine = lane < p.E;
    float s = z, c = z;
    if (p.sigmoid_scores) {
        s = rt_sigmoid(z);
        if (p.correction) c = s + (mine ? p.correction[lane] : 0.0f);
    } else if (p.chosen_softmax) {
        if (p.correction) c = s + (mine ? p.correction[lane] : 0.0f);
    } else {
        const float mx = wave_max(mine ? fmaxf(-INFINITY, z) : -INFINITY);
        const float v = mine ? expf(z - mx) : 0.0f;
        s = v / wave_sum(v);
        c = p.correction ? s + (mine ? p.correction[lane] : 0.0f) : s;
    }
    bool open = mine && c == c;
    float w = 0.0f, wsum = 0.0f;
    int at = 0;
    for (int k = 0; k < p.top; ++k) {
        const float best = wave_max(open ? c : -INFINITY);
        const unsigned long long m = __ballot(open && c == best);
        const int pick = m ? __ffsll(m) - 1 : 0;
        const float sp = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s), pick));
        wsum += sp;
        if (lane == k) w = sp, at = pick;
        if (lane == pick) open = false;
    }
    rt_store<PUBLISH>(p, t, lane, w, at, wsum);
}

// The plan, by one workgroup of NT threads; lds: [2 * experts + 1].  idx(i), wgt(i): a pair's choice and weight.
// (An LDS atomic a pair is the fastest way to its row: sums over a wave's lanes in its place, a ballot or a byte an expert, take 4.1 us for 1 to 256 tokens of two of 8 experts where this
// takes 2.8, 10.7 for 4096 where this takes 9.4.)
template <int NT, typename Idx, typename Wgt>
__device__ __forceinline__ void rt_plan(const i64h_moe_plan_args& p, int* lds, Idx idx, Wgt wgt) {
    int* cnt = lds;      // [experts + 1] counts, then offsets
    int* cur = lds + p.experts + 1;
    const int tid = threadIdx.x, E = p.experts;
    const int64_t pairs = p.n * p.top, base = p.shared ? p.n : 0;
    if (p.shared) {
        if (tid == 0) p.group_off[0] = 0;
        for (int64_t t = tid; t < p.n; t += NT) {
            p.pair_token[t] = (int)t;
            if (p.pair_wgt) p.pair_wgt[t] = 1.0f;
        }
    }
    int32_t* group_off = p.group_off + (p.shared ? 1 : 0);
    for (int e = tid; e <= E; e += NT) cnt[e] = 0;
    __syncthreads();
    for (int64_t i = tid; i < pairs; i += NT) {
        const int e = idx(i);
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int run = (int)base;
        for (int e = 0; e < E; ++e) {
            const int c = cnt[e];
            cnt[e] = run;
            cur[e] = run;
            run += c;
        }
        cnt[E] = run;
    }
    __syncthreads();
    for (int e = tid; e <= E; e += NT) group_off[e] = cnt[e];
    for (int64_t i = tid; i < pairs; i += NT) {
        const int e = idx(i);
        int r = -1;
        if (e >= 0 && e < E) {
            r = atomicAdd(&cur[e], 1);
            p.pair_token[r] = (int)((uint32_t)i / (uint32_t)p.top);
            if (p.pair_wgt) p.pair_wgt[r] = wgt(i);
        }
        p.pair_row[i] = r;
    }
}

#endif
