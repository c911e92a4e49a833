// Routing: bit-mask routing, int64 routing-table lookup, stable bucketing of (route, token) rows by
// (expert, route), row gather.  All index work is integer and bit-exact; no atomics decide an order.
//
// Bucketing is a three-phase stable counting sort in which every wave owns a contiguous range of source
// rows: (A) per-wave histograms, (B) a scan over waves per bucket plus the bucket offsets, (C) each wave
// walks its range in order and places rows with wave ballots.  Row order inside a bucket is therefore the
// source order, which is what a boolean-mask gather produces on the CPU.
#include "i64h_common.h"

// Rows a wave of the three launches: what it does is a chain of loads and exchanges, so many waves of few rows, the scan over the waves dealt to all threads of its workgroup, a row's place from
// ballots.  32768 rows, two layers, replayed: 16 buckets 31.7 -> 11.7 us, 128 buckets 71 -> 31 (512 rows a wave, one thread a bucket in the scan, a walk over the buckets before).
#define ROWS_PER_WAVE 128
#define SMALL_ROWS 512      // up to here a workgroup of 256 threads does all three phases, up to MID_ROWS one of 1024
#define MID_ROWS 4096
#define PLAN_THREADS 256
#define MAX_BUCKETS 256

// ---- route_tokens: expert = id & (E-1) -----------------------------------------------------------
__global__ void route_mask_kernel(const int64_t* __restrict__ ids, int32_t* __restrict__ out, int64_t n, int64_t mask) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (int32_t)(ids[i] & mask);
}

// ---- routing-table lookup: routes[k][t] = table[k][clamp(id[t], 0, V-1)] -----------------------------
__global__ void route_lookup_kernel(const int64_t* __restrict__ ids, const int64_t* __restrict__ table,
                                    int64_t* __restrict__ routes, int64_t n, int top_k, int64_t V) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * top_k) return;
    int k = (int)(i / n);
    int64_t t = i - (int64_t)k * n;
    int64_t id = ids[t];
    id = id < 0 ? 0 : (id >= V ? V - 1 : id);
    routes[i] = table[(int64_t)k * V + id];  // ids coalesced, table gather served by L2 (512 KB per layer)
}

// ---- phase A ---------------------------------------------------------------------------------------
// keys[l][s] for source row s = k*n + t, and per-wave histograms wave_counts[l][w][b].
// TABLE=true: key = table[l][k][clamp(id)] * top_k + k (bucket of the (route, token) row);
// TABLE=false: key = keys_in[s] (caller-supplied bucket ids, e.g. expert ids).
template <bool TABLE>
__global__ __launch_bounds__(PLAN_THREADS) void bucket_hist_kernel(
    const int64_t* __restrict__ ids, const int64_t* __restrict__ tables, int64_t table_layer_stride,
    const int32_t* __restrict__ keys_in, int32_t* __restrict__ keys, int64_t* __restrict__ routes, int32_t* __restrict__ tok_slots,
    int32_t* __restrict__ wave_counts, int n, int top_k, int64_t V, int nb, int num_waves) {
    __shared__ int hist[PLAN_THREADS / 64][MAX_BUCKETS];
    const int l = blockIdx.y;
    const int wib = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int gw = blockIdx.x * (PLAN_THREADS / 64) + wib;
    const int64_t R = (int64_t)n * top_k;
    for (int b = lane; b < nb; b += 64) hist[wib][b] = 0;
    __syncthreads();
    if (gw < num_waves && R > 0) {
        int64_t s0 = (int64_t)gw * ROWS_PER_WAVE;
        int64_t s1 = s0 + ROWS_PER_WAVE < R ? s0 + ROWS_PER_WAVE : R;
        constexpr int RPL = ROWS_PER_WAVE / 64;      // a lane's rows: their ids are asked for together, then their table entries
        int64_t e[RPL];
        int k[RPL];
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const int64_t s = min(s0 + lane + 64 * i, s1 - 1);
            k[i] = TABLE ? (int)(s / n) : 0;
            e[i] = TABLE ? ids[s - (int64_t)k[i] * n] : keys_in[s];
        }
        if (TABLE) {
#pragma unroll
            for (int i = 0; i < RPL; ++i) {
                const int64_t id = e[i] < 0 ? 0 : (e[i] >= V ? V - 1 : e[i]);
                e[i] = tables[(int64_t)l * table_layer_stride + (int64_t)k[i] * V + id];
            }
        }
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const int64_t s = s0 + lane + 64 * i;
            if (s >= s1) continue;
            int key = (int)e[i];
            if (TABLE) {
                if (routes) routes[(int64_t)l * R + s] = e[i];
                key = (int)e[i] * top_k + k[i];
                key = key < 0 ? 0 : (key >= nb ? nb - 1 : key);
                if (tok_slots) {  // per token: [0] = the call over all tokens, [1+k] = 1 + bucket of route k
                    int32_t* ts = tok_slots + ((int64_t)l * n + (s - (int64_t)k[i] * n)) * (1 + top_k);
                    ts[1 + k[i]] = 1 + key;
                    if (k[i] == 0) ts[0] = 0;
                }
            }
            key = key < 0 ? 0 : (key >= nb ? nb - 1 : key);  // memory safety only; valid inputs never clamp
            keys[(int64_t)l * R + s] = key;
            atomicAdd(&hist[wib][key], 1);  // LDS integer add: a count, order does not matter
        }
    }
    __syncthreads();
    if (gw < num_waves)
        for (int b = lane; b < nb; b += 64) wave_counts[((int64_t)l * num_waves + gw) * nb + b] = hist[wib][b];
}

// ---- phase B: exclusive scan over waves per bucket, then bucket offsets --------------------------------
__global__ __launch_bounds__(MAX_BUCKETS) void bucket_scan_kernel(int32_t* __restrict__ wave_counts, int32_t* __restrict__ offsets,
                                                                  int32_t* __restrict__ group_offsets, int group, int nb, int num_waves) {
    // the waves of a bucket are dealt to as many threads as there are (its count, then its running offsets: two rounds of loads that wait for nothing)
    __shared__ int tot[MAX_BUCKETS], part[MAX_BUCKETS];
    const int l = blockIdx.x, nbp = nb <= 1 ? 1 : 1 << (32 - __clz(nb - 1)), parts = MAX_BUCKETS / nbp;
    const int b = threadIdx.x & (nbp - 1), mine = threadIdx.x / nbp, per = (num_waves + parts - 1) / parts;
    const int w0 = min(num_waves, mine * per), w1 = min(num_waves, w0 + per);
    int32_t* p = wave_counts + (int64_t)l * num_waves * nb + min(b, nb - 1);
    int sum = 0;
#pragma unroll 8
    for (int w = w0; w < w1; ++w) sum += p[(int64_t)w * nb];
    part[threadIdx.x] = sum;
    __syncthreads();
    int run = 0;
    for (int j = 0; j < mine; ++j) run += part[j * nbp + b];
    if (b < nb) {
        if (mine == parts - 1) tot[b] = run + sum;
        for (int w = w0; w < w1; w += 8) {
            int c[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) c[j] = w + j < w1 ? p[(int64_t)(w + j) * nb] : 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (w + j < w1) p[(int64_t)(w + j) * nb] = run;
                run += c[j];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        int32_t* o = offsets + (int64_t)l * (nb + 1);
        for (int i = 0; i < nb; ++i) {
            o[i] = run;
            run += tot[i];
        }
        o[nb] = run;
        if (group_offsets) {  // offsets of every `group` consecutive buckets (= one expert's routes)
            int32_t* go = group_offsets + (int64_t)l * (nb / group + 1);
            for (int i = 0; i <= nb / group; ++i) go[i] = o[i * group];
        }
    }
}

// The lanes whose bucket is this lane's, of those in `valid`: a ballot a bit of the bucket
__device__ __forceinline__ uint64_t same_bucket(int key, uint64_t valid, int bits) {
    uint64_t m = valid;
    for (int i = 0; i < bits; ++i) {
        const uint64_t on = __ballot((key >> i) & 1);
        m &= ((key >> i) & 1) ? on : ~on;
    }
    return m;
}

// ---- phase C: stable placement ---------------------------------------------------------------------
__global__ __launch_bounds__(PLAN_THREADS) void bucket_place_kernel(
    const int32_t* __restrict__ keys, const int32_t* __restrict__ wave_counts, const int32_t* __restrict__ offsets,
    int32_t* __restrict__ perm, int32_t* __restrict__ inv, int32_t* __restrict__ sorted_bucket, int64_t R, int nb,
    int num_waves) {
    __shared__ int cursor[PLAN_THREADS / 64][MAX_BUCKETS];
    const int l = blockIdx.y;
    const int wib = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int gw = blockIdx.x * (PLAN_THREADS / 64) + wib;
    if (gw >= num_waves) return;  // no block-wide barrier below: each wave uses only its own LDS row
    for (int b = lane; b < nb; b += 64)
        cursor[wib][b] = offsets[(int64_t)l * (nb + 1) + b] + wave_counts[((int64_t)l * num_waves + gw) * nb + b];
    __builtin_amdgcn_wave_barrier();
    const int64_t s0 = (int64_t)gw * ROWS_PER_WAVE;
    const int64_t s1 = s0 + ROWS_PER_WAVE < R ? s0 + ROWS_PER_WAVE : R;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int bits = nb <= 1 ? 0 : 32 - __clz(nb - 1);
    for (int64_t base = s0; base < s1; base += 64) {
        const int64_t s = base + lane;
        const bool valid = s < s1;
        const int key = valid ? keys[(int64_t)l * R + s] : 0;
        const uint64_t m = same_bucket(key, __ballot(valid), bits);
        const int start = cursor[wib][key], rank = __popcll(m & lt), pos = start + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) cursor[wib][key] = start + __popcll(m);
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            perm[(int64_t)l * R + pos] = (int32_t)s;
            inv[(int64_t)l * R + s] = pos;
            if (sorted_bucket) sorted_bucket[(int64_t)l * R + pos] = key;
        }
    }
}

// embedding rows + stat-slot reset riding in the small plan launch (layers = number of plan workgroups in front; 0 riders when table == nullptr)
struct PlanEmbed {
    const float* table;
    float* out;
    uint32_t* stats;
    int64_t stat_words, emb_vocab;
    int H, layers;
};

// ---- all three phases in one launch for steps whose rows one workgroup covers, RPT rows a thread ------------------------------------------------
// One workgroup per layer; 64 rows are a group, whose counts by bucket lie in LDS.  A row's place among its group comes from ballots; as one wave's walk over the buckets that its 64 rows
// have, a dependent LDS read each, and in three launches from 513 rows on, two layers, replayed, before and after, us: 16 buckets, 2 rows 4.5 -> 4.2, 128 rows 6.4 -> 4.5, 512 14.0 -> 4.7, 1024
// 18.9 -> 6.9, 4096 20.5 -> 11.1 (1024 in the three launches as they are here: 4.0 + 4.0 + 5.1); 128 buckets, 128 rows 20 -> 5.4, 1024 56 -> 8.4.  Same keys, offsets, permutation: the results are identical to the three-launch path.
template <bool TABLE, int NT, int RPT>
__global__ __launch_bounds__(NT) void bucket_plan_small_kernel(
    const int64_t* __restrict__ ids, const int64_t* __restrict__ tables, int64_t table_layer_stride,
    const int32_t* __restrict__ keys_in, int32_t* __restrict__ keys, int64_t* __restrict__ routes, int32_t* __restrict__ tok_slots,
    int32_t* __restrict__ offsets, int32_t* __restrict__ group_offsets, int32_t* __restrict__ perm,
    int32_t* __restrict__ inv, int32_t* __restrict__ sorted_bucket, int n, int top_k, int64_t V, int nb, PlanEmbed em) {
    extern __shared__ int cnt[];      // [groups][nb]
    __shared__ int tot[MAX_BUCKETS], first[MAX_BUCKETS + 1];
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= em.layers) {
        // riders of the plan launch: the embedding rows of the same token ids and the start-of-forward reset of the stat slots
        // (both depend on nothing but the ids; as a launch of their own they cost a dispatch and ~4.6 us in front of layer 0)
        const int at = blockIdx.x - em.layers, t = at * (NT / MAX_BUCKETS) + tid / MAX_BUCKETS;
        for (int64_t i = (int64_t)at * NT + tid; i < em.stat_words; i += (int64_t)(gridDim.x - em.layers) * NT) em.stats[i] = I64H_ORDERED_ZERO;
        if (t >= n) return;
        int64_t id = ids[t];
        id = id < 0 ? 0 : (id >= em.emb_vocab ? em.emb_vocab - 1 : id);
        const float4* src = (const float4*)(em.table + id * em.H);
        float4* dst = (float4*)(em.out + (int64_t)t * em.H);
        for (int i = tid % MAX_BUCKETS; i < em.H / 4; i += MAX_BUCKETS) dst[i] = src[i];
        return;
    }
    const int l = blockIdx.x, lane = tid & 63, g0 = (tid >> 6) * RPT;
    const int R = n * top_k, groups = (R + 63) / 64, bits = nb <= 1 ? 0 : 32 - __clz(nb - 1);
    for (int i = tid; i < groups * nb; i += NT) cnt[i] = 0;
    int64_t e[RPT];
    int k[RPT], key[RPT], rank[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int s = min(64 * (g0 + j) + lane, R - 1);
        k[j] = TABLE ? s / n : 0;
        e[j] = TABLE ? ids[s - k[j] * n] : keys_in[s];
    }
    if (TABLE) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int64_t id = e[j] < 0 ? 0 : (e[j] >= V ? V - 1 : e[j]);
            e[j] = tables[(int64_t)l * table_layer_stride + (int64_t)k[j] * V + id];
        }
    }
    __syncthreads();
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int s = 64 * (g0 + j) + lane;
        const bool valid = s < R;
        key[j] = TABLE ? (int)e[j] * top_k + k[j] : (int)e[j];
        key[j] = key[j] < 0 ? 0 : (key[j] >= nb ? nb - 1 : key[j]);
        const uint64_t m = same_bucket(key[j], __ballot(valid), bits);
        rank[j] = __popcll(m & lt);
        if (!valid) continue;
        if (rank[j] == 0) cnt[(g0 + j) * nb + key[j]] = __popcll(m);
        keys[(int64_t)l * R + s] = key[j];
        if (TABLE) {
            if (routes) routes[(int64_t)l * R + s] = e[j];
            if (tok_slots) {
                int32_t* ts = tok_slots + ((int64_t)l * n + (s - k[j] * n)) * (1 + top_k);
                ts[1 + k[j]] = 1 + key[j];
                if (k[j] == 0) ts[0] = 0;
            }
        }
    }
    __syncthreads();
    if (tid < nb) {      // the rows of a bucket in front of every group
        int run = 0;
        for (int g = 0; g < groups; g += 8) {
            int c[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) c[j] = g + j < groups ? cnt[(g + j) * nb + tid] : 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (g + j < groups) cnt[(g + j) * nb + tid] = run;
                run += c[j];
            }
        }
        tot[tid] = run;
    }
    __syncthreads();
    for (int b = tid; b <= nb; b += NT) {
        int run = 0;
#pragma unroll 8
        for (int i = 0; i < b; ++i) run += tot[i];
        first[b] = run;
        offsets[(int64_t)l * (nb + 1) + b] = run;
        if (group_offsets && b % top_k == 0) group_offsets[(int64_t)l * (nb / top_k + 1) + b / top_k] = run;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int s = 64 * (g0 + j) + lane;
        if (s >= R) continue;
        const int pos = first[key[j]] + cnt[(g0 + j) * nb + key[j]] + rank[j];
        perm[(int64_t)l * R + pos] = (int32_t)s;
        inv[(int64_t)l * R + s] = pos;
        if (sorted_bucket) sorted_bucket[(int64_t)l * R + pos] = key[j];
    }
}

// ---- row gather: dst[i] = src[idx[i]] (rows of row_bytes bytes) ------------------------------------------
__global__ void gather_rows_kernel(const char* __restrict__ src, const int32_t* __restrict__ idx, char* __restrict__ dst,
                                   int64_t n_rows, int64_t row_bytes, int vec16) {
    const int64_t r = blockIdx.x;
    if (r >= n_rows) return;
    const int64_t sr = idx ? (int64_t)idx[r] : r;
    if (vec16) {
        const uint4* s = (const uint4*)(src + sr * row_bytes);
        uint4* d = (uint4*)(dst + r * row_bytes);
        for (int64_t i = threadIdx.x; i < row_bytes / 16; i += blockDim.x) d[i] = s[i];
    } else {
        const char* s = src + sr * row_bytes;
        char* d = dst + r * row_bytes;
        for (int64_t i = threadIdx.x; i < row_bytes; i += blockDim.x) d[i] = s[i];
    }
}

// ---- silu(gate) * up on a [n, 2I] matrix ------------------------------------------------------------
template <typename T>
__global__ void silu_mul_kernel(const T* __restrict__ gu, T* __restrict__ out, int64_t n, int I) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * I) return;
    int64_t r = i / I;
    int c = (int)(i - r * I);
    float g = (float)gu[r * 2 * I + c], u = (float)gu[r * 2 * I + I + c];
    out[i] = (T)((g / (1.0f + expf(-g))) * u);
}

// =====================================================================================================
extern "C" {

int i64h_route_tokens(const int64_t* token_ids, int32_t* expert_ids, int64_t n, int32_t num_experts, void* stream) {
    I64H_CHECK_ARG(n >= 0 && num_experts > 0, "route_tokens: bad sizes n=%lld E=%d", (long long)n, num_experts);
    I64H_CHECK_ARG((num_experts & (num_experts - 1)) == 0, "route_tokens: num_experts=%d is not a power of two", num_experts);
    if (n == 0) return 0;
    hipLaunchKernelGGL(route_mask_kernel, dim3(i64h_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, token_ids, expert_ids, n,
                       (int64_t)(num_experts - 1));
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_route_lookup(const int64_t* token_ids, const int64_t* table, int64_t* routes, int64_t n, int32_t top_k, int64_t vocab,
                      void* stream) {
    I64H_CHECK_ARG(n >= 0 && top_k > 0 && vocab > 0, "route_lookup: bad sizes");
    if (n == 0) return 0;
    hipLaunchKernelGGL(route_lookup_kernel, dim3(i64h_cdiv(n * top_k, 256)), dim3(256), 0, (hipStream_t)stream, token_ids, table,
                       routes, n, (int)top_k, vocab);
    I64H_CHECK_LAUNCH();
    return 0;
}

int64_t i64h_bucketize_workspace_bytes(int64_t rows, int32_t num_buckets, int32_t layers) {
    int64_t waves = (rows + ROWS_PER_WAVE - 1) / ROWS_PER_WAVE;
    if (waves < 1) waves = 1;
    return (int64_t)layers * waves * num_buckets * 4;
}

static int bucketize_common(bool table, const int64_t* ids, const int64_t* tables, int64_t layer_stride, const int32_t* keys_in,
                            int32_t* keys, int64_t* routes, int32_t* tok_slots, int32_t* offsets, int32_t* group_offsets, int32_t* perm,
                            int32_t* inv, int32_t* sorted_bucket, int32_t* workspace, int n, int top_k, int64_t V, int nb, int L,
                            hipStream_t st, const PlanEmbed* riders = nullptr, bool* riders_done = nullptr) {
    I64H_CHECK_ARG(nb > 0 && nb <= MAX_BUCKETS, "bucketize: %d buckets unsupported (max %d)", nb, MAX_BUCKETS);
    I64H_CHECK_ARG(n >= 0 && top_k > 0 && L > 0, "bucketize: bad sizes");
    const int64_t R = (int64_t)n * top_k;
    I64H_CHECK_ARG(R < (1ll << 31), "bucketize: too many rows");
    int num_waves = (int)((R + ROWS_PER_WAVE - 1) / ROWS_PER_WAVE);
    if (num_waves < 1) num_waves = 1;
    const int64_t lds = (R + 63) / 64 * nb * 4;
    if (R > 0 && R <= MID_ROWS && lds <= 32768) {  // one workgroup covers the rows: the three phases in one launch
        PlanEmbed em = {nullptr, nullptr, nullptr, 0, 0, 0, L};
        if (riders && table) {
            em = *riders;
            em.layers = L;
            *riders_done = true;
        }
        auto launch = [&](auto kern, int threads) {
            const int extra = em.table ? (int)i64h_cdiv(n, threads / MAX_BUCKETS) : 0;
            hipLaunchKernelGGL(kern, dim3(L + extra), dim3(threads), (size_t)lds, st, ids, tables, layer_stride, keys_in, keys, routes, tok_slots, offsets, group_offsets, perm, inv,
                               sorted_bucket, n, top_k, V, nb, em);
        };
        if (R <= SMALL_ROWS) table ? launch(bucket_plan_small_kernel<true, 256, 2>, 256) : launch(bucket_plan_small_kernel<false, 256, 2>, 256);
        else table ? launch(bucket_plan_small_kernel<true, 1024, 4>, 1024) : launch(bucket_plan_small_kernel<false, 1024, 4>, 1024);
        I64H_CHECK_LAUNCH();
        return 0;
    }
    const int wpb = PLAN_THREADS / 64;
    dim3 grid(i64h_cdiv(num_waves, wpb), L);
    if (table)
        hipLaunchKernelGGL(bucket_hist_kernel<true>, grid, dim3(PLAN_THREADS), 0, st, ids, tables, layer_stride, keys_in, keys,
                           routes, tok_slots, workspace, n, top_k, V, nb, num_waves);
    else
        hipLaunchKernelGGL(bucket_hist_kernel<false>, grid, dim3(PLAN_THREADS), 0, st, ids, tables, layer_stride, keys_in, keys,
                           routes, tok_slots, workspace, n, top_k, V, nb, num_waves);
    I64H_CHECK_LAUNCH();
    hipLaunchKernelGGL(bucket_scan_kernel, dim3(L), dim3(MAX_BUCKETS), 0, st, workspace, offsets, group_offsets, top_k, nb, num_waves);
    I64H_CHECK_LAUNCH();
    if (R > 0) {
        hipLaunchKernelGGL(bucket_place_kernel, grid, dim3(PLAN_THREADS), 0, st, keys, workspace, offsets, perm, inv, sorted_bucket,
                           R, nb, num_waves);
        I64H_CHECK_LAUNCH();
    }
    return 0;
}

int i64h_bucketize(const int32_t* keys_in, int32_t* keys, int32_t* offsets, int32_t* perm, int32_t* inv, int32_t* sorted_bucket,
                   int32_t* workspace, int64_t rows, int32_t num_buckets, void* stream) {
    I64H_CHECK_ARG(rows >= 0 && rows < (1ll << 31), "bucketize: bad row count");
    return bucketize_common(false, nullptr, nullptr, 0, keys_in, keys, nullptr, nullptr, offsets, nullptr, perm, inv, sorted_bucket,
                            workspace, (int)rows, 1, 0, num_buckets, 1, (hipStream_t)stream);
}

int i64h_moe_plan(const int64_t* token_ids, const int64_t* tables, int64_t table_layer_stride, int64_t* routes, int32_t* keys,
                  int32_t* tok_slots, int32_t* offsets, int32_t* expert_offsets, int32_t* perm, int32_t* inv, int32_t* sorted_bucket,
                  int32_t* workspace, int64_t n, int32_t top_k, int64_t vocab, int32_t num_experts, int32_t layers, void* stream) {
    I64H_CHECK_ARG(n >= 0 && n * top_k < (1ll << 31), "moe_plan: bad token count");
    return bucketize_common(true, token_ids, tables, table_layer_stride, nullptr, keys, routes, tok_slots, offsets, expert_offsets, perm,
                            inv, sorted_bucket, workspace, (int)n, top_k, vocab, num_experts * top_k, layers, (hipStream_t)stream);
}

int i64h_embedding_stats_reset(const int64_t* ids, const float* table, float* out, int64_t n, int32_t H, int64_t V, uint32_t* stats,
                               int64_t n_slots, void* stream);

int i64h_moe_plan_embedding(const int64_t* token_ids, const int64_t* tables, int64_t table_layer_stride, int64_t* routes, int32_t* keys,
                            int32_t* tok_slots, int32_t* offsets, int32_t* expert_offsets, int32_t* perm, int32_t* inv,
                            int32_t* sorted_bucket, int32_t* workspace, int64_t n, int32_t top_k, int64_t vocab, int32_t num_experts,
                            int32_t layers, const float* embed_table, float* embed_out, int32_t H, int64_t embed_vocab, uint32_t* stats,
                            int64_t n_slots, void* stream) {
    I64H_CHECK_ARG(n >= 0 && n * top_k < (1ll << 31), "moe_plan_embedding: bad token count");
    I64H_CHECK_ARG(embed_table && embed_out && H > 0 && H % 4 == 0 && embed_vocab > 0, "moe_plan_embedding: H=%d must be a positive multiple of 4", H);
    I64H_CHECK_ARG(n_slots == 0 || stats, "moe_plan_embedding: stats is NULL");
    PlanEmbed em = {embed_table, embed_out, stats, stats ? n_slots * I64H_SLOT_WORDS : 0, embed_vocab, H, 0};
    bool done = false;
    const int rc = bucketize_common(true, token_ids, tables, table_layer_stride, nullptr, keys, routes, tok_slots, offsets, expert_offsets,
                                    perm, inv, sorted_bucket, workspace, (int)n, top_k, vocab, num_experts * top_k, layers,
                                    (hipStream_t)stream, &em, &done);
    if (rc != 0 || done) return rc;
    return i64h_embedding_stats_reset(token_ids, embed_table, embed_out, n, H, embed_vocab, stats, n_slots, stream);
}

int i64h_gather_rows(const void* src, const int32_t* idx, void* dst, int64_t n_rows, int64_t row_bytes, void* stream) {
    I64H_CHECK_ARG(n_rows >= 0 && row_bytes > 0, "gather_rows: bad sizes");
    if (n_rows == 0) return 0;
    int vec16 = (row_bytes % 16 == 0) && (((uintptr_t)src | (uintptr_t)dst) % 16 == 0);
    int threads = 256;
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)n_rows), dim3(threads), 0, (hipStream_t)stream, (const char*)src, idx,
                       (char*)dst, n_rows, row_bytes, vec16);
    I64H_CHECK_LAUNCH();
    return 0;
}

// dtype: 0 = fp32, 1 = fp16, 2 = bf16
int i64h_silu_mul(const void* gate_up, void* out, int64_t n, int32_t inter, int32_t dtype, void* stream) {
    I64H_CHECK_ARG(n >= 0 && inter > 0, "silu_mul: bad sizes");
    if (n == 0) return 0;
    dim3 grid(i64h_cdiv(n * inter, 256)), block(256);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == 0)
        hipLaunchKernelGGL(silu_mul_kernel<float>, grid, block, 0, st, (const float*)gate_up, (float*)out, n, (int)inter);
    else if (dtype == 1)
        hipLaunchKernelGGL(silu_mul_kernel<_Float16>, grid, block, 0, st, (const _Float16*)gate_up, (_Float16*)out, n, (int)inter);
    else if (dtype == 2)
        hipLaunchKernelGGL(silu_mul_kernel<__bf16>, grid, block, 0, st, (const __bf16*)gate_up, (__bf16*)out, n, (int)inter);
    else
        I64H_CHECK_ARG(false, "silu_mul: unknown dtype %d", dtype);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
