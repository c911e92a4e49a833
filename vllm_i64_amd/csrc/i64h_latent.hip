// Latent attention of libi64hip_dense.so (include/i64h_dense.h): every token caches ONE row per layer - a normalised low-rank
// latent and a rotated key part shared by all heads.  The per-head key and value projections of the latent are never
// materialised: the caller carries the query through the key projection (q' = W_uk^T q, a batched Linear) and the attention
// output back through the value projection (a batched Linear over the summed latents), so a head's score is
// q'_latent . latent_j + q_rot . key_rot_j and all heads read the same cached rows.
//   latent_prep_kernel     : RMS norm of the latent, rotation of the shared key part and of every head's rotated query part,
//                            cache write - one workgroup per token
//   latent_attn_rows_kernel: bf16 caches of aligned widths, portions of prompts - four waves of 16 rows that share 32 keys at a time through LDS;
//                            latent_attn_rows_f32_kernel: the same for 32-bit caches, 32-bit products (latent_row in both where a value is no finite number)
//   latent_attn_mfma_decode_kernel: the same caches, rows that are one per sequence - a token's heads, 16 query vectors per wave
//   latent_attn_row_kernel : any width and cache type, true fp32 products: one wave per (token, head): 64 keys at a time, one key per lane for the scores (fp32 dot over the
//                            cached row), online softmax over the wave, weighted row sum with the columns spread over the lanes
#include "i64h_common.h"
#include "i64h_dense.h"
#include <type_traits>

__device__ __forceinline__ float lt_load(const void* cache, int dtype, int64_t idx) {
    return dtype == 0 ? ((const float*)cache)[idx] : __uint_as_float((uint32_t)((const uint16_t*)cache)[idx] << 16);
}
__device__ __forceinline__ void lt_store(void* cache, int dtype, int64_t idx, float v) {
    if (dtype == 0) {
        ((float*)cache)[idx] = v;
    } else {
        uint32_t u = __float_as_uint(v);
        u = (u & 0x7fffffffu) > 0x7f800000u ? ((u >> 16) | 0x40u) : ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        ((uint16_t*)cache)[idx] = (uint16_t)u;
    }
}

__global__ __launch_bounds__(256) void latent_prep_kernel(const i64h_latent_prep_args p) {
    __shared__ float red[4];
    const int tid = threadIdx.x;
    const int64_t t = blockIdx.x;
    const int pos = p.positions[t], slot = p.slot_ids[t];
    const int r = p.kv_rank, rd = p.rot_dim, D = r + rd, half = p.rot_dims / 2;
    const int64_t row = (int64_t)p.block_table[(int64_t)slot * p.max_blocks_per_seq + pos / p.block_size] * p.block_size + pos % p.block_size;
    const float* pr = p.P + t * p.ldp;
    const float* dkv = pr + p.dkv_off;
    float s = 0.0f;
    for (int c = tid; c < r; c += 256) s += dkv[c] * dkv[c];
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    const float den = sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)r + p.eps);
    for (int c = tid; c < r; c += 256) lt_store(p.cache, p.cache_dtype, row * D + c, dkv[c] / den * p.c_norm_w[c]);
    const float fpos = (float)pos;
    // the shared key part and every head's query part: index 0 is the key, 1 + h the heads
    for (int e = tid; e < (p.heads + 1) * rd; e += 256) {
        const int who = e / rd, c = e % rd;
        const float* src = who == 0 ? dkv + r : (p.Qsrc ? p.Qsrc + t * p.ldqs : pr) + p.q_off + (int64_t)(who - 1) * (p.dim + rd) + p.dim;
        float v;
        if (c < 2 * half) {
            float sn, cs;
            sincosf(fpos * p.inv_freq[c >> 1], &sn, &cs);
            sn *= p.rot_mult, cs *= p.rot_mult;
            const float a = src[c & ~1], b = src[c | 1];
            v = (c & 1) ? (b * cs + a * sn) : (a * cs - b * sn);
        } else {
            v = src[c];
        }
        if (who == 0) lt_store(p.cache, p.cache_dtype, row * D + r + c, v);
        else p.Q[(t * p.heads + (who - 1)) * D + r + c] = v;
    }
}

#define LT_MAXC 16  // latent columns per lane: kv_rank <= 64 * LT_MAXC

__global__ __launch_bounds__(256) void latent_attn_row_kernel(const i64h_latent_attn_args p) {
    extern __shared__ float lds[];  // [4][D] scaled queries, [4][64] weights, [4][64] cache rows
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t t = blockIdx.x;
    const int r = p.kv_rank, D = r + p.rot_dim;
    float* sq = lds + w * D;
    float* sp = lds + 4 * D + w * 64;
    int* srow = (int*)(lds + 4 * D + 256) + w * 64;
    const int h_raw = blockIdx.y * 4 + w;
    const bool active = h_raw < p.heads;
    const int h = active ? h_raw : p.heads - 1;
    const int pos = p.positions[t], slot = p.slot_ids[t];
    const float* q = p.Q + (t * p.heads + h) * D;
    for (int d = lane; d < D; d += 64) sq[d] = q[d] * p.scale;
    __syncthreads();
    const int j0 = p.window > 0 ? max(0, pos - p.window + 1) : 0;
    // the visible keys in order: the kept first positions in front of the window, then j0 .. pos
    const int kept = p.window > 0 ? min(p.keep_first, j0) : 0, total = kept + pos - j0 + 1;
    const int32_t* bt = p.block_table + (int64_t)slot * p.max_blocks_per_seq;
    // the sink: one more score (a learned one per head, or zero) that counts in the denominator and carries no value
    float m = p.sink ? (p.sink_w ? p.sink_w[h] : 0.0f) : -INFINITY, l = p.sink ? 1.0f : 0.0f, acc[LT_MAXC];
#pragma unroll
    for (int i = 0; i < LT_MAXC; ++i) acc[i] = 0.0f;
    for (int ib = 0; ib < total; ib += 64) {
        const int i = ib + lane;
        const bool valid = i < total;
        const int jj = valid ? (i < kept ? i : j0 + i - kept) : pos;
        const int64_t rj = (int64_t)bt[jj / p.block_size] * p.block_size + jj % p.block_size;
        float s = 0.0f;
        if (p.cache_dtype == 0) {
            const float* kr = (const float*)p.cache + rj * D;
            if ((D & 3) == 0) {
                for (int d = 0; d < D; d += 4) {
                    const float4 kv = *(const float4*)(kr + d);
                    s += sq[d] * kv.x; s += sq[d + 1] * kv.y; s += sq[d + 2] * kv.z; s += sq[d + 3] * kv.w;
                }
            } else {
                for (int d = 0; d < D; ++d) s += sq[d] * kr[d];
            }
        } else {
            const uint16_t* kr = (const uint16_t*)p.cache + rj * D;
            if ((D & 7) == 0) {
                for (int d = 0; d < D; d += 8) {
                    const uint4 kv = *(const uint4*)(kr + d);
                    const uint32_t kw[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s += sq[d + 2 * i] * __uint_as_float(kw[i] << 16);
                        s += sq[d + 2 * i + 1] * __uint_as_float(kw[i] & 0xffff0000u);
                    }
                }
            } else {
                for (int d = 0; d < D; ++d) s += sq[d] * __uint_as_float((uint32_t)kr[d] << 16);
            }
        }
        if (p.softcap > 0.0f) s = p.softcap * tanhf(s / p.softcap);
        s = valid ? s : -INFINITY;
        const float mn = fmaxf(m, wave_max(s));
        const float alpha = expf(m - mn);
        const float pj = valid ? expf(s - mn) : 0.0f;
        l = l * alpha + wave_sum(pj);
        m = mn;
        __syncthreads();  // the previous block's weights have been read by every lane
        sp[lane] = pj;
        srow[lane] = (int)rj;
        __syncthreads();
        const int cnt = min(64, total - ib);
#pragma unroll
        for (int i = 0; i < LT_MAXC; ++i) acc[i] *= alpha;
        for (int k = 0; k < cnt; ++k) {
            const float pk = sp[k];
            const int64_t base = (int64_t)srow[k] * D;
#pragma unroll
            for (int i = 0; i < LT_MAXC; ++i) {
                const int c = lane + 64 * i;
                if (c < r) acc[i] += pk * lt_load(p.cache, p.cache_dtype, base + c);
            }
        }
    }
    if (active) {
        float* o = p.out + (t * p.heads + h) * r;
#pragma unroll
        for (int i = 0; i < LT_MAXC; ++i) {
            const int c = lane + 64 * i;
            if (c < r) o[c] = acc[i] / l;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
#define LT_KD 10   // 32-wide steps over a cached row: kv_rank + rot_dim <= 320
#define LT_NB 16   // 16-column blocks of the output: kv_rank <= 256
#define LT_VLD 40  // halves per row of the transposed tile and of the weight planes (32 keys + 8: 16-byte aligned, conflict-poor)
typedef __bf16 lt_v8bf __attribute__((ext_vector_type(8)));
typedef float lt_v4f __attribute__((ext_vector_type(4)));
typedef short lt_v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t lt_rne(float f) {  // nearest even: the hardware conversion of this chip
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ void lt_split(float x, uint32_t& hi, uint32_t& lo) {
    hi = lt_rne(x);
    lo = lt_rne(x - __uint_as_float(hi << 16));
}

// two of them, the first in the low halves: both conversions in one instruction
__device__ __forceinline__ void lt_split_pair(float x, float y, uint32_t& hi, uint32_t& lo) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{x, y}), v2bf));
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{x - __uint_as_float(hi << 16), y - __uint_as_float(hi & 0xffff0000u)}), v2bf));
}

// a value, or four neighbours, of the result: rounded where the caller wants it so
__device__ __forceinline__ void lt_put(const i64h_latent_attn_args& p, int64_t at, float v) {
    if (p.out16) ((uint16_t*)p.out16)[at] = (uint16_t)lt_rne(v);
    else p.out[at] = v;
}
__device__ __forceinline__ void lt_put4(const i64h_latent_attn_args& p, int64_t at, const float4& v) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
    if (p.out16) *(uint2*)((uint16_t*)p.out16 + at) = __builtin_bit_cast(uint2, __builtin_convertvector((v4f{v.x, v.y, v.z, v.w}), v4bf));
    else if (((uintptr_t)p.out & 15) == 0) *(float4*)(p.out + at) = v;
    else p.out[at] = v.x, p.out[at + 1] = v.y, p.out[at + 2] = v.z, p.out[at + 3] = v.w;
}

// Matrix-core form (bf16 cache) of rows that are one per sequence.  One wave per task of 16 query vectors that walk the same cached rows: the (up to) 16
// heads of a group of one token, a share of its keys.
// Per tile of 32 keys: scores S^T[32, 16] = K Q^T on v_mfma_f32_16x16x32_bf16 with the cached rows read straight from memory as A
// fragments (8 consecutive values of one key per lane) and the scaled query carried as TWO bf16 terms (hi + lo, 16 mantissa bits);
// masking and the online softmax in fp32 as the accumulators lie - a lane holds eight keys of one query, whose weights, again as two bf16 terms, are
// the second product's operand without a move -; the tile's latent columns through LDS, written as they came and read transposed
// (ds_read_b64_tr_b16), out^T[kv_rank, 16] += V^T P^T in fp32.  Every product of two bf16 values is exact in fp32.
// What bounds it is the instructions of one wave a SIMD, and branches most of all: 64 tokens of 32 heads over one row of 288, 2048 keys, 63 | 40 us against
// the form with a branch around every step, score and query fragment (a tile 14000 cycles; the weights through LDS and columns transposed by 144 two-byte
// writes were the smaller part), one token, 500 keys 26 | 14, 32 heads of 64 over 8 key heads, 64 tokens, 1024 keys 38 | 30 (with the merge), 16 heads of 128 over 4,
// 2048 keys 88 | 51.  The general instance, 64 tokens, 2048 keys: one row of 256 with 32 heads 60 | 54, values of 128 and keys of 64 77 | 67, heads of 64
// with a soft cap 67 | 66.5 (72.5 with a branch around every score), with a bias 89 | 72 (88).
// Arranged around the memory latency of such launches: a tile's 18 fragment loads are requested together, the NEXT tile's are
// requested as soon as this tile's scores and transposed columns are done - under its softmax and second product - and the cache rows of the tile
// after that are looked up a tile ahead.  The workgroup is one wave, so LDS traffic needs program order only (no barrier, whose
// fence would wait for the loads in flight).  Registers: a whole SIMD's (one wave per SIMD is all such a launch has anyway).
// KD, NB: 32-wide steps over a cached row and 16-column blocks of the output that an instance holds registers for.  ANY: rows of at most 32 KD values,
// kv_rank <= 16 NB, key scales, soft cap, bias; else rows of exactly 32 KD values, kv_rank 16 NB, keys from step KO on and none of the others: without
// a branch around any, the query's fragments asked for together.
template <int KD, int NB, int KO, bool ANY>
__global__ __launch_bounds__(64) void latent_attn_mfma_decode_kernel(const i64h_latent_attn_args p, const int splits) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x, n = lane & 15, kg = lane >> 4;
    const int r = p.kv_rank, D = r + p.rot_dim, H = p.heads, bs = p.block_size, win = p.window;
    const int keep = p.chunk <= 0 && win > 0 ? p.keep_first : 0;
    const int vld = ANY ? r + 16 : 16 * NB + 16;      // halves per key in LDS (rows 8 banks apart where r is a multiple of 128)
    uint16_t* V = (uint16_t*)smem;            // [32][vld]
    int* rowoff = (int*)(V + 32 * vld);       // [2][32] cache rows of two tiles' keys
    const int64_t task = blockIdx.x;
    const int split = blockIdx.y;
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G, tpg = (rep + 15) / 16;
    const int hgroups = G * tpg;
    const int64_t tok = task / hgroups;
    const int sub = (int)(task % hgroups);
    const int hin = (sub % tpg) * 16;               // first of this wave's heads within its key head
    const int head0 = (sub / tpg) * rep + hin;
    const int rstride = p.row_stride > 0 ? p.row_stride : D;
    const int coff = (sub / tpg) * D;
    const int pos = p.positions[tok], slot = p.slot_ids[tok];
    const int lo = p.chunk > 0 ? (pos / p.chunk) * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0), hi = pos;
    const int32_t* bt = p.block_table + (int64_t)slot * p.max_blocks_per_seq;
    const uint16_t* cache = (const uint16_t*)p.cache;
    // tiles of 32 keys, dealt to the splits in turn: those of the kept first positions in front of the window's first tile, then the window's
    const int t0 = lo >> 5, kt = min((keep + 31) >> 5, t0), tiles = kt + (hi >> 5) - t0 + 1;
    auto first_key = [&](int tile) { return (tile < kt ? tile : t0 + tile - kt) * 32; };
    auto lookup = [&](int kb, int buf) {
        if (lane < 32) {
            const int jc = min(kb + lane, hi);
            rowoff[buf * 32 + lane] = bt[jc / bs] * bs + jc % bs;
        }
    };
    uint4 kf[2][KD];
    auto request = [&](int buf) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint16_t* rowp = cache + (int64_t)rowoff[buf * 32 + 16 * b + n] * rstride + coff;
#pragma unroll
            for (int ks = 0; ks < KD; ++ks) {
                const int d0 = ks * 32 + kg * 8;
                if (ANY) kf[b][ks] = (ks * 32 < D && d0 < D) ? *(const uint4*)(rowp + d0) : make_uint4(0, 0, 0, 0);
                else kf[b][ks] = *(const uint4*)(rowp + d0);
            }
        }
    };
    const int hq = min(head0 + n, H - 1);       // this lane's query (one without a head of its own: nobody reads its result)
    const float* q = p.Q + (tok * H + hq) * D;
    float4 qv[ANY ? 1 : 2 * KD];
    if (!ANY)
#pragma unroll
        for (int i = 0; i < 2 * KD; ++i) qv[i] = *(const float4*)(q + (i >> 1) * 32 + kg * 8 + 4 * (i & 1));
    if (split < tiles) {
        lookup(first_key(split), 0);
        if (split + splits < tiles) lookup(first_key(split + splits), 1);
        __builtin_amdgcn_wave_barrier();
        request(0);
    }
    // the query of row n (head head0 + n) times scale * log2(e), as two bf16 terms - converted while the first tile travels
    uint4 Qh[KD], Ql[KD];
    {
        const bool valid_n = hin + n < rep;
        const float qs = p.scale * 1.4426950408889634f;
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) {
            const int d0 = ks * 32 + kg * 8;
            uint32_t h[8], l[8];
            if (!ANY || (valid_n && d0 < D)) {
                const float4 a = ANY ? *(const float4*)(q + d0) : qv[ANY ? 0 : 2 * ks], b = ANY ? *(const float4*)(q + d0 + 4) : qv[ANY ? 0 : 2 * ks + 1];
                const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) lt_split(v[i] * qs, h[i], l[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) h[i] = l[i] = 0;
            }
            Qh[ks] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
            Ql[ks] = make_uint4(l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16), l[6] | (l[7] << 16));
        }
    }
    lt_v4f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = lt_v4f{0, 0, 0, 0};
    const bool sink = p.sink && split == 0;     // the extra score of zero counts once: in the first share of the keys
    const float capl = p.softcap * 1.4426950408889634f;     // the cap in the units of the scores (powers of two)
    float m = sink ? (p.sink_w ? p.sink_w[hq] * 1.4426950408889634f : 0.0f) : -INFINITY, l = sink && kg == 0 ? 1.0f : 0.0f;      // (the sum in four shares)
    int it = 0;
    for (int tile = split; tile < tiles; tile += splits, ++it) {
        const int cur = it & 1, kb = first_key(tile);
        lt_v4f S[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        float ksc[2][4];
        if (ANY && p.kscale) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) ksc[b][g] = p.kscale[rowoff[cur * 32 + 16 * b + 4 * kg + g]];
        }
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) {
            if (!ANY || ks * 32 < D) {
                const int d0 = ks * 32 + kg * 8;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const uint4 f = kf[b][ks];
                    if (ANY ? (ks + 1) * 32 > p.key_off : ks >= KO) {     // (a step of value-only columns: the query is zero there)
                        S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lt_v8bf, f), __builtin_bit_cast(lt_v8bf, Qh[ks]), S[b], 0, 0, 0);
                        S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lt_v8bf, f), __builtin_bit_cast(lt_v8bf, Ql[ks]), S[b], 0, 0, 0);
                    }
                    if (ANY ? d0 < r : ks < NB / 2) *(uint4*)&V[(16 * b + n) * vld + d0] = f;
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (tile + splits < tiles) request(cur ^ 1);          // the next tile travels under this tile's softmax and second product
        // scores of keys kb + 16 b + 4 kg + g; one branch around the eight of an option, whose chains then run side by side
        auto scores = [&](auto f) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) f(b, g, kb + 16 * b + 4 * kg + g);
        };
        if (ANY && p.kscale) scores([&](int b, int g, int) { S[b][g] *= ksc[b][g]; });
        if (ANY && capl > 0.0f) scores([&](int b, int g, int) { S[b][g] = capl * tanhf(S[b][g] / capl); });
        if (ANY && p.bias) {
            float add[2][4];
            scores([&](int b, int g, int j) { add[b][g] = p.bias[(int64_t)min(max(pos - j, 0), p.bias_rows - 1) * H + hq]; });
            scores([&](int b, int g, int) { S[b][g] += 1.4426950408889634f * add[b][g]; });
        }
        float mx = -INFINITY;
        scores([&](int b, int g, int j) {
            S[b][g] = (j <= pos && (j >= lo || j < keep)) ? S[b][g] : -INFINITY;
            mx = fmaxf(mx, S[b][g]);
        });
        const PairF m1 = swap_rows(mx);
        mx = fmaxf(m1.lo, m1.hi);
        const PairF m2 = swap_halves(mx);
        const float mn = fmaxf(m, fmaxf(m2.lo, m2.hi)), ms = mn == -INFINITY ? 0.0f : mn;
        const float al = __builtin_amdgcn_exp2f(m - ms);
        m = mn;
        float sum = 0.0f;
        uint32_t ph[4], pl[4];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int g = 0; g < 4; g += 2) {
                const float p0 = __builtin_amdgcn_exp2f(S[b][g] - ms), p1 = __builtin_amdgcn_exp2f(S[b][g + 1] - ms);
                sum += p0 + p1;
                uint32_t h0, l0, h1, l1;
                lt_split(p0, h0, l0);
                lt_split(p1, h1, l1);
                ph[b * 2 + g / 2] = h0 | (h1 << 16);
                pl[b * 2 + g / 2] = l0 | (l1 << 16);
            }
        l = l * al + sum;
        if (__ballot(al != 1.0f)) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int g = 0; g < 4; ++g) acc[nb][g] *= al;
        }
        const lt_v8bf Ph = __builtin_bit_cast(lt_v8bf, make_uint4(ph[0], ph[1], ph[2], ph[3])), Pl = __builtin_bit_cast(lt_v8bf, make_uint4(pl[0], pl[1], pl[2], pl[3]));
        // V^T fragments: lane 4 q + c of 16 addresses key 4 kg + q (and 16 keys further), columns 16 nb + 4 c .. + 3, and receives its own column of four keys
        const uint16_t* vp = &V[(4 * kg + (n >> 2)) * vld + 4 * (n & 3)];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (!ANY || nb * 16 < r) {
                const lt_v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lt_v4s*)(vp + nb * 16));
                const lt_v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lt_v4s*)(vp + 16 * vld + nb * 16));
                const lt_v8bf vf = __builtin_bit_cast(lt_v8bf, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Ph, acc[nb], 0, 0, 0);
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Pl, acc[nb], 0, 0, 0);
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (tile + 2 * splits < tiles) lookup(first_key(tile + 2 * splits), cur);   // rows of the tile after next, into the buffer this tile is done with
    }
    const PairF l1 = swap_rows(l);
    const PairF l2 = swap_halves(l1.lo + l1.hi);
    l = l2.lo + l2.hi;
    // query n's columns 16 nb + 4 kg .. + 3
    if (splits > 1) {
        float* o = p.workspace + ((int64_t)task * splits + split) * 16 * (r + 2) + n * (r + 2);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            if (!ANY || nb * 16 < r) {
                *(float2*)(o + nb * 16 + 4 * kg) = make_float2(acc[nb][0], acc[nb][1]);
                *(float2*)(o + nb * 16 + 4 * kg + 2) = make_float2(acc[nb][2], acc[nb][3]);
            }
        if (kg == 0) *(float2*)(o + r) = make_float2(m, l);
        return;
    }
    if (hin + n >= rep) return;
    const int64_t o = (tok * H + head0 + n) * r;
    const float inv = 1.0f / l;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
        if (!ANY || nb * 16 < r) lt_put4(p, o + nb * 16 + 4 * kg, make_float4(acc[nb][0] * inv, acc[nb][1] * inv, acc[nb][2] * inv, acc[nb][3] * inv));
}

// One row and head by one wave, over the keys that it sees only: a key per lane for the scores, the columns (at most 256) spread over the lanes for the
// sum, 32-bit products.  The kernels of prompt portions below multiply a tile's values for all rows of a wave, with weights of zero for keys that
// a row does not see (later ones, another sequence's).  Zero times an infinity is no number, and a sum stays no number from there on: such rows go here.
template <typename T>
__device__ __forceinline__ void latent_row(const i64h_latent_attn_args& p, const int64_t t, const int h) {
    const int lane = threadIdx.x & 63, r = p.kv_rank, D = r + p.rot_dim, bs = p.block_size, win = p.window;
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rstride = p.row_stride > 0 ? p.row_stride : D;
    const T* const cache = (const T*)p.cache + h / (p.heads / G) * D;
    auto value = [](T x) {
        if constexpr (sizeof(T) == 2) return __uint_as_float((uint32_t)x << 16);
        else return x;
    };
    const float* const q = p.Q + (t * p.heads + h) * D;
    const int pos = p.positions[t], slot = p.slot_ids[t], from = p.chunk > 0 ? pos / p.chunk * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0);
    const int kept = p.chunk <= 0 && win > 0 ? min(p.keep_first, from) : 0, total = slot < 0 ? 0 : kept + pos - from + 1;      // (no slot: no keys)
    const int32_t* const bt = p.block_table + (int64_t)slot * p.max_blocks_per_seq;
    auto key_of = [&](int i) { return i < kept ? i : from + i - kept; };      // the visible keys in order
    auto row_of = [&](int i) {
        const int j = key_of(i);
        return cache + ((int64_t)bt[j / bs] * bs + j % bs) * rstride;
    };
    float m = p.sink ? (p.sink_w ? p.sink_w[h] : 0.0f) : -INFINITY, l = p.sink ? 1.0f : 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i0 = 0; i0 < total; i0 += 64) {
        const int i = min(i0 + lane, total - 1), j = key_of(i);
        const T* const kr = row_of(i);
        float s = 0.0f;
        for (int d = p.key_off; d < D; ++d) s = fmaf(q[d] * p.scale, value(kr[d]), s);
        if (p.kscale) s *= p.kscale[(int64_t)bt[j / bs] * bs + j % bs];
        if (p.softcap > 0.0f) s = p.softcap * tanhf(s / p.softcap);
        if (p.bias) s += p.bias[(int64_t)min(pos - j, p.bias_rows - 1) * p.heads + h];
        if (i0 + lane >= total) s = -INFINITY;
        const float mn = fmaxf(m, wave_max(s)), ms = mn == -INFINITY ? 0.0f : mn, al = expf(m - ms), w = i0 + lane < total ? expf(s - ms) : 0.0f;
        l = l * al + wave_sum(w);
        m = mn;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] *= al;
        for (int k = 0; k < min(64, total - i0); ++k) {
            const float wk = __shfl(w, k);
            const T* const v = row_of(i0 + k);
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (lane + 64 * c < r) acc[c] = fmaf(wk, value(v[lane + 64 * c]), acc[c]);
        }
    }
    const int64_t o = (t * p.heads + h) * r;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < r) lt_put(p, o + lane + 64 * c, acc[c] / l);
}

// between words of LDS that a wave's lanes write and those that other lanes of the wave then read (such operations happen in their order: the compiler has to keep it)
__device__ __forceinline__ void lt_handed() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A tile's rows, [64] positions and [64] slots (-1: no such row) in LDS; lane l reads row l's.  (Every wave writes all of them, and reads what it wrote.)
// A run is a stretch of neighbouring rows of one sequence: rows s0 .. s1 - 1, the least and the largest position of them and of those
// among the wave's rows wr .. wr + 15.
struct lt_run {
    int s0, s1, slot, low, high, wlow, whigh;
};
#define LT_DPP(v, ctrl) __builtin_amdgcn_update_dpp(0, (v), (ctrl), 0xf, 0xf, true)
__device__ __forceinline__ uint64_t lt_run_starts(int slot) {
    const int lane = threadIdx.x & 63, before = __shfl_up(slot, 1);
    return __ballot(slot >= 0 && (lane == 0 || before != slot));
}
__device__ __forceinline__ lt_run lt_run_at(int s0, const int* info, int wr) {
    lt_run u;
    const int lane = threadIdx.x & 63, pos = info[lane], slot = info[64 + lane];
    u.s0 = s0;
    u.slot = __builtin_amdgcn_readlane(slot, s0);
    const uint64_t other = __ballot(slot != u.slot) & (~0ull << s0);
    u.s1 = other ? __ffsll((unsigned long long)other) - 1 : 64;
    const bool in = lane >= s0 && lane < u.s1;
    int hi = in ? pos : -1, lo = in ? pos : 0x7fffffff;      // over 16 lanes (lane ^ 1, lane ^ 2, half-row mirror, row mirror), then over the four rows of lanes
    hi = max(hi, LT_DPP(hi, 0xB1)), hi = max(hi, LT_DPP(hi, 0x4E)), hi = max(hi, LT_DPP(hi, 0x141)), hi = max(hi, LT_DPP(hi, 0x140));
    lo = min(lo, LT_DPP(lo, 0xB1)), lo = min(lo, LT_DPP(lo, 0x4E)), lo = min(lo, LT_DPP(lo, 0x141)), lo = min(lo, LT_DPP(lo, 0x140));
    u.whigh = __builtin_amdgcn_readlane(hi, wr), u.wlow = __builtin_amdgcn_readlane(lo, wr);
    u.high = max(max(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(hi, 16)), max(__builtin_amdgcn_readlane(hi, 32), __builtin_amdgcn_readlane(hi, 48)));
    u.low = min(min(__builtin_amdgcn_readlane(lo, 0), __builtin_amdgcn_readlane(lo, 16)), min(__builtin_amdgcn_readlane(lo, 32), __builtin_amdgcn_readlane(lo, 48)));
    return u;
}

// Portions of prompts: consecutive rows that share their sequences' cached rows.  A workgroup is four waves, each 16 rows of one head; the heads
// of a workgroup belong to one key head (HW of them; 4 / HW blocks of 16 rows), so that all four waves read the same 32 keys, staged
// in LDS once: row by row for the scores, the value columns transposed (a thread takes 4 keys x 8 columns) for the second product.
// Products are taken transposed, S^T = K Q^T and out^T = V^T P^T: a lane then holds one row's scores (its maximum needs two exchanges, its
// weights are the second product's operand as they lie, with the keys of the two 16-key blocks interleaved) and four neighbouring columns of
// that row's result.  The next tile is requested before this one's products and stored behind them into the other buffer, the rows of
// the one after that are looked up.  Query and weights are two bf16 terms each, as in the kernel above; sums, maxima and masks fp32.
//
// Bound by LDS and its latency: per 32 keys of 256 + 32 values a workgroup reads 136 KiB of fragments for 68 matrix instructions a wave, and
// the registers of two waves per SIMD leave few reads on their way (one wave per SIMD with all it wants: 194 us where two take 130).
// (For rows of 288, 128 and 256 values and for launches without an option the kernel behind this one; figures of both:)
// 8 prompts of 512 tokens, 16 heads over one cached row of 288: 304 -> 130 us against the form before (a wave per workgroup that read every
// fragment from memory itself and transposed it two bytes at a time), 16 heads of 64 over 4 key heads 120 -> 43 us, 32 heads of 64 over 8 key heads
// on prompts of 1531, 257, 64, 3 and 1101 tokens 285 -> 74 us, one prompt of 77 tokens 29 -> 19 and 17 -> 10 us.
// Which rows latent_row sums again is seen at the end, from sums that are no number: nothing between the products.  A tile's runs are found by lanes: as
// a walk over the rows in LDS they were 1 us of a launch of 16-row tiles and 5 of one of 64-row tiles (one prompt of 77 tokens 20.5 -> 19 us).
// KD: 32-wide steps over the columns that take part in the scores, NB: 16-column blocks of the result, EXTRA: key scales, a soft cap or a bias.
template <int KD, int NB, bool EXTRA>
__global__ __launch_bounds__(256, 2) void latent_attn_rows_kernel(const i64h_latent_attn_args p, const int hw) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, kg = lane >> 4;
    const int r = p.kv_rank, D = r + p.rot_dim, H = p.heads, bs = p.block_size, win = p.window, koff = p.key_off & ~31;
    const int keep = p.chunk <= 0 && win > 0 ? p.keep_first : 0;
    const int kld = D - koff + 8;             // halves per key row in LDS: the columns that take part in the scores, and eight zeros
    const int plane = 32 * kld + r * LT_VLD;
    uint16_t* const buf0 = (uint16_t*)smem;   // twice: keys [32][kld], values transposed [r][LT_VLD]
    int* const info = (int*)(buf0 + 2 * plane);
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G;
    const int rstride = p.row_stride > 0 ? p.row_stride : D;
    const int hgroups = H / hw, rows = 16 * (4 / hw), row_tiles = (int)((p.n + rows - 1) / rows);
    const int task = blockIdx.x, hg = task % hgroups, rt = row_tiles - 1 - task / hgroups;      // (the longest contexts first)
    const int head = hg * hw + wid % hw, coff = hg * hw / rep * D, wr = wid / hw * 16;
    const int64_t row0 = (int64_t)rt * rows;
    const bool row_l = lane < rows && row0 + lane < p.n;
    const int pos_l = row_l ? p.positions[row0 + lane] : -1, slot_l = row_l ? p.slot_ids[row0 + lane] : -1;
    const uint64_t starts = lt_run_starts(slot_l);
    if (blockIdx.y > 0 && (int)blockIdx.y >= __popcll(starts)) return;
    info[lane] = pos_l, info[64 + lane] = slot_l;
    lt_handed();
    bool mine = info[64 + wr + n] < 0 && blockIdx.y == 0;      // this workgroup's rows: those of its runs
    const int64_t tok = row0 + wr + n;
    const bool valid = tok < p.n;
    if (tid < 64) *(uint4*)&buf0[(tid >> 5) * plane + (tid & 31) * kld + D - koff] = make_uint4(0, 0, 0, 0);
    // the query of row n times scale * log2(e) (the softmax runs on powers of two), columns koff + ks * 32 + kg * 8 .. + 7, as two bf16 terms;
    // zeros past the end, as in the keys: no step and no block of columns has a branch of its own
    uint4 Qh[KD], Ql[KD];
    {
        const float* q = p.Q + ((valid ? tok : row0) * H + head) * D;
        const float qs = p.scale * 1.4426950408889634f;
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) {
            const int d0 = koff + ks * 32 + kg * 8;
            Qh[ks] = Ql[ks] = make_uint4(0, 0, 0, 0);
            if (valid && d0 < D) {
                const float4 a = *(const float4*)(q + d0), b = *(const float4*)(q + d0 + 4);
                const float v[8] = {a.x * qs, a.y * qs, a.z * qs, a.w * qs, b.x * qs, b.y * qs, b.z * qs, b.w * qs};
                uint32_t h[8], l[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) lt_split(v[i], h[i], l[i]);
                Qh[ks] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
                Ql[ks] = make_uint4(l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16), l[6] | (l[7] << 16));
            }
        }
    }
    lt_v4f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = lt_v4f{0, 0, 0, 0};
    // (the weight sum of a row is kept in four shares, one per group of keys: the sink belongs to one of them)
    float m = p.sink ? (p.sink_w ? p.sink_w[head] * 1.4426950408889634f : 0.0f) : -INFINITY, l = p.sink && kg == 0 ? 1.0f : 0.0f;
    const float capl = p.softcap * 1.4426950408889634f;
    const uint16_t* const cache = (const uint16_t*)p.cache + coff;
    auto first_seen = [&](int pos) { return p.chunk > 0 ? pos / p.chunk * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0); };
    // staging: this thread's four keys and its (at most two) groups of eight columns
    constexpr int PASS = NB > 8 ? 2 : 1;
    const int kq = tid & 7, cg = tid >> 3;
    const int groups = D >> 3;
    uint4 st[PASS][4];
    int64_t src[4];
    int turn = 0;
    for (uint64_t left = starts; left; left &= left - 1) {
        if ((turn++ & (gridDim.y - 1)) != blockIdx.y) continue;
        const lt_run u = lt_run_at(__ffsll((unsigned long long)left) - 1, info, wr);
        const bool in_run = wr + n >= u.s0 && wr + n < u.s1, whole = wr >= u.s0 && wr + 16 <= u.s1;      // (all of this wave's rows)
        mine |= in_run;
        const int pos = in_run ? info[wr + n] : -1, from = first_seen(max(pos, 0));
        // the keys of the run; of this wave's rows of it: the first and the last one that any sees, from where to where all see every key
        const int lo = first_seen(max(u.low, 0)), hi = u.high, wlo = first_seen(max(u.wlow, 0)), whi = u.whigh, wfrom = first_seen(max(whi, 0)), wall = whole ? u.wlow : -1;
        const int32_t* bt = p.block_table + (int64_t)u.slot * p.max_blocks_per_seq;
        // tiles of 32 keys: those of the kept first positions that lie in front of the window's first tile, then the window's
        const int t0 = lo >> 5, kt = min((keep + 31) >> 5, t0), tiles = hi < 0 ? 0 : kt + (hi >> 5) - t0 + 1;
        auto key_base = [&](int tile) { return (tile < kt ? tile : t0 + tile - kt) * 32; };
        auto look_up = [&](int tile) {
            const int j0 = key_base(min(tile, tiles - 1)) + kq * 4;
            if ((bs & 3) == 0) {      // four neighbours of one page
                const int f = min(j0, hi), pg = f / bs;
                const int64_t base = (int64_t)bt[pg] * bs - pg * bs;
#pragma unroll
                for (int i = 0; i < 4; ++i) src[i] = (base + min(j0 + i, hi)) * rstride;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = min(j0 + i, hi);
                    src[i] = ((int64_t)bt[j / bs] * bs + j % bs) * rstride;
                }
            }
        };
        auto request = [&]() {
#pragma unroll
            for (int q = 0; q < PASS; ++q)
                if (cg + 32 * q < groups)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st[q][i] = *(const uint4*)(cache + src[i] + (cg + 32 * q) * 8);
        };
        auto store = [&](int b) {
            uint16_t* K = buf0 + b * plane;
            uint16_t* V = K + 32 * kld;
#pragma unroll
            for (int q = 0; q < PASS; ++q) {
                const int c0 = (cg + 32 * q) * 8;
                if (c0 >= D) continue;
                if (c0 >= koff)
#pragma unroll
                    for (int i = 0; i < 4; ++i) *(uint4*)&K[(kq * 4 + i) * kld + c0 - koff] = st[q][i];
                if (c0 < r) {
                    // columns c0 + c of keys 4 kq .. + 3; a row of V holds the 32 keys as the second product's lanes take them:
                    // [key group kg][16-key block][4 keys]
                    const int at = (kq & 3) * 8 + (kq >> 2) * 4;
                    const uint32_t a[4][4] = {{st[q][0].x, st[q][0].y, st[q][0].z, st[q][0].w}, {st[q][1].x, st[q][1].y, st[q][1].z, st[q][1].w},
                                              {st[q][2].x, st[q][2].y, st[q][2].z, st[q][2].w}, {st[q][3].x, st[q][3].y, st[q][3].z, st[q][3].w}};
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const uint32_t sel = c & 1 ? 0x07060302u : 0x05040100u;
                        *(uint2*)&V[(c0 + c) * LT_VLD + at] = make_uint2(__builtin_amdgcn_perm(a[1][c >> 1], a[0][c >> 1], sel), __builtin_amdgcn_perm(a[3][c >> 1], a[2][c >> 1], sel));
                    }
                }
            }
        };
        if (tiles > 0) {
            look_up(0);
            request();
            look_up(1);
            store(0);
        }
        __syncthreads();
        for (int tile = 0; tile < tiles; ++tile) {
            const int kb = key_base(tile);
            if (tile + 1 < tiles) {
                request();
                look_up(tile + 2);
            }
            const uint16_t* K = buf0 + (tile & 1) * plane;
            const uint16_t* V = K + 32 * kld;
            if (kb <= whi && (kb + 31 >= wlo || kb < keep)) {      // (something that a row of this wave sees)
                lt_v4f S[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
                for (int ks = 0; ks < KD; ++ks) {
                    const int d0 = ks * 32 + kg * 8;
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const lt_v8bf kf = __builtin_bit_cast(lt_v8bf, *(const uint4*)&K[(16 * b + n) * kld + min(d0, D - koff)]);
                        S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, __builtin_bit_cast(lt_v8bf, Qh[ks]), S[b], 0, 0, 0);
                        S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, __builtin_bit_cast(lt_v8bf, Ql[ks]), S[b], 0, 0, 0);
                    }
                }
                if (EXTRA) {
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int j = kb + 16 * b + kg * 4 + g, jc = min(j, hi);
                            if (p.kscale) S[b][g] *= p.kscale[(int64_t)bt[jc / bs] * bs + jc % bs];
                            if (capl > 0.0f) S[b][g] = capl * tanhf(S[b][g] / capl);
                            if (p.bias) S[b][g] += 1.4426950408889634f * p.bias[(int64_t)min(max(pos - j, 0), p.bias_rows - 1) * H + head];
                        }
                }
                if (kb + 31 > wall || kb < wfrom) {
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int j = kb + 16 * b + kg * 4 + g;
                            S[b][g] = j <= pos && (j >= from || j < keep) ? S[b][g] : -INFINITY;
                        }
                }
                float mx = fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])), fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.0f : mn;
                const float al = __builtin_amdgcn_exp2f(m - ms);
                m = mn;
                float w[2][4], sum = 0.0f;
                uint32_t ph[4], pl[4];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        w[b][g] = __builtin_amdgcn_exp2f(S[b][g] - ms);
                        sum += w[b][g];
                    }
#pragma unroll
                    for (int g = 0; g < 4; g += 2) {
                        uint32_t h0, l0, h1, l1;
                        lt_split(w[b][g], h0, l0);
                        lt_split(w[b][g + 1], h1, l1);
                        ph[b * 2 + g / 2] = h0 | (h1 << 16);
                        pl[b * 2 + g / 2] = l0 | (l1 << 16);
                    }
                }
                l = l * al + sum;
                if (__ballot(al != 1.0f)) {
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                        for (int g = 0; g < 4; ++g) acc[nb][g] *= al;
                }
                const lt_v8bf Ph = __builtin_bit_cast(lt_v8bf, make_uint4(ph[0], ph[1], ph[2], ph[3])), Pl = __builtin_bit_cast(lt_v8bf, make_uint4(pl[0], pl[1], pl[2], pl[3]));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const lt_v8bf vf = __builtin_bit_cast(lt_v8bf, *(const uint4*)&V[min(nb * 16 + n, r - 1) * LT_VLD + kg * 8]);
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Ph, acc[nb], 0, 0, 0);
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Pl, acc[nb], 0, 0, 0);
                }
            }
            if (tile + 1 < tiles) store((tile + 1) & 1);
            __syncthreads();
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    bool nan = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int g = 0; g < 4; ++g) nan |= acc[nb][g] != acc[nb][g];
    const uint64_t lanes = __ballot(valid && mine && nan);
    const uint32_t by_key = (uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu;      // rows of this wave
    for (uint32_t left = by_key; left; left &= left - 1) latent_row<uint16_t>(p, row0 + wr + __ffs((int)left) - 1, head);
    if (!valid || !mine || (by_key >> n & 1)) return;
    const int64_t o = (tok * H + head) * r;
    const float inv = 1.0f / l;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
        if (nb * 16 < r) lt_put4(p, o + nb * 16 + kg * 4, make_float4(acc[nb][0] * inv, acc[nb][1] * inv, acc[nb][2] * inv, acc[nb][3] * inv));
}

// The same for rows of exactly D values, the first R of them value columns, keys from column KO on, without key scales, soft cap or bias.  A tile's rows go
// from memory to LDS by themselves, 16 bytes a lane, two tiles ahead, and lie there once: score fragments are read as rows, value fragments transposed
// (ds_read_b64_tr_b16).  The chunk of 16 bytes at place c of row i is chunk c ^ lt_swizzle(i): rows whose pitch is a multiple of the banks would meet in
// the same ones.  The kernel above moves a tile through registers, 40 of which it holds for it, and writes the value columns a second time, transposed.
// Bound by vector instructions and the chain barrier - scores - softmax - second product (heads of 64), by these, the fragments' way out of LDS and the
// query and result rows (latent rows: 142 MB at 8 x 512, 30 us at a copy's rate).  Two heads a wave, which reads every fragment once for both: 31 us as
// well for heads of 64, 113 for latent rows, whose 320 registers do not stay where the products take them.  Microseconds, the kernel above | this:
//   16 heads over one row of 288: 8 prompts of 512 125 | 74, one of 77 19 | 12.5, 64 portions of 3 behind 500 69 | 41; 32 heads, 229 behind 512 83 | 43
//   16 heads of 64 over 4: 8 x 512 44 | 31, one of 77 9.8 | 9.5; 32 over 8, prompts of 1531, 257, 64, 3, 1101 73 | 51; 24 heads of 128 over 8, 8 x 512 89 | 62
// Heads of 128 whose every context is one tile are slower, by the tiles past the end that are loaded all the same: 24 over 8, 40 prompts of 16 17.7 | 19.4, 300 portions of 2
// behind 30 67 | 75.  (A way of their own for such runs took 70, and 3 to 40 % more in the other launches of this kernel: registers.)
template <int D>
__device__ __forceinline__ int lt_swizzle(int row) {
    if constexpr (D % 128 == 0) return (row & 7) << 1 | (row >> 3 & 1);      // every row starts in bank 0: sixteen places, neighbours in pairs
    else return (row >> 1 & 2) | (row >> 3 & 1);                             // (rows a quarter of the banks apart: four places)
}
struct lt_place {      // a cached row: its page, its place in the page
    int page, in;
};
template <int D, int R, int KO>
__global__ __launch_bounds__(256, 2) void latent_attn_rows_direct_kernel(const i64h_latent_attn_args p, const int hw) {
    static_assert(D % 32 == 0 && (D % 128 == 0 || D % 128 == 32) && R % 16 == 0 && KO % 32 == 0, "");
    constexpr int KD = (D - KO) / 32, NB = R / 16, CH = D / 8, NL = CH / 2, LW = (NL + 3) / 4;      // chunks of a row, a tile's loads of 64 chunks, a wave's
    __shared__ __attribute__((aligned(1024))) uint16_t s0[32 * D], s1[32 * D], s2[32 * D];
    __shared__ int info[128];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, kg = lane >> 4;
    const int H = p.heads, bs = p.block_size, win = p.window;
    const int keep = p.chunk <= 0 && win > 0 ? p.keep_first : 0;
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G;
    const int rstride = p.row_stride > 0 ? p.row_stride : D;
    const int hgroups = H / hw, rows = 16 * (4 / hw), row_tiles = (int)((p.n + rows - 1) / rows);
    const int task = blockIdx.x, hg = task % hgroups, rt = row_tiles - 1 - task / hgroups;      // (the longest contexts first)
    const int head = hg * hw + wid % hw, coff = hg * hw / rep * D, wr = wid / hw * 16;
    const int64_t row0 = (int64_t)rt * rows;
    const bool row_l = lane < rows && row0 + lane < p.n;
    const int pos_l = row_l ? p.positions[row0 + lane] : -1, slot_l = row_l ? p.slot_ids[row0 + lane] : -1;
    const uint64_t starts = lt_run_starts(slot_l);
    if (blockIdx.y > 0 && (int)blockIdx.y >= __popcll(starts)) return;
    info[lane] = pos_l, info[64 + lane] = slot_l;
    __syncthreads();
    bool mine = info[64 + wr + n] < 0 && blockIdx.y == 0;      // this workgroup's rows: those of its runs
    const int64_t tok = row0 + wr + n;
    const bool valid = tok < p.n;
    // the query of row n times scale * log2(e) (the softmax runs on powers of two), columns KO + ks * 32 + kg * 8 .. + 7, as two bf16 terms
    uint4 Qh[KD], Ql[KD];
    {
        const float* q = p.Q + ((valid ? tok : row0) * H + head) * D + KO + kg * 8;
        const float qs = valid ? p.scale * 1.4426950408889634f : 0.0f;
        float4 v[2 * KD];
#pragma unroll
        for (int i = 0; i < 2 * KD; ++i) v[i] = *(const float4*)(q + (i >> 1) * 32 + 4 * (i & 1));
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) {
            const float4 a = v[2 * ks], b = v[2 * ks + 1];
            const float x[8] = {a.x * qs, a.y * qs, a.z * qs, a.w * qs, b.x * qs, b.y * qs, b.z * qs, b.w * qs};
            uint32_t h[4], l[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) lt_split_pair(x[2 * i], x[2 * i + 1], h[i], l[i]);
            Qh[ks] = make_uint4(h[0], h[1], h[2], h[3]);
            Ql[ks] = make_uint4(l[0], l[1], l[2], l[3]);
        }
    }
    lt_v4f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = lt_v4f{0, 0, 0, 0};
    // (the weight sum of a row is kept in four shares, one per group of keys: the sink belongs to one of them)
    float m = p.sink ? (p.sink_w ? p.sink_w[head] * 1.4426950408889634f : 0.0f) : -INFINITY, l = p.sink && kg == 0 ? 1.0f : 0.0f;
    const uint16_t* const cache = (const uint16_t*)p.cache + coff;
    auto first_seen = [&](int pos) { return p.chunk > 0 ? pos / p.chunk * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0); };
    // this lane's chunk of a load of its wave: the key it belongs to and its first column (a wave without a last load of its own repeats the tile's)
    int key_l[LW], col_l[LW];
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int at = min(i * 4 + wid, NL - 1) * 64 + lane;
        key_l[i] = at / CH, col_l[i] = (at % CH ^ lt_swizzle<D>(at / CH)) * 8;
    }
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    constexpr std::integral_constant<int, 2> S2{};
    auto stage = [&](auto set) -> uint16_t* {      // (variables of their own: the compiler then knows which loads a read of one has to wait for)
        constexpr int S = decltype(set)::value;
        return S == 0 ? s0 : S == 1 ? s1 : s2;
    };
    const int krow = n * D, ksw = lt_swizzle<D>(n);
    const int vrow = (4 * kg + (n >> 2)) * D + (n & 1) * 4, vsw = ((n & 3) >> 1) ^ lt_swizzle<D>(4 * kg + (n >> 2));
    int turn = 0;
    for (uint64_t left = starts; left; left &= left - 1) {
        if ((turn++ & (gridDim.y - 1)) != blockIdx.y) continue;
        const lt_run u = lt_run_at(__ffsll((unsigned long long)left) - 1, info, wr);
        const bool in_run = wr + n >= u.s0 && wr + n < u.s1, whole = wr >= u.s0 && wr + 16 <= u.s1;      // (all of this wave's rows)
        mine |= in_run;
        const int pos = in_run ? info[wr + n] : -1, from = first_seen(max(pos, 0));
        // the keys of the run; of this wave's rows of it: the first and the last one that any sees, from where to where all see every key
        const int lo = first_seen(max(u.low, 0)), hi = u.high, wlo = first_seen(max(u.wlow, 0)), whi = u.whigh, wfrom = first_seen(max(whi, 0)), wall = whole ? u.wlow : -1;
        const int32_t* bt = p.block_table + (int64_t)u.slot * p.max_blocks_per_seq;
        // tiles of 32 keys: those of the kept first positions that lie in front of the window's first tile, then the window's
        const int t0 = lo >> 5, kt = min((keep + 31) >> 5, t0), tiles = hi < 0 ? 0 : kt + (hi >> 5) - t0 + 1;
        if (tiles == 0) continue;
        auto key_base = [&](int tile) { return (tile < kt ? tile : t0 + tile - kt) * 32; };
        // lane l < 32: the tile's key l
        auto look_up = [&](int tile) {
            const int j = min(key_base(min(tile, tiles - 1)) + (lane & 31), hi), pg = j / bs;
            return lt_place{bt[pg], j - pg * bs};
        };
        auto load = [&](lt_place at, auto set) {
            uint16_t* sm = stage(set);
            const int row = at.page * bs + at.in;
            int src[LW];
#pragma unroll
            for (int i = 0; i < LW; ++i) src[i] = __shfl(row, key_l[i]);
#pragma unroll
            for (int i = 0; i < LW; ++i)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(cache + (int64_t)src[i] * rstride + col_l[i]),
                                                 (__attribute__((address_space(3))) void*)(sm + min(i * 4 + wid, NL - 1) * 512), 16, 0, 0);
        };
        // this wave's loads of the tile are in LDS, its reads of the one before done; then everybody's.  On their way: the loads of the next tile
        lt_place next;      // of the tile after the next
        auto meet = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0070 | (LW & 15));      // vmcnt LW, lgkmcnt 0
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto step = [&](int tile, auto cur, auto free) {
            meet();
            // (past the end the last tile again, which nobody reads: without a branch the loads on their way are the same everywhere)
            const lt_place then = look_up(tile + 3);
            load(next, free);
            next = then;
            const int kb = key_base(tile);
            if (kb > whi || (kb + 31 < wlo && kb >= keep)) return;      // (nothing that a row of this wave sees)
            const uint16_t* T = stage(cur);
            lt_v4f S[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
            __builtin_amdgcn_sched_barrier(0);
            lt_v8bf kf[KD][2];
#pragma unroll
            for (int ks = 0; ks < KD; ++ks)
#pragma unroll
                for (int b = 0; b < 2; ++b) kf[ks][b] = __builtin_bit_cast(lt_v8bf, *(const uint4*)&T[krow + 16 * b * D + ((KO / 8 + ks * 4 + kg) ^ ksw) * 8]);
#pragma unroll
            for (int ks = 0; ks < KD; ++ks) {
#pragma unroll
                for (int b = 0; b < 2; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks][b], __builtin_bit_cast(lt_v8bf, Qh[ks]), S[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < 2; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks][b], __builtin_bit_cast(lt_v8bf, Ql[ks]), S[b], 0, 0, 0);
            }
            // four steps' fragments on their way
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * (KD < 4 ? KD : 4), 0);
#pragma unroll
            for (int ks = 0; ks < KD; ++ks) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                if (ks + 4 < KD) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (kb + 31 > wall || kb < wfrom) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int j = kb + 16 * b + kg * 4 + g;
                        S[b][g] = j <= pos && (j >= from || j < keep) ? S[b][g] : -INFINITY;
                    }
            }
            float mx = fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])), fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
            const PairF m1 = swap_rows(mx);
            mx = fmaxf(m1.lo, m1.hi);
            const PairF m2 = swap_halves(mx);
            const float mn = fmaxf(m, fmaxf(m2.lo, m2.hi)), ms = mn == -INFINITY ? 0.0f : mn;
            const float al = __builtin_amdgcn_exp2f(m - ms);
            m = mn;
            float w[2][4], sum = 0.0f;
            uint32_t ph[4], pl[4];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    w[b][g] = __builtin_amdgcn_exp2f(S[b][g] - ms);
                    sum += w[b][g];
                }
#pragma unroll
                for (int g = 0; g < 4; g += 2) lt_split_pair(w[b][g], w[b][g + 1], ph[b * 2 + g / 2], pl[b * 2 + g / 2]);
            }
            l = l * al + sum;
            if (__ballot(al != 1.0f)) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int g = 0; g < 4; ++g) acc[nb][g] *= al;
            }
            const lt_v8bf Ph = __builtin_bit_cast(lt_v8bf, make_uint4(ph[0], ph[1], ph[2], ph[3])), Pl = __builtin_bit_cast(lt_v8bf, make_uint4(pl[0], pl[1], pl[2], pl[3]));
            // V^T fragments: lane 4 q + c of 16 addresses key 4 kg + q (and 16 keys further), columns 16 nb + 4 c .. + 3, and receives its own column of four keys
            __builtin_amdgcn_sched_barrier(0);
            lt_v4s va[NB][2];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const uint16_t* vp = &T[vrow + ((2 * nb) ^ vsw) * 8];
#pragma unroll
                for (int b = 0; b < 2; ++b) va[nb][b] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lt_v4s*)(vp + 16 * b * D));
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const lt_v8bf vf = __builtin_bit_cast(lt_v8bf, __builtin_shufflevector(va[nb][0], va[nb][1], 0, 1, 2, 3, 4, 5, 6, 7));
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Ph, acc[nb], 0, 0, 0);
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, Pl, acc[nb], 0, 0, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * (NB < 6 ? NB : 6), 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                if (nb + 6 < NB) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        __syncthreads();      // (the run before has been read)
        const lt_place at0 = look_up(0), at1 = look_up(1);
        next = look_up(2);
        load(at0, S0);
        load(at1, S1);
        int tile = 0;
        for (; tile + 3 <= tiles; tile += 3) {
            step(tile, S0, S2);
            step(tile + 1, S1, S0);
            step(tile + 2, S2, S1);
        }
        if (tile < tiles) step(tile, S0, S2);
        if (tile + 1 < tiles) step(tile + 1, S1, S0);
        __builtin_amdgcn_s_waitcnt(0x0f70);      // (nothing is on its way into LDS when a run ends)
    }
    const PairF l1 = swap_rows(l), l2 = swap_halves(l1.lo + l1.hi);
    bool nan = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int g = 0; g < 4; ++g) nan |= acc[nb][g] != acc[nb][g];
    const uint64_t lanes = __ballot(valid && mine && nan);
    const uint32_t by_key = (uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu;      // rows of this wave
    for (uint32_t left = by_key; left; left &= left - 1) latent_row<uint16_t>(p, row0 + wr + __ffs((int)left) - 1, head);
    if (!valid || !mine || (by_key >> n & 1)) return;
    const int64_t o = (tok * H + head) * R + kg * 4;
    const float inv = 1.0f / (l2.lo + l2.hi);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) lt_put4(p, o + nb * 16, make_float4(acc[nb][0] * inv, acc[nb][1] * inv, acc[nb][2] * inv, acc[nb][3] * inv));
}

// The same for caches of 32-bit rows, with 32-bit products: keys and transposed values once in LDS (twice would be a workgroup per CU), the next tile
// waiting in registers.  Bound by the matrix instructions at their 32-bit rate (272 a wave and 32 keys of 256 + 32 values).  16 heads over one
// cached row of 288, prompts of 300, 75 and 1 tokens: 315 -> 96 us against latent_attn_row_kernel, which reads every key again for each query (the
// widest rows with a SIMD's registers to themselves: 109 us at two waves, whose spills cost more).
#define LT_FLD 36  // values per row of the transposed tile (32 keys + 4)
template <int KC, int NB, bool EXTRA>
__global__ __launch_bounds__(256, NB > 8 ? 1 : 2) void latent_attn_rows_f32_kernel(const i64h_latent_attn_args p, const int hw) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, kg = lane >> 4;
    const int r = p.kv_rank, D = r + p.rot_dim, H = p.heads, bs = p.block_size, win = p.window, koff = p.key_off & ~15;
    const int keep = p.chunk <= 0 && win > 0 ? p.keep_first : 0;
    const int kld = D - koff + 4;             // values per key row in LDS: the columns that take part in the scores, and four zeros
    float* const K = (float*)smem;            // keys [32][kld], values transposed [r][LT_FLD]
    float* const V = K + 32 * kld;
    int* const info = (int*)(V + r * LT_FLD);
    int* const odd = info + 128;                   // a value of a tile that some row sees a part of is no finite number
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G;
    const int rstride = p.row_stride > 0 ? p.row_stride : D;
    const int hgroups = H / hw, rows = 16 * (4 / hw), row_tiles = (int)((p.n + rows - 1) / rows);
    const int task = blockIdx.x, hg = task % hgroups, rt = row_tiles - 1 - task / hgroups;      // (the longest contexts first)
    const int head = hg * hw + wid % hw, coff = hg * hw / rep * D, wr = wid / hw * 16;
    const int64_t row0 = (int64_t)rt * rows;
    const bool row_l = lane < rows && row0 + lane < p.n;
    const int pos_l = row_l ? p.positions[row0 + lane] : -1, slot_l = row_l ? p.slot_ids[row0 + lane] : -1;
    const uint64_t starts = lt_run_starts(slot_l);
    if (blockIdx.y > 0 && (int)blockIdx.y >= __popcll(starts)) return;
    info[lane] = pos_l, info[64 + lane] = slot_l;
    lt_handed();
    bool mine = info[64 + wr + n] < 0 && blockIdx.y == 0;      // this workgroup's rows: those of its runs
    const int64_t tok = row0 + wr + n;
    const bool valid = tok < p.n;
    if (tid < 32) *(lt_v4f*)&K[tid * kld + D - koff] = lt_v4f{0, 0, 0, 0};
    if (tid == 0) *odd = 0;
    // the query of row n times scale * log2(e), columns koff + c * 16 + kg * 4 .. + 3; zeros past the end, as in the keys
    lt_v4f Q[KC];
    {
        const float* q = p.Q + ((valid ? tok : row0) * H + head) * D;
        const float qs = p.scale * 1.4426950408889634f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const int d0 = koff + c * 16 + kg * 4;
            Q[c] = lt_v4f{0, 0, 0, 0};
            if (valid && d0 < D) Q[c] = *(const lt_v4f*)(q + d0) * qs;
        }
    }
    lt_v4f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = lt_v4f{0, 0, 0, 0};
    // (the weight sum of a row is kept in four shares, one per group of keys: the sink belongs to one of them)
    float m = p.sink ? (p.sink_w ? p.sink_w[head] * 1.4426950408889634f : 0.0f) : -INFINITY, l = p.sink && kg == 0 ? 1.0f : 0.0f;
    const float capl = p.softcap * 1.4426950408889634f;
    const float* const cache = (const float*)p.cache + coff;
    auto first_seen = [&](int pos) { return p.chunk > 0 ? pos / p.chunk * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0); };
    // staging: this thread's four keys and its (at most three) groups of four columns
    constexpr int PASS = NB > 8 ? 3 : 2;
    const int kq = tid & 7, cg = tid >> 3;
    const int groups = D >> 2;
    lt_v4f st[PASS][4];
    int64_t src[4];
    int turn = 0;
    for (uint64_t left = starts; left; left &= left - 1) {
        if ((turn++ & (gridDim.y - 1)) != blockIdx.y) continue;
        const lt_run u = lt_run_at(__ffsll((unsigned long long)left) - 1, info, wr);
        const bool in_run = wr + n >= u.s0 && wr + n < u.s1, whole = wr >= u.s0 && wr + 16 <= u.s1;      // (all of this wave's rows)
        mine |= in_run;
        const int pos = in_run ? info[wr + n] : -1, from = first_seen(max(pos, 0));
        // the keys of the run; of this wave's rows of it: the first and the last one that any sees, from where to where all see every key
        const int lo = first_seen(max(u.low, 0)), hi = u.high, wlo = first_seen(max(u.wlow, 0)), whi = u.whigh, wfrom = first_seen(max(whi, 0)), wall = whole ? u.wlow : -1;
        const int all = u.s0 == 0 && u.s1 == rows ? u.low : -1, last = first_seen(max(hi, 0));      // the same of the workgroup's rows
        const int32_t* bt = p.block_table + (int64_t)u.slot * p.max_blocks_per_seq;
        // tiles of 32 keys: those of the kept first positions that lie in front of the window's first tile, then the window's
        const int t0 = lo >> 5, kt = min((keep + 31) >> 5, t0), tiles = hi < 0 ? 0 : kt + (hi >> 5) - t0 + 1;
        auto key_base = [&](int tile) { return (tile < kt ? tile : t0 + tile - kt) * 32; };
        auto look_up = [&](int tile) {
            const int j0 = key_base(min(tile, tiles - 1)) + kq * 4;
            if ((bs & 3) == 0) {      // four neighbours of one page
                const int f = min(j0, hi), pg = f / bs;
                const int64_t base = (int64_t)bt[pg] * bs - pg * bs;
#pragma unroll
                for (int i = 0; i < 4; ++i) src[i] = (base + min(j0 + i, hi)) * rstride;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = min(j0 + i, hi);
                    src[i] = ((int64_t)bt[j / bs] * bs + j % bs) * rstride;
                }
            }
        };
        auto request = [&]() {
#pragma unroll
            for (int q = 0; q < PASS; ++q)
                if (cg + 32 * q < groups)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st[q][i] = *(const lt_v4f*)(cache + src[i] + (cg + 32 * q) * 4);
        };
        auto store = [&](bool partial) {
#pragma unroll
            for (int q = 0; q < PASS; ++q) {
                const int c0 = (cg + 32 * q) * 4;
                if (c0 < D && c0 >= koff)
#pragma unroll
                    for (int i = 0; i < 4; ++i) *(lt_v4f*)&K[(kq * 4 + i) * kld + c0 - koff] = st[q][i];
            }
            if (partial) {      // a sum of zeros unless a value is infinite or no number
                float z = 0.0f;
#pragma unroll
                for (int q = 0; q < PASS; ++q)
                    if ((cg + 32 * q) * 4 < r)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int c = 0; c < 4; ++c) z = fmaf(st[q][i][c], 0.0f, z);
                if (z != 0.0f) *odd = 1;
            }
#pragma unroll
            for (int q = 0; q < PASS; ++q) {
                const int c0 = (cg + 32 * q) * 4;
                if (c0 < r)      // columns c0 + c of keys 4 kq .. + 3
#pragma unroll
                    for (int c = 0; c < 4; ++c) *(lt_v4f*)&V[(c0 + c) * LT_FLD + kq * 4] = lt_v4f{st[q][0][c], st[q][1][c], st[q][2][c], st[q][3][c]};
            }
        };
        if (tiles > 0) {
            look_up(0);
            request();
            look_up(1);
        }
        for (int tile = 0; tile < tiles; ++tile) {
            const int kb = key_base(tile);
            __syncthreads();      // (the tile before has been read)
            store(kb + 31 > all || kb < last);      // (true: a row does not see every key)
            __syncthreads();
            if (tile + 1 < tiles) {
                request();
                look_up(tile + 2);
            }
            if (kb <= whi && (kb + 31 >= wlo || kb < keep)) {      // (something that a row of this wave sees)
                lt_v4f S[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
                for (int c = 0; c < KC; ++c) {
                    const int d0 = c * 16 + kg * 4;
#pragma unroll
                    for (int b = 0; b < 2; ++b) {      // (a lane's four neighbouring columns go to four products)
                        const lt_v4f kf = *(const lt_v4f*)&K[(16 * b + n) * kld + min(d0, D - koff)];
#pragma unroll
                        for (int g = 0; g < 4; ++g) S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[g], Q[c][g], S[b], 0, 0, 0);
                    }
                }
                if (EXTRA) {
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int j = kb + 16 * b + kg * 4 + g, jc = min(j, hi);
                            if (p.kscale) S[b][g] *= p.kscale[(int64_t)bt[jc / bs] * bs + jc % bs];
                            if (capl > 0.0f) S[b][g] = capl * tanhf(S[b][g] / capl);
                            if (p.bias) S[b][g] += 1.4426950408889634f * p.bias[(int64_t)min(max(pos - j, 0), p.bias_rows - 1) * H + head];
                        }
                }
                if (kb + 31 > wall || kb < wfrom) {
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int j = kb + 16 * b + kg * 4 + g;
                            S[b][g] = j <= pos && (j >= from || j < keep) ? S[b][g] : -INFINITY;
                        }
                }
                float mx = fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])), fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.0f : mn;
                const float al = exp2f(m - ms);
                m = mn;
                float w[2][4], sum = 0.0f;
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        w[b][g] = exp2f(S[b][g] - ms);
                        sum += w[b][g];
                    }
                l = l * al + sum;
                if (__ballot(al != 1.0f)) {
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                        for (int g = 0; g < 4; ++g) acc[nb][g] *= al;
                }
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const lt_v4f vf = *(const lt_v4f*)&V[min(nb * 16 + n, r - 1) * LT_FLD + b * 16 + kg * 4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[g], w[b][g], acc[nb], 0, 0, 0);
                    }
            }
        }
    }
    __syncthreads();
    if (*odd) {      // zero times such a value is no zero: these rows key by key, each the keys that it sees
        const uint32_t rows16 = (uint32_t)__ballot(valid && mine) & 0xffffu;
        for (uint32_t left = rows16; left; left &= left - 1) latent_row<float>(p, row0 + wr + __ffs((int)left) - 1, head);
        return;
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (!valid || !mine) return;
    const int64_t o = (tok * H + head) * r;
    const float inv = 1.0f / l;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
        if (nb * 16 < r) lt_put4(p, o + nb * 16 + kg * 4, make_float4(acc[nb][0] * inv, acc[nb][1] * inv, acc[nb][2] * inv, acc[nb][3] * inv));
}

// The same for rows of exactly D values without an option (as latent_attn_rows_direct_kernel), in launches whose workgroups of four heads would leave CUs
// without work: a workgroup takes 16 rows of ONE head, its four waves share every tile's products.  A wave multiplies its quarter of the key columns,
// the waves hand each other the sums through LDS, and each takes its quarter of the value columns: a tile's chain of matrix instructions is a quarter as
// long.  The tile lies in LDS once, as its rows come from memory (the 32-bit products take single values, so no order of them has to be turned), the next
// one on its way into the other buffer; exactly half of a CU's LDS for latent rows.  Bound by that chain in short launches (a tile 1.6 us where it was 4), by the
// matrix instructions at their 32-bit rate in long ones.  Microseconds, the kernel above | this:
//   16 heads over one row of 288: 16 rows 18 | 10, 77 33 | 14, 300 85 | 35, 600 153 | 67, 2000 509 | 456, 8 x 512 391 | 286
//   heads of 64, 16 over 4: 16 rows 8.8 | 9.1, 77 12.5 | 9.4, 300 30 | 17, 1000 86 | 52, 2000 106 | 110, 4000 198 | 242; 32 over 8: 1000 98 | 77, 2000 160 | 213;
//   16 over 16, windows of 128: 300 23 | 13.5, 1000 22.9 | 21.7, 2000 30 | 37; heads of 128, 24 over 8: 300 49 | 24, 1000 157 | 109, 2000 285 | 305
template <int D, int R, int KO>
__global__ __launch_bounds__(256, 2) void latent_attn_rows_f32_quarters_kernel(const i64h_latent_attn_args p) {
    constexpr int KC = (D - KO) / 16, CW = (KC + 3) / 4, NBW = R / 64, CH = D / 4, LW = CH / 8;      // 16-column steps, a wave's of them and its column blocks; chunks of a row, a wave's loads
    static_assert(D % 32 == 0 && R % 64 == 0 && KO % 16 == 0 && (D % 64 == 0 || D % 64 == 32), "");
    __shared__ __attribute__((aligned(1024))) float s0[32 * D], s1[32 * D];
    __shared__ __attribute__((aligned(16))) float ex[4 * 2 * 64 * 4];
    int* const info = (int*)ex;
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, kg = lane >> 4;
    const int H = p.heads, bs = p.block_size, win = p.window;
    const int keep = p.chunk <= 0 && win > 0 ? p.keep_first : 0;
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G;
    const int rstride = p.row_stride > 0 ? p.row_stride : D;
    const int row_tiles = (int)((p.n + 15) / 16), task = blockIdx.x, head = task % H, rt = row_tiles - 1 - task / H;      // (the longest contexts first)
    const int64_t row0 = (int64_t)rt * 16;
    const bool row_l = lane < 16 && row0 + lane < p.n;
    const int pos_l = row_l ? p.positions[row0 + lane] : -1, slot_l = row_l ? p.slot_ids[row0 + lane] : -1;
    const uint64_t starts = lt_run_starts(slot_l);
    if (blockIdx.y > 0 && (int)blockIdx.y >= __popcll(starts)) return;
    bool mine = __shfl(slot_l, n) < 0 && blockIdx.y == 0;      // this workgroup's rows: those of its runs
    const int64_t tok = row0 + n;
    const bool valid = tok < p.n;
    // (key place c of a row lies at c ^ swizzle: rows a multiple of the banks apart would meet in the same ones)
    auto swizzle = [](int row) { return D % 64 == 0 ? row & 15 : row >> 1 & 7; };
    // the query of row n times scale * log2(e), this wave's steps: columns KO + (4 i + wid) * 16 + kg * 4 .. + 3
    lt_v4f Q[CW];
    {
        const float* q = p.Q + ((valid ? tok : row0) * H + head) * D + KO + kg * 4;
        const float qs = valid ? p.scale * 1.4426950408889634f : 0.0f;
#pragma unroll
        for (int i = 0; i < CW; ++i) Q[i] = *(const lt_v4f*)(q + min(4 * i + wid, KC - 1) * 16) * (4 * i + wid < KC ? qs : 0.0f);
    }
    lt_v4f acc[NBW];
#pragma unroll
    for (int i = 0; i < NBW; ++i) acc[i] = lt_v4f{0, 0, 0, 0};
    // (the weight sum of a row is kept in four shares, one per group of keys: the sink belongs to one of them)
    float m = p.sink ? (p.sink_w ? p.sink_w[head] * 1.4426950408889634f : 0.0f) : -INFINITY, l = p.sink && kg == 0 ? 1.0f : 0.0f;
    const float* const cache = (const float*)p.cache + head / rep * D;
    auto first_seen = [&](int pos) { return p.chunk > 0 ? pos / p.chunk * p.chunk : (win > 0 ? max(0, pos - win + 1) : 0); };
    int key_l[LW], col_l[LW];      // this lane's chunk of a load of its wave
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int at = (i * 4 + wid) * 64 + lane;
        key_l[i] = at / CH, col_l[i] = (at % CH ^ swizzle(at / CH)) * 4;
    }
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    auto stage = [&](auto set) -> float* { return decltype(set)::value == 0 ? s0 : s1; };      // (variables of their own: see above)
    const int krow = n * D, ksw = swizzle(n);
    int turn = 0;
    for (uint64_t left = starts; left; left &= left - 1) {
        if ((turn++ & (gridDim.y - 1)) != blockIdx.y) continue;
        __syncthreads();      // (the run before has been read)
        info[lane] = pos_l, info[64 + lane] = slot_l;
        __syncthreads();
        const lt_run u = lt_run_at(__ffsll((unsigned long long)left) - 1, info, 0);
        __syncthreads();
        const bool in_run = n >= u.s0 && n < u.s1;
        mine |= in_run;
        const int pos = in_run ? __shfl(pos_l, n) : -1, from = first_seen(max(pos, 0));
        // the keys of the run; from where to where all rows see every key
        const int lo = first_seen(max(u.low, 0)), hi = u.high, wfrom = first_seen(max(hi, 0)), wall = u.s0 == 0 && u.s1 >= 16 ? u.low : -1;
        const int32_t* bt = p.block_table + (int64_t)u.slot * p.max_blocks_per_seq;
        // tiles of 32 keys: those of the kept first positions that lie in front of the window's first tile, then the window's
        const int t0 = lo >> 5, kt = min((keep + 31) >> 5, t0), tiles = hi < 0 ? 0 : kt + (hi >> 5) - t0 + 1;
        if (tiles == 0) continue;
        auto key_base = [&](int tile) { return (tile < kt ? tile : t0 + tile - kt) * 32; };
        // lane l < 32: the tile's key l
        auto look_up = [&](int tile) {
            const int j = min(key_base(min(tile, tiles - 1)) + (lane & 31), hi), pg = j / bs;
            return lt_place{bt[pg], j - pg * bs};
        };
        auto load = [&](lt_place at, auto set) {
            float* sm = stage(set);
            const int row = at.page * bs + at.in;
            int src[LW];
#pragma unroll
            for (int i = 0; i < LW; ++i) src[i] = __shfl(row, key_l[i]);
#pragma unroll
            for (int i = 0; i < LW; ++i)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(cache + (int64_t)src[i] * rstride + col_l[i]),
                                                 (__attribute__((address_space(3))) void*)(sm + (i * 4 + wid) * 256), 16, 0, 0);
        };
        lt_place next;
        auto step = [&](int tile, auto cur, auto other) {
            // this wave's loads of the tile are in LDS, its reads of the one before done; then everybody's
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0070);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            const lt_place then = look_up(tile + 2);
            load(next, other);      // (past the end the last tile again, which nobody reads)
            next = then;
            const int kb = key_base(tile);
            const float* T = stage(cur);
            lt_v4f S[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                lt_v4f kf[2];
#pragma unroll
                for (int b = 0; b < 2; ++b) kf[b] = *(const lt_v4f*)&T[krow + 16 * b * D + ((KO / 4 + min(4 * i + wid, KC - 1) * 4 + kg) ^ ksw) * 4];
                if (KC % 4 == 0 || 4 * i + wid < KC)
#pragma unroll
                    for (int g = 0; g < 4; ++g)      // (a lane's four neighbouring columns go to four products)
#pragma unroll
                        for (int b = 0; b < 2; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][g], Q[i][g], S[b], 0, 0, 0);
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) *(lt_v4f*)&ex[((wid * 2 + b) * 64 + lane) * 4] = S[b];
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt 0; the next tile's loads stay on their way
            asm volatile("s_barrier" ::: "memory");
            {
                lt_v4f part[4][2];
#pragma unroll
                for (int w = 0; w < 4; ++w)
#pragma unroll
                    for (int b = 0; b < 2; ++b) part[w][b] = *(const lt_v4f*)&ex[((w * 2 + b) * 64 + lane) * 4];
#pragma unroll
                for (int b = 0; b < 2; ++b) S[b] = (part[0][b] + part[1][b]) + (part[2][b] + part[3][b]);
            }
            if (kb + 31 > wall || kb < wfrom) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int j = kb + 16 * b + kg * 4 + g;
                        S[b][g] = j <= pos && (j >= from || j < keep) ? S[b][g] : -INFINITY;
                    }
            }
            float mx = fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])), fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
            const PairF m1 = swap_rows(mx);
            mx = fmaxf(m1.lo, m1.hi);
            const PairF m2 = swap_halves(mx);
            const float mn = fmaxf(m, fmaxf(m2.lo, m2.hi)), ms = mn == -INFINITY ? 0.0f : mn;
            const float al = exp2f(m - ms);
            m = mn;
            float w[2][4], sum = 0.0f;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    w[b][g] = exp2f(S[b][g] - ms);
                    sum += w[b][g];
                }
            l = l * al + sum;
#pragma unroll
            for (int i = 0; i < NBW; ++i) acc[i] *= al;
            // a value fragment's lane holds column n of key 4 kg + g, the order that the weights lie in
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int i = 0; i < NBW; ++i) {
                        const int key = 4 * kg + g;
                        const float vf = T[(16 * b + key) * D + (((wid * NBW + i) * 4 + (n >> 2)) ^ swizzle(key)) * 4 + (n & 3)];
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf, w[b][g], acc[i], 0, 0, 0);
                    }
        };
        const lt_place at0 = look_up(0);
        next = look_up(1);
        load(at0, S0);
        int tile = 0;
        for (; tile + 2 <= tiles; tile += 2) {
            step(tile, S0, S1);
            step(tile + 1, S1, S0);
        }
        if (tile < tiles) step(tile, S0, S1);
        __builtin_amdgcn_s_waitcnt(0x0f70);      // (nothing is on its way into LDS when a run ends)
    }
    const PairF l1 = swap_rows(l), l2 = swap_halves(l1.lo + l1.hi);
    bool nan = false;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) nan |= acc[i][g] != acc[i][g];
    // a value that is no finite number under a weight of zero: such rows key by key, each the keys that it sees (any wave's columns speak for the row)
    const uint64_t lanes = __ballot(valid && mine && nan);
    __syncthreads();
    if (lane == 0) info[wid] = (int)((uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu);
    __syncthreads();
    const uint32_t by_key = (uint32_t)(info[0] | info[1] | info[2] | info[3]);
    for (uint32_t left = by_key, k = 0; left; left &= left - 1, ++k)
        if ((int)(k & 3) == wid) latent_row<float>(p, row0 + __ffs((int)left) - 1, head);
    if (!valid || !mine || (by_key >> n & 1)) return;
    const int64_t o = (tok * H + head) * R + wid * NBW * 16 + kg * 4;
    const float inv = 1.0f / (l2.lo + l2.hi);
#pragma unroll
    for (int i = 0; i < NBW; ++i) lt_put4(p, o + i * 16, make_float4(acc[i][0] * inv, acc[i][1] * inv, acc[i][2] * inv, acc[i][3] * inv));
}

// the shares of a token's keys, merged: one wave per (token, head); lane s holds share s's maximum and weight sum (at most 64
// shares), then every lane sums its columns over the shares, eight loads in flight at a time
template <int NC>      // columns a lane takes at a time: kv_rank <= 64, 128 or more
__global__ __launch_bounds__(64) void latent_attn_merge_kernel(const i64h_latent_attn_args p, const int splits) {
    __shared__ float sf[64];
    const int lane = threadIdx.x;
    const int r = p.kv_rank, H = p.heads;
    const int G = p.kv_groups > 1 ? p.kv_groups : 1, rep = H / G, tpg = (rep + 15) / 16;
    const int hgroups = G * tpg;
    const int64_t task = blockIdx.x, tok = task / hgroups;
    const int m = blockIdx.y;
    const int sub = (int)(task % hgroups);
    if ((sub % tpg) * 16 + m >= rep) return;
    const int head = (sub / tpg) * rep + (sub % tpg) * 16 + m;
    const float* w = p.workspace + (task * splits * 16 + m) * (r + 2);      // share s: + s * 16 * (r + 2)
    const int64_t stride = (int64_t)16 * (r + 2);
    const float* mine = w + (int64_t)min(lane, splits - 1) * stride;
    // eight shares of the columns on their way together, the first in front of the maximum: column by column behind the maximum
    // 7 tokens of 16 heads in 23 shares of 256 columns took 19 us with the attention, so 15
    float v[NC][8];
    auto fetch = [&](int c0, int s0) {
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u) v[i][u] = w[(int64_t)min(s0 + u, splits - 1) * stride + min(c0 + 64 * i, r - 1)];
    };
    const float ms = lane < splits ? mine[r] : -INFINITY, ls = lane < splits ? mine[r + 1] : 0.0f;
    fetch(lane, 0);
    const float mx = wave_max(ms);
    const float f = __builtin_amdgcn_exp2f(ms - mx);      // share `lane`'s factor (0 for an empty share)
    const float den = wave_sum(f * ls);
    sf[lane] = lane < splits ? f : 0.0f;
    __syncthreads();
    for (int c0 = lane; c0 < r; c0 += 64 * NC) {
        float num[NC] = {};
        for (int s0 = 0; s0 < splits; s0 += 8) {
            if (c0 > lane || s0 > 0) fetch(c0, s0);
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int u = 0; u < 8; ++u) num[i] += sf[(s0 + u) & 63] * (s0 + u < splits ? v[i][u] : 0.0f);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i)
            if (c0 + 64 * i < r) lt_put(p, (tok * H + head) * r + c0 + 64 * i, num[i] / den);
    }
}

// Heads of a key head that share a workgroup of the kernels of prompt portions, and their grid: tiles of 16 * (4 / hw) rows times the shares that
// a tile's runs - rows of one sequence each - are dealt to.  Short portions would follow each other in one workgroup otherwise; where a tile is
// one run, the other shares leave at once.  16 heads of 64 over 16 key heads, bf16, one share | four | eight: a portion of 1500 rows beside 64 of three
// with 500 cached tokens each 568 | 172 | 106 us (20 rows in 64 sequences: 17 | 14 | 14; 8 x 512: 46 | 46 | 46); 24 heads of 128 over 8 on 8 x 512, where
// 1536 workgroups fill the chip twice, 90 | 91 | 91, with 16 shares 96.
static int lt_heads_per_group(int rep) { return rep % 4 == 0 ? 4 : (rep % 2 == 0 ? 2 : 1); }
static dim3 lt_rows_grid(const i64h_latent_attn_args& d, int hw) {
    const int rows = 16 * (4 / hw);
    const int64_t wgs = (d.n + rows - 1) / rows * (d.heads / hw);
    int shares = 4;
    while (shares < rows && wgs * shares < 2048) shares *= 2;
    while (shares > d.n) shares /= 2;
    return dim3((unsigned)wgs, (unsigned)shares);
}

// portions of prompts over 32-bit caches (i64h_latent_attn, and i64h_kattn with its key heads, chunks, key scales and bias)
bool latent_rows_f32_ok(const i64h_latent_attn_args& d) {
    const int D = d.kv_rank + d.rot_dim;
    return d.mode == 3 && d.cache_dtype == 0 && D % 4 == 0 && d.kv_rank % 16 == 0 && d.kv_rank <= 256 && D <= 320 && (uintptr_t)d.Q % 16 == 0 &&
           (uintptr_t)d.cache % 16 == 0 && d.row_stride % 4 == 0;
}

int latent_rows_f32_run(const i64h_latent_attn_args& d, void* stream) {
    const int D = d.kv_rank + d.rot_dim;
    const int G = d.kv_groups > 1 ? d.kv_groups : 1;
    I64H_CHECK_ARG(d.heads % G == 0, "latent_attn: %d heads over %d key heads", d.heads, G);
    const int hw = lt_heads_per_group(d.heads / G);
    I64H_CHECK_ARG((d.n + 15) / 16 * d.heads < (1ll << 31), "latent_attn: too many tiles");
    const dim3 grid = lt_rows_grid(d, hw);
    const int kcols = D - (d.key_off & ~15), chunks = (kcols + 15) / 16;
    const size_t bytes = ((size_t)32 * (kcols + 4) + (size_t)d.kv_rank * LT_FLD) * 4 + 129 * 4;
    const bool extra = d.kscale || d.bias || d.softcap > 0.0f;
    auto exact = [&](int width, int rank, int off) { return !extra && D == width && d.kv_rank == rank && d.key_off == off; };
    // quarters: for latent rows always (they were faster in every launch timed), for heads of 64 and 128 while the workgroups of four waves on their own rows would be at most
    // 400 (256 CUs, two or more a CU; the figures beside the kernel: 1000 rows of 32 heads over 8 would be 504 and still gain, 2000 of them and 2000 of 24 heads of 128 over 8 lose), 256
    // where a row sees few keys.  Several sequences in 16 rows are as many workgroups, of which a quarter's
    // reads for itself what four heads of the other form share.  Microseconds, four heads over their rows | quarters: 64 portions of 3 behind 500, 32 heads over 8 (96 of six sequences)
    // 84 | 100, 16 over 4 (48 of six) 62.5 | 62.5, 8 over 2 62 | 57; 300 of 2 behind 30, 8 over 2 (76 of eight) 12.7 | 19.4; 40 of 16, 32 over 8 (320) 11.9 | 12.6
    const int64_t wgs = (d.n + 15) / 16 * d.heads;
    int shares = 4;
    while (shares < 16 && wgs * shares < 2048) shares *= 2;
    while (shares > d.n) shares /= 2;
    const int64_t many = hw > 1 && d.seqs > 0 && d.seqs <= d.n ? ((int64_t)d.seqs * 16 + d.n - 1) / d.n : 1;      // sequences in 16 rows
    const bool brief = (d.window > 0 && d.window <= 256) || (hw > 1 && d.seqs > 0 && d.n <= 16 * (int64_t)d.seqs), few = grid.x * many <= (brief ? 256 : 400);
    auto quarters = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)wgs, (unsigned)shares), dim3(256), 0, (hipStream_t)stream, d); };
#define LT_ROWS(KC, NB) do { \
        if (extra) hipLaunchKernelGGL((latent_attn_rows_f32_kernel<KC, NB, true>), grid, dim3(256), bytes, (hipStream_t)stream, d, hw); \
        else hipLaunchKernelGGL((latent_attn_rows_f32_kernel<KC, NB, false>), grid, dim3(256), bytes, (hipStream_t)stream, d, hw); \
    } while (0)
    if (exact(288, 256, 0)) quarters(latent_attn_rows_f32_quarters_kernel<288, 256, 0>);
    else if (few && exact(128, 64, 64)) quarters(latent_attn_rows_f32_quarters_kernel<128, 64, 64>);
    else if (few && exact(256, 128, 128)) quarters(latent_attn_rows_f32_quarters_kernel<256, 128, 128>);
    else if (chunks <= 4 && d.kv_rank <= 64) LT_ROWS(4, 4);
    else if (chunks <= 8 && d.kv_rank <= 128) LT_ROWS(8, 8);
    else if (chunks <= 18) LT_ROWS(18, 16);
    else LT_ROWS(20, 16);
#undef LT_ROWS
    I64H_CHECK_LAUNCH();
    return 0;
}

static int g_decode_form = 1;
bool latent_decode_form() { return g_decode_form; }

extern "C" {

int i64h_latent_prep(const i64h_latent_prep_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "latent_prep: no descriptor");
    const i64h_latent_prep_args& d = *dp;
    I64H_CHECK_ARG(d.n >= 0 && d.heads > 0 && d.dim > 0 && d.rot_dim >= 0 && d.kv_rank > 0 && d.block_size > 0, "latent_prep: bad sizes");
    I64H_CHECK_ARG(d.rot_dims >= 0 && d.rot_dims <= d.rot_dim && d.rot_dims % 2 == 0, "latent_prep: %d rotated dimensions of %d", d.rot_dims, d.rot_dim);
    I64H_CHECK_ARG(d.cache_dtype == 0 || d.cache_dtype == 2, "latent_prep: cache dtype %d", d.cache_dtype);
    I64H_CHECK_ARG(d.P && d.c_norm_w && d.positions && d.slot_ids && d.block_table && d.cache && d.Q && (d.inv_freq || d.rot_dims == 0), "latent_prep: null operand");
    if (d.n == 0) return 0;
    hipLaunchKernelGGL(latent_prep_kernel, dim3((unsigned)d.n), dim3(256), 0, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_set_latent_attn_decode_form(int32_t on) {  // tuning / test knob: 0 = rows that are one per sequence by a wave per row and head, 32-bit products
    g_decode_form = on;
    return 0;
}

int64_t i64h_latent_attn_workspace_floats(int64_t n, int32_t heads, int32_t kv_rank, int32_t splits) {
    if (splits <= 1) return 0;
    return n * ((heads + 15) / 16) * (int64_t)(splits > 64 ? 64 : splits) * 16 * (kv_rank + 2);
}

int i64h_latent_attn(const i64h_latent_attn_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "latent_attn: no descriptor");
    const i64h_latent_attn_args& d = *dp;
    I64H_CHECK_ARG(d.n >= 0 && d.heads > 0 && d.kv_rank > 0 && d.rot_dim >= 0 && d.block_size > 0, "latent_attn: bad sizes");
    I64H_CHECK_ARG(d.kv_rank <= 64 * LT_MAXC, "latent_attn: kv_rank %d above %d", d.kv_rank, 64 * LT_MAXC);
    I64H_CHECK_ARG(d.cache_dtype == 0 || d.cache_dtype == 2, "latent_attn: cache dtype %d", d.cache_dtype);
    I64H_CHECK_ARG(d.Q && d.cache && d.block_table && d.slot_ids && d.positions && (d.out || d.out16), "latent_attn: null operand");
    I64H_CHECK_ARG(d.key_off >= 0 && d.key_off <= d.kv_rank, "latent_attn: %d value-only columns of %d value columns", d.key_off, d.kv_rank);
    if (d.n == 0) return 0;
    const int D = d.kv_rank + d.rot_dim;
    const bool mfma_ok = d.cache_dtype == 2 && D % 8 == 0 && d.kv_rank % 16 == 0 && d.kv_rank <= 16 * LT_NB && D <= 32 * LT_KD &&
                         (uintptr_t)d.Q % 16 == 0 && (uintptr_t)d.cache % 16 == 0 && d.row_stride % 8 == 0 && (d.mode == 3 || g_decode_form || d.out16);
    I64H_CHECK_ARG(mfma_ok || (d.kv_groups <= 1 && d.row_stride <= 0 && d.chunk <= 0 && !d.kscale && !d.bias),
                   "latent_attn: key heads, chunks, key scales and bias are built for the matrix-core form only");
    I64H_CHECK_ARG(!d.sink_w || d.sink, "latent_attn: sink scores without the sink");
    I64H_CHECK_ARG(!d.out16 || (mfma_ok && d.mode != 1 && (uintptr_t)d.out16 % 16 == 0), "latent_attn: a result in bf16 belongs to the matrix-core form, at 16 bytes");
    I64H_CHECK_ARG(d.keep_first >= 0, "latent_attn: %d kept positions", d.keep_first);
    if (d.mode != 1 && mfma_ok) {
        const int row_tiles = d.mode == 3;
        const int G = d.kv_groups > 1 ? d.kv_groups : 1;
        I64H_CHECK_ARG(d.heads % G == 0, "latent_attn: %d heads over %d key heads", d.heads, G);
        const int64_t tasks = row_tiles ? (d.n + 15) / 16 * d.heads : d.n * G * ((d.heads / G + 15) / 16);
        I64H_CHECK_ARG(tasks < (1ll << 31), "latent_attn: too many tiles");
        const int splits = (!row_tiles && d.workspace && d.splits > 1) ? (d.splits > 64 ? 64 : d.splits) : 1;
        const size_t bytes = (size_t)32 * (d.kv_rank + 16) * 2 + 64 * 4;
        const dim3 grid((unsigned)tasks, (unsigned)splits);
        hipStream_t st = (hipStream_t)stream;
        const int size = (D <= 64 && d.kv_rank <= 64) ? 0 : ((D <= 128 && d.kv_rank <= 128) ? 1 : 2);     // the narrowest instance that holds the rows
        if (row_tiles) {
            const int hw = lt_heads_per_group(d.heads / G);
            const dim3 grid_rows = lt_rows_grid(d, hw);
            const size_t lds = ((size_t)32 * (D - (d.key_off & ~31) + 8) + (size_t)d.kv_rank * LT_VLD) * 4 + 128 * 4;
            const bool extra = d.kscale || d.bias || d.softcap > 0.0f;
#define LT_ROWS(KD, NB) do { \
                if (extra) hipLaunchKernelGGL((latent_attn_rows_kernel<KD, NB, true>), grid_rows, dim3(256), lds, st, d, hw); \
                else hipLaunchKernelGGL((latent_attn_rows_kernel<KD, NB, false>), grid_rows, dim3(256), lds, st, d, hw); \
            } while (0)
            const int steps = (D - (d.key_off & ~31) + 31) / 32;
            auto exact = [&](int width, int rank, int off) { return !extra && D == width && d.kv_rank == rank && d.key_off == off; };
            auto direct = [&](auto kern) { hipLaunchKernelGGL(kern, grid_rows, dim3(256), 0, st, d, hw); };
            if (exact(288, 256, 0)) direct(latent_attn_rows_direct_kernel<288, 256, 0>);                // a latent row of 256 + 32
            else if (exact(128, 64, 64)) direct(latent_attn_rows_direct_kernel<128, 64, 64>);           // values and keys of 64
            else if (exact(256, 128, 128)) direct(latent_attn_rows_direct_kernel<256, 128, 128>);       // ... of 128
            else if (steps <= 2 && d.kv_rank <= 64) LT_ROWS(2, 4);
            else if (steps <= 4 && d.kv_rank <= 128) LT_ROWS(4, 8);
            else if (steps <= 9) LT_ROWS(9, LT_NB);
            else LT_ROWS(LT_KD, LT_NB);
#undef LT_ROWS
        } else {
            const bool plain = !d.kscale && !d.bias && d.softcap <= 0.0f;
            auto exact = [&](int kd, int nb, int ko) { return plain && D == 32 * kd && d.kv_rank == 16 * nb && d.key_off / 32 == ko; };
            auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64), bytes, st, d, splits); };
            if (exact(9, 16, 0)) launch(latent_attn_mfma_decode_kernel<9, 16, 0, false>);             // a latent row of 256 + 32
            else if (exact(4, 4, 2)) launch(latent_attn_mfma_decode_kernel<4, 4, 2, false>);          // values and keys of 64
            else if (exact(8, 8, 4)) launch(latent_attn_mfma_decode_kernel<8, 8, 4, false>);          // ... of 128
            else if (size == 0) launch(latent_attn_mfma_decode_kernel<2, 4, 0, true>);
            else if (size == 1) launch(latent_attn_mfma_decode_kernel<4, 8, 0, true>);
            else launch(latent_attn_mfma_decode_kernel<LT_KD, LT_NB, 0, true>);
        }
        I64H_CHECK_LAUNCH();
        if (splits > 1) {
            auto merge = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)tasks, 16), dim3(64), 0, st, d, splits); };
            if (d.kv_rank <= 64) merge(latent_attn_merge_kernel<1>);
            else if (d.kv_rank <= 128) merge(latent_attn_merge_kernel<2>);
            else merge(latent_attn_merge_kernel<4>);
            I64H_CHECK_LAUNCH();
        }
        return 0;
    }
    if (latent_rows_f32_ok(d)) return latent_rows_f32_run(d, stream);
    const size_t lds = (size_t)(4 * D + 512) * 4;
    I64H_CHECK_ARG(lds <= 64 * 1024, "latent_attn: cached rows of %d values do not fit", D);
    hipLaunchKernelGGL(latent_attn_row_kernel, dim3((unsigned)d.n, (unsigned)((d.heads + 3) / 4)), dim3(256), lds, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
