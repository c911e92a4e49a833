// The recurrences of i64h_gdn_scan (delta rule) and i64h_gla_scan (keys of their own), runs of rows in tiles of 16 tokens on the 32-bit matrix
// instruction (include/i64h_dense.h).  With P_t the product of a tile's decays up to token t (per key channel), S the state in front of the tile:
//   scan_pairs_kernel : per tile and head k P, q P and k P_16 / P as the operands' registers hold them, and what tokens of a tile are to each other: A_ts = sum_c k_t k_s P_t / P_s (s < t) and B_ts with q_t in
//                       k_t's place (s <= t), the quotients as running products of the decays between (nothing is divided: decays may underflow);
//                       delta rule: T = (1 + diag(beta) A)^-1 diag(beta) by forward substitution
//                       (RAW: from the projections, with what else stands between them and the recurrence)
//   scan_tile_kernel  : U = T (V - (k P)^T S)  (linear attention: U = V);   O = (q P)^T S + B U;   S <- P_16 S + (k P_16 / P)^T U
// Every product's result already lies in the registers as the next product's operand (which of a product's terms an instruction sums is free), so
// a tile is a chain of matrix instructions; four waves share the key channels and meet once a tile, in LDS.
// All arithmetic fp32.  A row that holds no finite number reaches no token before it, as in the scans token by token.
#include <type_traits>

#include "i64h_dense_dev.h"
#include "i64h_scan_dev.h"

typedef float stf4 __attribute__((ext_vector_type(4)));
enum { ST_TOK = 16, ST_PAIR = ST_TOK * ST_TOK };

// tile `i` of run `seg` keeps its pairs at slot (r0 >> 4) + seg + i: slots of different runs never meet, and there are at most n / 16 + nseg
__device__ __forceinline__ int64_t st_slot(int64_t r0, int seg) { return (r0 >> 4) + seg; }

// what one tile of a head leaves for the scan, in floats: three operands, P_16, B and (delta rule) T
__host__ __device__ constexpr int st_floats(int NP) { return 3 * ST_TOK * NP + NP + 2 * ST_PAIR; }

// What stands in front of the pairs, for a tile of one head that is read from the projections as they are (i64h_rec_step's operands; RAW): the convolutions of q, k and v, unit
// vectors, write strengths, and the decays' low-rank map on the bf16 matrix instruction, into sQ, sK, sF, sBeta; v goes to the values' columns of X.  (Every 16 rows of a convolution read three
// more; carried inputs are read only here, and stored by a launch behind.)
template <int NP, bool DELTA>
__device__ __forceinline__ void st_raw(const i64h_gdn_args& p, const i64h_rec_step_args& r, int a, int64_t r0, int64_t r1, int64_t t0, float (*sQ)[NP + 4], float (*sK)[NP + 4], float (*sF)[NP + 4],
                                       float* sBeta) {
    static_assert(NP <= 128, "a thread per channel of q and k, two per channel of v");
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, N = p.dim, V = p.vdim, H = p.heads;
    const int cnt = (int)min((int64_t)ST_TOK, r1 - t0);
    const float* rows = r.P + t0 * r.ldp;
    // the convolutions' inputs are asked for first: COUNT tokens of a channel from token `from` of the tile on, behind the three before them (before the run: carried)
    constexpr int HALF = ST_TOK / 2;
    float in[DELTA ? ST_TOK + 3 : 1], inv[DELTA ? HALF + 3 : 1], wt[4], wv[4];
    const int part = tid / NP, qc = tid % NP, ch = (part * H + a) * N + qc, vc = tid % V, vfrom = tid / V * HALF, vch = 2 * H * N + a * V + vc, T = DELTA ? r.taps : 0;
    const bool qk = part < 2 && qc < N, val = tid < 2 * V;
    if constexpr (DELTA) {
        // (no branch at a load: a run's first tile repeats its first row, then takes what is carried; rows past the end repeat the last one and nobody uses them)
        const int C = H * (2 * N + V), pos = p.positions[t0], before = t0 == r0 ? 0 : 3;
        const float* st = r.conv + (int64_t)p.slot_ids[r0] * (T - 1) * C;
        auto load = [&](int c, int from, auto count, float* x, float* wx) {
            const float* in0 = rows + r.q_off + c;
#pragma unroll
            for (int j = 0; j < decltype(count)::value + 3; ++j) x[j] = in0[(int64_t)min(max(from + j - 3, -before), cnt - 1) * r.ldp];
#pragma unroll
            for (int d = 0; d < 4; ++d) wx[d] = d < T ? r.conv_w[(int64_t)c * T + T - 1 - d] : 0.0f;
            if (before == 0 && from == 0) {
#pragma unroll
                for (int j = 0; j < 3; ++j) x[j] = 3 - j < T && pos + j >= 3 ? st[(int64_t)(T + j - 4) * C + c] : 0.0f;
            }
        };
        if (qk) load(ch, 0, std::integral_constant<int, ST_TOK>(), in, wt);
        if (val) load(vch, vfrom, std::integral_constant<int, HALF>(), inv, wv);
    }
    // decays: a wave takes every fourth block of 16 channels; lane (c, g): token c, channels 4 g .. of a block
    {
        const int c = lane & 15, g = lane >> 4;
        const float* arow = rows + min(c, cnt - 1) * r.ldp + r.a_off;
        const uint16_t* map = (const uint16_t*)r.A + (int64_t)a * N * r.a_rank;
        dn_v4f acc[NP / 64];
#pragma unroll
        for (int b = 0; b < NP / 64; ++b) acc[b] = dn_v4f{0, 0, 0, 0};
#pragma unroll 4
        for (int k0 = 0; k0 < r.a_rank; k0 += 32) {
            // (no branch at a load: past the rank both factors are zeros - an infinite weight times a zero would be no number -, past the last channel nobody uses the sum; four steps' loads
            // asked for together take 139 registers for 79 and longer, 70 us for 58)
            const int k = min(k0 + 8 * g, r.a_rank - 8);
            const bool past = k != k0 + 8 * g;
            const dn_v4f u = *(const dn_v4f*)(arow + k), v = *(const dn_v4f*)(arow + k + 4);
            dn_v4u x{dn_bf16_pair(u[0], u[1]), dn_bf16_pair(u[2], u[3]), dn_bf16_pair(v[0], v[1]), dn_bf16_pair(v[2], v[3])};
            if (past) x = dn_v4u{0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < NP / 64; ++b) {
                dn_v4u m = *(const dn_v4u*)(map + (int64_t)min(16 * (w + 4 * b) + c, N - 1) * r.a_rank + k);
                if (past) m = dn_v4u{0, 0, 0, 0};
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, m), __builtin_bit_cast(dn_v8bf, x), acc[b], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < NP / 64; ++b) {
            const int c0 = 16 * (w + 4 * b) + 4 * g;
            stf4 f = (stf4)1.0f;
            if (c0 < N && c < cnt) {
                const stf4 rate = *(const stf4*)(r.a_rate + a * N + c0), bias = *(const stf4*)(r.a_bias + a * N + c0);
#pragma unroll
                for (int i = 0; i < 4; ++i) f[i] = expf(-rate[i] * dn_softplus(acc[b][i] + bias[i]));
            }
            *(stf4*)&sF[c][c0] = f;
        }
    }
    if constexpr (!DELTA) {
        for (int e = tid; e < ST_TOK * NP / 4; e += 256) {
            const int i = e / (NP / 4), c = e % (NP / 4) * 4;
            const bool ok = i < cnt && c < N;
            const float* row = rows + i * r.ldp + a * N + c;
            *(stf4*)&sK[i][c] = ok ? *(const stf4*)(row + r.k_off) : (stf4)0.0f;
            *(stf4*)&sQ[i][c] = ok ? *(const stf4*)(row + r.q_off) : (stf4)0.0f;
        }
    } else {
        auto silu = [&](const float* x, const float* wx, int j) {      // token j of what was loaded
            float o = 0.0f;
#pragma unroll
            for (int d = 3; d > 0; --d) o = d < T ? o + wx[d] * x[j + 3 - d] : o;
            o += wx[0] * x[j + 3];
            return dn_gated(o, o);
        };
        if (part < 2) {
            float (*dst)[NP + 4] = part ? sK : sQ;
#pragma unroll
            for (int i = 0; i < ST_TOK; ++i) {
                const float o = silu(in, wt, i);
                dst[i][qc] = qk && i < cnt ? o : 0.0f;
            }
        }
        if (val) {
            float* out = p.X + (t0 + vfrom) * p.ldx + p.v_off + a * V + vc;
#pragma unroll
            for (int i = 0; i < HALF; ++i) {
                const float o = silu(inv, wv, i);
                if (vfrom + i < cnt) out[i * p.ldx] = o;
            }
        }
        if (tid < ST_TOK) sBeta[tid] = tid < cnt ? dn_sigmoid(rows[tid * r.ldp + r.b_off + a]) : 0.0f;
        __syncthreads();
        const int s = tid >> 4, l = tid & 15;      // 16 lanes a token
        auto unit = [&](float (*x)[NP + 4], float scale) {
            stf4 v[NP / 64];
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < NP / 64; ++i) {
                v[i] = *(const stf4*)&x[s][64 * i + 4 * l];
                ss += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
            }
            const float f = 1.0f / sqrtf(group_sum(ss, 16) + r.unit_eps) * scale;
#pragma unroll
            for (int i = 0; i < NP / 64; ++i) *(stf4*)&x[s][64 * i + 4 * l] = v[i] * f;
        };
        unit(sQ, r.q_scale);
        unit(sK, 1.0f);
    }
}

// One workgroup per (slot, head), 154 MB through memory for 3008 rows and 16 heads of 128 (38 us): 16 lanes walk from a token s to the tile's end, k_s times the decays so far in their registers; then a thread per
// channel takes the products from the tile's start and from its end.  RAW: from the projections (st_raw), 58 us where convolution, gates,
// the decays' Linear and this took 41 + 16 + 21 + 40 (linear attention 34 for 20 + 27): nothing but the values and the operands is written and read again.
template <int NP, bool DELTA, bool RAW>
__global__ __launch_bounds__(256) void scan_pairs_kernel(const i64h_gdn_args p, const i64h_rec_step_args raw) {
    constexpr int KPT = NP / 16, LD = NP + 4;
    __shared__ __attribute__((aligned(16))) float sF[ST_TOK][LD], sK[ST_TOK][LD], sQ[ST_TOK][LD];
    __shared__ float sA[ST_TOK][ST_TOK + 1], sB[ST_TOK][ST_TOK + 1], sBeta[ST_TOK];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int a = blockIdx.x % p.heads, slot = blockIdx.x / p.heads, N = p.dim;
    int seg = -1;
    for (int b = 0; b < p.nseg; b += 64) {      // the last run that starts at or before this slot (run starts grow)
        const int s = b + lane;
        const int c = __popcll(__ballot(s < p.nseg && st_slot(p.seg_start[min(s, p.nseg - 1)], s) <= slot));
        seg += c;
        if (c < 64) break;
    }
    if (seg < 0) return;
    const int64_t r0 = p.seg_start[seg], r1 = p.seg_start[seg + 1];
    const int64_t t0 = r0 + ST_TOK * (slot - st_slot(r0, seg));
    if (t0 >= r1) return;      // (the whole workgroup)
    if constexpr (RAW) st_raw<NP, DELTA>(p, raw, a, r0, r1, t0, sQ, sK, sF, sBeta);
    else {
        const int kh = a / (p.heads / p.kv_heads);
#pragma unroll
        for (int e = tid; e < ST_TOK * NP / 4; e += 256) {      // (tokens behind the run's end neither decay, write nor read; nor do channels behind the last)
            const int i = e / (NP / 4), c = e % (NP / 4) * 4;
            const int64_t t = t0 + i;
            const bool ok = t < r1 && c < N;
            const stf4 zero = (stf4)0.0f;
            const float* row = p.X + t * p.ldx + kh * N + c;
            *(stf4*)&sK[i][c] = ok ? *(const stf4*)(row + p.k_off) : zero;
            *(stf4*)&sQ[i][c] = ok ? *(const stf4*)(row + p.q_off) : zero;
            if (p.F) *(stf4*)&sF[i][c] = ok ? *(const stf4*)(p.F + t * p.ldf + a * N + c) : (stf4)1.0f;
            else *(stf4*)&sF[i][c] = (stf4)(t < r1 ? p.G[t * 2 * p.heads + p.heads + a] : 1.0f);
        }
        if (DELTA && tid < ST_TOK) sBeta[tid] = t0 + tid < r1 ? p.G[(t0 + tid) * 2 * p.heads + a] : 0.0f;
    }
    __syncthreads();
    {
        const int s = tid >> 4, l = tid & 15;
        stf4 wk[KPT / 4];
#pragma unroll
        for (int i = 0; i < KPT / 4; ++i) wk[i] = *(const stf4*)&sK[s][4 * l + 64 * i];
        auto walk = [&](int t, bool on) {
            float x0 = 0.0f, x1 = 0.0f, y0 = 0.0f, y1 = 0.0f;
#pragma unroll
            for (int i = 0; i < KPT / 4; ++i) {
                const stf4 f = *(const stf4*)&sF[t][4 * l + 64 * i], q = *(const stf4*)&sQ[t][4 * l + 64 * i];
                wk[i] = on ? wk[i] * f : wk[i];
                y0 = fmaf(wk[i][0], q[0], y0), y1 = fmaf(wk[i][1], q[1], y1), y0 = fmaf(wk[i][2], q[2], y0), y1 = fmaf(wk[i][3], q[3], y1);
                if (DELTA) {
                    const stf4 k = *(const stf4*)&sK[t][4 * l + 64 * i];
                    x0 = fmaf(wk[i][0], k[0], x0), x1 = fmaf(wk[i][1], k[1], x1), x0 = fmaf(wk[i][2], k[2], x0), x1 = fmaf(wk[i][3], k[3], x1);
                }
            }
            const float y = group_sum(y0 + y1, 16), x = DELTA ? group_sum(x0 + x1, 16) : 0.0f;
            if (l == 0) {
                sB[t][s] = y;
                if (DELTA) sA[t][s] = x;
            }
        };
        for (int t = 4 * w; t < 4 * w + 4; ++t) walk(t, t > s);      // (a wave holds the tokens 4 w .. 4 w + 3)
        for (int t = 4 * w + 4; t < ST_TOK; ++t) walk(t, true);
    }
    __syncthreads();
    float* out = p.work + ((int64_t)slot * p.heads + a) * st_floats(NP);
    // a channel's products: from the tile's start (first NP threads), to its end (next NP)
    float x[(2 * NP + 255) / 256][2 * ST_TOK];
#pragma unroll
    for (int u = 0; u < (2 * NP + 255) / 256; ++u) {
        const int e = tid + 256 * u, c = e % NP;
        if (e < NP) {
            float P = 1.0f;
#pragma unroll
            for (int t = 0; t < ST_TOK; ++t) {
                P *= sF[t][c];
                x[u][t] = sQ[t][c] * P;
                if (DELTA) x[u][ST_TOK + t] = sK[t][c] * P;
            }
            out[3 * ST_TOK * NP + c] = P;
        } else if (e < 2 * NP) {
            float E = 1.0f;
#pragma unroll
            for (int t = ST_TOK - 1; t >= 0; --t) {
                x[u][t] = sK[t][c] * E;
                E *= sF[t][c];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < (2 * NP + 255) / 256; ++u) {
        const int e = tid + 256 * u, c = e % NP;
#pragma unroll
        for (int t = 0; t < ST_TOK; ++t) {
            if (e < NP) {
                sQ[t][c] = x[u][t];
                if (DELTA) sK[t][c] = x[u][ST_TOK + t];
            } else if (e < 2 * NP) sF[t][c] = x[u][t];
        }
    }
    out += 3 * ST_TOK * NP + NP;
    out[tid] = (tid & 15) <= (tid >> 4) ? sB[tid >> 4][tid & 15] : 0.0f;
    if (DELTA && tid < ST_TOK) {
        const int j = tid;      // a column of T
        float col[ST_TOK];
#pragma unroll
        for (int t = 0; t < ST_TOK; ++t) {
            float s0 = t == j ? 1.0f : 0.0f;
#pragma unroll
            for (int s = 0; s < t; ++s) s0 = s >= j ? fmaf(-sA[t][s], col[s], s0) : s0;
            col[t] = t >= j ? sBeta[t] * s0 : 0.0f;
            out[ST_PAIR + t * ST_TOK + j] = col[t];
        }
    }
    __syncthreads();
    out -= 3 * ST_TOK * NP + NP;
#pragma unroll
    for (int e = tid; e < ST_TOK * NP / 4; e += 256) {      // lane (g, c) of block b: token c, channels 4 g ..; tokens 4 g .., channel c
        const int b = e >> 6, g = (e >> 4) & 3, c = e & 15;
        *(stf4*)(out + 4 * e) = *(const stf4*)&sQ[c][16 * b + 4 * g];
        *(stf4*)(out + ST_TOK * NP + 4 * e) = stf4{sF[4 * g][16 * b + c], sF[4 * g + 1][16 * b + c], sF[4 * g + 2][16 * b + c], sF[4 * g + 3][16 * b + c]};
        if (DELTA) *(stf4*)(out + 2 * ST_TOK * NP + 4 * e) = *(const stf4*)&sK[c][16 * b + 4 * g];
    }
}

// a descriptor of `bytes` from `base` on (the same in every lane, which the compiler doesn't see where they run along with a loop)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t st_buffer(const float* base, uint32_t bytes) {
    const uint64_t b = (uint64_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0, (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// One workgroup per (16 value columns, head, run); wave w holds the key channels [16 BPW w, + 16 BPW) of the state, lane (g, c) of column c the
// channels 4 g .. 4 g + 3 of every block of 16.  Operands come two tiles ahead, straight into registers.
// What bounds a long run is a tile's chain - 8 matrix instructions, LDS and a barrier, 4, 8 more - and what one wave a SIMD has to issue beside it: 0.88 us of 16
// tokens of 128 channels (token by token 2.5), of which the 29 matrix instructions are 930 cycles of 2000 and the loads' addresses 350.  Loads through descriptors
// (no 64-bit address a lane, no branch for rows behind the end) and in four groups that stand between the products, the read-out's products around the exchange,
// its sums and stores behind the next tile's barrier; before that 1.13 us.  Tiles that load nothing more (a run's last ones) are code of their own, and a run of one or two
// tiles asks for no more than it has: three sets of operands then take 168 registers where they took 254.  us, before and after: 1531 rows, 16 heads 107 -> 84, five ragged runs
// 110 -> 89, 8 of 512 over 8 heads 56 -> 49, 32 of 2048 949 -> 759, 64 of 256 over 16 heads 532 -> 438, 27 single rows beside 229 and 256 52 -> 31, 64 channels 76 -> 57; linear
// attention 68 -> 55, 84 -> 59, 38 -> 34, 572 -> 530, 294 -> 289, 45 -> 21, 52 -> 37.  All of a tile's loads in front of its products: 101 for the first; reloading an operand's registers
// behind its last product instead of a third set: 85, linear attention 71.  Reading q, k and decays here and taking the products in every workgroup was 2.0 us a tile.
// The workgroups of a head are a multiple of eight apart where there are eight heads: one die's L2 then serves them all.
template <int BPW, bool DELTA>
__global__ __launch_bounds__(256, BPW > 2 ? (DELTA ? 1 : 2) : 3) void scan_tile_kernel(const i64h_gdn_args p) {
    constexpr int NP = 64 * BPW, FL = st_floats(NP), SETS = 3;
    __shared__ stf4 sX[2][DELTA ? 4 : 1][64], sY[2][4][64];
    const int N = p.dim, P = p.vdim;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int a = blockIdx.x % p.heads, seg = gd_run(p.seg_start, p.nseg, blockIdx.y);
    const int col = blockIdx.x / p.heads * 16 + c;
    const bool cok = col < P;
    const int64_t r0 = p.seg_start[seg], r1 = p.seg_start[seg + 1];
    if (r1 <= r0) return;      // (the whole workgroup)
    const int ch0 = 16 * BPW * w + 4 * g;
    float* gS = p.state + (((int64_t)p.slot_ids[r0] * p.heads + a) * P + (cok ? col : 0)) * N;
    const bool fresh = p.positions[r0] == 0;
    stf4 S[BPW];
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
        S[b] = (stf4)0.0f;
        if (!fresh && cok && ch0 + 16 * b < N) S[b] = *(const stf4*)(gS + ch0 + 16 * b);
    }
    const int nt = (int)((r1 - r0 + ST_TOK - 1) / ST_TOK);
    const float* tiles = p.work + (st_slot(r0, seg) * p.heads + a) * FL;
    const int64_t tstep = (int64_t)p.heads * FL, vstep = ST_TOK * p.ldx;
    const int rows_last = (int)(r1 - r0) - ST_TOK * (nt - 1);      // of the last tile
    const float* values = p.X + r0 * p.ldx + p.v_off + a * P;
    // what a lane reads lies at the same offsets of every tile (16 rows span less than 4 GiB: the launch's check); value rows behind the run's end read as zeros
    const uint32_t ldx4 = 4 * (uint32_t)p.ldx, at = 4 * (256 * BPW * w + 4 * lane), at_B = 4 * (c * ST_TOK + 4 * g + w), at_T = 4 * (c * ST_TOK + 4 * g);
    uint32_t at_v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) at_v[r] = (4 * g + r) * ldx4 + (cok ? 4 * col : 0);
    auto at4 = [](const __amdgpu_buffer_rsrc_t& m, uint32_t lane_at, uint32_t step) { return __builtin_bit_cast(stf4, __builtin_amdgcn_raw_buffer_load_b128(m, lane_at, step, 0)); };
    auto at1 = [](const __amdgpu_buffer_rsrc_t& m, uint32_t lane_at, uint32_t step) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(m, lane_at, step, 0)); };
    struct Ops {      // k P and q P (lane: token c, channels 4 g ..), k P_16 / P (tokens 4 g .., channel c), P_16 (channels 4 g ..), values (tokens 4 g ..)
        stf4 qp[BPW], kd[BPW], kp[DELTA ? BPW : 1], tot[BPW], T;
        float v[4], B;
    };
    struct Tile {
        __amdgpu_buffer_rsrc_t m, v;
    };
    auto where = [&](int i) {
        i = min(i, nt - 1);      // (past the end: the last tile once more, nobody reads it)
        return Tile{st_buffer(tiles + i * tstep, 4 * FL), st_buffer(values + i * vstep, (i < nt - 1 ? ST_TOK - 1 : rows_last - 1) * ldx4 + 4 * (uint32_t)P)};
    };
    // a tile's loads in four parts, which stand apart: a wave's sixteen bytes a lane keep the unit that takes them, one for four waves, busy for 16 cycles
    auto load = [&](const Tile& t, Ops& u, int part) {
        __builtin_amdgcn_sched_barrier(0);
        if (part == 0) {
#pragma unroll
            for (int b = 0; b < BPW; ++b)
                if (DELTA) u.kp[b] = at4(t.m, at, 4 * (2 * ST_TOK * NP + 256 * b));
        } else if (part == 1) {
#pragma unroll
            for (int b = 0; b < BPW; ++b) u.qp[b] = at4(t.m, at, 4 * 256 * b);
        } else if (part == 2) {
#pragma unroll
            for (int b = 0; b < BPW; ++b) u.tot[b] = at4(t.m, 4 * ch0, 4 * (3 * ST_TOK * NP + 16 * b));
#pragma unroll
            for (int r = 0; r < 4; ++r) u.v[r] = at1(t.v, at_v[r], 0);
            if (DELTA) u.T = at4(t.m, at_T, 4 * (3 * ST_TOK * NP + NP + ST_PAIR));
        } else {
#pragma unroll
            for (int b = 0; b < BPW; ++b) u.kd[b] = at4(t.m, at, 4 * (ST_TOK * NP + 256 * b));
            u.B = at1(t.m, at_B, 4 * (3 * ST_TOK * NP + NP));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // a tile's read-out, once every wave's share lies in LDS: wave w stores the tokens 4 g + w
    float* o_next = p.out + (r0 + 4 * g + w) * p.ldo + a * P + col;
    const int64_t ostep = ST_TOK * p.ldo;
    auto store = [&](const float y[4], int rows) {
        const float o = (y[0] + y[1]) + (y[2] + y[3]);
        if (cok && 4 * g + w < rows) *o_next = DELTA ? o : o * p.q_scale;
        o_next += ostep;
    };
    // M v over the tokens up to and with a row's own, term by term: the terms from `first` on, every `stride`th
    auto below = [&](const float* M, const stf4& v, int first, int stride, stf4 o) {
        const __amdgpu_buffer_rsrc_t m = st_buffer(M, 4 * ST_PAIR);
        int g4 = 4 * g;
        asm volatile("" : "+v"(g4));      // (its addresses are not kept in registers through all tiles)
#pragma unroll 1
        for (int s = first; s < ST_TOK; s += stride) {
            const float lo = (s & 1) ? v[1] : v[0], hi = (s & 1) ? v[3] : v[2];
            const float vs = __shfl((s & 2) ? hi : lo, 16 * (s >> 2) + c);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (s <= g4 + r) o[r] = fmaf(at1(m, 4 * ((g4 + r) * ST_TOK + s), 0), vs, o[r]);
        }
        return o;
    };
    // What a tile waits for is its chain, so whatever else there is stands where the chain waits: the read-out's products around the exchange of the shares of
    // k P S, the sums and stores of the tile before behind the barrier that this exchange needs, the state times P_16 in front of its last products.
    stf4 O = (stf4)0.0f;      // a wave's share of the read-out of the tile before
    auto tile = [&](int i, const Ops& o, Ops& ahead, auto more) {      // more: a tile's operands are loaded meanwhile
        const int pb = i & 1;
        constexpr bool LOAD = decltype(more)::value;
        const Tile next = LOAD ? where(i + SETS - 1) : Tile{};
        if constexpr (DELTA) {
            stf4 x[2] = {(stf4)0.0f, (stf4)0.0f};
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int b = 0; b < BPW; ++b) x[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kp[b][r], S[b][r], x[b & 1], 0, 0, 0);
            sY[pb][w][lane] = O;
            if constexpr (LOAD) load(next, ahead, 0);
            sX[pb][w][lane] = BPW > 1 ? x[0] + x[1] : x[0];
        } else sY[pb][w][lane] = O;
        stf4 y[2] = {(stf4)0.0f, (stf4)0.0f};
        auto read_out = [&](int r0, int r1) {
#pragma unroll
            for (int r = r0; r < r1; ++r)
#pragma unroll
                for (int b = 0; b < BPW; ++b) y[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.qp[b][r], S[b][r], y[b & 1], 0, 0, 0);
        };
        read_out(0, 1);
        // one barrier a tile: LDS holds two tiles' shares, and the one that is written again was read in front of it
        __syncthreads();
        stf4 xs[4];
        float ys[4];
        if constexpr (DELTA) {
#pragma unroll
            for (int j = 0; j < 4; ++j) xs[j] = sX[pb][j][lane];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) ys[j] = ((const float*)&sY[pb][j][lane])[w];
        if constexpr (LOAD) load(next, ahead, 1);
        read_out(1, 4);
        if constexpr (LOAD) load(next, ahead, 2);
#pragma unroll
        for (int b = 0; b < BPW; ++b) S[b] = S[b] * o.tot[b];
        stf4 W, U;      // (rows behind the run's end: no value, no key, no write strength)
#pragma unroll
        for (int r = 0; r < 4; ++r) W[r] = o.v[r];
        if constexpr (DELTA) W = W - ((xs[0] + xs[1]) + (xs[2] + xs[3]));
        // a sum over all 16 tokens would carry what is no finite number to tokens in front of it, through a zero: such a tile is summed term by term
        auto odd = [](const stf4& x) { return __ballot(!((fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3])) < INFINITY)) != 0; };
        const float* pr = tiles + i * tstep + 3 * ST_TOK * NP + NP;
        U = W;
        if constexpr (DELTA) {
            stf4 u0 = (stf4)0.0f, u1 = (stf4)0.0f;
            u0 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.T[0], W[0], u0, 0, 0, 0);
            u1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.T[2], W[2], u1, 0, 0, 0);
            u0 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.T[1], W[1], u0, 0, 0, 0);
            u1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.T[3], W[3], u1, 0, 0, 0);
            if (odd(W)) u0 = below(pr + ST_PAIR, W, 0, 1, (stf4)0.0f), u1 = (stf4)0.0f;
            U = u0 + u1;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int b = 0; b < BPW; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kd[b][r], U[r], S[b], 0, 0, 0);
        if constexpr (LOAD) load(next, ahead, 3);
        if (i > 0) store(ys, ST_TOK);
        // a wave's share of the read-out: its channels of the state, and every fourth token's write
        O = BPW > 1 ? y[0] + y[1] : y[0];
        if (odd(U)) O = below(pr, U, w, 4, O);
        else O = __builtin_amdgcn_mfma_f32_16x16x4f32(o.B, w == 0 ? U[0] : (w == 1 ? U[1] : (w == 2 ? U[2] : U[3])), O, 0, 0, 0);
    };
    Ops u[SETS];
    auto whole = [&](int i, Ops& o) {
        const Tile t = where(i);
#pragma unroll
        for (int part = 0; part < 4; ++part) load(t, o, part);
    };
    constexpr std::false_type none{};
    if (nt < SETS) {      // (a run of a tile or two loads no more than it has: beside a prompt most of a step's runs are single rows)
        whole(0, u[0]);
        if (nt > 1) whole(1, u[1]);
        tile(0, u[0], u[0], none);
        if (nt > 1) tile(1, u[1], u[1], none);
    } else {
#pragma unroll
        for (int j = 0; j < SETS - 1; ++j) {      // (the sets' loads stay apart: waiting for one must not wait for the next)
            whole(j, u[j]);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        int i = 0;
        for (; i + SETS <= nt; i += SETS) {      // (not left in the middle: round the loop every set is as many loads behind the next)
#pragma unroll
            for (int j = 0; j < SETS; ++j) tile(i + j, u[j], u[(j + SETS - 1) % SETS], std::true_type{});
        }
#pragma unroll
        for (int j = 0; j < SETS - 1; ++j)
            if (i + j < nt) tile(i + j, u[j], u[j], none);
    }
    sY[nt & 1][w][lane] = O;
    __syncthreads();
    float ys[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) ys[j] = ((const float*)&sY[nt & 1][j][lane])[w];
    store(ys, rows_last);
#pragma unroll
    for (int b = 0; b < BPW; ++b)
        if (cok && ch0 + 16 * b < N) *(stf4*)(gS + ch0 + 16 * b) = S[b];
}

static int st_padded(int dim) { return dim <= 64 ? 64 : (dim <= 128 ? 128 : 256); }

extern "C" int64_t i64h_scan_work_floats(int64_t n, int32_t nseg, int32_t heads, int32_t dim) {
    return (n / ST_TOK + nseg) * heads * st_floats(st_padded(dim));
}

template <bool RAW>
static int st_run(const i64h_gdn_args& d, const i64h_rec_step_args& raw, bool delta, void* stream) {
    const dim3 pairs((unsigned)((d.n / ST_TOK + d.nseg) * d.heads)), tiles((unsigned)(d.heads * ((d.vdim + 15) / 16)), (unsigned)d.nseg);
    auto run = [&](auto a, auto b) {
        hipLaunchKernelGGL(a, pairs, dim3(256), 0, (hipStream_t)stream, d, raw);
        hipLaunchKernelGGL(b, tiles, dim3(256), 0, (hipStream_t)stream, d);
    };
    auto pick = [&](auto bpw) {
        constexpr int B = decltype(bpw)::value;
        if (delta) run(scan_pairs_kernel<64 * B, true, RAW>, scan_tile_kernel<B, true>);
        else run(scan_pairs_kernel<64 * B, false, RAW>, scan_tile_kernel<B, false>);
    };
    if (d.dim <= 64) pick(std::integral_constant<int, 1>());
    else if (d.dim <= 128) pick(std::integral_constant<int, 2>());
    else if constexpr (!RAW) pick(std::integral_constant<int, 4>());
    I64H_CHECK_LAUNCH();
    return 0;
}

// both launches; the caller (the scans' own dispatch) has checked sizes, alignment and the workspace
int i64h_scan_tiles(const i64h_gdn_args& d, bool delta, void* stream) { return st_run<false>(d, {}, delta, stream); }
// the same from the projections (the caller, i64h_rec_tiles, has checked)
int i64h_scan_tiles_raw(const i64h_gdn_args& d, const i64h_rec_step_args& raw, bool delta, void* stream) { return st_run<true>(d, raw, delta, stream); }
