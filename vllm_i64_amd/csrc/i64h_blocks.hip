// Kernels of libi64hip_dense.so for gated linear recurrences and mixtures of experts (include/i64h_dense.h):
//   gla_gates_kernel   : query activation and bounded forget gate, in place on the projection rows
//   gdn_gates_kernel / gdn_scan_kernel : gated delta rule - unit-vector queries and keys, write strength and decay; the recurrence with the
//                        correction S^T k summed over the DPP row before the write, the read-out after it; a decay per head or per key channel;
//                        without the correction: gated linear attention, with keys of its own or one minus the decay as the key
//   gdn_tile_kernel    : the same recurrence for long runs, tokens staged through LDS
//   route_topk_kernel  : softmax scores (over all entries or the chosen ones) or sigmoid scores, corrected choice, groups of
//                        neighbours, top-k and normalised (or raw) weights, one wave per row (few rows: a workgroup per row)
//   moe_plan_kernel    : (token, choice) pairs grouped by expert: offsets, the token of every grouped row, the row of every pair
//   moe_combine_kernel : weighted sum of the chosen experts' rows, pass-through entries and the shared expert's row
// A row continues the row before it iff slot and position say so; state is taken as empty at position 0.  All arithmetic fp32.
#include "i64h_common.h"
#include "i64h_dense.h"
#include "i64h_route_dev.h"
#include "i64h_scan_dev.h"

int i64h_scan_tiles(const i64h_gdn_args& d, bool delta, void* stream);      // i64h_scan_tile.hip

__device__ __forceinline__ float bl_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gla_gates_kernel(const i64h_gla_args p) {
    const int64_t t = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= p.heads * p.dim) return;
    float* row = p.P + t * p.ldp;
    if (p.q_act) {
        const float q = row[p.q_off + c];
        row[p.q_off + c] = q * bl_sigmoid(q);
    }
    const float lo = p.lower ? p.lower[c] : 0.0f;
    row[p.f_off + c] = lo + (1.0f - lo) * bl_sigmoid(row[p.f_off + c]);
}

// ---------------------------------------------------------------------------------------------------------------------------
// Gated delta rule.  gdn_gates_kernel: one workgroup per token - the heads of query and key become unit vectors in place (the query also
// scaled), and threads turn the raw gate projections into the write strength and the decay of every head.
// VEC (16-byte rows): 16 lanes take a head, the loads of GT_ROUNDS rounds of 16 heads on their way together; else a wave takes a head, one
// after the other.  What bounds it is the way to memory and back of a row's heads: 3008 rows of 2 x 16 heads of 128, 28 | 16 us beside nothing else.
__device__ __forceinline__ float bl_softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

#define GT_ROUNDS 2
template <int VEC>      // stripes of 64 channels a head has; 0: any row
__global__ __launch_bounds__(256) void gdn_gates_kernel(const i64h_gdn_args p) {
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    float* row = p.X + t * p.ldx;
    if (VEC && (p.unit_eps >= 0.0f || p.q_scale != 1.0f)) {
        const int l = threadIdx.x & 15;
        for (int u0 = threadIdx.x >> 4; u0 < 2 * p.kv_heads; u0 += 16 * GT_ROUNDS) {
            float4 v[GT_ROUNDS][VEC ? VEC : 1];
            auto head = [&](int u) { return row + (u < p.kv_heads ? p.q_off + u * p.dim : p.k_off + (u - p.kv_heads) * p.dim); };
#pragma unroll
            for (int r = 0; r < GT_ROUNDS; ++r)
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const int u = u0 + 16 * r, d = 64 * i + 4 * l;
                    v[r][i] = make_float4(0, 0, 0, 0);
                    if (u < 2 * p.kv_heads && d < p.dim) v[r][i] = *(const float4*)(head(u) + d);
                }
#pragma unroll
            for (int r = 0; r < GT_ROUNDS; ++r) {
                const int u = u0 + 16 * r;
                float s = 0.0f;
#pragma unroll
                for (int i = 0; i < VEC; ++i) s += (v[r][i].x * v[r][i].x + v[r][i].y * v[r][i].y) + (v[r][i].z * v[r][i].z + v[r][i].w * v[r][i].w);
                s = group_sum(s, 16);
                float f = p.unit_eps >= 0.0f ? 1.0f / sqrtf(s + p.unit_eps) : 1.0f;
                if (u < p.kv_heads) f *= p.q_scale;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const int d = 64 * i + 4 * l;
                    if (u < 2 * p.kv_heads && d < p.dim) *(float4*)(head(u) + d) = make_float4(v[r][i].x * f, v[r][i].y * f, v[r][i].z * f, v[r][i].w * f);
                }
            }
        }
    } else if (p.unit_eps >= 0.0f || p.q_scale != 1.0f) {
        for (int u = wid; u < 2 * p.kv_heads; u += 4) {
            const bool isq = u < p.kv_heads;
            float* x = row + (isq ? p.q_off + u * p.dim : p.k_off + (u - p.kv_heads) * p.dim);
            float s = 0.0f;
            for (int d = lane; d < p.dim; d += 64) s += x[d] * x[d];
            s = wave_sum(s);
            float f = p.unit_eps >= 0.0f ? 1.0f / sqrtf(s + p.unit_eps) : 1.0f;
            if (isq) f *= p.q_scale;
            for (int d = lane; d < p.dim; d += 64) x[d] *= f;
        }
    }
    for (int a = threadIdx.x; a < p.heads; a += 256) {
        const float* r = p.R + t * p.ldr;
        p.G[t * 2 * p.heads + a] = bl_sigmoid(r[p.b_off + a]);
        if (p.a_off >= 0) p.G[t * 2 * p.heads + p.heads + a] = expf(-expf(p.A_log[a]) * bl_softplus(r[p.a_off + a] + p.dt_bias[a]));
    }
}

// gdn_scan_kernel: one workgroup per (head, 16 * CPT value columns, run of rows); the 16 lanes of a DPP row share CPT value columns and hold
// KPT key channels of each in registers, a wave has four such rows.  Per token the state decays, the row sums S^T k with DPP
// moves (every lane of the row ends with the sum), the correction along k is written, and a second row sum reads the state out with
// the query - after the write.  No LDS and no barrier, the tokens of a run strictly in their order (the same sums in the same order however
// a prompt is cut); loads run TG tokens ahead in two alternating register sets.  State layout [slot, head, value column, key channel].
// CHD: a decay per head and key channel (F) in the place of one per head.  RULE: the delta rule's correction and write strength, or gated
// linear attention: the token writes k v^T as it is, the read-out is multiplied by q_scale; the keys are the row's own or one minus the decay.
// TG is chosen so that two waves fit a SIMD's registers (the loads in flight are most of them); one where every run is a single row.
template <int KPT, int CPT, bool CHD, int TG, int RULE>
__global__ __launch_bounds__(256) void gdn_scan_kernel(const i64h_gdn_args p, const int ctiles, const int vec) {
    const int N = p.dim, P = p.vdim;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nlane = lane & 15, cl = lane >> 4;
    const int a = blockIdx.x / ctiles, seg = blockIdx.y;
    const int kh = a / (p.heads / p.kv_heads);
    const int cbase = (blockIdx.x % ctiles) * 16 * CPT + (w * 4 + cl) * CPT;
    const int64_t r0 = p.seg_start[seg], r1 = p.seg_start[seg + 1];
    if (r1 <= r0) return;
    float S[CPT][KPT];
    float* gS = p.state + ((int64_t)p.slot_ids[r0] * p.heads + a) * P * N;      // + column * N
    const bool fresh = p.positions[r0] == 0;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        const bool cok = cbase + j < P;
        const float* src = gS + (int64_t)(cok ? cbase + j : 0) * N;
#pragma unroll
        for (int k = 0; k < KPT; ++k) S[j][k] = 0.0f;
        if (!fresh && cok) {
            if (vec) {
#pragma unroll
                for (int k = 0; k < KPT; k += 4)
                    if (gd_channel<KPT>(nlane, k) < N) {
                        const float4 v = *(const float4*)(src + gd_channel<KPT>(nlane, k));
                        S[j][k] = v.x, S[j][k + 1] = v.y, S[j][k + 2] = v.z, S[j][k + 3] = v.w;
                    }
            } else {
#pragma unroll
                for (int k = 0; k < KPT; ++k)
                    if (gd_channel<KPT>(nlane, k) < N) S[j][k] = src[gd_channel<KPT>(nlane, k)];
            }
        }
    }
    const int qoff = p.q_off + kh * N, koff = p.k_off + kh * N, foff = a * N;
    struct Tok {
        float q[KPT], k[RULE == GD_FORGET ? 1 : KPT], f[CHD ? KPT : 1], v[CPT], beta;
    };
    auto fetch = [&](int64_t t, Tok& u) {
        if (t >= r1) return;
        const float* row = p.X + t * p.ldx;
        if (vec) {      // KPT % 4 == 0 and every slice starts at a multiple of four floats and lies inside the row
#pragma unroll
            for (int k = 0; k < KPT; k += 4) {
                float4 q = make_float4(0, 0, 0, 0), kk = q, f = RULE == GD_FORGET ? make_float4(1, 1, 1, 1) : q;
                if (gd_channel<KPT>(nlane, k) < N) {
                    q = *(const float4*)(row + qoff + gd_channel<KPT>(nlane, k));
                    if (RULE != GD_FORGET) kk = *(const float4*)(row + koff + gd_channel<KPT>(nlane, k));
                    if (CHD) f = *(const float4*)(p.F + t * p.ldf + foff + gd_channel<KPT>(nlane, k));
                }
                u.q[k] = q.x, u.q[k + 1] = q.y, u.q[k + 2] = q.z, u.q[k + 3] = q.w;
                if (RULE != GD_FORGET) u.k[k] = kk.x, u.k[k + 1] = kk.y, u.k[k + 2] = kk.z, u.k[k + 3] = kk.w;
                if (CHD) u.f[k] = f.x, u.f[k + 1] = f.y, u.f[k + 2] = f.z, u.f[k + 3] = f.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < KPT; ++k) {
                const int c = gd_channel<KPT>(nlane, k);
                const bool ok = c < N;
                u.q[k] = ok ? row[qoff + c] : 0.0f;
                if (RULE != GD_FORGET) u.k[k] = ok ? row[koff + c] : 0.0f;
                if (CHD) u.f[k] = ok ? p.F[t * p.ldf + foff + c] : (RULE == GD_FORGET ? 1.0f : 0.0f);
            }
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) u.v[j] = cbase + j < P ? row[p.v_off + a * P + cbase + j] : 0.0f;
        if (RULE == GD_DELTA) u.beta = p.G[t * 2 * p.heads + a];
        if (!CHD) u.f[0] = p.G[t * 2 * p.heads + p.heads + a];
    };
    auto step = [&](int64_t t, const Tok& u) {
        if (t >= r1) return;
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            float part;
            if constexpr (RULE == GD_DELTA) part = gd_delta<KPT, CHD>(S[j], u.f, u.k, u.q, u.v[j], u.beta);
            else part = gd_linear<KPT, CHD, RULE == GD_FORGET>(S[j], u.f, u.k, u.q, u.v[j]);
            if (nlane == 0 && cbase + j < P) p.out[t * p.ldo + a * P + cbase + j] = RULE == GD_DELTA ? part : part * p.q_scale;
        }
    };
    Tok A[TG], B[TG];
#pragma unroll
    for (int i = 0; i < TG; ++i) fetch(r0 + i, A[i]);
    for (int64_t t = r0; t < r1; t += 2 * TG) {
#pragma unroll
        for (int i = 0; i < TG; ++i) fetch(t + TG + i, B[i]);
#pragma unroll
        for (int i = 0; i < TG; ++i) step(t + i, A[i]);
#pragma unroll
        for (int i = 0; i < TG; ++i) fetch(t + 2 * TG + i, A[i]);
#pragma unroll
        for (int i = 0; i < TG; ++i) step(t + TG + i, B[i]);
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        if (cbase + j >= P) continue;
        float* dst = gS + (int64_t)(cbase + j) * N;
        if (vec) {
#pragma unroll
            for (int k = 0; k < KPT; k += 4)
                if (gd_channel<KPT>(nlane, k) < N) *(float4*)(dst + gd_channel<KPT>(nlane, k)) = make_float4(S[j][k], S[j][k + 1], S[j][k + 2], S[j][k + 3]);
        } else {
#pragma unroll
            for (int k = 0; k < KPT; ++k)
                if (gd_channel<KPT>(nlane, k) < N) dst[gd_channel<KPT>(nlane, k)] = S[j][k];
        }
    }
}

// gdn_tile_kernel: the same recurrence, bit for bit, for runs of many rows.  What every wave of a workgroup reads of a token (query, key,
// decays) is loaded once per workgroup, TT tokens at a time, into one of two LDS tiles while the other one is computed: the loads of a
// tile have the arithmetic of a whole tile to arrive, and the waves read 16 bytes per lane from LDS one token ahead.  Needs 16-byte rows.
// What bounds it is the chain from token to token - decay, row sum, correction - and the reads of the tile: the 16 tokens of a tile are one
// stretch of code without a branch, so that a token's read-out runs beside the next one's sums, its result waiting in a lane until
// the tile's end; 16 heads of 128, one run of 1531 rows: 334 -> 245 us (218 -> 160 ns a token), linear attention, 1500 rows, 278 -> 213 us.
template <int KPT, int CPT, bool CHD, int RULE>
__global__ __launch_bounds__(256) void gdn_tile_kernel(const i64h_gdn_args p, const int ctiles) {
    static_assert(KPT % 4 == 0, "whole 16-byte slices per lane");
    constexpr int TT = KPT > 8 ? 8 : 16;      // tokens per tile
    constexpr int NP = 16 * KPT, PARTS = CHD && RULE != GD_FORGET ? 3 : 2, LPP = TT * NP / 4 / 256, WC = 16 * CPT;     // LPP: 16-byte loads per thread and part
    constexpr int VPT = (TT * WC + 255) / 256;
    __shared__ __attribute__((aligned(16))) float sX[2][PARTS][TT][NP];
    __shared__ float sV[2][TT][WC];
    __shared__ float sG[2][TT][2];      // write strength, decay per head
    const int N = p.dim, P = p.vdim;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int nlane = lane & 15, cl = lane >> 4;
    const int a = blockIdx.x / ctiles, seg = gd_run(p.seg_start, p.nseg, blockIdx.y);
    const int kh = a / (p.heads / p.kv_heads);
    const int wg0 = (blockIdx.x % ctiles) * WC, cw = (w * 4 + cl) * CPT, cbase = wg0 + cw;
    const int64_t r0 = p.seg_start[seg], r1 = p.seg_start[seg + 1];
    if (r1 <= r0) return;      // (the whole workgroup)
    float S[CPT][KPT];
    float* gS = p.state + ((int64_t)p.slot_ids[r0] * p.heads + a) * P * N;
    const bool fresh = p.positions[r0] == 0;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        const bool cok = cbase + j < P;
        const float* src = gS + (int64_t)(cok ? cbase + j : 0) * N;
#pragma unroll
        for (int k = 0; k < KPT; k += 4) {
            const int c = gd_channel<KPT>(nlane, k);
            float4 v = make_float4(0, 0, 0, 0);
            if (!fresh && cok && c < N) v = *(const float4*)(src + c);
            S[j][k] = v.x, S[j][k + 1] = v.y, S[j][k + 2] = v.z, S[j][k + 3] = v.w;
        }
    }
    float4 st[PARTS][LPP];
    float sv[VPT], sg = 0.0f;
    auto gload = [&](int64_t t0) {
#pragma unroll
        for (int u = 0; u < LPP; ++u) {
            const int e = tid + 256 * u, c = (e % (NP / 4)) * 4;
            const int64_t t = t0 + e / (NP / 4);
            const bool ok = t < r1 && c < N;
            const float* row = p.X + t * p.ldx;
            st[0][u] = ok ? *(const float4*)(row + p.q_off + kh * N + c) : make_float4(0, 0, 0, 0);
            if (RULE != GD_FORGET) st[1][u] = ok ? *(const float4*)(row + p.k_off + kh * N + c) : make_float4(0, 0, 0, 0);
            const float pad = RULE == GD_FORGET ? 1.0f : 0.0f;
            if (CHD) st[PARTS - 1][u] = ok ? *(const float4*)(p.F + t * p.ldf + a * N + c) : make_float4(pad, pad, pad, pad);
        }
#pragma unroll
        for (int u = 0; u < VPT; ++u) {
            const int e = tid + 256 * u, c = wg0 + e % WC;
            const int64_t t = t0 + e / WC;
            sv[u] = (t < r1 && c < P) ? p.X[t * p.ldx + p.v_off + a * P + c] : 0.0f;
        }
        if (tid < 2 * TT) {
            const int64_t t = t0 + (tid >> 1);
            sg = (t < r1 && (RULE == GD_DELTA || (tid & 1)) && !(CHD && (tid & 1))) ? p.G[t * 2 * p.heads + (tid & 1) * p.heads + a] : 0.0f;
        }
    };
    auto lstore = [&](int b) {
#pragma unroll
        for (int u = 0; u < LPP; ++u) {
            const int e = tid + 256 * u;
#pragma unroll
            for (int x = 0; x < PARTS; ++x) *(float4*)&sX[b][x][e / (NP / 4)][(e % (NP / 4)) * 4] = st[x][u];
        }
#pragma unroll
        for (int u = 0; u < VPT; ++u)
            if (tid + 256 * u < TT * WC) sV[b][(tid + 256 * u) / WC][(tid + 256 * u) % WC] = sv[u];
        if (tid < 2 * TT) sG[b][tid >> 1][tid & 1] = sg;
    };
    struct Tok {
        float q[KPT], k[RULE == GD_FORGET ? 1 : KPT], f[CHD ? KPT : 1], v[CPT], beta;
    };
    auto fetch = [&](int b, int i, Tok& u) {
#pragma unroll
        for (int k = 0; k < KPT; k += 4) {
            const int c = gd_channel<KPT>(nlane, k);
            const float4 q = *(const float4*)&sX[b][0][i][c];
            u.q[k] = q.x, u.q[k + 1] = q.y, u.q[k + 2] = q.z, u.q[k + 3] = q.w;
            if (RULE != GD_FORGET) {
                const float4 kk = *(const float4*)&sX[b][1][i][c];
                u.k[k] = kk.x, u.k[k + 1] = kk.y, u.k[k + 2] = kk.z, u.k[k + 3] = kk.w;
            }
            if (CHD) {
                const float4 f = *(const float4*)&sX[b][PARTS - 1][i][c];
                u.f[k] = f.x, u.f[k + 1] = f.y, u.f[k + 2] = f.z, u.f[k + 3] = f.w;
            }
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) u.v[j] = sV[b][i][cw + j];
        u.beta = sG[b][i][0];
        if (!CHD) u.f[0] = sG[b][i][1];
    };
    auto step = [&](int j, const Tok& u) {
        if constexpr (RULE == GD_DELTA) return gd_delta<KPT, CHD>(S[j], u.f, u.k, u.q, u.v[j], u.beta);
        else return gd_linear<KPT, CHD, RULE == GD_FORGET>(S[j], u.f, u.k, u.q, u.v[j]) * p.q_scale;
    };
    gload(r0);
    lstore(0);
    __syncthreads();
    int b = 0;
    for (int64_t t0 = r0; t0 < r1; t0 += TT, b ^= 1) {
        const int cnt = (int)min((int64_t)TT, r1 - t0);
        const bool more = t0 + TT < r1;
        if (more) gload(t0 + TT);
        Tok A, B;
        fetch(b, 0, A);
        if (cnt == TT) {
            // a whole tile without a branch: a token's read-out runs beside the next token's decay and sums.  All 16 lanes of a row end with
            // a token's result: lane i keeps that of token i, stored once a tile
            float o[CPT];
#pragma unroll
            for (int j = 0; j < CPT; ++j) o[j] = 0.0f;
#pragma unroll
            for (int i = 0; i < TT; i += 2) {
                fetch(b, i + 1, B);
#pragma unroll
                for (int j = 0; j < CPT; ++j) {
                    const float part = step(j, A);
                    o[j] = nlane == i ? part : o[j];
                }
                if (i + 2 < TT) fetch(b, i + 2, A);
#pragma unroll
                for (int j = 0; j < CPT; ++j) {
                    const float part = step(j, B);
                    o[j] = nlane == i + 1 ? part : o[j];
                }
            }
            if (nlane < TT)
#pragma unroll
                for (int j = 0; j < CPT; ++j)
                    if (cbase + j < P) p.out[(t0 + nlane) * p.ldo + a * P + cbase + j] = o[j];
        } else {
            for (int i = 0; i < cnt; ++i) {
                if (i > 0) fetch(b, i, A);
#pragma unroll
                for (int j = 0; j < CPT; ++j) {
                    const float part = step(j, A);
                    if (nlane == 0 && cbase + j < P) p.out[(t0 + i) * p.ldo + a * P + cbase + j] = part;
                }
            }
        }
        if (more) lstore(b ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        if (cbase + j >= P) continue;
        float* dst = gS + (int64_t)(cbase + j) * N;
#pragma unroll
        for (int k = 0; k < KPT; k += 4) {
            const int c = gd_channel<KPT>(nlane, k);
            if (c < N) *(float4*)(dst + c) = make_float4(S[j][k], S[j][k + 1], S[j][k + 2], S[j][k + 3]);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
// the lane that holds the largest value, ties to the lower index; (value, index) pairs with index < 0 do not take part
__device__ __forceinline__ int bl_wave_argmax(float v, int idx, float& best) {
    best = wave_max(idx >= 0 ? v : -INFINITY);
    const int cand = (idx >= 0 && v == best) ? idx : 0x7fffffff;
    return -wave_max_i(-cand);
}

// SPLIT: a workgroup per row - four waves share the columns of the router's products, four such groups (or one) the entries, eight at a time, the first
// wave goes on with their sums (few rows: one wave's chain of loads is what a launch would wait for).
// One group | four, rows of 2048: 16 entries 64 rows 10.4 | 8.0 us, 256 rows 10.5 | 8.3, 512 rows 10.9 | 12.0; 64 entries 28.4 | 13.8, 28.6 | 14.5,
// 29.1 | 19.0.  Without SPLIT 1024 rows of 16 entries take 25 us and of 64 entries 87, with it 33.
#define RT_WIDE_ROWS 256       // launches of at most so many rows have the four groups; all of more than RT_MANY entries do
#define RT_MANY 32
#define RT_SPLIT_ROWS 512      // launches of at most so many rows are split; twice as many over more than RT_MANY entries
// NINE: the last entry behind a multiple of eight goes with the eight before it (eight experts and a gate's row, 3008 rows of 2048: 20 | 15 us, 64 and a gate
// 53 | 34); a kernel of its own, for its registers cost the launches beside it where there is no such entry (a step of 4096 rows 0.6 %).
template <bool SPLIT, bool NINE>
__global__ __launch_bounds__(SPLIT ? 1024 : 256) void route_topk_kernel(const i64h_route_args p) {
    extern __shared__ float rt_lds[];   // per wave: [E] scores, [E] choice values, [groups] group flags; SPLIT: once, and [4][E + 1] partial products
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t t = SPLIT ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wid;
    if (t >= p.n) return;     // (a whole wave leaves; without SPLIT there is no workgroup barrier below)
    const int E = p.E, G = p.groups > 1 ? p.groups : 1, gsz = E / G;
    // volatile: lanes read what another lane of the wave wrote (one wave: program order is enough, no barrier)
    volatile float* sc = rt_lds + (SPLIT ? 0 : (size_t)wid * (2 * E + G));
    float* part = rt_lds + 2 * E + G;
    volatile float* ch = sc + E;
    volatile float* gflag = ch + E;
    if (p.W) {      // the router's own products: eight entries at a time, every lane a share of the columns, fp32 throughout
        const float* h = p.h + t * p.ldh;
        const uint16_t* W = (const uint16_t*)p.W;
        const int K = p.K;
        const bool vec = (K & 3) == 0 && (p.ldh & 3) == 0 && ((uintptr_t)p.h & 15) == 0 && ((uintptr_t)p.W & 7) == 0;
        const int rows = p.gate_out ? E + 1 : E;
        bool nine = false;
        for (int e0 = SPLIT ? wid / 4 * 8 : 0; e0 < rows; e0 += SPLIT ? blockDim.x / 32 : (NINE && nine ? 9 : 8)) {
            float acc[9] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            nine = NINE && rows - e0 == 9;
            if (NINE && vec && rows - e0 >= 8) {
                const uint16_t* we = W + (int64_t)e0 * K;
#pragma unroll 2
                for (int k = lane * 4; k < K; k += 256) {
                    const float4 x = *(const float4*)(h + k);
                    uint2 w[9];
#pragma unroll
                    for (int j = 0; j < 8; ++j) w[j] = *(const uint2*)(we + (int64_t)j * K + k);
                    w[8] = nine ? *(const uint2*)(we + (int64_t)8 * K + k) : make_uint2(0, 0);
#pragma unroll
                    for (int j = 0; j < 9; ++j) {
                        acc[j] = fmaf(x.x, __uint_as_float(w[j].x << 16), acc[j]);
                        acc[j] = fmaf(x.y, __uint_as_float(w[j].x & 0xffff0000u), acc[j]);
                        acc[j] = fmaf(x.z, __uint_as_float(w[j].y << 16), acc[j]);
                        acc[j] = fmaf(x.w, __uint_as_float(w[j].y & 0xffff0000u), acc[j]);
                    }
                }
            } else if (vec) {
                for (int k = (SPLIT ? threadIdx.x & 255 : lane) * 4; k < K; k += SPLIT ? 1024 : 256) {
                    const float4 x = *(const float4*)(h + k);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        if (e0 + j < rows) {
                            const uint2 w = *(const uint2*)(W + (int64_t)(e0 + j) * K + k);
                            acc[j] = fmaf(x.x, __uint_as_float(w.x << 16), acc[j]);
                            acc[j] = fmaf(x.y, __uint_as_float(w.x & 0xffff0000u), acc[j]);
                            acc[j] = fmaf(x.z, __uint_as_float(w.y << 16), acc[j]);
                            acc[j] = fmaf(x.w, __uint_as_float(w.y & 0xffff0000u), acc[j]);
                        }
                    }
                }
            } else {
                for (int k = SPLIT ? threadIdx.x & 255 : lane; k < K; k += SPLIT ? 256 : 64) {
                    const float x = h[k];
#pragma unroll
                    for (int j = 0; j < (NINE ? 9 : 8); ++j)
                        if (j < 8 ? e0 + j < rows : nine) acc[j] = fmaf(x, __uint_as_float((uint32_t)W[(int64_t)(e0 + j) * K + k] << 16), acc[j]);
                }
            }
            auto keep = [&](int e, float v) {
                if (SPLIT) part[(wid & 3) * rows + e] = v;
                else if (e < E) ch[e] = p.bias ? v + p.bias[e] : v;
                else if (p.gate_out) p.gate_out[t] = bl_sigmoid(v);
            };
            const float v8 = rt_sum8(acc);
            if ((lane & 7) == 0 && e0 + (lane >> 3) < rows) keep(e0 + (lane >> 3), v8);
            if (NINE && nine) {
                const float v9 = wave_sum(acc[8]);
                if (lane == 0) keep(e0 + 8, v9);
            }
        }
        if (SPLIT) {
            __syncthreads();
            if (wid > 0) return;
            for (int e = lane; e < rows; e += 64) {
                const float v = (part[e] + part[rows + e]) + (part[2 * rows + e] + part[3 * rows + e]);
                if (e < E) ch[e] = p.bias ? v + p.bias[e] : v;
                else p.gate_out[t] = bl_sigmoid(v);
            }
        }
    } else {
        const float* z = p.logits + t * p.ld;
        for (int e = lane; e < E; e += 64) ch[e] = p.bias ? z[e] + p.bias[e] : z[e];
    }
    if (E <= 64 && G == 1) {
        rt_choose_few<false>(p, t, lane, lane < E ? ch[lane] : 0.0f);
        return;
    }
    if (p.sigmoid_scores) {     // scores of their own, in the logits' order: the choice falls on the logits unless it is corrected
        for (int e = lane; e < E; e += 64) {
            const float s = bl_sigmoid(ch[e]);
            sc[e] = s;
            if (p.correction) ch[e] = s + p.correction[e];
        }
    } else if (p.chosen_softmax) {     // the choice falls on the logits themselves
        for (int e = lane; e < E; e += 64) {
            const float s = ch[e];
            sc[e] = s;
            if (p.correction) ch[e] = s + p.correction[e];
        }
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) mx = fmaxf(mx, ch[e]);
        mx = wave_max(mx);
        float sum = 0.0f;
        for (int e = lane; e < E; e += 64) {
            const float v = expf(ch[e] - mx);
            sc[e] = v;
            sum += v;
        }
        sum = wave_sum(sum);
        for (int e = lane; e < E; e += 64) {
            const float s = sc[e] / sum;
            sc[e] = s;
            ch[e] = p.correction ? s + p.correction[e] : s;
        }
    }
    if (G > 1) {   // a group's score: its largest choice value; the `keep` best groups stay, the entries of the others cannot be chosen
        for (int g = lane; g < G; g += 64) {
            float b = -INFINITY;
            for (int i = 0; i < gsz; ++i) b = fmaxf(b, ch[g * gsz + i]);
            gflag[g] = b;
        }
        // (LDS traffic of one wave needs program order only)
        for (int r = 0; r < p.keep; ++r) {
            float bv = -INFINITY;
            int bi = -1;
            for (int g = lane; g < G; g += 64) {
                const float v = gflag[g];
                if (!(v != v) && v != INFINITY && (bi < 0 || v > bv)) bv = v, bi = g;     // +inf marks a group already kept
            }
            float best;
            const int pick = bl_wave_argmax(bv, bi, best);
            if (pick != 0x7fffffff && lane == 0) gflag[pick] = INFINITY;
        }
        for (int e = lane; e < E; e += 64)
            if (gflag[e / gsz] != INFINITY) ch[e] = -INFINITY;
    }
    float wsum = 0.0f;
    float mine_w = 0.0f;      // lane k keeps the k-th choice
    int mine_i = 0;
    for (int k = 0; k < p.top; ++k) {
        float bv = -INFINITY;
        int bi = -1;
        for (int e = lane; e < E; e += 64) {
            const float v = ch[e];
            if (v == v && (bi < 0 || v > bv)) bv = v, bi = e;
        }
        float best;
        int pick = bl_wave_argmax(bv, bi, best);
        if (pick == 0x7fffffff) pick = 0;
        const float s = sc[pick];
        wsum += s;
        if (lane == k) mine_w = s, mine_i = pick;
        if (lane == 0) ch[pick] = __builtin_nanf("");     // taken: out of every later comparison
    }
    rt_store<false>(p, t, lane, mine_w, mine_i, wsum);
}

// ---------------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void moe_plan_kernel(const i64h_moe_plan_args p) {
    extern __shared__ int pl_lds[];
    rt_plan<1024>(p, pl_lds, [&](int64_t i) { return p.idx[i]; }, [&](int64_t i) { return p.wgt[i]; });
}

// A thread's loads of four choices are on their way together (as one after the other, each behind its row's number: 7.9 us for 64 rows of
// 2048, 4 choices and a shared part, 3.6 so; 4096 rows 37 -> 29); VEC columns at a time.
template <int VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(const i64h_moe_combine_args p) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const int64_t t = blockIdx.x;
    const int W = p.W;
    for (int c = threadIdx.x * VEC; c < W; c += 256 * VEC) {
        vec a = 0.0f, sh = 0.0f;
        if (p.shared) sh = *(const vec*)(p.shared + t * W + c);
        for (int k0 = 0; k0 < p.top; k0 += 4) {
            vec v[4];
            float w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = min(k0 + i, p.top - 1), r = p.pair_row[t * p.top + k];
                v[i] = *(const vec*)(r >= 0 ? p.Y + (int64_t)r * W + c : p.h + t * W + c);
                w[i] = p.wgt ? p.wgt[t * p.top + k] : 1.0f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (k0 + i < p.top) a += w[i] * v[i];
        }
        if (p.shared) a += p.shared_gate ? p.shared_gate[t] * sh : sh;
        *(vec*)(p.out + t * W + c) = a;
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
extern "C" {

static int gla_check(const i64h_gla_args& d, const char* what) {
    I64H_CHECK_ARG(d.heads > 0 && d.dim > 0 && d.vdim > 0 && d.n >= 0, "%s: heads %d, dim %d, vdim %d", what, d.heads, d.dim, d.vdim);
    I64H_CHECK_ARG(d.P && d.q_off >= 0 && d.f_off >= 0 && d.v_off >= 0, "%s: null operand or negative column", what);
    return 0;
}

int i64h_gla_gates(const i64h_gla_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "gla_gates: no descriptor");
    const i64h_gla_args& d = *dp;
    if (gla_check(d, "gla_gates")) return 1;
    I64H_CHECK_ARG(d.n <= 65535, "gla_gates: %lld rows in one launch (at most 65535)", (long long)d.n);
    if (d.n == 0) return 0;
    hipLaunchKernelGGL(gla_gates_kernel, dim3((unsigned)((d.heads * d.dim + 255) / 256), (unsigned)d.n), dim3(256), 0, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

static int gdn_check(const i64h_gdn_args& d, const char* what) {
    I64H_CHECK_ARG(d.heads > 0 && d.kv_heads > 0 && d.heads % d.kv_heads == 0 && d.dim > 0 && d.vdim > 0 && d.n >= 0, "%s: heads %d, query / key heads %d, dim %d, vdim %d",
                   what, d.heads, d.kv_heads, d.dim, d.vdim);
    I64H_CHECK_ARG(d.X && d.q_off >= 0 && d.k_off >= 0 && d.v_off >= 0, "%s: null operand or negative column", what);
    return 0;
}

int i64h_gdn_gates(const i64h_gdn_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "gdn_gates: no descriptor");
    const i64h_gdn_args& d = *dp;
    if (gdn_check(d, "gdn_gates")) return 1;
    I64H_CHECK_ARG(d.G && d.R && d.b_off >= 0 && (d.a_off < 0 || (d.A_log && d.dt_bias)), "gdn_gates: null operand or negative column");
    if (d.n == 0) return 0;
    auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)d.n), dim3(256), 0, (hipStream_t)stream, d); };
    const bool vec = d.dim % 4 == 0 && d.dim <= 256 && d.ldx % 4 == 0 && d.q_off % 4 == 0 && d.k_off % 4 == 0 && (uintptr_t)d.X % 16 == 0;
    if (!vec) launch(gdn_gates_kernel<0>);
    else if (d.dim <= 64) launch(gdn_gates_kernel<1>);
    else if (d.dim <= 128) launch(gdn_gates_kernel<2>);
    else launch(gdn_gates_kernel<4>);
    I64H_CHECK_LAUNCH();
    return 0;
}

static int g_gdn_form = 0;
int i64h_set_gdn_scan_form(int32_t form) {
    I64H_CHECK_ARG(form >= 0 && form <= 5, "gdn_scan: form %d", form);
    g_gdn_form = form;
    return 0;
}

// Tiles of 16 tokens on the matrix cores are two launches and a tile costs the same however few rows it holds; token by token a launch takes as long as
// its longest run.  So it is the longest run that decides.  Microseconds in replayed graphs, token by token | in tiles, delta rule (linear attention), heads
// of 128: 16 heads, a run of 1531 rows 242 | 106 (215 | 71), of 160 28 | 21 (27 | 15), of 96 17.9 | 17.5 (17.1 | 13.0: too little for a workspace of 27 KB a tile and head), 40 single rows beside 200
// 39 | 44 (33 | 33), beside 280 51 | 46 (45 | 34), 20 beside 128 26 | 30 (23 | 22), 16 runs of 24 30 | 31 (27 | 22), 4 of 64 22 | 22 (19 | 15); 8 heads, 8 runs of 512 125 | 77 (96 | 52), 20 single rows
// beside 128 25 | 22 (22 | 17); 8 heads of 64, 8 runs of 17 5.6 | 11.9 (5.0 | 9.3), 16 of 64 14.6 | 16.6 (11.6 | 12.2), 4 of 96 13.9 | 14.4 (11.3 | 10.9).  Narrow heads in thousands of workgroups
// are little more than their reads either way (32 heads of 64, 32 runs of 192 rows 193 | 182, 140 | 135), as are many short runs (64 of 17 rows, delta rule 41 | 48).
int32_t i64h_scan_in_tiles(int64_t n, int32_t nseg, int32_t longest, int32_t heads, int32_t dim, int32_t vdim, int32_t delta) {
    const int64_t groups = (int64_t)heads * ((vdim + 15) / 16) * nseg;      // workgroups of the second launch
    return dim % 4 == 0 && dim <= 256 && n >= 96 && n >= 8 * (int64_t)nseg && longest >= (delta ? 144 : 112) && (n >= 32 * (int64_t)nseg || groups < 6144) &&
           (dim > 64 || groups <= 2048);
}

// From the projections three launches stand for four or six that read and write the rows between them, so tiles pay earlier, against the number of runs, each a tile at least (in workgroups
// of the second launch).  Microseconds as above, in launches of their own token
// by token | in tiles: 16 heads of 128, a run of 32 rows 27 | 26 (14.6 | 16.3), of 64 36 | 28 (20 | 17), of 96 44 | 29 (26 | 19), 8 single rows beside 40 33 | 32 (18 | 20), beside 60 39 | 33 (22 | 21),
// 20 beside 64 42 | 44 (24 | 28), beside 100 51 | 45 (29 | 29), 40 beside 100 58 | 61 (36 | 40), beside 150 65 | 64 (39 | 43), beside 200 75 | 66 (45 | 44), 64 beside 200 82 | 86 (53 | 59), beside 400
// 114 | 95 (73 | 62), 32 runs of 17 85 | 73 (53 | 48), 16 of 24 73 | 52 (41 | 34); 8 heads, 40 beside 48 38 | 43 (22 | 27), beside 100 47 | 43 (28 | 27), 20 beside 64 36 | 32 (21 | 21);
// 32 heads of 64, a run of 32 26 | 22, 40 beside 100 52 | 53, 20 beside 64 37 | 36.
int32_t i64h_rec_in_tiles(int64_t n, int32_t nseg, int32_t longest, int32_t heads, int32_t dim, int32_t vdim, int32_t delta) {
    const int64_t groups = (int64_t)heads * ((vdim + 15) / 16) * nseg;
    return i64h_scan_in_tiles(n, nseg, longest, heads, dim, vdim, delta) ||
           (dim % 4 == 0 && dim <= 128 && (longest >= (delta ? 28 + groups / 48 : 44 + groups / 36) || (n >= 128 && n >= 16 * (int64_t)nseg)) && (dim > 64 || groups <= 2048));
}

// the recurrence's launch, with the delta rule's correction or (a decay per key channel, every head its own keys) without it
extern "C++" {
template <int RULE>
static int gdn_launch(const i64h_gdn_args& d, void* stream) {
    const int kpt = (d.dim + 15) / 16;
    auto vec_ok = [&](int K) {
        return K % 4 == 0 && d.dim % 4 == 0 && d.ldx % 4 == 0 && d.q_off % 4 == 0 && d.k_off % 4 == 0 && (uintptr_t)d.X % 16 == 0 && (uintptr_t)d.state % 16 == 0 &&
               (!d.F || (d.ldf % 4 == 0 && (uintptr_t)d.F % 16 == 0));
    };
    const int kround = kpt <= 4 ? 4 : (kpt <= 8 ? 8 : 16);
    // runs nobody measured: the mean says whether one of them may be long
    const bool several = d.n >= 8 * (int64_t)d.nseg;
    const bool tiles = i64h_scan_in_tiles(d.n, d.nseg, d.longest > 0 ? d.longest : INT32_MAX, d.heads, d.dim, d.vdim, RULE == GD_DELTA);
    if (RULE != GD_FORGET && d.work && ((g_gdn_form == 0 && tiles) || g_gdn_form == 5) && vec_ok(4) && (uintptr_t)d.work % 16 == 0 && d.ldx < (1 << 25) &&
        (d.n / 16 + d.nseg) * (int64_t)d.heads < (1ll << 31)) {
        I64H_CHECK_ARG(d.work_floats >= i64h_scan_work_floats(d.n, d.nseg, d.heads, d.dim), "scan: a workspace of %lld floats, %lld needed", (long long)d.work_floats,
                       (long long)i64h_scan_work_floats(d.n, d.nseg, d.heads, d.dim));
        return i64h_scan_tiles(d, RULE == GD_DELTA, stream);
    }
    // Staged through LDS, 16 tokens at a time, from a mean of eight rows a run or one run of 16 on: 16 heads, linear attention (delta rule), straight into registers | staged, 40 single rows
    // beside 17 rows 23 | 23 us (24 | 23), beside 100 64 | 25 (75 | 27), beside 280 155 | 45 (184 | 51), 3 beside 20 13.5 | 7.1 (15.8 | 7.7); 32 runs of 7 24 | 27 (26.5 | 28), 64 of 3 27 | 32 (28 | 35).
    if (g_gdn_form != 1 && vec_ok(kround) && (g_gdn_form > 1 || several || d.longest >= 16)) {
        // One value column per lane: a token then takes the longest run least time, and it is the longest run that the launch waits for (16
        // heads of 128, runs of 1531, 257, 64, 3 and 1101 rows: 264 us, two columns 448; 27 single rows beside 229 and 256: 68 and 100).  Two
        // columns (fewer reads of the tile) only where many workgroups wait for a CU and the runs are long (8 runs of 512 rows: 220 and 199 us, 32 of 128
        // 212 and 203, 64 of 64 rows and 32 heads 419 and 389).  Short runs in such numbers would rather have two (64 of 17: 70 and 66), but are not to be
        // told from single rows beside a prompt by their count.
        const int cpt = g_gdn_form > 1 ? (g_gdn_form == 4 ? 4 : g_gdn_form - 1) : ((int64_t)d.heads * ((d.vdim + 15) / 16) * d.nseg >= 1024 && d.n >= 64 * (int64_t)d.nseg ? 2 : 1);
        const int ctiles = (d.vdim + 16 * cpt - 1) / (16 * cpt);
        const dim3 grid((unsigned)(d.heads * ctiles), (unsigned)d.nseg);
        auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, d, ctiles); };
#define GDN_TILE(C, CHD)                                             \
    if (kround == 4) launch(gdn_tile_kernel<4, C, CHD, RULE>);      \
    else if (kround == 8) launch(gdn_tile_kernel<8, C, CHD, RULE>); \
    else launch(gdn_tile_kernel<16, C, CHD, RULE>);
        if (RULE != GD_DELTA || d.F) {
            if (cpt == 1) { GDN_TILE(1, true) } else if (cpt == 2) { GDN_TILE(2, true) } else { GDN_TILE(4, true) }
        } else if constexpr (RULE == GD_DELTA) {
            if (cpt == 1) { GDN_TILE(1, false) } else if (cpt == 2) { GDN_TILE(2, false) } else { GDN_TILE(4, false) }
        }
#undef GDN_TILE
        I64H_CHECK_LAUNCH();
        return 0;
    }
    // columns per lane: query and key are loaded once for both - unless the launch would then leave most of the chip idle
    // (two columns also give the two row sums of a token independent work to overlap: measured faster from 256 workgroups on)
    const int cpt = (d.vdim > 16 && (int64_t)d.heads * ((d.vdim + 31) / 32) * d.nseg >= 256) ? 2 : 1;
    const int ctiles = (d.vdim + 16 * cpt - 1) / (16 * cpt);
    const dim3 grid((unsigned)(d.heads * ctiles), (unsigned)d.nseg);
    auto launch = [&](auto kern, int K) {
        const int vec = vec_ok(K);
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, d, ctiles, vec);
    };
#define GDN_PICK(C, CHD, ONE)                                                                    \
    if (kpt <= 1) launch(gdn_scan_kernel<1, C, CHD, ONE ? 1 : 4, RULE>, 1);                       \
    else if (kpt <= 2) launch(gdn_scan_kernel<2, C, CHD, ONE ? 1 : 4, RULE>, 2);                  \
    else if (kpt <= 4) launch(gdn_scan_kernel<4, C, CHD, ONE ? 1 : 4, RULE>, 4);                  \
    else if (kpt <= 8) launch(gdn_scan_kernel<8, C, CHD, ONE ? 1 : (CHD ? 2 : 4), RULE>, 8);      \
    else launch(gdn_scan_kernel<16, C, CHD, ONE ? 1 : (CHD ? 1 : 2), RULE>, 16);
#define GDN_PICK2(C, CHD) \
    if (d.nseg == d.n) { GDN_PICK(C, CHD, true) } else { GDN_PICK(C, CHD, false) }
    if (RULE != GD_DELTA || d.F) {
        if (cpt == 2) { GDN_PICK2(2, true) } else { GDN_PICK2(1, true) }
    } else if constexpr (RULE == GD_DELTA) {
        if (cpt == 2) { GDN_PICK2(2, false) } else { GDN_PICK2(1, false) }
    }
#undef GDN_PICK2
#undef GDN_PICK
    I64H_CHECK_LAUNCH();
    return 0;
}
}

int i64h_gdn_scan(const i64h_gdn_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "gdn_scan: no descriptor");
    const i64h_gdn_args& d = *dp;
    if (gdn_check(d, "gdn_scan")) return 1;
    I64H_CHECK_ARG(d.G && d.seg_start && d.positions && d.slot_ids && d.state && d.out, "gdn_scan: null operand");
    I64H_CHECK_ARG(d.dim <= 16 * 16, "gdn_scan: dim %d above 256", d.dim);
    I64H_CHECK_ARG(d.nseg <= 65535, "gdn_scan: %d runs in one launch", d.nseg);
    if (d.nseg <= 0 || d.n == 0) return 0;
    return gdn_launch<GD_DELTA>(d, stream);
}

int i64h_gla_scan(const i64h_gla_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "gla_scan: no descriptor");
    const i64h_gla_args& d = *dp;
    if (gla_check(d, "gla_scan")) return 1;
    I64H_CHECK_ARG(d.seg_start && d.positions && d.slot_ids && d.state && d.out, "gla_scan: null operand");
    I64H_CHECK_ARG(d.dim <= 16 * 16, "gla_scan: dim %d above 256", d.dim);
    I64H_CHECK_ARG(d.nseg <= 65535, "gla_scan: %d runs in one launch", d.nseg);
    I64H_CHECK_ARG(!d.F || d.ldf >= d.f_off + (int64_t)d.heads * d.dim, "gla_scan: the decays' rows are shorter than their columns");
    if (d.nseg <= 0 || d.n == 0) return 0;
    i64h_gdn_args a = {};
    a.X = d.P, a.ldx = d.ldp, a.q_off = d.q_off, a.k_off = d.k_off >= 0 ? d.k_off : 0, a.v_off = d.v_off, a.heads = a.kv_heads = d.heads, a.dim = d.dim, a.vdim = d.vdim;
    a.F = (d.F ? d.F : d.P) + d.f_off, a.ldf = d.F ? d.ldf : d.ldp, a.q_scale = d.q_scale, a.seg_start = d.seg_start, a.nseg = d.nseg;
    a.positions = d.positions, a.slot_ids = d.slot_ids, a.state = d.state, a.out = d.out, a.ldo = d.ldo, a.n = d.n;
    a.work = d.work, a.work_floats = d.work_floats, a.longest = d.longest;
    return d.k_off >= 0 ? gdn_launch<GD_KEYS>(a, stream) : gdn_launch<GD_FORGET>(a, stream);
}

int i64h_route_topk(const i64h_route_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "route_topk: no descriptor");
    const i64h_route_args& d = *dp;
    I64H_CHECK_ARG(d.E > 0 && d.E <= 1024 && d.top > 0 && d.top <= RT_MAX_TOP && d.top <= d.E, "route_topk: %d entries (at most 1024), top %d (at most %d)", d.E, d.top, RT_MAX_TOP);
    I64H_CHECK_ARG(d.groups <= 1 || (d.E % d.groups == 0 && d.keep >= 1 && d.keep <= d.groups), "route_topk: %d entries in %d groups, %d kept", d.E, d.groups, d.keep);
    I64H_CHECK_ARG(!d.sigmoid_scores || !d.chosen_softmax, "route_topk: sigmoid scores, or the softmax over the chosen logits");
    I64H_CHECK_ARG(!d.gate_out || d.W, "route_topk: the gate's row lies behind the router's rows");
    I64H_CHECK_ARG(d.groups <= 1 || d.keep * (d.E / d.groups) >= d.top, "route_topk: %d kept groups of %d entries hold fewer than top %d", d.keep, d.E / (d.groups > 0 ? d.groups : 1), d.top);
    I64H_CHECK_ARG(d.idx && d.wgt && ((d.logits && d.ld >= d.E) || (d.W && d.h && d.K > 0 && d.ldh >= d.K)), "route_topk: null operand or row stride below the row");
    if (d.n == 0) return 0;
    const size_t own = (size_t)(2 * d.E + (d.groups > 1 ? d.groups : 1));
    const int many = d.E > RT_MANY;
    if (d.W && d.n <= (RT_SPLIT_ROWS << many))
        hipLaunchKernelGGL((route_topk_kernel<true, false>), dim3((unsigned)d.n), dim3(many || d.n <= RT_WIDE_ROWS ? 1024 : 256), (own + 4 * (size_t)(d.E + 1)) * 4, (hipStream_t)stream, d);
    else {
        const int rows = d.E + (d.gate_out ? 1 : 0);
        auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)((d.n + 3) / 4)), dim3(256), 4 * own * 4, (hipStream_t)stream, d); };
        if (d.W && rows > 8 && rows % 8 == 1) launch(route_topk_kernel<false, true>);
        else launch(route_topk_kernel<false, false>);
    }
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_moe_plan(const i64h_moe_plan_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "moe_plan: no descriptor");
    const i64h_moe_plan_args& d = *dp;
    I64H_CHECK_ARG(d.experts > 0 && d.experts <= 4096 && d.top > 0 && d.n >= 0, "moe_plan: %d experts (at most 4096), top %d", d.experts, d.top);
    I64H_CHECK_ARG(d.idx && d.group_off && d.pair_token && d.pair_row, "moe_plan: null operand");
    I64H_CHECK_ARG(d.n * ((int64_t)d.top + (d.shared ? 1 : 0)) < (1ll << 31), "moe_plan: too many pairs");
    I64H_CHECK_ARG(!d.pair_wgt || d.wgt, "moe_plan: weights per row come from the weights per choice");
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), (size_t)(2 * d.experts + 1) * 4, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_moe_combine(const i64h_moe_combine_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "moe_combine: no descriptor");
    const i64h_moe_combine_args& d = *dp;
    I64H_CHECK_ARG(d.top > 0 && d.W > 0 && d.n >= 0, "moe_combine: top %d, width %d", d.top, d.W);
    I64H_CHECK_ARG(d.Y && d.pair_row && d.h && d.out, "moe_combine: null operand");
    if (d.n == 0) return 0;
    const bool vec = d.W % 4 == 0 && (((uintptr_t)d.Y | (uintptr_t)d.h | (uintptr_t)d.shared | (uintptr_t)d.out) & 15) == 0;
    if (vec) hipLaunchKernelGGL(moe_combine_kernel<4>, dim3((unsigned)d.n), dim3(256), 0, (hipStream_t)stream, d);
    else hipLaunchKernelGGL(moe_combine_kernel<1>, dim3((unsigned)d.n), dim3(256), 0, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
