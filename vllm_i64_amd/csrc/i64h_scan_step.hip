// A decode step of the recurrences (include/i64h_dense.h, i64h_rec_step): everything between a layer's projections and its out-projection that belongs to one head
// of one row - convolution and unit vectors (delta rule), the low-rank decays and output gates, the recurrence's one step, the head's norm and gate -
// in one workgroup, so that a layer waits for one launch in the place of six (linear attention: three).
// What bounds it: few rows the chain inside a workgroup (loads of the sequence's slot, of the state behind it, sums, norm), many rows the state's way from memory and
// back; the low-rank maps' 64 KB a head come from L2.  7 rows of 8 heads of 128 in a graph: six launches of the delta rule 23 us, this one 9, a step of eight such layers 510 -> 404; 64 rows
// of 16 heads, linear attention: 37 -> 24 alone; beside an attention over 134 MB the launch takes 59 and the attention 58 where it took 37, together 268 MB at the copy rate, a step 1524 -> 1508.
#include "i64h_dense_dev.h"
#include "i64h_scan_dev.h"

int i64h_conv_carry(const i64h_causal_conv_args& d, void* stream);      // i64h_hybrid.hip
int i64h_scan_tiles_raw(const i64h_gdn_args& d, const i64h_rec_step_args& raw, bool delta, void* stream);      // i64h_scan_tile.hip

// 512 threads: the 16 lanes of a DPP row share CPT value columns and hold KPT key channels of each in registers; a workgroup has 32 such rows.
// DELTA: the delta rule behind a convolution; else linear attention with keys of its own, its gates columns of P.
template <int KPT, int CPT, bool DELTA>
__global__ __launch_bounds__(512) void rec_step_kernel(const i64h_rec_step_args p) {
    constexpr int NP = 16 * KPT, RPT = NP / 32;      // RPT: rows of the decays' map a DPP row takes
    __shared__ __attribute__((aligned(16))) float sX[DELTA ? 2 * NP + 32 * CPT : 4], sF[NP], sS[32];
    const int tid = threadIdx.x, l = tid & 15, g = tid >> 4;
    const int N = p.dim, V = p.vdim, a = blockIdx.x % p.heads;
    const int64_t t = blockIdx.x / p.heads;
    const float* row = p.P + t * p.ldp;
    const int64_t slot = p.slot_ids[t];
    const int pos = p.positions[t];
    // the maps' input rows, rounded as the Linears round them, and the products: 16 lanes a row of the map, eight values a lane and stripe of 128
    auto map = [&](const void* M, int off, int rank, int first, int count, int top, auto& sum) {
        constexpr int R = sizeof(sum) / sizeof(float);
#pragma unroll
        for (int r = 0; r < R; ++r) sum[r] = 0.0f;
        for (int k = 8 * l; k < rank; k += 128) {
            dn_v4u w[R];
#pragma unroll
            for (int r = 0; r < R; ++r) w[r] = first + r < top ? *(const dn_v4u*)((const uint16_t*)M + ((int64_t)a * top + first + r) * rank + k) : (dn_v4u)0u;
            float x[8];
            *(dn_v4f*)x = *(const dn_v4f*)(row + off + k), *(dn_v4f*)(x + 4) = *(const dn_v4f*)(row + off + k + 4);
            if (!p.exact) {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = dn_bf16_to_f32(dn_bf16_rne(x[i]));
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s0 = fmaf(x[2 * i], __uint_as_float(w[r][i] << 16), s0);
                    s1 = fmaf(x[2 * i + 1], __uint_as_float(w[r][i] & 0xffff0000u), s1);
                }
                sum[r] += s0 + s1;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) sum[r] = group_sum(sum[r], 16);
    };
    // ---- what does not wait for the sequence's slot: decays and gates ----
    float zs[CPT], fs[RPT];
    map(p.A, p.a_off, p.a_rank, RPT * g, RPT, N, fs);
    if (DELTA) map(p.Z, p.z_off, p.z_rank, CPT * g, CPT, V, zs);
    // ---- the state, on its way from here on ----
    float S[CPT][KPT];
    float* gS = p.state + ((slot * p.heads + a) * V + CPT * g) * N;
#pragma unroll
    for (int j = 0; j < CPT; ++j)
#pragma unroll
        for (int k = 0; k < KPT; k += 4) {
            const int c = gd_channel<KPT>(l, k);
            dn_v4f v = {0, 0, 0, 0};
            if (pos != 0 && CPT * g + j < V && c < N) v = *(const dn_v4f*)(gS + j * N + c);
            *(dn_v4f*)&S[j][k] = v;
        }
    if (l < RPT) {
        const int c = RPT * g + l;
        float f = fs[0];
#pragma unroll
        for (int r = 1; r < RPT; ++r) f = l == r ? fs[r] : f;
        sF[c] = c < N ? expf(-p.a_rate[a * N + c] * dn_softplus(f + p.a_bias[a * N + c])) : 1.0f;
    }
    float q[KPT], k[KPT], f[KPT], v[CPT], beta = 0.0f;
    if constexpr (DELTA) {      // a thread per channel of q | k | v: its convolution, and the carried inputs one position on
        const int part = tid < NP ? 0 : (tid < 2 * NP ? 1 : 2), c = tid - part * NP;
        if (tid < 2 * NP + 32 * CPT) {
            float o = 0.0f;
            if (c < (part < 2 ? N : V)) {
                const int H = p.heads, ch = part < 2 ? (part * H + a) * N + c : 2 * H * N + a * V + c, C = H * (2 * N + V), T = p.taps;
                const float* w = p.conv_w + (int64_t)ch * T;
                float* st = p.conv + slot * (T - 1) * C + ch;
                const float x = row[p.q_off + ch];
                float in[7];
#pragma unroll
                for (int d = 1; d < 8; ++d) in[d - 1] = d < T && pos >= d ? st[(int64_t)(T - 1 - d) * C] : 0.0f;
                for (int d = T - 1; d > 0; --d) {
                    float y = in[0];
#pragma unroll
                    for (int i = 1; i < 7; ++i) y = d == i + 1 ? in[i] : y;
                    o += w[T - 1 - d] * y;
                }
                o += w[T - 1] * x;
                o = o / (1.0f + expf(-o));
#pragma unroll
                for (int d = 1; d < 7; ++d)
                    if (d < T - 1) st[(int64_t)(T - 2 - d) * C] = in[d - 1];
                st[(int64_t)(T - 2) * C] = x;
            }
            sX[tid] = o;
        }
        beta = dn_sigmoid(row[p.b_off + a]);
    } else {
#pragma unroll
        for (int i = 0; i < KPT; i += 4) {
            const int c = gd_channel<KPT>(l, i);
            dn_v4f x = {0, 0, 0, 0}, y = x;
            if (c < N) x = *(const dn_v4f*)(row + p.q_off + a * N + c), y = *(const dn_v4f*)(row + p.k_off + a * N + c);
            *(dn_v4f*)&q[i] = x, *(dn_v4f*)&k[i] = y;
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = CPT * g + j;
            v[j] = c < V ? row[p.v_off + a * V + c] : 0.0f, zs[j] = c < V ? row[p.z_off + a * V + c] : 0.0f;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KPT; i += 4) {
        const int c = gd_channel<KPT>(l, i);
        *(dn_v4f*)&f[i] = *(const dn_v4f*)&sF[c];
        if constexpr (DELTA) *(dn_v4f*)&q[i] = *(const dn_v4f*)&sX[c], *(dn_v4f*)&k[i] = *(const dn_v4f*)&sX[NP + c];
    }
    if constexpr (DELTA) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) v[j] = sX[2 * NP + CPT * g + j];
        auto unit = [&](float (&x)[KPT], float scale) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < KPT; i += 4) s += (x[i] * x[i] + x[i + 1] * x[i + 1]) + (x[i + 2] * x[i + 2] + x[i + 3] * x[i + 3]);
            const float u = 1.0f / sqrtf(group_sum(s, 16) + p.unit_eps) * scale;
#pragma unroll
            for (int i = 0; i < KPT; ++i) x[i] *= u;
        };
        unit(q, p.q_scale);
        unit(k, 1.0f);
    }
    float o[CPT], ss = 0.0f;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        if constexpr (DELTA) o[j] = gd_delta<KPT, true>(S[j], f, k, q, v[j], beta);
        else o[j] = gd_linear<KPT, true, false>(S[j], f, k, q, v[j]) * p.q_scale;
        ss += CPT * g + j < V ? o[j] * o[j] : 0.0f;
    }
    if (l == 0) sS[g] = ss;
#pragma unroll
    for (int j = 0; j < CPT; ++j)
#pragma unroll
        for (int i = 0; i < KPT; i += 4) {
            const int c = gd_channel<KPT>(l, i);
            if (CPT * g + j < V && c < N) *(dn_v4f*)(gS + j * N + c) = *(const dn_v4f*)&S[j][i];
        }
    __syncthreads();
    float all = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        const dn_v4f s = *(const dn_v4f*)&sS[i];
        all += (s[0] + s[1]) + (s[2] + s[3]);
    }
    const int c = CPT * g + l;
    if (l >= CPT || c >= V) return;
    float y = o[0], z = zs[0];
#pragma unroll
    for (int j = 1; j < CPT; ++j) y = l == j ? o[j] : y, z = l == j ? zs[j] : z;
    y = y / sqrtf(all / (float)V + p.eps) * p.norm_w[c] * (p.gate_act ? dn_sigmoid(z) : z / (1.0f + expf(-z)));
    if (p.out) p.out[t * p.ldo + a * V + c] = y;
    if (p.out16) ((uint16_t*)p.out16)[t * p.ldo + a * V + c] = (uint16_t)dn_bf16_rne(y);
}

// Norm and gate of many rows whose gate is a low-rank map: a workgroup per 16 rows of one head takes the map's products on the bf16 matrix instruction - lane (c, g): row c, columns 4 g ..
// of a block of 16, as the norm's operands lie - so that the gates never pass memory (2956 rows of 16 heads of 128: a Linear of 12 us and gate_norm_kernel's 17, 23 together).
template <int NV>      // blocks of 16 columns a wave has at most
__global__ __launch_bounds__(256) void gate_map_kernel(const i64h_rec_step_args p, const float* y, const int64_t ldy) {
    __shared__ float sS[4][16];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, g = lane >> 4;
    const int V = p.vdim, a = blockIdx.x % p.heads;
    const int64_t t = (int64_t)(blockIdx.x / p.heads) * 16 + c;
    const bool ok = t < p.n;
    const float* row = p.P + (ok ? t : p.n - 1) * p.ldp + p.z_off;
    const uint16_t* map = (const uint16_t*)p.Z + (int64_t)a * V * p.z_rank;
    dn_v4f v[NV], acc[NV];
    float ss = 0.0f;
#pragma unroll
    for (int b = 0; b < NV; ++b) {
        const int col = 16 * (NV * w + b) + 4 * g;
        v[b] = acc[b] = dn_v4f{0, 0, 0, 0};
        if (ok && col < V) v[b] = *(const dn_v4f*)(y + t * ldy + a * V + col);
    }
    for (int k0 = 0; k0 < p.z_rank; k0 += 128) {      // (four steps' loads together, none behind a branch: past the rank both factors are zeros, past the last column nobody uses the sum)
        dn_v4f u[4][2];
        dn_v4u m[4][NV];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = min(k0 + 32 * s + 8 * g, p.z_rank - 8);
            u[s][0] = *(const dn_v4f*)(row + k), u[s][1] = *(const dn_v4f*)(row + k + 4);
#pragma unroll
            for (int b = 0; b < NV; ++b) m[s][b] = *(const dn_v4u*)(map + (int64_t)min(16 * (NV * w + b) + c, V - 1) * p.z_rank + k);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            dn_v4u x{dn_bf16_pair(u[s][0][0], u[s][0][1]), dn_bf16_pair(u[s][0][2], u[s][0][3]), dn_bf16_pair(u[s][1][0], u[s][1][1]), dn_bf16_pair(u[s][1][2], u[s][1][3])};
            if (k0 + 32 * s + 8 * g >= p.z_rank) {
                x = dn_v4u{0, 0, 0, 0};
#pragma unroll
                for (int b = 0; b < NV; ++b) m[s][b] = dn_v4u{0, 0, 0, 0};
            }
#pragma unroll
            for (int b = 0; b < NV; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, m[s][b]), __builtin_bit_cast(dn_v8bf, x), acc[b], 0, 0, 0);
        }
    }
#pragma unroll
    for (int b = 0; b < NV; ++b) ss += (v[b][0] * v[b][0] + v[b][1] * v[b][1]) + (v[b][2] * v[b][2] + v[b][3] * v[b][3]);
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) sS[w][c] = ss;
    __syncthreads();
    const float den = sqrtf(((sS[0][c] + sS[1][c]) + (sS[2][c] + sS[3][c])) / (float)V + p.eps);
#pragma unroll
    for (int b = 0; b < NV; ++b) {
        const int col = 16 * (NV * w + b) + 4 * g;
        if (!ok || col >= V) continue;
        const dn_v4f nw = *(const dn_v4f*)(p.norm_w + col);
        dn_v4f o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = v[b][i] / den * nw[i] * dn_gated(p.gate_act && acc[b][i] == acc[b][i] ? 1.0f : acc[b][i], acc[b][i]);
        if (p.out) *(dn_v4f*)(p.out + t * p.ldo + a * V + col) = o;
        if (p.out16) *(dn_v2u*)((uint16_t*)p.out16 + t * p.ldo + a * V + col) = dn_v2u{dn_bf16_pair(o[0], o[1]), dn_bf16_pair(o[2], o[3])};
    }
}

extern "C" {

static int rec_check(const i64h_rec_step_args& d, const char* what) {
    const bool delta = d.conv_w != nullptr;
    I64H_CHECK_ARG(d.heads > 0 && d.dim > 0 && d.dim <= 128 && d.dim % 4 == 0 && d.vdim > 0 && d.vdim <= 128 && d.n >= 0,
                   "%s: heads %d, dim %d, vdim %d (dims to 128, key channels in fours)", what, d.heads, d.dim, d.vdim);
    I64H_CHECK_ARG(d.P && d.positions && d.slot_ids && d.state && d.A && d.a_bias && d.a_rate && d.norm_w && (d.out || d.out16), "%s: null operand", what);
    I64H_CHECK_ARG(d.q_off >= 0 && d.a_off >= 0 && d.z_off >= 0 && (delta ? d.b_off >= 0 : d.k_off >= 0 && d.v_off >= 0), "%s: negative column", what);
    I64H_CHECK_ARG(!delta || (d.conv && d.Z && d.taps >= 2 && d.taps <= 8 && d.z_rank > 0), "%s: the delta rule takes a convolution of 2 to 8 taps (%d) and a low-rank gate", what, d.taps);
    I64H_CHECK_ARG(d.a_rank > 0 && d.a_rank % 8 == 0 && (!delta || d.z_rank % 8 == 0), "%s: ranks %d and %d, multiples of eight", what, d.a_rank, d.z_rank);
    I64H_CHECK_ARG((((uintptr_t)d.P | (uintptr_t)d.A | (uintptr_t)d.Z | (uintptr_t)d.state) & 15) == 0 && d.ldp % 4 == 0 && d.a_off % 4 == 0 &&
                   (delta ? d.z_off % 4 == 0 : d.q_off % 4 == 0 && d.k_off % 4 == 0), "%s: rows and states are read 16 bytes at a time", what);
    I64H_CHECK_ARG(d.n * d.heads < (1ll << 31), "%s: %lld rows of %d heads", what, (long long)d.n, d.heads);
    const int64_t nd = (int64_t)d.heads * d.dim, rv = (int64_t)d.heads * d.vdim;
    auto inside = [&](int64_t off, int64_t width) { return off + width <= d.ldp; };
    I64H_CHECK_ARG(d.ldo >= rv && inside(d.a_off, d.a_rank) && (delta ? inside(d.q_off, 2 * nd + rv) && inside(d.b_off, d.heads) && inside(d.z_off, d.z_rank)
                                                                   : inside(d.q_off, nd) && inside(d.k_off, nd) && inside(d.v_off, rv) && inside(d.z_off, rv)), "%s: columns behind the row's end", what);
    return 0;
}

int i64h_rec_step(const i64h_rec_step_args* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "rec_step: no descriptor");
    const i64h_rec_step_args& d = *dp;
    const bool delta = d.conv_w != nullptr;
    if (rec_check(d, "rec_step")) return 1;
    if (d.n == 0) return 0;
    auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)(d.n * d.heads)), dim3(512), 0, (hipStream_t)stream, d); };
#define REC_PICK(K, C)                                  \
    if (delta) launch(rec_step_kernel<K, C, true>);     \
    else launch(rec_step_kernel<K, C, false>);
    if (d.dim <= 64) {
        if (d.vdim <= 64) { REC_PICK(4, 2) } else { REC_PICK(4, 4) }
    } else {
        if (d.vdim <= 64) { REC_PICK(8, 2) } else { REC_PICK(8, 4) }
    }
#undef REC_PICK
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_rec_tiles(const i64h_rec_step_args* dp, const i64h_gdn_args* sp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr && sp != nullptr, "rec_tiles: no descriptor");
    const i64h_rec_step_args& d = *dp;
    const bool delta = d.conv_w != nullptr;
    if (rec_check(d, "rec_tiles")) return 1;
    I64H_CHECK_ARG(!d.exact && d.dim % 4 == 0 && d.vdim % 4 == 0 && (!delta || d.taps <= 4), "rec_tiles: products of bf16 values, columns in fours, at most 4 taps");
    i64h_gdn_args a = *sp;
    I64H_CHECK_ARG(a.seg_start && a.nseg > 0 && a.nseg <= 65535 && a.out && a.ldo >= (int64_t)d.heads * d.vdim && (!delta || (a.X && a.v_off >= 0 && a.ldx >= a.v_off + (int64_t)d.heads * d.vdim)) && a.work && a.work_floats >= i64h_scan_work_floats(d.n, a.nseg, d.heads, d.dim),
                   "rec_tiles: runs, a workspace and rows for the read-out");
    I64H_CHECK_ARG((((uintptr_t)a.work | (uintptr_t)a.out | (uintptr_t)d.norm_w | (uintptr_t)d.a_rate | (uintptr_t)d.a_bias | (uintptr_t)d.out | (uintptr_t)d.out16) & 15) == 0 && a.ldo % 4 == 0 && d.ldo % 4 == 0 &&
                   d.ldp < (1 << 25) && a.ldx < (1 << 25) && (d.n / 16 + a.nseg) * (int64_t)d.heads < (1ll << 31), "rec_tiles: rows are read 16 bytes at a time");
    if (d.n == 0) return 0;
    a.heads = a.kv_heads = d.heads, a.dim = d.dim, a.vdim = d.vdim, a.positions = d.positions, a.slot_ids = d.slot_ids, a.state = d.state, a.n = d.n, a.q_scale = d.q_scale;
    if (!delta) a.X = const_cast<float*>(d.P), a.ldx = d.ldp, a.v_off = d.v_off;
    if (i64h_scan_tiles_raw(a, d, delta, stream)) return 1;
    if (!delta) {      // (the gates are columns)
        i64h_gate_norm_args g = {};
        g.y = a.out, g.ldy = a.ldo, g.z = d.P + d.z_off, g.ldz = d.ldp, g.w = d.norm_w, g.width = d.heads * d.vdim, g.groups = d.heads, g.eps = d.eps, g.out = d.out, g.out16 = d.out16, g.ldo = d.ldo;
        g.n = d.n, g.gate_after = 1, g.w_len = d.vdim, g.gate_act = d.gate_act;
        return i64h_gate_norm(&g, stream);
    }
    i64h_causal_conv_args c = {};
    c.P = d.P, c.ldp = d.ldp, c.off = d.q_off, c.channels = d.heads * (2 * d.dim + d.vdim), c.taps = d.taps, c.positions = d.positions, c.slot_ids = d.slot_ids, c.state = d.conv, c.n = d.n;
    c.seg_start = a.seg_start, c.nseg = a.nseg;
    if (i64h_conv_carry(c, stream)) return 1;
    const dim3 grid((unsigned)((d.n + 15) / 16 * d.heads));
    if (d.vdim <= 64) hipLaunchKernelGGL(gate_map_kernel<1>, grid, dim3(256), 0, (hipStream_t)stream, d, (const float*)a.out, a.ldo);
    else hipLaunchKernelGGL(gate_map_kernel<2>, grid, dim3(256), 0, (hipStream_t)stream, d, (const float*)a.out, a.ldo);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
