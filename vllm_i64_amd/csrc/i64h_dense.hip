// Kernels of libi64hip_dense.so for decoder models with bf16 weights and a 32-bit residual stream (include/i64h_dense.h):
//   linear_tile_kernel   : C = epilogue(A W^T), 64 x 64 tiles, four waves of 32 x 32, on v_mfma_f32_16x16x32_bf16 (A rounded to
//                          bf16 while staged) or v_mfma_f32_16x16x4_f32 (W widened while staged: true 32-bit); batched over
//                          blockIdx.z (per-head weights on column blocks of wider matrices); epilogues: gelu_tanh(gate) * up
//                          on two accumulators, * sigmoid(E), logit soft cap and others; an RMS norm of its input on the way.  The form
//                          of operands that 16-byte loads cannot read; every other launch of more than a few rows is
//                          linear_block_kernel's (i64h_linear_block.hip)
//   linear_skinny_kernel : the same product for at most I64H_SKINNY_ROWS rows (decode steps): the rows sit in LDS as bf16, every
//                          wave streams four weight rows at a time with 16-byte loads and reduces over its lanes
//   linear_rows_kernel   : at most 64 rows of a small product: 16 output columns per workgroup, the k steps dealt to its waves, every operand read
//                          from memory as a matrix-core fragment, partial tiles summed through LDS
//   embed_scaled_kernel  : bf16 table row * scale -> fp32
//   gated_postnorm_kernel: alpha * x + sigmoid(gate) * y -> RMS norm in groups -> (optional) weighted sum over the outputs of
//                          all earlier layers; one workgroup per row, the row held in LDS between the passes
//   sample_rows_kernel   : greedy / temperature / top-k / top-p draw of one token per row
#include "i64h_dense_dev.h"
#include <type_traits>

// ---------------------------------------------------------------------------------------------------------------------------
template <bool EXACT, int EPI>
__global__ __launch_bounds__(256) void linear_tile_kernel(const i64h_linear p, const int vecA, const int vecW) {
    constexpr bool DUAL = dn_dual(EPI);
    constexpr int LD = EXACT ? 33 : 40;  // 33 words: conflict-free column reads; 40 halves = 80 bytes: 16-byte aligned fragments
    using T = typename std::conditional<EXACT, float, uint16_t>::type;
    __shared__ __attribute__((aligned(16))) T sA[2][64][LD];
    __shared__ __attribute__((aligned(16))) T sB[2][64][LD];
    __shared__ __attribute__((aligned(16))) T sB2[DUAL ? 2 : 1][DUAL ? 64 : 1][LD];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wm = wid >> 1, wn = wid & 1;
    const int64_t b = blockIdx.z;
    int64_t m0 = (int64_t)blockIdx.y * 64;
    const int n0 = blockIdx.x * 64;
    int64_t rows = p.M;
    if (p.group_off) {   // this batch's share of the rows; m0 becomes the tile's first row among all rows
        const int64_t g0 = p.group_off[b];
        rows = min(rows, (int64_t)p.group_off[b + 1] - g0);
        if (m0 >= rows) return;
        rows += g0;
        m0 += g0;
    }
    const int M = (int)min((int64_t)64, rows - m0);  // rows of this tile
    const int N = p.N, K = p.K;
    const int lr = tid >> 2, lc = (tid & 3) * 8;
    constexpr bool INN = EPI == I64H_EPI_IN_NORM;
    __shared__ float sRow[INN ? 64 : 1];
    float ssq = 0.0f;
    const bool aok = lr < M, bok = n0 + lr < N;
    const int64_t arow = aok ? (p.a_rows ? (int64_t)p.a_rows[m0 + lr] : m0 + lr) : 0;
    const float* pa = p.A + b * p.a_batch + arow * p.lda;
    const uint16_t* pw = (const uint16_t*)p.W + b * p.w_batch + (int64_t)(bok ? n0 + lr : 0) * K;
    const uint16_t* pw2 = pw + (int64_t)N * K;
    float ra[8], rn[INN ? 8 : 1];
    uint16_t rb[8], rb2[8];
    auto gload = [&](int k0) {
        const int k = k0 + lc;
        if (INN) {
            if (vecA && k + 8 <= K) {
                const float4 u = *(const float4*)(p.in_norm_w + k), v = *(const float4*)(p.in_norm_w + k + 4);
                const float w[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) rn[INN ? i : 0] = w[i];
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) rn[INN ? i : 0] = k + i < K ? p.in_norm_w[k + i] : 0.0f;
            }
        }
        if (aok && vecA && k + 8 <= K) {
            const float4 u = *(const float4*)(pa + k), v = *(const float4*)(pa + k + 4);
            ra[0] = u.x; ra[1] = u.y; ra[2] = u.z; ra[3] = u.w; ra[4] = v.x; ra[5] = v.y; ra[6] = v.z; ra[7] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) ra[i] = (aok && k + i < K) ? pa[k + i] : 0.0f;
        }
        if (bok && vecW && k + 8 <= K) {
            *(uint4*)rb = *(const uint4*)(pw + k);
            if (DUAL) *(uint4*)rb2 = *(const uint4*)(pw2 + k);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                rb[i] = (bok && k + i < K) ? pw[k + i] : (uint16_t)0;
                if (DUAL) rb2[i] = (bok && k + i < K) ? pw2[k + i] : (uint16_t)0;
            }
        }
    };
    auto lstore = [&](int buf) {
        if (INN) {      // the row's squares as they come, the norm's weights on what is staged
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                ssq = fmaf(ra[i], ra[i], ssq);
                ra[i] *= rn[INN ? i : 0];
            }
        }
        if (EXACT) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sA[buf][lr][lc + i] = (T)ra[i];
                sB[buf][lr][lc + i] = (T)dn_bf16_to_f32(rb[i]);
                if (DUAL) sB2[buf][lr][lc + i] = (T)dn_bf16_to_f32(rb2[i]);
            }
        } else {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = dn_bf16_rne(ra[2 * i]) | (dn_bf16_rne(ra[2 * i + 1]) << 16);
            *(uint4*)&sA[buf][lr][lc] = make_uint4(w[0], w[1], w[2], w[3]);
            *(uint4*)&sB[buf][lr][lc] = *(const uint4*)rb;
            if (DUAL) *(uint4*)&sB2[buf][lr][lc] = *(const uint4*)rb2;
        }
    };
    dn_v4f acc[2][2], acc2[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[i][j] = dn_v4f{0, 0, 0, 0};
            acc2[i][j] = dn_v4f{0, 0, 0, 0};
        }
    const int fr = lane & 15, fk = lane >> 4;
    gload(0);
    lstore(0);
    __syncthreads();
    const int KT = (K + 31) / 32;
    for (int kt = 0; kt < KT; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < KT) gload((kt + 1) * 32);  // the next tile is in flight behind the matrix instructions of this one
        if (EXACT) {
#pragma unroll
            for (int kk = 0; kk < 32; kk += 4) {
                float a[2], bb[2], b2[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) a[i] = (float)sA[cur][wm * 32 + i * 16 + fr][kk + fk];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bb[j] = (float)sB[cur][wn * 32 + j * 16 + fr][kk + fk];
                    if (DUAL) b2[j] = (float)sB2[cur][wn * 32 + j * 16 + fr][kk + fk];
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], bb[j], acc[i][j], 0, 0, 0);
                        if (DUAL) acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b2[j], acc2[i][j], 0, 0, 0);
                    }
            }
        } else {
            dn_v8bf a[2], bb[2], b2[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = *(const dn_v8bf*)&sA[cur][wm * 32 + i * 16 + fr][fk * 8];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bb[j] = *(const dn_v8bf*)&sB[cur][wn * 32 + j * 16 + fr][fk * 8];
                if (DUAL) b2[j] = *(const dn_v8bf*)&sB2[cur][wn * 32 + j * 16 + fr][fk * 8];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bb[j], acc[i][j], 0, 0, 0);
                    if (DUAL) acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b2[j], acc2[i][j], 0, 0, 0);
                }
        }
        if (kt + 1 < KT) lstore(cur ^ 1);
        __syncthreads();
    }
    if (INN) {      // four neighbouring lanes hold a row's shares
        ssq += __shfl_xor(ssq, 1);
        ssq += __shfl_xor(ssq, 2);
        if ((tid & 3) == 0) sRow[INN ? lr : 0] = 1.0f / sqrtf(ssq / (float)K + p.in_eps);
        __syncthreads();
    }
    float* C = p.C + b * p.c_batch;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int reg = 0; reg < 4; ++reg) {
            const int rl = wm * 32 + i * 16 + fk * 4 + reg;
            if (rl >= M) continue;
            const int64_t r = m0 + rl;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int c = n0 + wn * 32 + j * 16 + fr;
                if (c < N) C[r * p.ldc + c] = dn_epilogue<EPI>(p, INN ? acc[i][j][reg] * sRow[INN ? rl : 0] : acc[i][j][reg], acc2[i][j][reg], b, r, c);
            }
        }
}


// ---------------------------------------------------------------------------------------------------------------------------
// One or two rows.  They are rounded to bf16 into LDS once per workgroup (M * K halves); a wave takes CPW = 4 weight rows at a time, every lane
// 8 consecutive k of each per iteration (one 16-byte load per weight row), products in fp32.  The products are what bounds it: 1024 x 1024
// in a replayed graph 4.2 us at one row, 5.0 at two, 6.4 at four, 8.4 at seven; on the matrix cores 5.4 us at any of them.
template <int EPI>
__global__ __launch_bounds__(256) void linear_skinny_kernel(const i64h_linear p, const int cols_per_block) {
    constexpr bool DUAL = dn_dual(EPI);
    constexpr int CPW = 4, MR = I64H_SKINNY_ROWS;
    constexpr bool INN = EPI == I64H_EPI_IN_NORM;
    __shared__ float sRow[INN ? MR : 1][4];
    extern __shared__ __attribute__((aligned(16))) uint16_t sa[];  // [M][K]
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t b = blockIdx.z;
    const int M = (int)p.M, N = p.N, K = p.K;
    for (int m = 0; m < M; ++m) {
        const int64_t arow = p.a_rows ? (int64_t)p.a_rows[m] : m;
        const float* pa = p.A + b * p.a_batch + arow * p.lda;
        float ssq = 0.0f;
        for (int k = tid * 4; k < K; k += 1024) {
            float4 v = *(const float4*)(pa + k);
            if (INN) {
                ssq = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ssq))));
                const float4 w = *(const float4*)(p.in_norm_w + k);
                v.x *= w.x, v.y *= w.y, v.z *= w.z, v.w *= w.w;
            }
            *(uint2*)&sa[m * K + k] = make_uint2(dn_bf16_rne(v.x) | (dn_bf16_rne(v.y) << 16), dn_bf16_rne(v.z) | (dn_bf16_rne(v.w) << 16));
        }
        if (INN) {
            ssq = wave_sum(ssq);
            if (lane == 0) sRow[INN ? m : 0][wid] = ssq;
        }
    }
    __syncthreads();
    const uint16_t* W = (const uint16_t*)p.W + b * p.w_batch;
    float* C = p.C + b * p.c_batch;
    const int c_end = min(N, (int)(blockIdx.x + 1) * cols_per_block);
    for (int c0 = blockIdx.x * cols_per_block + wid * CPW; c0 < c_end; c0 += 4 * CPW) {
        float acc[CPW][MR], acc2[DUAL ? CPW : 1][MR];
#pragma unroll
        for (int j = 0; j < CPW; ++j)
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                acc[j][m] = 0.0f;
                if (DUAL) acc2[j][m] = 0.0f;
            }
        for (int k = lane * 8; k < K; k += 512) {
            uint4 w[CPW], w2[DUAL ? CPW : 1];
#pragma unroll
            for (int j = 0; j < CPW; ++j) {
                const int c = min(c0 + j, N - 1);
                w[j] = *(const uint4*)(W + (int64_t)c * K + k);
                if (DUAL) w2[j] = *(const uint4*)(W + (int64_t)(c + N) * K + k);
            }
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                if (m >= M) break;
                const uint4 a = *(const uint4*)&sa[m * K + k];
                const uint32_t aw[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int j = 0; j < CPW; ++j) {
                    const uint32_t ww[4] = {w[j].x, w[j].y, w[j].z, w[j].w};
                    float s = acc[j][m];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        s = fmaf(__uint_as_float(aw[q] << 16), __uint_as_float(ww[q] << 16), s);
                        s = fmaf(__uint_as_float(aw[q] & 0xffff0000u), __uint_as_float(ww[q] & 0xffff0000u), s);
                    }
                    acc[j][m] = s;
                    if (DUAL) {
                        const uint32_t w2w[4] = {w2[j].x, w2[j].y, w2[j].z, w2[j].w};
                        float s2 = acc2[j][m];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            s2 = fmaf(__uint_as_float(aw[q] << 16), __uint_as_float(w2w[q] << 16), s2);
                            s2 = fmaf(__uint_as_float(aw[q] & 0xffff0000u), __uint_as_float(w2w[q] & 0xffff0000u), s2);
                        }
                        acc2[j][m] = s2;
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < CPW; ++j)
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                if (m >= M) break;
                float s = wave_sum(acc[j][m]);
                if (INN) {
                    const float* q = sRow[INN ? m : 0];
                    s *= 1.0f / sqrtf(((q[0] + q[1]) + (q[2] + q[3])) / (float)K + p.in_eps);
                }
                const float s2 = DUAL ? wave_sum(acc2[j][m]) : 0.0f;
                const int c = c0 + j;
                if (lane == 0 && c < c_end) C[(int64_t)m * p.ldc + c] = dn_epilogue<EPI>(p, s, s2, b, m, c);
            }
    }
}


// ---------------------------------------------------------------------------------------------------------------------------
// At most 16 MB rows of a small product, bf16 form.  A workgroup owns 16 output columns; its NW waves deal the 32-wide k steps among them, each with the
// 16-row blocks of A against the one weight fragment, all operands read straight from memory as matrix-core fragments (no staging, no barrier
// inside the loop); the partial tiles meet in LDS, then the epilogue.  Its launch is one round of loads and one reduction: 7 x 1024 x 1024 5.4 us in a
// replayed graph against 5.9 us of the 16 x 64 tiles of linear_block_kernel, 7 x 1024 x 128 3.2 against 4.1 us.
constexpr int dn_rows_waves(int epi, int mb) { return dn_dual(epi) && mb > 1 ? 4 : 8; }      // (the gate / up pair of 64 rows needs twice the LDS)
template <int EPI, int MB>
__global__ __launch_bounds__(64 * dn_rows_waves(EPI, MB)) void linear_rows_kernel(const i64h_linear p) {
    constexpr bool DUAL = dn_dual(EPI), INN = EPI == I64H_EPI_IN_NORM;
    constexpr int NW = dn_rows_waves(EPI, MB), U = 2;
    __shared__ float red[DUAL ? 2 : 1][NW][16 * MB][17];
    __shared__ float sRow[INN ? NW : 1][16 * MB];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n = lane & 15, kg = lane >> 4;
    const int64_t b = blockIdx.z;
    const int n0 = blockIdx.x * 16;
    const int N = p.N, K = p.K;
    int M = (int)p.M;
    int64_t g0 = 0;      // this batch's first row among all rows, where the rows are dealt to the batches by group_off
    if (p.group_off) {
        g0 = p.group_off[b];
        M = min(M, p.group_off[b + 1] - (int)g0);
        if (M <= 0) return;
    }
    const int blocks = MB > 1 ? (M + 15) / 16 : 1;
    const bool cok = n0 + n < N;
    const uint16_t* pw = (const uint16_t*)p.W + b * p.w_batch + (int64_t)(cok ? n0 + n : 0) * K;
    const uint16_t* pw2 = pw + (int64_t)N * K;
    const float* pa[MB];
    bool rok[MB];
    float ssq[MB];
    dn_v4f acc[MB], acc2[DUAL ? MB : 1];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = i * 16 + n;
        rok[i] = m < M;
        const int64_t arow = rok[i] ? (p.a_rows ? (int64_t)p.a_rows[g0 + m] : g0 + m) : 0;
        pa[i] = p.A + b * p.a_batch + arow * p.lda;
        ssq[i] = 0.0f;
        acc[i] = dn_v4f{0, 0, 0, 0};
        acc2[DUAL ? i : 0] = dn_v4f{0, 0, 0, 0};
    }
    const int KT = (K + 31) / 32;
    for (int kt = wv; kt < KT; kt += U * NW) {      // the loads of U steps are requested before the first matrix instruction
        uint4 wf[U], wf2[U];
        float4 au[U][MB], av[U][MB], nu[INN ? U : 1], nv[INN ? U : 1];
#pragma unroll
        for (int h = 0; h < U; ++h) {
            const int k = (kt + h * NW) * 32 + kg * 8;
            const bool kin = kt + h * NW < KT && k < K;
            wf[h] = wf2[h] = make_uint4(0, 0, 0, 0);
            if (INN) {
                nu[INN ? h : 0] = kin ? *(const float4*)(p.in_norm_w + k) : make_float4(0, 0, 0, 0);
                nv[INN ? h : 0] = kin ? *(const float4*)(p.in_norm_w + k + 4) : make_float4(0, 0, 0, 0);
            }
            if (cok && kin) {
                wf[h] = *(const uint4*)(pw + k);
                if (DUAL) wf2[h] = *(const uint4*)(pw2 + k);
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                au[h][i] = av[h][i] = make_float4(0, 0, 0, 0);
                if (i < blocks && rok[i] && kin) {
                    au[h][i] = *(const float4*)(pa[i] + k);
                    av[h][i] = *(const float4*)(pa[i] + k + 4);
                }
            }
        }
#pragma unroll
        for (int h = 0; h < U; ++h)
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                if (i >= blocks) break;
                float4 u = au[h][i], v = av[h][i];
                if (INN) {
                    ssq[i] = fmaf(u.x, u.x, fmaf(u.y, u.y, fmaf(u.z, u.z, fmaf(u.w, u.w, ssq[i]))));
                    ssq[i] = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ssq[i]))));
                    u.x *= nu[INN ? h : 0].x, u.y *= nu[INN ? h : 0].y, u.z *= nu[INN ? h : 0].z, u.w *= nu[INN ? h : 0].w;
                    v.x *= nv[INN ? h : 0].x, v.y *= nv[INN ? h : 0].y, v.z *= nv[INN ? h : 0].z, v.w *= nv[INN ? h : 0].w;
                }
                const uint4 af = make_uint4(dn_bf16_pair(u.x, u.y), dn_bf16_pair(u.z, u.w), dn_bf16_pair(v.x, v.y), dn_bf16_pair(v.z, v.w));
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, af), __builtin_bit_cast(dn_v8bf, wf[h]), acc[i], 0, 0, 0);
                if (DUAL) acc2[DUAL ? i : 0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, af), __builtin_bit_cast(dn_v8bf, wf2[h]), acc2[DUAL ? i : 0], 0, 0, 0);
            }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            red[0][wv][i * 16 + kg * 4 + g][n] = acc[i][g];
            if (DUAL) red[DUAL ? 1 : 0][wv][i * 16 + kg * 4 + g][n] = acc2[DUAL ? i : 0][g];
        }
        if (INN) {      // lanes n, n + 16, n + 32, n + 48 hold shares of row n of a block
            float q = ssq[i];
            q += __shfl_xor(q, 16);
            q += __shfl_xor(q, 32);
            if (kg == 0) sRow[INN ? wv : 0][i * 16 + n] = q;
        }
    }
    __syncthreads();
    float* C = p.C + b * p.c_batch;
#pragma unroll
    for (int h = 0; h < (256 * MB + 64 * NW - 1) / (64 * NW); ++h) {
        const int m = (tid + h * 64 * NW) >> 4, c = tid & 15;
        if (m >= M || n0 + c >= N) continue;
        float s = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            s += red[0][w][m][c];
            if (DUAL) s2 += red[DUAL ? 1 : 0][w][m][c];
        }
        if (INN) {
            float q = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) q += sRow[INN ? w : 0][m];
            s *= 1.0f / sqrtf(q / (float)K + p.in_eps);
        }
        C[(g0 + m) * p.ldc + n0 + c] = dn_epilogue<EPI>(p, s, s2, b, g0 + m, n0 + c);
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void embed_scaled_kernel(const int64_t* __restrict__ ids, const uint16_t* __restrict__ table, float scale,
                                                           float* __restrict__ out, int W, int64_t V) {
    const int64_t t = blockIdx.x;
    int64_t id = ids[t];
    id = id < 0 ? 0 : (id >= V ? V - 1 : id);
    const uint16_t* row = table + id * W;
    for (int c = threadIdx.x; c < W; c += 256) out[t * W + c] = dn_bf16_to_f32(row[c]) * scale;
}

// ---------------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gated_postnorm_kernel(const i64h_postnorm p) {
    extern __shared__ float sv[];  // [W] the row before the norm, then [groups] root mean squares
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t m = blockIdx.x;
    const int W = p.W;
    const int64_t xr = p.x_rows ? (int64_t)p.x_rows[m] : m;
    const float* x = p.x + xr * W;
    for (int c = tid; c < W; c += 256) {
        float v = p.alpha * x[c];
        if (p.y) {
            float g = 1.0f;
            if (p.gate_pre) g = dn_sigmoid(p.gate_pre[m * p.ldg + c] + (p.gate_bias ? p.gate_bias[c] : 0.0f));
            v = v + g * p.y[m * p.ldy + c];
        }
        sv[c] = v;
    }
    __syncthreads();
    const int gs = W / p.groups;
    for (int g = wid; g < p.groups; g += 4) {
        float s = 0.0f;
        for (int c = lane; c < gs; c += 64) {
            const float v = sv[g * gs + c];
            s += v * v;
        }
        s = wave_sum(s);
        if (lane == 0) sv[W + g] = sqrtf(s / (float)gs + p.eps);
    }
    __syncthreads();
    const int64_t plane = p.n * (int64_t)W;
    if ((W & 3) == 0 && ((uintptr_t)p.norm_w & 15) == 0 && ((uintptr_t)p.out & 15) == 0 && ((uintptr_t)p.hist & 15) == 0 && ((uintptr_t)p.mix_out & 15) == 0 &&
        gs % 4 == 0) {
        // four columns per thread and 16-byte accesses; the history planes are read four at a time (independent loads in flight)
        for (int c = tid * 4; c < W; c += 1024) {
            const float den = sv[W + c / gs];
            const float4 nw = *(const float4*)(p.norm_w + c);
            float4 o;
            o.x = sv[c] / den * nw.x; o.y = sv[c + 1] / den * nw.y; o.z = sv[c + 2] / den * nw.z; o.w = sv[c + 3] / den * nw.w;
            if (p.out) *(float4*)(p.out + m * W + c) = o;
            if (p.mix_w) {
                const float* h = p.hist + m * W + c;
                *(float4*)(p.hist + p.hist_index * plane + m * W + c) = o;
                float4 a = make_float4(0, 0, 0, 0);
                int j = 0;
                for (; j + 4 <= p.hist_index; j += 4) {
                    float4 v[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = *(const float4*)(h + (j + u) * plane);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float wj = p.mix_w[j + u];
                        a.x += wj * v[u].x; a.y += wj * v[u].y; a.z += wj * v[u].z; a.w += wj * v[u].w;
                    }
                }
                for (; j < p.hist_index; ++j) {
                    const float4 v = *(const float4*)(h + j * plane);
                    const float wj = p.mix_w[j];
                    a.x += wj * v.x; a.y += wj * v.y; a.z += wj * v.z; a.w += wj * v.w;
                }
                const float wl = p.mix_w[p.hist_index];
                a.x += wl * o.x; a.y += wl * o.y; a.z += wl * o.z; a.w += wl * o.w;
                *(float4*)(p.mix_out + m * W + c) = a;
            }
        }
        return;
    }
    for (int c = tid; c < W; c += 256) {
        const float o = sv[c] / sv[W + c / gs] * p.norm_w[c];
        if (p.out) p.out[m * W + c] = o;
        if (p.mix_w) {
            p.hist[p.hist_index * plane + m * W + c] = o;
            float a = 0.0f;
            for (int j = 0; j < p.hist_index; ++j) a += p.mix_w[j] * p.hist[j * plane + m * W + c];
            a += p.mix_w[p.hist_index] * o;
            p.mix_out[m * W + c] = a;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
// One workgroup per row.  Thresholds are found by bisection over the bits of the order-preserving integer image of a float:
// top-k: the largest key with at least k values at or above it; top-p: the largest key whose values at or above it hold at
// least p of the mass.  The draw takes the first kept value, in index order, behind which the running sum exceeds u of the total.
//
// What bounds it is the chain of dependent sums, one per bit, so each is made short.  With top-k of at most half as many as there are threads the row
// is read once: a bound that at least k of the threads' maxima reach and few others do is found by one wave that holds them all, the values above it
// (at most one a thread, sorted by index) lie one to a thread from there on - and up to 128 of them in one wave, whose sums need no barrier.  Without
// top-k the row's keys and weights stay in registers (NV float4 per thread; NV = 0: read again, vocabularies beyond 32768).  64 rows of 32000, top-k 50 and
// top-p 0.95: 1280 us with four waves that read the row again for every bit, 33 us with sixteen and a barrier a bit, 15.3 with one wave's sums.  Without
// top-k, top-p 0.9, 45.8 us with a maximum and its index looked for together, 54 where the weights were taken again for every bit, 42.8; rows of
// 50257 drawn without either 56, 71 (read once more for a NaN and again for the maximum's place), 53.  Up to 4096
// values four waves have the shorter sums: 64 rows of 1000 drawn without top-k 11 us, sixteen waves 16, rows of 4000 13 and 17.
template <int NV, int SR_WAVES>
__global__ __launch_bounds__(64 * SR_WAVES) void sample_rows_kernel(const float* __restrict__ logits, int64_t* __restrict__ out, int V, const int vec,
                                                                 const float* __restrict__ temperature, const int32_t* __restrict__ top_k,
                                                                 const float* __restrict__ top_p, const float* __restrict__ u) {
    constexpr int SR_THREADS = 64 * SR_WAVES, SR_LIST = SR_THREADS, SR_TOPK = SR_LIST / 2;
    __shared__ float redf[2][SR_WAVES];
    __shared__ int redi[2][SR_WAVES];
    __shared__ uint32_t lkey[SR_LIST], skey[SR_LIST], svalue[128];
    __shared__ int lidx[SR_LIST], sidx[SR_LIST];
    __shared__ int listed, chosen, sarg;
    __shared__ uint32_t sbound;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t r = blockIdx.x;
    const float* x = logits + r * V;
    int turn = 0;      // the sums alternate between two buffers: one barrier each
    auto sum_i = [&](int v) {      // v: a wave's share, the same in all of its lanes
        if (lane == 0) redi[turn & 1][wid] = v;
        __syncthreads();
        int s = 0;
#pragma unroll
        for (int w = 0; w < SR_WAVES; ++w) s += redi[turn & 1][w];
        ++turn;
        return s;
    };
    auto sum_f = [&](float v) {      // v: a thread's share
        v = wave_sum(v);
        if (lane == 0) redf[turn & 1][wid] = v;
        __syncthreads();
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < SR_WAVES; ++w) s += redf[turn & 1][w];
        ++turn;
        return s;
    };
    auto wave_count = [&](bool b) { return __popcll(__ballot(b)); };
    constexpr int STEP = 4 * SR_THREADS;
    const int chunks = (V + STEP - 1) / STEP;
    auto load4 = [&](int i, uint32_t* k) {      // the keys of four neighbouring values; past the end 0, which no number has
        const int c = i * STEP + tid * 4;
        if (vec && c + 4 <= V) {
            const float4 v = *(const float4*)(x + c);
            k[0] = f32_to_ordered(v.x), k[1] = f32_to_ordered(v.y), k[2] = f32_to_ordered(v.z), k[3] = f32_to_ordered(v.w);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) k[j] = c + j < V ? f32_to_ordered(x[c + j]) : 0u;
        }
    };
    uint32_t key[NV > 0 ? NV : 1][4];
    // the largest number (kbest: its key, of what is no NaN; 0: none) and the largest key; where the first value that large lies is looked up behind them
    constexpr uint32_t KINF = 0xff800000u, KNINF = 0x007fffffu;      // the keys of the infinities: beyond them lie the NaNs
    uint32_t kmax = 0, kbest = 0, kmin = ~0u;      // (NV = 0: the smallest key too, and the chunk of the first value that large)
    int where = 0;
    auto lowest = [&](int i, const uint32_t* q) {
        if (i < V / STEP) kmin = min(min(min(q[0], q[1]), min(q[2], q[3])), kmin);
        else
#pragma unroll
            for (int j = 0; j < 4; ++j) kmin = i * STEP + tid * 4 + j < V ? min(kmin, q[j]) : kmin;
    };
    auto look = [&](int i, const uint32_t* k) {
        const uint32_t front = kbest;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            kmax = max(kmax, k[j]);
            kbest = max(kbest, k[j] <= KINF ? k[j] : 0u);
        }
        if (NV == 0 && kbest != front && !(kbest == 0x80000000u && front == 0x7fffffffu)) where = i;
    };
    if (NV > 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) load4(i, key[i]);
#pragma unroll
        for (int i = 0; i < NV; ++i) look(i, key[i]);
    } else {
        for (int i = 0; i < chunks; ++i) {
            load4(i, key[0]);
            look(i, key[0]);
            lowest(i, key[0]);
        }
    }
    auto max16 = [](uint32_t v) {      // over sixteen neighbouring lanes
        v = max(v, __float_as_uint(I64H_DPPF(__uint_as_float(v), 0x128)));
        v = max(v, __float_as_uint(I64H_DPPF(__uint_as_float(v), 0x124)));
        v = max(v, __float_as_uint(I64H_DPPF(__uint_as_float(v), 0x4E)));
        return max(v, __float_as_uint(I64H_DPPF(__uint_as_float(v), 0xB1)));
    };
    auto max64 = [&](uint32_t v) {
        v = max16(v);
        const uint32_t a = max((uint32_t)__builtin_amdgcn_readlane((int)v, 0), (uint32_t)__builtin_amdgcn_readlane((int)v, 16));
        const uint32_t b = max((uint32_t)__builtin_amdgcn_readlane((int)v, 32), (uint32_t)__builtin_amdgcn_readlane((int)v, 48));
        return max(a, b);
    };
    const uint32_t wbest = max64(kbest), wmax = max64(kmax);
    if (lane == 0) skey[wid] = wbest, skey[SR_WAVES + wid] = wmax;
    lkey[tid] = kmax;
    if (tid == 0) listed = 0, chosen = V, sarg = V;
    __syncthreads();
    static_assert(SR_WAVES <= 16, "");
    const uint32_t rbest = (uint32_t)__builtin_amdgcn_readfirstlane((int)max16(skey[lane & (SR_WAVES - 1)]));
    const uint32_t rmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)max16(skey[SR_WAVES + (lane & (SR_WAVES - 1))]));
    // (two zeros are equal, their keys are not: the first of either)
    const uint32_t twin = rbest == 0x80000000u ? rbest - 1 : rbest;
    if (rbest >= KNINF && kbest >= rbest - 1) {      // (a few threads)
        int first = V;
        auto find4 = [&](int i, const uint32_t* k) {
#pragma unroll
            for (int j = 3; j >= 0; --j) first = k[j] == rbest || k[j] == twin ? i * STEP + tid * 4 + j : first;
        };
        if (NV > 0) {
#pragma unroll
            for (int i = NV - 1; i >= 0; --i) find4(i, key[i]);
        } else {
            load4(where, key[0]);
            find4(where, key[0]);
        }
        if (first < V) atomicMin(&sarg, first);
    }
    __syncthreads();
    const int arg = sarg < V ? sarg : 0;
    const float best = rbest >= KNINF ? ordered_to_f32(rbest) : -INFINITY;      // (nothing but NaNs: token 0)
    const float T = temperature ? temperature[r] : 0.0f;
    if (!(T > 0.0f) || (u && u[r] < 0.0f)) {
        if (tid == 0) out[r] = arg;
        return;
    }
    const float invT = 1.0f / T, mx = best, pp = top_p ? top_p[r] : 1.0f, uu = u ? u[r] : 0.5f;
    const int k = top_k ? top_k[r] : 0;
    auto weight = [&](uint32_t q) { return expf((ordered_to_f32(q) - mx) * invT); };
    // the largest key that `enough` holds for, bit by bit; keys above every value of the row hold nothing
    auto bisect = [&](auto enough) {
        uint32_t thr = 0;
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = thr | (1u << bit);
            if (cand > rmax) continue;
            const int e = enough(cand);
            if (e) thr = cand;
            if (e > 1) break;      // exactly what was asked for: lower bits exclude nothing more
        }
        return thr;
    };
    if (k > 0 && k < V && k <= SR_TOPK) {
        // a key that at least k of the threads' maxima reach and no more than k or a wave's width: one wave looks for it, without a barrier a bit
        if (wid == 0) {
            uint32_t mine[SR_WAVES];
#pragma unroll
            for (int w = 0; w < SR_WAVES; ++w) mine[w] = lkey[w * 64 + lane];
            const int most = max(k, 64);
            const uint32_t found = bisect([&](uint32_t cand) {
                int n = 0;
#pragma unroll
                for (int w = 0; w < SR_WAVES; ++w) n += wave_count(mine[w] >= cand);
                return n < k ? 0 : (n <= most ? 2 : 1);
            });
            if (lane == 0) sbound = found;
        }
        __syncthreads();
        const uint32_t bound = sbound;
        auto list4 = [&](int i, const uint32_t* q) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (q[j] >= bound && i * STEP + tid * 4 + j < V) {
                    const int at = atomicAdd(&listed, 1);
                    if (at < SR_LIST) lkey[at] = q[j], lidx[at] = i * STEP + tid * 4 + j;
                }
        };
        if (NV > 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) list4(i, key[i]);
        } else {
            for (int i = 0; i < chunks; ++i) {
                load4(i, key[0]);
                list4(i, key[0]);
            }
        }
        __syncthreads();
        const int n = listed;
        // One wave holds up to 128 of them, one or two a lane, and needs no barrier.  Sorted by index (the order of the sums, which are added as those of two waves
        // are below) and by value: the k-th largest is top-k's bound, and top-p's lies at one of the values, found in as many sums as their number has bits.
        auto few = [&](auto per) {
            constexpr int PER = decltype(per)::value;
            int c[PER], at[PER] = {}, above[PER] = {};
            uint32_t q[PER];
            float w[PER], run[PER], total[PER], sum = 0.0f;
#pragma unroll
            for (int h = 0; h < PER; ++h) {
                const bool mine = h * 64 + lane < n;
                c[h] = mine ? lidx[h * 64 + lane] : V;
                q[h] = mine ? lkey[h * 64 + lane] : 0u;
            }
#pragma unroll
            for (int g = 0; g < PER; ++g)
                for (int j = 0; j < min(n - g * 64, 64); ++j) {
                    const int oc = __builtin_amdgcn_readlane(c[g], j);
                    const uint32_t oq = (uint32_t)__builtin_amdgcn_readlane((int)q[g], j);
#pragma unroll
                    for (int h = 0; h < PER; ++h) {
                        const bool front = oc < c[h];
                        at[h] += front ? 1 : 0;
                        above[h] += oq > q[h] || (oq == q[h] && front) ? 1 : 0;
                    }
                }
#pragma unroll
            for (int h = 0; h < PER; ++h)
                if (h * 64 + lane < n) skey[at[h]] = q[h], sidx[at[h]] = c[h], svalue[above[h]] = q[h];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            uint32_t thr = svalue[k - 1];
#pragma unroll
            for (int h = 0; h < PER; ++h) {
                q[h] = h * 64 + lane < n ? skey[h * 64 + lane] : 0u;      // (0: past the end; no bound is that low)
                w[h] = h * 64 + lane < n ? weight(q[h]) : 0.0f;
            }
            auto mass = [&](uint32_t cut) {
                float s = 0.0f;
#pragma unroll
                for (int h = 0; h < PER; ++h) s += wave_sum(h * 64 + lane < n && q[h] >= cut ? w[h] : 0.0f);
                return s;
            };
            if (pp < 1.0f) {
                const float need = pp * mass(thr);
                if (!(need > 0.0f)) {      // nothing is asked for (or the sum is no number): the most likely token
                    if (lane == 0) out[r] = arg;
                    return;
                }
                int lo = 0, hi = 0;      // the first place of the values in descending order whose values at or above it hold enough: in [lo, hi]
#pragma unroll
                for (int h = 0; h < PER; ++h) hi += wave_count(h * 64 + lane < n && q[h] >= thr);
                --hi;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (mass(svalue[mid]) >= need) hi = mid;
                    else lo = mid + 1;
                }
                thr = svalue[lo];
            }
#pragma unroll
            for (int h = 0; h < PER; ++h) {      // running sums in index order
                run[h] = h * 64 + lane < n && q[h] >= thr ? w[h] : 0.0f;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const float up = __shfl_up(run[h], d);
                    run[h] += lane >= d ? up : 0.0f;
                }
                total[h] = __shfl(run[h], 63);
                sum += total[h];
            }
            int pick = -1;
            float before = 0.0f;
#pragma unroll
            for (int h = 0; h < PER; ++h) {
                const unsigned long long past = __ballot(h * 64 + lane < n && q[h] >= thr && before + run[h] > uu * sum);
                if (pick < 0 && past) pick = sidx[h * 64 + __ffsll(past) - 1];
                before += total[h];
            }
            if (lane == 0) out[r] = pick >= 0 ? pick : arg;  // rounding at the far end of the walk: the most likely token
        };
        if (n <= 128) {
            if (wid > 0) return;
            if (n <= 64) few(std::integral_constant<int, 1>{});
            else few(std::integral_constant<int, 2>{});
            return;
        }
        if (n <= SR_LIST) {
            if (tid < n) {
                const int c = lidx[tid];
                int at = 0;
                for (int j = 0; j < n; ++j) at += lidx[j] < c ? 1 : 0;
                skey[at] = lkey[tid];
                sidx[at] = c;
            }
            __syncthreads();
            const uint32_t q = tid < n ? skey[tid] : 0u;
            uint32_t thr = bisect([&](uint32_t cand) {
                const int m = sum_i(wave_count(q >= cand));
                return m == k ? 2 : (m > k ? 1 : 0);
            });
            const bool mine = tid < n;
            const float w = mine ? weight(q) : 0.0f;
            if (pp < 1.0f) {
                const float need = pp * sum_f(mine && q >= thr ? w : 0.0f);
                if (!(need > 0.0f)) {      // nothing is asked for (or the sum is no number): the most likely token
                    if (tid == 0) out[r] = arg;
                    return;
                }
                const uint32_t t2 = bisect([&](uint32_t cand) { return sum_f(mine && q >= max(cand, thr) ? w : 0.0f) >= need ? 1 : 0; });
                thr = max(thr, t2);
            }
            // running sums in index order: within the wave, then over the waves in front
            float run = mine && q >= thr ? w : 0.0f;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const float up = __shfl_up(run, d);
                run += lane >= d ? up : 0.0f;
            }
            if (lane == 63) redf[turn & 1][wid] = run;
            __syncthreads();
            float before = 0.0f, total = 0.0f;
#pragma unroll
            for (int v = 0; v < SR_WAVES; ++v) {
                if (v == wid) before = total;
                total += redf[turn & 1][v];
            }
            if (mine && q >= thr && before + run > uu * total) atomicMin(&chosen, sidx[tid]);
            __syncthreads();
            if (tid == 0) out[r] = chosen < V ? chosen : arg;  // rounding at the far end of the walk: the most likely token
            return;
        }
    }
    // the row as a whole
    auto each = [&](auto f) {      // f(chunk, four keys)
        if (NV > 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) f(i, key[i]);
        } else {
            for (int i = 0; i < chunks; ++i) {
                load4(i, key[0]);
                f(i, key[0]);
            }
        }
    };
    uint32_t thr = 0;
    if (k > 0 && k < V)
        thr = bisect([&](uint32_t cand) {
            int n = 0;
            each([&](int, const uint32_t* q) {
#pragma unroll
                for (int j = 0; j < 4; ++j) n += wave_count(q[j] >= cand);
            });
            n = sum_i(n);
            return n == k ? 2 : (n > k ? 1 : 0);
        });
    if (thr == 0u) {      // the NaN of all bits set is kept: the sum is no number
        if (NV > 0)
#pragma unroll
            for (int i = 0; i < NV; ++i) lowest(i, key[i]);
        if (sum_i(wave_count(kmin == 0u)) > 0) {
            if (tid == 0) out[r] = arg;
            return;
        }
    }
    thr = max(thr, 1u);      // (0: the places past the end)
    // (NV > 0: the weights beside their keys: left to the compiler they were taken again for every bit, a branch around each)
    float held[NV > 0 ? NV : 1][4];
    if (NV > 0)
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) held[i][j] = weight(key[i][j]);
    auto weight_of = [&](int i, int j, uint32_t q) { return NV > 0 ? held[i][j] : weight(q); };
    auto mass = [&](uint32_t cut) {
        float s = 0.0f;
        each([&](int i, const uint32_t* q) {
#pragma unroll
            for (int j = 0; j < 4; ++j) s += q[j] >= cut ? weight_of(i, j, q[j]) : 0.0f;
        });
        return sum_f(s);
    };
    if (pp < 1.0f) {
        const float need = pp * mass(thr);
        if (!(need > 0.0f)) {
            if (tid == 0) out[r] = arg;
            return;
        }
        const uint32_t t2 = bisect([&](uint32_t cand) { return mass(max(cand, thr)) >= need ? 1 : 0; });
        thr = max(thr, t2);
    }
    const float target = uu * mass(thr);
    // 4096 values at a time until the running sum passes the target, then inside that stretch
    float base = 0.0f;
    bool open = true;
    each([&](int i, const uint32_t* q) {
        if (!open || i >= chunks) return;
        float w[4], s = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = q[j] >= thr ? weight_of(i, j, q[j]) : 0.0f, s += w[j];
        float run = s;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const float up = __shfl_up(run, d);
            run += lane >= d ? up : 0.0f;
        }
        if (lane == 63) redf[turn & 1][wid] = run;
        __syncthreads();
        float before = 0.0f, total = 0.0f;
#pragma unroll
        for (int v = 0; v < SR_WAVES; ++v) {
            if (v == wid) before = total;
            total += redf[turn & 1][v];
        }
        ++turn;
        if (base + total > target) {
            float a = base + (before + (run - s));
            int pick = V;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                a += w[j];
                if (pick == V && q[j] >= thr && a > target) pick = i * STEP + tid * 4 + j;
            }
            if (pick < V) atomicMin(&chosen, pick);
            open = false;
        }
        base += total;
    });
    __syncthreads();
    if (tid == 0) out[r] = chosen < V ? chosen : arg;
}

// ---------------------------------------------------------------------------------------------------------------------------
template <bool EXACT>
static void launch_tile(const i64h_linear& d, dim3 grid, hipStream_t s, int vecA, int vecW) {
    switch (d.epilogue) {
        case I64H_EPI_GELU_MUL: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_GELU_MUL>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_SILU_MUL: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_SILU_MUL>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_CLAMP_GLU: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_CLAMP_GLU>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_MUL_SIGMOID: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_MUL_SIGMOID>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_SOFTCAP: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_SOFTCAP>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_GELU_ERF: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_GELU_ERF>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_XIELU: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_XIELU>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_RELU_SQ: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_RELU_SQ>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_ADD: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_ADD>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_DECAY: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_DECAY>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_ROW_SIGMOID: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_ROW_SIGMOID>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_IN_NORM: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_IN_NORM>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        case I64H_EPI_SCALE: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_SCALE>), grid, dim3(256), 0, s, d, vecA, vecW); break;
        default: hipLaunchKernelGGL((linear_tile_kernel<EXACT, I64H_EPI_STORE>), grid, dim3(256), 0, s, d, vecA, vecW); break;
    }
}

template <int MB>
static void launch_rows_of(const i64h_linear& d, hipStream_t s) {
    const dim3 grid((unsigned)((d.N + 15) / 16), 1, (unsigned)d.batch);
#define DN_ROWS(E) case E: hipLaunchKernelGGL((linear_rows_kernel<E, MB>), grid, dim3(64 * dn_rows_waves(E, MB)), 0, s, d); break;
    switch (d.epilogue) {
        DN_ROWS(I64H_EPI_GELU_MUL) DN_ROWS(I64H_EPI_SILU_MUL) DN_ROWS(I64H_EPI_CLAMP_GLU) DN_ROWS(I64H_EPI_MUL_SIGMOID) DN_ROWS(I64H_EPI_SOFTCAP) DN_ROWS(I64H_EPI_GELU_ERF) DN_ROWS(I64H_EPI_XIELU) DN_ROWS(I64H_EPI_RELU_SQ)
        DN_ROWS(I64H_EPI_ADD) DN_ROWS(I64H_EPI_DECAY) DN_ROWS(I64H_EPI_ROW_SIGMOID) DN_ROWS(I64H_EPI_IN_NORM) DN_ROWS(I64H_EPI_SCALE)
        default: hipLaunchKernelGGL((linear_rows_kernel<I64H_EPI_STORE, MB>), grid, dim3(512), 0, s, d); break;
    }
#undef DN_ROWS
}
static void launch_rows(const i64h_linear& d, hipStream_t s) { d.M <= 16 ? launch_rows_of<1>(d, s) : launch_rows_of<4>(d, s); }

// Launches of few rows for linear_rows_kernel: those whose 16-column workgroups find a CU each (beyond, and with more rows over long k, linear_block_kernel
// has more of the weights on their way at a time), and rows dealt to experts whose weights are small or, with one or two tokens, whose few
// experts have no other way to spread theirs over the CUs.  Microseconds in replayed graphs, linear_block_kernel by size | here:
//    3 rows   1024 x 1024  6.1 | 4.3   33 x 4096  11.8 | 8.6    4096 x 2048  8.7 | 7.0   5760 x 1024  6.7 | 6.5   a pair of 1000 x 2752  14.9 | 9.8
//   16 rows   1024 x 1024  6.1 | 5.1   33 x 4096  11.8 | 12.9   4096 x 2048  8.7 | 8.7   5760 x 1024  6.7 | 8.6   a pair of 1000 x 2752  14.9 | 12.9
//   24 rows   1024 x 512  5.3 | 5.0   1024 x 1024  6.2 | 6.7    normed 1024 x 512  6.5 | 5.8   1024 x 1024  8.1 | 7.9
//   64 rows   1024 x 128  4.6 | 4.5   256 x 256  4.6 | 5.3      normed 1024 x 128  5.2 | 5.3   256 x 256  5.3 | 6.3
//   experts   8 of 1024 x 896, 3 tokens of two  7.3 | 4.4, 24 tokens  7.7 | 7.0, 64  1.09 times the other;  64 of pairs of 512 x 2048, 7 tokens of six  1.16 times;
//             32 of pairs of 256 x 512, 24 tokens of four  8.0 | 6.9;  4 of 256 x 128, 64 tokens of two  5.5 | 4.2
static bool rows_form(const i64h_linear& d) {
    const int64_t cols = (int64_t)d.N * d.batch, work = d.M * d.K;
    const bool dual = dn_dual(d.epilogue), normed = d.epilogue == I64H_EPI_IN_NORM;
    if (d.group_off) {
        if (d.M <= 16) return (d.rows_total > 0 && d.rows_total <= 4) || cols <= 16384;
        return cols <= 8192 && d.rows_total > 0 && d.rows_total * d.K <= (dual ? 5120 : 8960) * (int64_t)d.batch;
    }
    if (cols > 4096) return false;
    if (d.M <= 16) return dual || normed || work <= 49152;
    return !dual && (d.M <= 32 ? work <= (normed ? 20480 : 12288) : d.K <= 128);
}

static int g_skinny = 1, g_rows = 1, g_block = 1, g_form = -1;

extern "C" {

// tuning / test knob, bit 0: launches of at most I64H_SKINNY_ROWS rows on the weight-streaming kernel; bit 1: small launches of at most 64 rows on
// the fragment-streaming kernel; bit 2: all launches of at most 64 rows on it; bits 4 and up: one more than the form of linear_block_kernel to take whatever the size (default 3;
// 0 = every launch on the 64 x 64 tile kernel)
int i64h_set_linear_skinny(int32_t on) {
    g_skinny = on & 1;
    g_rows = on & 4 ? 2 : (on >> 1) & 1;
    g_block = on != 0;
    g_form = (on >> 4) - 1;
    return 0;
}

int i64h_linear_form(const i64h_linear* d) {
    return d && d->M > 0 && d->N > 0 && d->K > 0 && d->batch > 0 ? dn_linear_wide_form(*d) : -1;
}

int i64h_linear_run(const i64h_linear* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "linear: no descriptor");
    const i64h_linear& d = *dp;
    I64H_CHECK_ARG(d.M >= 0 && d.N > 0 && d.K > 0 && d.batch > 0, "linear: bad sizes M=%lld N=%d K=%d batch=%d", (long long)d.M, d.N, d.K, d.batch);
    I64H_CHECK_ARG((d.A || d.A16) && d.W && (d.C || (d.A16 && d.C16)), "linear: null operand");
    I64H_CHECK_ARG(d.epilogue >= 0 && d.epilogue <= I64H_EPI_IN_NORM, "linear: epilogue %d", d.epilogue);
    I64H_CHECK_ARG((d.epilogue != I64H_EPI_MUL_SIGMOID && d.epilogue != I64H_EPI_ADD && d.epilogue != I64H_EPI_DECAY && d.epilogue != I64H_EPI_ROW_SIGMOID) || d.E, "linear: epilogue %d needs E", d.epilogue);
    I64H_CHECK_ARG(d.epilogue != I64H_EPI_CLAMP_GLU || d.act_b > 0.0f, "linear: bound %g of the clamped gate / up epilogue", (double)d.act_b);
    I64H_CHECK_ARG(d.epilogue != I64H_EPI_SOFTCAP || d.softcap > 0.0f, "linear: soft cap %g", (double)d.softcap);
    I64H_CHECK_ARG(!dn_dual(d.epilogue) || !d.bias, "linear: the gate / up epilogues take no bias");
    I64H_CHECK_ARG((d.epilogue == I64H_EPI_IN_NORM) == (d.in_norm_w != nullptr), "linear: the normed input and its weights come together");
    I64H_CHECK_ARG(dn_dual(d.epilogue) || !d.row_scale, "linear: row factors belong to the gate / up epilogues");
    I64H_CHECK_ARG(d.lda >= d.K || d.M <= 1, "linear: lda %lld < K %d", (long long)d.lda, d.K);
    I64H_CHECK_ARG(d.batch <= 65535 && (d.M + 63) / 64 <= 65535, "linear: grid too large");
    I64H_CHECK_ARG(d.A16 || !d.C16, "linear: results in bf16 belong to input rows in bf16");
    if (d.A16) {
        I64H_CHECK_ARG(!d.exact && (dn_dual(d.epilogue) || d.epilogue == I64H_EPI_STORE || d.epilogue == I64H_EPI_SCALE || d.epilogue == I64H_EPI_ADD || d.epilogue == I64H_EPI_ROW_SIGMOID),
                       "linear: input rows in bf16 with epilogue %d or 32-bit products", d.epilogue);
        I64H_CHECK_ARG(d.K % 64 == 0 && d.lda % 8 == 0 && d.a_batch % 8 == 0 && d.w_batch % 8 == 0 && ((uintptr_t)d.A16 | (uintptr_t)d.W) % 16 == 0,
                       "linear: input rows in bf16 need K a multiple of 64 (%d) and rows at 16 bytes", d.K);
        if (d.M == 0) return 0;
        I64H_CHECK_ARG(dn_linear_wide(d, g_form, (hipStream_t)stream), "linear: input rows in bf16 beyond 32-bit offsets");
        I64H_CHECK_LAUNCH();
        return 0;
    }
    if (d.M == 0) return 0;
    const int vecA = (uintptr_t)d.A % 16 == 0 && d.lda % 4 == 0 && d.a_batch % 4 == 0 && (uintptr_t)d.in_norm_w % 16 == 0;
    const int vecW = (uintptr_t)d.W % 16 == 0 && d.K % 8 == 0 && d.w_batch % 8 == 0;
    hipStream_t s = (hipStream_t)stream;
    const size_t lds = (size_t)d.M * d.K * 2;
    if (g_skinny && !d.group_off && !d.exact && d.M <= I64H_SKINNY_ROWS && vecA && vecW && lds <= 64 * 1024) {
        int cpb = 64;  // columns per workgroup: at least about two workgroups per CU, a wave takes four columns at a time
        while (cpb > 16 && (int64_t)((d.N + cpb - 1) / cpb) * d.batch < 512) cpb >>= 1;
        const dim3 grid((unsigned)((d.N + cpb - 1) / cpb), 1, (unsigned)d.batch);
        switch (d.epilogue) {
            case I64H_EPI_GELU_MUL: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_GELU_MUL>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_SILU_MUL: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_SILU_MUL>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_CLAMP_GLU: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_CLAMP_GLU>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_MUL_SIGMOID: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_MUL_SIGMOID>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_SOFTCAP: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_SOFTCAP>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_GELU_ERF: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_GELU_ERF>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_XIELU: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_XIELU>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_RELU_SQ: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_RELU_SQ>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_ADD: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_ADD>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_DECAY: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_DECAY>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_ROW_SIGMOID: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_ROW_SIGMOID>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_IN_NORM: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_IN_NORM>), grid, dim3(256), lds, s, d, cpb); break;
            case I64H_EPI_SCALE: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_SCALE>), grid, dim3(256), lds, s, d, cpb); break;
            default: hipLaunchKernelGGL((linear_skinny_kernel<I64H_EPI_STORE>), grid, dim3(256), lds, s, d, cpb); break;
        }
        I64H_CHECK_LAUNCH();
        return 0;
    }
    const bool rows_ok = g_rows && !d.exact && d.M <= 64 && vecA && vecW;
    if (rows_ok && (g_rows > 1 || rows_form(d))) {
        launch_rows(d, s);
        I64H_CHECK_LAUNCH();
        return 0;
    }
    if (g_block && vecA && vecW && dn_linear_block(d, g_form, s)) {
        I64H_CHECK_LAUNCH();
        return 0;
    }
    // operands beyond 32-bit offsets (gathered rows of a matrix of 4 GiB or of unknown height): eight rows under 32000 x 2048 36 us, there 56; 16 rows 46 and 47
    if (rows_ok && d.M <= 8) {
        launch_rows(d, s);
        I64H_CHECK_LAUNCH();
        return 0;
    }
    const dim3 grid((unsigned)((d.N + 63) / 64), (unsigned)((d.M + 63) / 64), (unsigned)d.batch);
    if (d.exact) launch_tile<true>(d, grid, s, vecA, vecW);
    else launch_tile<false>(d, grid, s, vecA, vecW);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_embed_scaled(const int64_t* ids, const void* table_bf16, float scale, float* out, int64_t n, int32_t W, int64_t V, void* stream) {
    I64H_CHECK_ARG(n >= 0 && W > 0 && V > 0, "embed_scaled: bad sizes");
    if (n == 0) return 0;
    hipLaunchKernelGGL(embed_scaled_kernel, dim3((unsigned)n), dim3(256), 0, (hipStream_t)stream, ids, (const uint16_t*)table_bf16, scale, out,
                       (int)W, V);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_gated_postnorm(const i64h_postnorm* dp, void* stream) {
    I64H_CHECK_ARG(dp != nullptr, "gated_postnorm: no descriptor");
    const i64h_postnorm& d = *dp;
    I64H_CHECK_ARG(d.n >= 0 && d.W > 0 && d.groups > 0 && d.W % d.groups == 0, "gated_postnorm: W %d does not split into %d groups", d.W, d.groups);
    I64H_CHECK_ARG(d.x && d.norm_w, "gated_postnorm: null operand");
    I64H_CHECK_ARG(!d.mix_w || (d.hist && d.mix_out && d.hist_index >= 0), "gated_postnorm: the depth mix needs hist and mix_out");
    I64H_CHECK_ARG(d.out || d.mix_w, "gated_postnorm: no output");
    const size_t lds = ((size_t)d.W + d.groups) * 4;
    I64H_CHECK_ARG(lds <= 64 * 1024, "gated_postnorm: a row of %d values does not fit the kernel's LDS buffer", d.W);
    if (d.n == 0) return 0;
    hipLaunchKernelGGL(gated_postnorm_kernel, dim3((unsigned)d.n), dim3(256), lds, (hipStream_t)stream, d);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_sample_rows(const float* logits, int64_t* out, int64_t rows, int32_t V, const float* temperature, const int32_t* top_k,
                     const float* top_p, const float* u, void* stream) {
    I64H_CHECK_ARG(rows >= 0 && V > 0 && logits && out, "sample_rows: bad arguments");
    if (rows == 0) return 0;
    const int vec = (uintptr_t)logits % 16 == 0 && V % 4 == 0;
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](auto kern, int threads) { hipLaunchKernelGGL(kern, dim3((unsigned)rows), dim3(threads), 0, s, logits, out, (int)V, vec, temperature, top_k, top_p, u); };
    if (V <= 4096) launch(sample_rows_kernel<4, 4>, 256);
    else if (V <= 32768) launch(sample_rows_kernel<8, 16>, 1024);
    else launch(sample_rows_kernel<0, 16>, 1024);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
