// C = epilogue(A W^T), A fp32, W bf16 [N, K], on v_mfma_f32_16x16x32_bf16 (A rounded to bf16 while it is staged, or in three parts for 32-bit products): BM x BN tiles staged
// through LDS, four waves a tile and KG groups of four waves that share a tile's k steps.
//
// What bounds it.  Large launches: the step from memory to LDS - A is read as 32-bit values and rounded on the way, so a 128 x 128 tile moves
// 48 KiB a step for 512 cycles of matrix instructions; hence 128 x 128 before anything smaller, two steps of registers on their way, the
// next step's LDS writes between this step's matrix instructions (2956 x 11008 x 2048: 247 us with one step ahead, 224 with two, 199 with the
// writes interleaved; the 64 x 64 kernel with 32-wide steps that this one replaces: 360 us, 370 TFLOP/s against 670).  Small launches: the
// latency of a load per step, hence groups that share the steps, their sums added in LDS in a fixed order (64 x 2048 x 2048: 19.6 us with
// fragments straight from memory before, 15.1 with a group a tile, 8.3 with 16 x 64 tiles and four; 64 x 32000 x 2048, whose 131 MB take 28 us at
// the rate of a large copy: 133 -> 31 us).
#include "i64h_dense_dev.h"
#include <type_traits>

// EX: products of 32-bit rows.  W is bf16, so a row's value x = hi + mid + lo, three bf16 of eight bits each cut off in turn, makes x w the sum of three products that the bf16
// instruction takes exactly, summed in 32 bits: three instructions in the place of eight v_mfma_f32_16x16x4_f32 of twice their length.  (lo and mid first.)
template <int EPI, int BM, int BN, int KG, bool EX>
__global__ __launch_bounds__(256 * KG, KG == 1 ? 2 : KG) void linear_block_kernel(const i64h_linear p, const int n_tiles, const int m_tiles, const int vecC) {
    constexpr bool DUAL = dn_dual(EPI), INN = EPI == I64H_EPI_IN_NORM;
    constexpr int BK = 64, CH = 8, PARTS = EX ? 3 : 1;      // values of a step, of a thread's chunk; bf16 rows a staged row of A becomes
    constexpr int NWM = BM >= 64 ? 2 : 1, NWN = 4 / NWM;      // waves of a group over rows and columns
    constexpr int WM = BM / NWM, WN = BN / NWN, FM = WM / 16, FN = WN / 16;
    static_assert(FM > 0 && FN > (DUAL ? 1 : 0), "");
    constexpr int PA = (BM + 31) / 32, PB = BN / 32;       // staging passes: 32 rows of 64 values, 8 values a thread
    constexpr int COLS = DUAL ? BN / 2 : BN;               // output columns of a tile
    constexpr int PLANE = (PARTS * BM + BN) * 64;          // (in 16-bit units)
    // [buffer][group][A rows (EX: hi, mid, lo), W rows]; (variables of their own, so that the writes of one step may be scheduled between the reads of the other)
    __shared__ __attribute__((aligned(16))) uint16_t s0[KG * PLANE], s1[KG * PLANE];
    __shared__ float sRow[INN ? KG : 1][INN ? BM : 1];
    const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int tid = threadIdx.x & 255, lane = tid & 63, wid = tid >> 6, wm = wid / NWN, wn = wid % NWN;
    const int N = p.N, K = p.K;
    const dn_tile t = dn_find_tile<BM>(p, n_tiles, m_tiles, lane);
    if (!t.any) return;
    const int64_t b = t.b, g0 = t.g0, rows = t.rows;
    const int mt = t.mt, nt = t.nt;
    const int n0 = nt * COLS;
    const int64_t m0 = g0 + (int64_t)mt * BM;
    const int M = (int)min((int64_t)BM, rows - (int64_t)mt * BM);
    const int lr = tid >> 3, lc = tid & 7;                 // staging: row within a pass, chunk of eight k
    // (rows past the end repeat the last one and are not stored)
    const __amdgpu_buffer_rsrc_t bufA = dn_buffer(p.A + b * p.a_batch + (p.a_rows ? 0 : m0 * p.lda)), bufW = dn_buffer((const uint16_t*)p.W + b * p.w_batch + (int64_t)n0 * K);
    uint32_t oa[PA], ow[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int r = min(i * 32 + lr, M - 1);
        oa[i] = (uint32_t)((p.a_rows ? p.a_rows[m0 + r] : r) * p.lda + lc * CH) * 4u;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int r = i * 32 + lr;
        // gate and up rows of the same columns go to the same wave: its first half of fragments, its second half
        const int c = DUAL ? (r / WN) * (WN / 2) + r % (WN / 2) : r;
        ow[i] = (uint32_t)((int64_t)(min(c, N - 1 - n0) + (DUAL && r % WN >= WN / 2 ? N : 0)) * K + lc * CH) * 2u;
    }
    dn_v4u ra[2][PA][2], rb[2][PB], rn[2][2];      // two steps on their way
    float ssq[PA];
#pragma unroll
    for (int i = 0; i < PA; ++i) ssq[i] = 0.0f;
    // this group's steps: KT of them from k_base on, the last group's past the end of K reading zeros
    const int KT = ((K + BK - 1) / BK + KG - 1) / KG, k_base = grp * KT * BK, k_end = KG > 1 ? min(K, k_base + KT * BK) : K;
    auto gload = [&](int kt, auto set) {
        constexpr int S = decltype(set)::value;
        const int k0 = k_base + kt * BK;
        const uint32_t past = k0 + lc * CH >= k_end ? DN_BUF_END : 0u;      // (K is a multiple of eight)
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            ra[S][i][0] = dn_load16(bufA, oa[i] | past, k0 * 4);
            ra[S][i][1] = dn_load16(bufA, (oa[i] + 16) | past, k0 * 4);
        }
#pragma unroll
        for (int i = 0; i < PB; ++i) rb[S][i] = dn_load16(bufW, ow[i] | past, k0 * 2);
        if (INN) {
            const float* nw = p.in_norm_w + (past ? 0 : k0 + lc * CH);
            rn[S][0] = *(const dn_v4u*)nw;
            rn[S][1] = *(const dn_v4u*)(nw + 4);
        }
    };
    // 128-byte rows; a row's chunks are stored exclusive-or its number, so that the 16 rows of a fragment read lie in different banks
    auto lstore = [&](auto set) {      // into the buffer of the same number
        constexpr int S = decltype(set)::value;
        uint16_t* sm = (S ? s1 : s0) + grp * PLANE;
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            dn_v4f u = __builtin_bit_cast(dn_v4f, ra[S][i][0]), v = __builtin_bit_cast(dn_v4f, ra[S][i][1]);
            if (INN) {      // the row's squares as they come, the norm's weights on what is staged
                const dn_v4f nu = __builtin_bit_cast(dn_v4f, rn[S][0]), nv = __builtin_bit_cast(dn_v4f, rn[S][1]);
#pragma unroll
                for (int g = 0; g < 4; ++g) ssq[i] = fmaf(u[g], u[g], ssq[i]);
#pragma unroll
                for (int g = 0; g < 4; ++g) ssq[i] = fmaf(v[g], v[g], ssq[i]);
#pragma unroll
                for (int g = 0; g < 4; ++g) u[g] *= nu[g], v[g] *= nv[g];
            }
            const int r = i * 32 + lr, at = r * 64 + ((lc ^ (r & 7)) << 3);
            if constexpr (EX) {
                dn_v4u w[PARTS];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    uint32_t part[2][PARTS];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float x = g < 2 ? u[2 * g + e] : v[2 * g - 4 + e];
                        const float hi = __uint_as_float(__float_as_uint(x) & 0xffff0000u), rest = x == hi ? 0.0f : x - hi;      // (an infinity leaves none)
                        const float mid = __uint_as_float(__float_as_uint(rest) & 0xffff0000u);
                        part[e][0] = __float_as_uint(hi), part[e][1] = __float_as_uint(mid), part[e][2] = __float_as_uint(rest - mid);
                    }
#pragma unroll
                    for (int q = 0; q < PARTS; ++q) w[q][g] = __builtin_amdgcn_perm(part[1][q], part[0][q], 0x07060302u);      // the upper halves
                }
#pragma unroll
                for (int q = 0; q < PARTS; ++q)
                    if (BM >= 32 || lr < BM) *(dn_v4u*)&sm[q * BM * 64 + at] = w[q];
            } else {
                const dn_v4u w{dn_bf16_pair(u[0], u[1]), dn_bf16_pair(u[2], u[3]), dn_bf16_pair(v[0], v[1]), dn_bf16_pair(v[2], v[3])};
                if (BM >= 32 || lr < BM) *(dn_v4u*)&sm[at] = w;
            }
        }
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const int r = i * 32 + lr;
            *(dn_v4u*)&sm[(PARTS * BM + r) * 64 + ((lc ^ (r & 7)) << 3)] = rb[S][i];
        }
    };
    dn_v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = dn_v4f{0, 0, 0, 0};
    const int fr = lane & 15, fk = lane >> 4;
    auto multiply = [&](auto set) {
        constexpr int S = decltype(set)::value;
        const uint16_t* sm = (S ? s1 : s0) + grp * PLANE;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int ch = ((kk * 4 + fk) ^ (fr & 7)) << 3;
            dn_v4u a[PARTS][FM], w[FN];
#pragma unroll
            for (int q = 0; q < PARTS; ++q)
#pragma unroll
                for (int i = 0; i < FM; ++i) a[q][i] = *(const dn_v4u*)&sm[(q * BM + wm * WM + i * 16 + fr) * 64 + ch];
#pragma unroll
            for (int j = 0; j < FN; ++j) w[j] = *(const dn_v4u*)&sm[(PARTS * BM + wn * WN + j * 16 + fr) * 64 + ch];
#pragma unroll
            for (int q = PARTS - 1; q >= 0; --q)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, w[j]), __builtin_bit_cast(dn_v8bf, a[q][i]), acc[i][j], 0, 0, 0);
        }
    };
    // the next tile's writes and the loads behind it between the matrix instructions; small tiles are faster as the compiler orders them
    auto interleave = [&]() {
        if (EX || BN < 128 || BM < 64) return;
        constexpr int MF = 2 * FM * FN, DR = 2 * (FM + FN), DW = PA + PB, VM = 2 * PA + PB;
        __builtin_amdgcn_sched_group_barrier(0x100, DR / 2, 0);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, MF / 8, 0);
            if (g < 4) __builtin_amdgcn_sched_group_barrier(0x100, DR / 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, (DW + 7) / 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, (VM + 7) / 8, 0);
        }
    };
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    // a step's operands are requested two steps ahead (a workgroup alone on its CU waits for them otherwise), past the end as zeros
    gload(0, S0);
    gload(1, S1);
    lstore(S0);
    __syncthreads();
    for (int kt = 0; kt + 1 < KT; kt += 2) {
        gload(kt + 2, S0);
        multiply(S0);
        lstore(S1);
        interleave();
        __syncthreads();
        gload(kt + 3, S1);
        multiply(S1);
        lstore(S0);
        interleave();
        __syncthreads();
    }
    if (KT & 1) multiply(S0);
    if (INN) {      // eight neighbouring lanes hold a row's shares
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            float q = ssq[i];
            q += __shfl_xor(q, 1);
            q += __shfl_xor(q, 2);
            q += __shfl_xor(q, 4);
            if (lc == 0 && (BM >= 32 || lr < BM)) sRow[INN ? grp : 0][INN ? i * 32 + lr : 0] = q;
        }
        if (KG == 1) __syncthreads();
    }
    if (KG > 1) {      // the groups' sums meet in LDS, added in the groups' order by the first one
        constexpr int TILE = 4 * 64 * FM * FN;      // fragments of four values
        static_assert((KG - 1) * TILE * 16 <= 2 * KG * PLANE * 2, "");
        constexpr int HALF = (KG * PLANE * 2) / (TILE * 16);      // tiles that fit the first buffer
        __syncthreads();
        dn_v4f* dst = grp - 1 < HALF ? (dn_v4f*)s0 + (grp - 1) * TILE : (dn_v4f*)s1 + (grp - 1 - HALF) * TILE;
        if (grp > 0) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) dst[(i * FN + j) * 256 + tid] = acc[i][j];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 0; g < KG - 1; ++g) {
            const dn_v4f* src = g < HALF ? (const dn_v4f*)s0 + g * TILE : (const dn_v4f*)s1 + (g - HALF) * TILE;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] += src[(i * FN + j) * 256 + tid];
        }
    }
    // the weights are the left operand: a lane holds four neighbouring columns of a row
    // An infinite weight makes no number of a part that is zero: such sums are taken again term by term, unless the row itself holds what is no number.  376 x 5760 x 1024, us: 31; a row of NaN 30,
    // one at the end of a row 56, an infinite weight 85 (every such sum taken term by term 475, 476, 140).
    if constexpr (EX) {
        auto row = [&](int64_t rl) { return p.A + b * p.a_batch + (p.a_rows ? (int64_t)p.a_rows[m0 + rl] : m0 + rl) * p.lda; };
        auto again = [&](const float* x, int c) {      // (K is a multiple of eight)
            const uint16_t* w = (const uint16_t*)p.W + b * p.w_batch + (int64_t)c * K;
            float v = 0.0f;
            for (int k = 0; k < K && v == v; k += 8)
#pragma unroll
                for (int i = 0; i < 8; ++i) v = fmaf(INN ? x[k + i] * p.in_norm_w[k + i] : x[k + i], dn_bf16_to_f32(w[k + i]), v);
            return v;
        };
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int rl = wm * WM + i * 16 + fr;
            bool odd = false;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) odd |= acc[i][j][g] != acc[i][j][g];
            if (rl >= M || !odd) continue;
            const float* x = row(rl);
            bool lost = false;
            for (int k = 0; k < K && !lost; k += 8)
#pragma unroll
                for (int e = 0; e < 8; ++e) lost |= x[k + e] != x[k + e];
            if (lost) continue;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int c = n0 + wn * (COLS / NWN) + (DUAL ? j % (FN / 2) : j) * 16 + fk * 4;
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    if (c + g < N && acc[i][j][g] != acc[i][j][g]) acc[i][j][g] = again(x, c + g + (DUAL && j >= FN / 2 ? N : 0));
            }
        }
    }
    float* C = p.C + b * p.c_batch;
    // (a bias and factors of rows are asked for once, not at every value)
    i64h_linear q = p;
    q.bias = nullptr, q.row_scale = nullptr;
    float add[DUAL ? 1 : FN][4];
    if constexpr (!DUAL) {
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) add[j][g] = -0.0f;      // (changes no value, not even a zero's sign)
        if (p.bias) {
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) add[j][g] = p.bias[b * p.bias_batch + min(n0 + wn * (COLS / NWN) + j * 16 + fk * 4 + g, N - 1)];
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int rl = wm * WM + i * 16 + fr;
        if (rl >= M) continue;
        const int64_t r = m0 + rl;
        if (DUAL && p.row_scale) {
            const float factor = p.row_scale[r];
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] *= factor;
        }
        float f = 1.0f;
        if (INN) {
            float q = 0.0f;
#pragma unroll
            for (int g = 0; g < KG; ++g) q += sRow[INN ? g : 0][INN ? rl : 0];
            f = 1.0f / sqrtf(q / (float)K + p.in_eps);
        }
#pragma unroll
        for (int j = 0; j < (DUAL ? FN / 2 : FN); ++j) {
            const int c = n0 + wn * (COLS / NWN) + j * 16 + fk * 4;
            auto out = [&](int g) { return DUAL ? dn_epilogue<EPI>(q, acc[i][j][g], acc[i][DUAL ? j + FN / 2 : j][g], b, r, c + g) : dn_epilogue<EPI>(q, (INN ? acc[i][j][g] * f : acc[i][j][g]) + add[DUAL ? 0 : j][g], 0.0f, b, r, c + g); };
            float* dst = C + r * p.ldc + c;
            if (vecC && c + 4 <= N) {
                *(float4*)dst = make_float4(out(0), out(1), out(2), out(3));
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    if (c + g < N) dst[g] = out(g);
            }
        }
    }
}

enum { PLAIN = 1, PAIR = 2 };      // the epilogues that a form is built for: all but the gate / up pairs, those, both
template <int BM, int BN, int KG, int FOR = PLAIN | PAIR, bool EX = false>
static void launch(const i64h_linear& d, hipStream_t s) {
    const int cols = dn_dual(d.epilogue) ? BN / 2 : BN;
    const int nt = (d.N + cols - 1) / cols;
    int64_t mt = (d.M + BM - 1) / BM;
    if (d.group_off) {      // at most one partly filled row tile per batch beside the full ones
        const int64_t most = mt * d.batch;
        mt = d.rows_total > 0 ? (most < d.rows_total / BM + d.batch ? most : d.rows_total / BM + d.batch) : most;
    }
    const int vecC = (uintptr_t)d.C % 16 == 0 && d.ldc % 4 == 0 && d.c_batch % 4 == 0;
    const dim3 grid((unsigned)(mt * nt), 1, d.group_off ? 1u : (unsigned)d.batch);
#define DN_BLOCK(E) case E: if constexpr (FOR & (dn_dual(E) ? PAIR : PLAIN)) hipLaunchKernelGGL((linear_block_kernel<E, BM, BN, KG, EX>), grid, dim3(256 * KG), 0, s, d, nt, (int)mt, vecC); break;
    switch (d.epilogue) {
        DN_BLOCK(I64H_EPI_GELU_MUL) DN_BLOCK(I64H_EPI_SILU_MUL) DN_BLOCK(I64H_EPI_CLAMP_GLU) DN_BLOCK(I64H_EPI_MUL_SIGMOID) DN_BLOCK(I64H_EPI_SOFTCAP)
        DN_BLOCK(I64H_EPI_GELU_ERF) DN_BLOCK(I64H_EPI_XIELU) DN_BLOCK(I64H_EPI_RELU_SQ) DN_BLOCK(I64H_EPI_ADD) DN_BLOCK(I64H_EPI_DECAY) DN_BLOCK(I64H_EPI_ROW_SIGMOID)
        DN_BLOCK(I64H_EPI_IN_NORM) DN_BLOCK(I64H_EPI_SCALE)
        default: if constexpr (FOR & PLAIN) hipLaunchKernelGGL((linear_block_kernel<I64H_EPI_STORE, BM, BN, KG, EX>), grid, dim3(256 * KG), 0, s, d, nt, (int)mt, vecC); break;
    }
#undef DN_BLOCK
}

// Workgroups of a launch in BM x BN tiles (all columns of a gate / up pair count twice).
static int64_t tiles(const i64h_linear& d, int BM, int BN) {
    int64_t mt = (d.M + BM - 1) / BM * d.batch;
    if (d.group_off && d.rows_total > 0 && d.rows_total / BM + d.batch < mt) mt = d.rows_total / BM + d.batch;
    const int64_t cols = dn_dual(d.epilogue) ? 2 * (int64_t)d.N : d.N;
    return mt * ((cols + BN - 1) / BN);
}

bool dn_linear_block(const i64h_linear& d, int form, hipStream_t s) {
    const bool dual = dn_dual(d.epilogue);
    // the buffer descriptors' 32-bit offsets: rows of a tile, or whatever a_rows may name; the weights of a tile, of a pair from gate to up
    const int64_t span = (d.a_rows ? d.a_height : 128) * d.lda * 4;
    if ((d.a_rows && d.a_height <= 0) || span >= (int64_t)DN_BUF_END - 64 || ((dual ? (int64_t)d.N : 0) + 128) * 2 * d.K >= (int64_t)DN_BUF_END - 64) return false;
    if (tiles(d, 16, 64) > 0x7fffffff) return false;
    // rows that share a batch's weights: taller tiles would only repeat the last one
    const int64_t tall = d.group_off && d.rows_total > 0 ? (d.rows_total + d.batch - 1) / d.batch : d.M;
    // Short k and many tiles: two steps of registers and LDS on their way are little use, and the plainer kernel's smaller workgroups overlap their loads and
    // stores better.  Microseconds, here | there: 12000 x 4096 x 64 62 | 35, x 128 80 | 48, 4096 x 1024 x 128 11.1 | 9.7, 1000 x 4096 x 64 10.0 | 7.8, 320 x 4096 x 128 6.6 | 6.4, 1000 x
    // 1024 x 128 5.2 | 5.7 (a gate / up pair: 2048 x 4096 x 128 25.3 | 23.3, 1000 x 4096 15.2 | 13.5, 1000 x 1024 6.2 | 8.4).
    auto short_k = [&](int64_t many) { return (d.K <= 32 && !dual) || (d.K <= 128 && tiles(d, 64, 64) >= many); };
    if (d.exact) {
        // A third of the bf16 rate, and the parts are made while rows are staged (eight instructions a value), so a row is better staged for many columns; small launches are bound as those
        // of bf16 are.  Microseconds in replayed graphs, in front v_mfma_f32_16x16x4_f32 in the form that was best for it:
        //   rows x columns x k                 before   64x128  32x128/2  32x64  32x64/2  16x64/4  16x128/2 (a gate / up pair)
        //   4096 x 5760 x 1024                   368      172      250      211      234      531
        //    900 x 5760 x 1024                             49       66       55       58      123
        //    376 x 5760 x 1024                    53       33       36       29       29       55
        //   12000 x 4096 x 64                     92       84      197       64
        //    150 x 5760 x 1024                             23       13       15       14       26
        //    600 x 1024 x 2752                    50       48       26       31       28       34
        //    376 x 1024 x 1024                    14       22       12       11        9       13
        //     40 x 1024 x 1024                     9       21       12       11        9        7
        //      3 x 32000 x 1024                   16       20       14       14       14       17
        //   2000 x 2752 x 1024, pair             178       85      114                                 173
        //    376 x 2752 x 1024, pair              55       30       33                                  42
        //    100 x 2752 x 1024, pair              22       21       12                                  18
        //  8 x 25 x 896 x 1024, pair              26       22       13                                  11
        // Errors against 64 bits are 0.55 to 0.8 of what they were (376 x 5760 x 1024: 3.4e-7 of the result, 5.7e-7 before): fewer roundings of a sum.
        if (form < 0) {
            if (d.K < 64 && !dual) return false;      // (less than a step: 4096 x 1024 x 32 9.3, there 8.2; 512 rows 3.7 and 4.2)
            if (dual) form = tiles(d, 16, 128) <= (tall <= 32 ? 512 : 256) ? 6 : (tiles(d, 32, 128) <= 256 ? 7 : 2);
            else if (tiles(d, 16, 64) <= 256) form = 5;
            else if (tall <= 16 || tiles(d, 32, 64) <= 256) form = 4;
            else if (d.K >= 512 && tiles(d, 32, 128) <= 256) form = 7;
            else form = d.K < 512 || tiles(d, 64, 128) < 384 ? 1 : 2;
        }
        switch (form) {
            case 1: if (!dual) { launch<32, 64, 1, PLAIN, true>(d, s); break; } [[fallthrough]];
            case 4: if (!dual) { launch<32, 64, 2, PLAIN, true>(d, s); break; } [[fallthrough]];
            case 5: if (!dual) { launch<16, 64, 4, PLAIN, true>(d, s); break; } [[fallthrough]];
            case 6: if (dual) { launch<16, 128, 2, PAIR, true>(d, s); break; } [[fallthrough]];
            case 7: launch<32, 128, 2, PLAIN | PAIR, true>(d, s); break;
            default: launch<64, 128, 1, PLAIN | PAIR, true>(d, s); break;
        }
        return true;
    }
    if (form < 0) {
        // Large tiles as long as (nearly) every CU gets one: their operands are read least often.  Below that, a tile's k steps follow each
        // other at the latency of a load and what counts is how few of them a workgroup has and how many CUs work: four groups a tile
        // while its workgroups (one a CU, LDS) run in one round, two groups while there is a CU for each.  Microseconds in replayed graphs:
        //   rows x columns x k       128x128  64x128   64x64  64x64/2  32x64/4  16x64/4
        //   4096 x 5760 x 1024           98     110     133
        //   2000 x 1024 x 1024         18.8    13.7    13.6     14.4     24.0     34.8
        //    512 x 6464 x 2048         31.2    30.7    39.7     40.4     59.2     83.7
        //    512 x 2048 x 2048         28.3    21.3    16.8     13.9     18.2     27.2
        //    512 x 1024 x 1024         15.7    12.5     9.4      8.5      7.3     10.5
        //     64 x 11392 x 2048                        16.3     13.5     18.6     21.1
        //     64 x 2048 x 2048                         15.1     12.3      9.6      8.3
        // Few rows under weights that take longer than everything else: 32 x 128 tiles, two groups (8 experts of 16 rows x 3584 x 2048: 24.4 us, in 128
        // x 128 tiles 33, in 64 x 64 30; 7 x 32000 x 1024 12.7, 64x64 13.4).
        const bool longer = d.K > 128, wide = (dual ? 2 * (int64_t)d.N : d.N) > 64;      // (half of a 128-column tile would be idle)
        if (short_k(dual ? 2000 : 700)) return false;
        if (longer && wide && tall > 64 && tiles(d, 128, 128) >= 200) form = 0;
        else if (longer && wide && tall > 32 && tiles(d, 64, 128) >= 250) form = 1;
        else if (dual ? tiles(d, 16, 128) <= 256 : tiles(d, 16, 64) <= 256) form = dual ? 6 : 5;
        else if (!dual && d.K >= 512 && tiles(d, 32, 64) <= 256) form = 4;
        else if (d.K >= 512 && wide && tall <= 32) form = 7;
        else if (d.K >= 512 && tiles(d, 64, 64) <= 256) form = 3;
        else form = 2;
    }
    switch (form) {
        case 0: launch<128, 128, 1>(d, s); break;
        case 1: launch<64, 128, 1>(d, s); break;
        case 7: launch<32, 128, 2>(d, s); break;
        case 3: launch<64, 64, 2>(d, s); break;
        case 4: if (!dual) { launch<32, 64, 4, PLAIN>(d, s); break; } [[fallthrough]];
        case 5: if (!dual) { launch<16, 64, 4, PLAIN>(d, s); break; } [[fallthrough]];
        case 6: if (dual) { launch<16, 128, 2, PAIR>(d, s); break; } [[fallthrough]];      // 64 columns of a gate / up pair: 64 x 1792 x 2048 15.0 us, 64x64/2 17.5
        default: launch<64, 64, 1>(d, s); break;
    }
    return true;
}
