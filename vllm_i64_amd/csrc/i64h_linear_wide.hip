// C = epilogue(A W^T) with both operands in bf16 (i64h_linear's A16): the products of linear_block_kernel on rows that their producer rounded once
// instead of every tile that reads them, summed in the order of k.
//
// What bounds it.  Large launches: the matrix instructions and, at k of 1024, a round's stores.  The kernel that rounds while it stages moved 48 KiB
// a step of a 128 x 128 tile through registers; here 32 KiB go from memory to LDS by themselves, a wave's registers hold fragments alone and the
// reads of one half step lie under the products of the other.  Small launches: the latency of a step, hence three or four steps on their way where a
// stage is small enough (512 x 2048 x 5504 in 64 x 64 tiles: 41.8 us with two stages, 24.7 with three, 21.6 with four).  Microseconds in replayed
// graphs, the weights of eight launches in turn:
//   rows x columns x k            rounded while staged   256x256  256x128  192x128  128x128  64x128  64x64
//   4096 x 5760 x 1024                  92                  60       59       52       55      67      80
//   4096 x 1024 x 1024                  20                  27       18       18       16      15      17
//   4096 x 2752 x 1024, pair            77                  55       52       48       50      58      77
//   2956 x 8352 x 2048                 168                  98      113      106      114     128     149
//   2956 x 5504 x 2048, pair           197                 142      140      124      137     150     184
//   2956 x 2048 x 5504                 123                 100       62       73       70      79     101
//   8 batches, 5912 x 2048 x 1792       95                  55       61       64       70      73      86
//    512 x 5504 x 2048, pair            50                  42       26       36       28      30      36
//    512 x 2048 x 2048                  13.5                39       22       25       22      13       9.5
//    200 x 5760 x 1024                  13.3                24       15       16       14       9.1     9.8
//     77 x 1024 x 1024                   5.9                23       14       12       10       7.1     5.5
// Wider shares of a tile for a wave cost LDS reads the least (a 64 x 64 share reads as many bytes of LDS a cycle as the products take), so the large
// tiles win as soon as their rounds fill the chip.
#include "i64h_dense_dev.h"
#include <cmath>
#include <type_traits>

// 16 bytes a lane from memory to LDS without registers between: the wave's 1024 bytes land one lane after the other
__device__ __forceinline__ void dn_load_lds(__amdgpu_buffer_rsrc_t r, uint16_t* lds, uint32_t lane_bytes, uint32_t step_bytes) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, lane_bytes, step_bytes, 0, 0);
}

constexpr uint32_t DN_STORE_END = 0x7fffff00u;      // offsets from here on are not stored

template <bool DUAL, int BM, int BN, int NWM, int NWN, int NS, int PER_CU>
__global__ __launch_bounds__(64 * NWM * NWN, PER_CU * NWM * NWN / 4) void linear_wide_kernel(const i64h_linear p, const int n_tiles, const int m_tiles, const int vecC) {
    constexpr int NW = NWM * NWN, WM = BM / NWM, WN = BN / NWN, FM = WM / 16, FN = WN / 16;
    constexpr int COLS = DUAL ? BN / 2 : BN;               // output columns of a tile
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW;      // loads of a wave a step: eight rows of 64 values each
    static_assert(LA > 0 && LB > 0 && FN > (DUAL ? 1 : 0), "");
    // (variables of their own: the compiler then knows which loads a read of one has to wait for)
    constexpr int STAGE = (BM + BN) * 64;
    static_assert(NS >= 2 && NS <= 4, "");
    __shared__ __attribute__((aligned(1024))) uint16_t s0[STAGE], s1[STAGE], s2[NS > 2 ? STAGE : 8], s3[NS > 3 ? STAGE : 8];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wid / NWN, wn = wid % NWN;
    const int N = p.N, K = p.K;
    const dn_tile t = dn_find_tile<BM>(p, n_tiles, m_tiles, lane);
    if (!t.any) return;
    const int64_t b = t.b;
    const int n0 = t.nt * COLS;
    const int64_t m0 = t.g0 + (int64_t)t.mt * BM;
    const int M = (int)min((int64_t)BM, t.rows - (int64_t)t.mt * BM);
    const uint16_t *baseA = (const uint16_t*)p.A16 + b * p.a_batch + (p.a_rows ? 0 : m0 * p.lda), *baseW = (const uint16_t*)p.W + b * p.w_batch + (int64_t)n0 * K;
    // 128-byte rows in LDS; the lane that fills chunk c of row r brings chunk c ^ (r & 7), so that the 16 rows of a fragment read lie in different banks
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 16;
    uint32_t oa[LA], ow[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) {      // (rows past the end are zeros that nobody asks memory for, and are not stored)
        const int r = (i * NW + wid) * 8 + lr, at = min(r, M - 1);
        oa[i] = r < M ? (uint32_t)((p.a_rows ? p.a_rows[m0 + at] : at) * p.lda) * 2u + lc : DN_BUF_END;
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
        const int r = (i * NW + wid) * 8 + lr;
        // gate and up rows of the same columns go to the same wave: its first half of fragments, its second half
        const int c = DUAL ? (r / WN) * (WN / 2) + r % (WN / 2) : r;
        ow[i] = (uint32_t)((int64_t)(min(c, N - 1 - n0) + (DUAL && r % WN >= WN / 2 ? N : 0)) * K) * 2u + lc;
    }
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    constexpr std::integral_constant<int, 2> S2{};
    constexpr std::integral_constant<int, 3> S3{};
    auto stage = [&](auto set) -> uint16_t* {
        constexpr int S = decltype(set)::value;
        return S == 0 ? s0 : S == 1 ? s1 : S == 2 ? s2 : s3;
    };
    const int KT = K / 64;
    // (a step past the end asks for nothing: a buffer of no bytes)
    auto load = [&](int kt, auto set) {
        uint16_t* sm = stage(set);
        const uint32_t bytes = kt < KT ? DN_BUF_END : 0u;
        const __amdgpu_buffer_rsrc_t bufA = __builtin_amdgcn_make_buffer_rsrc((void*)baseA, 0, (int)bytes, 0x00020000), bufW = __builtin_amdgcn_make_buffer_rsrc((void*)baseW, 0, (int)bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < LA; ++i) dn_load_lds(bufA, sm + (i * NW + wid) * 512, oa[i], kt * 128);
#pragma unroll
        for (int i = 0; i < LB; ++i) dn_load_lds(bufW, sm + BM * 64 + (i * NW + wid) * 512, ow[i], kt * 128);
    };
    dn_v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = dn_v4f{0, 0, 0, 0};
    const int fr = lane & 15, fk = lane >> 4;
    dn_v4u a[2][FM], w[2][FN];      // the fragments of a step's two halves
    auto fragments = [&](auto set, auto half) {
        constexpr int H = decltype(half)::value;
        const uint16_t* sm = stage(set);
        const int ch = ((H * 4 + fk) ^ (fr & 7)) << 3;
#pragma unroll
        for (int i = 0; i < FM; ++i) a[H][i] = *(const dn_v4u*)&sm[(wm * WM + i * 16 + fr) * 64 + ch];
#pragma unroll
        for (int j = 0; j < FN; ++j) w[H][j] = *(const dn_v4u*)&sm[(BM + wn * WN + j * 16 + fr) * 64 + ch];
    };
    auto multiply = [&](auto half) {
        constexpr int H = decltype(half)::value;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, w[H][j]), __builtin_bit_cast(dn_v8bf, a[H][i]), acc[i][j], 0, 0, 0);
    };
    // this wave's loads of the step after this one are in LDS and its fragments in registers; then everybody's
    auto meet = [&]() {
        constexpr int LEFT = (NS - 2) * (LA + LB);      // loads of later steps
        static_assert(LEFT < 64, "");
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | (LEFT & 15) | (LEFT >> 4) << 14);      // vmcnt LEFT, lgkmcnt 0
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // reads (and loads) from the first product on, one between two products
    auto interleave = [&](auto loads) {
        constexpr int MF = FM * FN, DR = FM + FN, VM = decltype(loads)::value ? LA + LB : 0;
#pragma unroll
        for (int g = 0; g < DR; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (g < VM) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
            if (MF >= 2 * DR) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    load(0, S0);
    load(1, S1);
    if constexpr (NS > 2) load(2, S2);
    if constexpr (NS > 3) load(3, S3);
    {
        constexpr int LEFT = (NS - 1) * (LA + LB);
        __builtin_amdgcn_s_waitcnt(0x0f70 | (LEFT & 15) | (LEFT >> 4) << 14);
        asm volatile("s_barrier" ::: "memory");
    }
    fragments(S0, S0);
    // The second half's fragments are read under the first half's products.  Behind them the step's buffer is free: the loads of the step NS further on
    // go there, and the next step's first fragments are read under the second half's products.
    // (Without a branch in the loop: where paths meet the compiler waits for whatever either may have on its way.)
    auto step = [&](int kt, auto cur, auto nxt) {
        fragments(cur, S1);
        multiply(S0);
        interleave(S0);
        meet();
        load(kt + NS, cur);
        fragments(nxt, S0);
        multiply(S1);
        interleave(S1);
    };
    int kt = 0;
    for (; kt + NS <= KT; kt += NS) {
        if constexpr (NS == 2) {
            step(kt, S0, S1);
            step(kt + 1, S1, S0);
        } else if constexpr (NS == 3) {
            step(kt, S0, S1);
            step(kt + 1, S1, S2);
            step(kt + 2, S2, S0);
        } else {
            step(kt, S0, S1);
            step(kt + 1, S1, S2);
            step(kt + 2, S2, S3);
            step(kt + 3, S3, S0);
        }
    }
    if (kt < KT) step(kt, S0, S1);
    if constexpr (NS > 2)
        if (kt + 1 < KT) step(kt + 1, S1, S2);
    if constexpr (NS > 3)
        if (kt + 2 < KT) step(kt + 2, S2, S3);
    __builtin_amdgcn_s_waitcnt(0x0f70);      // (nothing is on its way into LDS when the workgroup ends)
    // The weights are the left operand: a lane holds four neighbouring columns of a row, a block of 16 rows 64 bytes (bf16: 32) of each.  Stored so, half or a
    // quarter of a line at a time, a round of 256 x 256 tiles took 10.5 us to end, in fp32 and in bf16 alike: the lines, not the bytes.  So 16 rows at a time pass
    // through LDS of the wave's own and leave as whole lines.  What a launch may have or not (a bias, factors of the rows) is asked once, not at every value, and rows and
    // columns past the end are stored where the buffer ends.  8192 x 2048 x 64 in 256 x 256 / 128 x 128 tiles, us: fp32 16.8 / 20.4 -> 15.6 / 17.8 (67 MB), bf16
    // 16.1 / 16.4 -> 11.9 / 12.9; a pair to bf16, 8192 x 896 x 64, 16.2 / 17.1 -> 12.4 / 13.5 (9.9 of it without the activation); 4096 x 5760 x 1024 in 192 x 128 tiles
    // 53.5 -> 50, as a pair of 2752 51.5 -> 46.
    constexpr int FO = DUAL ? FN / 2 : FN;      // blocks of output columns
    auto finish = [&](auto epi, auto vec) {      // (vec: a lane's four columns at a time)
        constexpr int EPI = decltype(epi)::value;
        int at_lane = lane, at_row = wm * WM, at_col = wn * (COLS / NWN);
        asm volatile("" : "+v"(at_lane), "+s"(at_row), "+s"(at_col));      // (nothing of what follows is worked out, and kept, ahead of the loop, nor shared with its addresses)
        const int c0 = at_col + (at_lane >> 4) * 4, r0 = at_row + (at_lane & 15);      // this lane's first column and row in the tile
        if constexpr (decltype(vec)::value) {
            i64h_linear q = p;      // (what the values below have already)
            q.bias = nullptr, q.row_scale = nullptr;
            float add[DUAL ? 1 : FO][4];
            if constexpr (!DUAL) {
#pragma unroll
                for (int j = 0; j < FO; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) add[j][g] = -0.0f;      // (changes no value, not even a zero's sign)
                if (p.bias) {
#pragma unroll
                    for (int j = 0; j < FO; ++j)
#pragma unroll
                        for (int g = 0; g < 4; ++g) add[j][g] = p.bias[b * p.bias_batch + min(n0 + c0 + j * 16 + g, N - 1)];
                }
            }
            // 16 rows at a time through LDS of the wave's own, so that a store takes whole lines
            constexpr int OC = FO * 16, PITCH = OC + 4;
            static_assert(NW * 16 * PITCH * 4 <= STAGE * 2, "");
            float* const own = (float*)s0 + wid * 16 * PITCH;
            const int64_t at = b * p.c_batch + m0 * p.ldc + n0;
            const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(p.C + at, 0, (int)DN_STORE_END, 0x00020000);
            const __amdgpu_buffer_rsrc_t buf16 = __builtin_amdgcn_make_buffer_rsrc((uint16_t*)p.C16 + at, 0, (int)DN_STORE_END, 0x00020000);
            const bool eight = ((N | (int)p.ldc | (int)p.c_batch) & 7) == 0;
            const int cw = at_col, ldc = (int)p.ldc;
            // (a lane reads what others of its wave wrote: LDS operations of a wave happen in their order, and the fence keeps the compiler to it)
            auto handed = [&]() {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            };
            __syncthreads();
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int64_t r = m0 + min(r0 + i * 16, M - 1);
                if (DUAL && p.row_scale) {
                    const float factor = p.row_scale[r];
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] *= factor;
                }
                float gate = 1.0f;
                if constexpr (EPI == I64H_EPI_ROW_SIGMOID) gate = dn_sigmoid(p.E[b * p.e_batch + r * p.lde]);
#pragma unroll
                for (int j = 0; j < FO; ++j) {
                    const int c = min(n0 + c0 + j * 16, N - 4);
                    dn_v4f o;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        if constexpr (DUAL) o[g] = dn_epilogue<EPI>(q, acc[i][j][g], acc[i][j + FN / 2][g], b, r, c + g);
                        else if constexpr (EPI == I64H_EPI_ROW_SIGMOID) o[g] = (acc[i][j][g] + add[j][g]) * gate;
                        else o[g] = dn_epilogue<EPI>(q, acc[i][j][g] + add[j][g], 0.0f, b, r, c + g);
                    }
                    *(dn_v4f*)&own[(at_lane & 15) * PITCH + j * 16 + (at_lane >> 4) * 4] = o;
                }
                handed();
                const int r1 = at_row + i * 16;
                if (p.C16) {
                    if (eight) {
#pragma unroll
                        for (int t = 0; t < (FO + 1) / 2; ++t) {
                            const int e = t * 64 + at_lane, row = e / (OC / 8), c = e % (OC / 8) * 8;
                            const dn_v4f x = *(const dn_v4f*)&own[min(row, 15) * PITCH + c], y = *(const dn_v4f*)&own[min(row, 15) * PITCH + c + 4];
                            const uint32_t off = r1 + row < M && row < 16 && n0 + cw + c < N ? (uint32_t)((r1 + row) * ldc + cw + c) * 2 : DN_STORE_END;
                            __builtin_amdgcn_raw_buffer_store_b128(dn_v4u{dn_bf16_pair(x[0], x[1]), dn_bf16_pair(x[2], x[3]), dn_bf16_pair(y[0], y[1]), dn_bf16_pair(y[2], y[3])}, buf16, off, 0, 0);
                        }
                    } else {
#pragma unroll
                        for (int t = 0; t < FO; ++t) {
                            const int e = t * 64 + at_lane, row = e / (OC / 4), c = e % (OC / 4) * 4;
                            const dn_v4f x = *(const dn_v4f*)&own[row * PITCH + c];
                            const uint32_t off = r1 + row < M && n0 + cw + c < N ? (uint32_t)((r1 + row) * ldc + cw + c) * 2 : DN_STORE_END;
                            __builtin_amdgcn_raw_buffer_store_b64(dn_v2u{dn_bf16_pair(x[0], x[1]), dn_bf16_pair(x[2], x[3])}, buf16, off, 0, 0);
                        }
                    }
                }
                if (p.C) {
#pragma unroll
                    for (int t = 0; t < FO; ++t) {
                        const int e = t * 64 + at_lane, row = e / (OC / 4), c = e % (OC / 4) * 4;
                        const dn_v4f x = *(const dn_v4f*)&own[row * PITCH + c];
                        const uint32_t off = r1 + row < M && n0 + cw + c < N ? (uint32_t)((r1 + row) * ldc + cw + c) * 4 : DN_STORE_END;
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(dn_v4u, x), buf, off, 0, 0);
                    }
                }
                if (i + 1 < FM) {      // (a row's work at a time: the registers are full)
                    handed();
#pragma unroll
                    for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(acc[i + 1 < FM ? i + 1 : i][j]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int rl = r0 + i * 16;
                if (rl >= M) continue;
                const int64_t r = m0 + rl, row = b * p.c_batch + r * p.ldc;
#pragma unroll
                for (int j = 0; j < FO; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int c = n0 + c0 + j * 16 + g;
                        if (c >= N) continue;
                        const float v = dn_epilogue<EPI>(p, acc[i][j][g], DUAL ? acc[i][DUAL ? j + FN / 2 : j][g] : 0.0f, b, r, c);
                        if (p.C16) ((uint16_t*)p.C16)[row + c] = (uint16_t)dn_bf16_rne(v);
                        if (p.C) p.C[row + c] = v;
                    }
            }
        }
    };
#define DN_FINISH(E) case E: if (vecC) finish(std::integral_constant<int, E>{}, S1); else finish(std::integral_constant<int, E>{}, S0); break;
    if constexpr (DUAL) {
        switch (p.epilogue) { DN_FINISH(I64H_EPI_CLAMP_GLU) DN_FINISH(I64H_EPI_GELU_MUL) DN_FINISH(I64H_EPI_SILU_MUL) }
    } else {
        switch (p.epilogue) { DN_FINISH(I64H_EPI_SCALE) DN_FINISH(I64H_EPI_ADD) DN_FINISH(I64H_EPI_ROW_SIGMOID) DN_FINISH(I64H_EPI_STORE) }
    }
#undef DN_FINISH
}

template <int BM, int BN, int NWM, int NWN, int NS, int PER_CU>
static void launch(const i64h_linear& d, hipStream_t s) {
    const bool dual = dn_dual(d.epilogue);
    const int cols = dual ? BN / 2 : BN;
    const int nt = (d.N + cols - 1) / cols;
    int64_t mt = (d.M + BM - 1) / BM;
    if (d.group_off) {      // at most one partly filled row tile per batch beside the full ones
        const int64_t most = mt * d.batch;
        mt = d.rows_total > 0 ? (most < d.rows_total / BM + d.batch ? most : d.rows_total / BM + d.batch) : most;
    }
    const int vecC = ((uintptr_t)d.C | (uintptr_t)d.C16) % 16 == 0 && d.ldc % 4 == 0 && d.c_batch % 4 == 0 && d.N % 4 == 0 && d.ldc < (DN_STORE_END / 4 - 256) / 256;
    const dim3 grid((unsigned)(mt * nt), 1, d.group_off ? 1u : (unsigned)d.batch);
    if (dual) hipLaunchKernelGGL((linear_wide_kernel<true, BM, BN, NWM, NWN, NS, PER_CU>), grid, dim3(64 * NWM * NWN), 0, s, d, nt, (int)mt, vecC);
    else hipLaunchKernelGGL((linear_wide_kernel<false, BM, BN, NWM, NWN, NS, PER_CU>), grid, dim3(64 * NWM * NWN), 0, s, d, nt, (int)mt, vecC);
}

// ---- up to 128 rows under few columns: 16 columns and 64 rows a workgroup, the steps of k dealt to its waves ------------------------------------
// What bounds it: the latency of a step, a few of them on their way.  A 64 x 64 tile walks all of k alone, and 1024 or 2048 columns are 16 or 32 of them on 256 CUs.
// Here every wave takes every NW-th step of 64 k for 16 columns and all rows, with loads, LDS and waits of its own: nobody meets before the end, where the waves' sums
// are added in their order.  The rows are read once for 16 columns, from L2: at 64 rows of 5504 that is 90 MB, and the launch's time.  Microseconds in replayed graphs, the
// weights of twelve launches in turn, the fp32 rows' kernels | 64 x 64 tiles | here (more than 64 rows: two tiles of them):
//   rows:                   3                     16                   64                   77                  128
//   1024 x 1024     3.5 | 4.9 | 3.5     4.6 | 5.0 | 3.4      5.8 | 5.1 | 4.3      5.7 | 5.1 | 4.5      5.8 | 5.1 | 4.5
//   1024 x 2752     6.6 | 9.3 | 4.7     9.6 | 9.3 | 5.1      9.4 | 10.5 | 7.6     9.3 | 9.4 | 6.9      9.5 | 10.1 | 7.6
//   2048 x 2048     5.7 | 7.8 | 4.7     7.9 | 7.8 | 4.8      8.3 | 8.2 | 6.6      8.3 | 7.9 | 6.4      8.5 | 8.2 | 6.9
//   2048 x 5504     11.8 | 21.6 | 8.2   23.8 | 22.1 | 9.5    22.5 | 27.1 | 16.6   22.0 | 22.2 | 13.2   22.1 | 25.9 | 16.5
//   4352 x 2048                         8.4 | 8.1 | 8.4      9.8 | 8.5 | 12.5
// (more than 256 tiles, the last row: a second round, worth it only under a long k)
template <int MB, int NW, int NS, int EPI>
__global__ __launch_bounds__(64 * NW, NW / 4) void linear_thin_kernel(const i64h_linear p, const int vecC) {
    constexpr int LA = 2 * MB, LB = 2, ROWS = 16 * MB + 16, STAGE = NW * ROWS * 64;      // loads a step: eight rows of 64 values each
    static_assert(NS == 3 || NS == 4, "");
    __shared__ __attribute__((aligned(1024))) uint16_t s0[STAGE], s1[STAGE], s2[STAGE], s3[NS > 3 ? STAGE : 8];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N = p.N, K = p.K, KT = K / 64;
    const int n0 = blockIdx.x * 16;
    const int64_t b = blockIdx.z, m0 = (int64_t)blockIdx.y * (16 * MB);
    const int M = (int)min((int64_t)16 * MB, p.M - m0);
    const uint16_t *baseA = (const uint16_t*)p.A16 + b * p.a_batch + m0 * p.lda, *baseW = (const uint16_t*)p.W + b * p.w_batch + (int64_t)n0 * K;
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 16;      // (chunks permuted per row, as above)
    uint32_t oa[LA], ow[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) oa[i] = i * 8 + lr < M ? (uint32_t)((i * 8 + lr) * p.lda) * 2u + lc : DN_BUF_END;
#pragma unroll
    for (int i = 0; i < LB; ++i) ow[i] = (uint32_t)(min(i * 8 + lr, N - 1 - n0) * K) * 2u + lc;
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    constexpr std::integral_constant<int, 2> S2{};
    constexpr std::integral_constant<int, 3> S3{};
    auto stage = [&](auto set) -> uint16_t* {
        constexpr int S = decltype(set)::value;
        return (S == 0 ? s0 : S == 1 ? s1 : S == 2 ? s2 : s3) + wid * ROWS * 64;
    };
    auto load = [&](int t, auto set) {      // (a step past the end asks for nothing: a buffer of no bytes)
        const int kt = t * NW + wid;
        uint16_t* sm = stage(set);
        const uint32_t bytes = kt < KT ? DN_BUF_END : 0u;
        const __amdgpu_buffer_rsrc_t bufA = __builtin_amdgcn_make_buffer_rsrc((void*)baseA, 0, (int)bytes, 0x00020000), bufW = __builtin_amdgcn_make_buffer_rsrc((void*)baseW, 0, (int)bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < LB; ++i) dn_load_lds(bufW, sm + (16 * MB + i * 8) * 64, ow[i], kt * 128);
#pragma unroll
        for (int i = 0; i < LA; ++i) dn_load_lds(bufA, sm + i * 512, oa[i], kt * 128);
    };
    dn_v4f acc[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i] = dn_v4f{0, 0, 0, 0};
    const int fr = lane & 15, fk = lane >> 4;
    auto step = [&](int t, auto cur) {
        constexpr int LEFT = (NS - 1) * (LA + LB);
        static_assert(LEFT < 64, "");
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0f70 | (LEFT & 15) | (LEFT >> 4) << 14);      // this step's loads are in LDS (the wave's own)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint16_t* sm = stage(cur);
        dn_v4u a[2][MB], w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int ch = ((h * 4 + fk) ^ (fr & 7)) << 3;
            w[h] = *(const dn_v4u*)&sm[(16 * MB + fr) * 64 + ch];
#pragma unroll
            for (int i = 0; i < MB; ++i) a[h][i] = *(const dn_v4u*)&sm[(i * 16 + fr) * 64 + ch];
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt 0: they are in registers, the place is free
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load(t + NS, cur);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_v8bf, w[h]), __builtin_bit_cast(dn_v8bf, a[h][i]), acc[i], 0, 0, 0);
    };
    load(0, S0);
    load(1, S1);
    load(2, S2);
    if constexpr (NS > 3) load(3, S3);
    const int T = (KT + NW - 1) / NW;
    int t = 0;
    for (; t + NS <= T; t += NS) {
        step(t, S0);
        step(t + 1, S1);
        step(t + 2, S2);
        if constexpr (NS > 3) step(t + 3, S3);
    }
    if (t < T) step(t, S0);
    if (t + 1 < T) step(t + 1, S1);
    if constexpr (NS > 3)
        if (t + 2 < T) step(t + 2, S2);
    __builtin_amdgcn_s_waitcnt(0x0f70);      // (nothing is on its way into LDS)
    __syncthreads();
    // the waves' sums meet in LDS; wave i adds those of rows 16 i .. in the waves' order
    dn_v4f* sum = (dn_v4f*)s0;
    static_assert(NW * MB * 64 * 16 <= STAGE * 2 && MB <= NW, "");
#pragma unroll
    for (int i = 0; i < MB; ++i) sum[(wid * MB + i) * 64 + lane] = acc[i];
    __syncthreads();
    if (wid >= MB) return;
    dn_v4f o = sum[wid * 64 + lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) o += sum[(w * MB + wid) * 64 + lane];
    const int c = n0 + fk * 4;
    if (wid * 16 + fr >= M) return;
    const int64_t r = m0 + wid * 16 + fr;
    const int64_t at = b * p.c_batch + r * p.ldc + c;
#pragma unroll
    for (int g = 0; g < 4; ++g)
        if (c + g < N) o[g] = dn_epilogue<EPI>(p, o[g], 0.0f, b, r, c + g);
    if (vecC && c < N) {
        if (p.C16) *(uint2*)((uint16_t*)p.C16 + at) = make_uint2(dn_bf16_pair(o[0], o[1]), dn_bf16_pair(o[2], o[3]));
        if (p.C) *(dn_v4f*)(p.C + at) = o;
        return;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        if (c + g >= N) continue;
        if (p.C16) ((uint16_t*)p.C16)[at + g] = (uint16_t)dn_bf16_rne(o[g]);
        if (p.C) p.C[at + g] = o[g];
    }
}

static bool thin_fits(const i64h_linear& d) {
    return !dn_dual(d.epilogue) && !d.a_rows && !d.group_off && d.batch <= 65535 && d.M <= 64 * 65535;
}
template <int EPI>
static void launch_thin(const i64h_linear& d, hipStream_t s) {
    const int vecC = ((uintptr_t)d.C | (uintptr_t)d.C16) % 16 == 0 && d.ldc % 4 == 0 && d.c_batch % 4 == 0 && d.N % 4 == 0;
    const dim3 grid((unsigned)((d.N + 15) / 16), (unsigned)((d.M + 63) / 64), (unsigned)d.batch);
    if (d.M <= 16) hipLaunchKernelGGL((linear_thin_kernel<1, 8, 4, EPI>), grid, dim3(512), 0, s, d, vecC);
    else if (d.M <= 32) hipLaunchKernelGGL((linear_thin_kernel<2, 8, 3, EPI>), grid, dim3(512), 0, s, d, vecC);
    else hipLaunchKernelGGL((linear_thin_kernel<4, 4, 3, EPI>), grid, dim3(256), 0, s, d, vecC);
}
static void launch_thin(const i64h_linear& d, hipStream_t s) {
    switch (d.epilogue) {
        case I64H_EPI_SCALE: launch_thin<I64H_EPI_SCALE>(d, s); break;
        case I64H_EPI_ADD: launch_thin<I64H_EPI_ADD>(d, s); break;
        case I64H_EPI_ROW_SIGMOID: launch_thin<I64H_EPI_ROW_SIGMOID>(d, s); break;
        default: launch_thin<I64H_EPI_STORE>(d, s); break;
    }
}

// The form of a launch by what it costs: its workgroups' rounds on the 256 CUs times a round's microseconds, fitted to the measurements above (weights
// that come from memory: a step is not shorter than the microsecond that its loads take, divided by the steps on their way).
struct dn_wide_form {
    int BM, BN;
    bool alone;           // one workgroup a CU: every round ends with its stores, in the open; two a CU: the one's stores lie under the other's products
    float first, step;    // a step of 64 k: of a workgroup alone on its CU, of a round (of two workgroups a CU)
    float end;            // a round's stores
};

enum { DN_WIDE_FORMS = 6 };      // tile forms; the number itself stands for linear_thin_kernel

// -1: operands beyond what the tiles' 32-bit offsets reach
int dn_linear_wide_form(const i64h_linear& d) {
    const bool dual = dn_dual(d.epilogue);
    const int64_t span = (d.a_rows ? d.a_height : 256) * d.lda * 2;
    if ((d.a_rows && d.a_height <= 0) || span >= (int64_t)DN_BUF_END - 64 || ((dual ? (int64_t)d.N : 0) + 256) * 2 * d.K >= (int64_t)DN_BUF_END - 64) return -1;
    const int64_t cols = dual ? 2 * (int64_t)d.N : d.N;
    if ((d.M + 63) / 64 * d.batch * ((cols + 63) / 64) > 0x7fffffff) return -1;
    // few tiles of 16 columns: one for every CU at most (its LDS holds three or four steps of all its waves), two where up to 32 rows walk a long k.  Microseconds, here | 64 x 64
    // tiles | rows in 32 bits: 5120 x 4096, 3 rows 14.3 | 19.4 | 18.5, 32 rows 19.4 | 20.3 | 19.5, 48 rows 23.6 | 21.1 | 18.9; 8192 x 3072, 16 rows 15.0 | 16.8 | 20.1; 4352 x 2048, 16 rows 9.0 |
    // 8.6 | 8.7
    const int64_t thin_tiles = (d.M + 63) / 64 * ((d.N + 15) / 16) * d.batch;
    if (thin_fits(d) && d.M <= 128 && d.K >= 256 && (thin_tiles <= 256 || (thin_tiles <= 512 && d.M <= 32 && d.K >= 3072))) return DN_WIDE_FORMS;
    static const dn_wide_form forms[DN_WIDE_FORMS] = {{256, 256, true, 1.3f, 1.3f, 12.0f}, {256, 128, true, 0.72f, 0.72f, 7.0f}, {192, 128, false, 1.0f, 1.7f, 0.0f},
                                                      {128, 128, false, 1.0f, 1.2f, 0.0f}, {64, 128, false, 0.5f, 0.75f, 0.0f}, {64, 64, false, 0.33f, 0.4f, 0.0f}};
    int form = 0;
    float best = 0.0f;
    for (int i = 0; i < DN_WIDE_FORMS; ++i) {
        const dn_wide_form& f = forms[i];
        int64_t mt = (d.M + f.BM - 1) / f.BM * d.batch;
        // rows dealt to batches: half a tile more than the rows fill, on average
        if (d.group_off && d.rows_total > 0 && d.rows_total / f.BM + (d.batch + 1) / 2 < mt) mt = d.rows_total / f.BM + (d.batch + 1) / 2;
        const float q = (float)(mt * ((cols + f.BN - 1) / f.BN)) / 256.0f;
        const float step = f.alone ? ceilf(q) * f.step : fmaxf(f.first, fmaxf(0.5f * q, q > 1.0f ? 0.75f : 0.0f) * f.step);
        const float cost = (float)(d.K / 64) * step + (f.alone ? ceilf(q) * f.end : 0.0f);
        if (i == 0 || cost < best) best = cost, form = i;
    }
    // At most 64 rows, dealt to batches by chance: a launch waits for the weights of the batches that have any (one of them perhaps with all).  Where 64 x 128 tiles of these
    // fill a round of the 256 CUs by half and no more than once, they read the rows half as often for the same wait.  Microseconds, 64 x 128 | 64 x 64: 9 batches, pairs of 1792
    // x 2048 (252 tiles), 12 tokens 34.4 | 35.6, 64 tokens 35.1 | 37.8; 2048 x 1792 (144), 40 tokens 18.3 | 20.8; 13 batches, pairs of 896 x 1024 (182), 64 tokens 14.2 | 16.3.  Less
    // than half: 8 batches, pairs of 896 x 1024 (112), 64 tokens 10.6 | 9.3.  More than once, or longer k, where the four steps that a 64 x 64 tile has on their way count: 12
    // batches, pairs of 1792 x 2048 (336), 12 tokens 44.0 | 41.8; 8 of 5504 x 2048 (688), 64 tokens 87.7 | 81.6; 15 of 1024 x 4096 (240), 27 tokens 63.4 | 58.7; but 64 of 2048 x 768
    // (1024), 40 tokens 42.4 | 47.3.  (Taller tiles are never the fastest there: 59 to 107 us for these.)  Where 64 x 64 tiles under a longer
    // k are one to one and a half of a round, 64 x 128 ones are faster alone, 9 of 2048 x 5504 (144), 64 tokens 61.9 | 73.2, but not beside a second stream's scan (92 | 85): of steps with
    // such experts one with the recurrent branch beside them took 747 | 718, one without 1024 | 1058.
    if (form >= 4 && d.group_off && d.rows_total > 0 && d.M <= 64) {
        const float others = (float)(d.batch - 1), live = others > 0.0f ? 1.0f + others * (1.0f - expf(-fmaxf(0.0f, (float)(d.rows_total - d.M)) / others)) : 1.0f;
        const float tiles = live * (float)((cols + 127) / 128);
        if (form == 5 && d.K <= 2048 && tiles >= 128.0f && tiles < 256.0f) form = 4;
        else if (form == 4 && d.K >= 2048 && tiles >= 256.0f) form = 5;
    }
    return form;
}

bool dn_linear_wide(const i64h_linear& d, int form, hipStream_t s) {
    const int by_size = dn_linear_wide_form(d);
    if (by_size < 0) return false;
    if (form < 0) form = by_size;
    if (form == DN_WIDE_FORMS && thin_fits(d)) {
        launch_thin(d, s);
        return true;
    }
    switch (form) {
        case 0: launch<256, 256, 2, 4, 2, 1>(d, s); break;
        case 1: launch<256, 128, 4, 2, 3, 1>(d, s); break;
        case 2: launch<192, 128, 2, 2, 2, 2>(d, s); break;
        case 3: launch<128, 128, 2, 2, 2, 2>(d, s); break;
        case 4: launch<64, 128, 2, 2, 3, 2>(d, s); break;
        default: launch<64, 64, 2, 2, 4, 2>(d, s); break;
    }
    return true;
}
