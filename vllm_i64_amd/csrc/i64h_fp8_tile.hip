// e4m3 Linears of a few hundred rows (mixed steps, short prompts) on rows quantized beforehand: C[r, c] = (sum_k A[r, k] B[c, k]) * (a_scale[r] *
// b_scale[c]), the arithmetic and the order of the sums of gemm_fp8_skinny_kernel, so that both give the same bits.
//
// What bounds it.  gemm_fp8_skinny_kernel quantizes its 16 rows in front of every 64 columns: 3.3 us of vector instructions a row tile and workgroup, which
// is nothing while a launch is one round of the chip and everything beyond (512 rows x 1536 x 1024: 18.6 us; with tiles of 32 and 64 rows 21.8 and 16.9, the
// quantizing being the same).  Here the codes are written once and a 64 x 64 tile's steps of 128 bytes go from memory to LDS by direct loads, three
// steps on their way: 512 rows of the products of a layer (qkv with its tail, o, gate / up and down of eight experts and a shared one) 23, 11, 42 and 27 us
// before, 12.0, 7.4, 13.9 and 9.8 here, and two launches of 3.5 to 4 us for the codes.  A tile's chain (codes, steps, epilogue) bounds it now.
#include "i64h_common.h"
#include "i64h_gemm_dev.h"
#include "i64h.h"
#include <type_traits>

typedef float ft_v4f __attribute__((ext_vector_type(4)));
#define FT_BM 64
#define FT_BN 64
#define FT_NS 4

struct Fp8CodesPair {
    i64h_fp8_codes_desc p[2];
    int nblk0;  // workgroups [0, nblk0) run p[0], the rest p[1]
};

// workgroups are dealt to the 8 XCDs in turn: with the column tiles padded to a multiple of 8 the row tiles that read the same weights share an L2
__host__ __device__ __forceinline__ int ft_pad_tiles(int n_tiles) { return n_tiles >= 6 ? (n_tiles + 7) & ~7 : n_tiles; }

// EPI 0: store (c_add: on top of the residual); 1: silu(gate) * up; 2: a tile's columns are one head of the fused qkv projection - QK norm, rotation, cache
template <int EPI>
__global__ __launch_bounds__(256, 2) void gemm_fp8_tile_kernel(const Fp8CodesPair pp, const RowTailArgs ta) {
    constexpr int STAGE = (FT_BM + FT_BN) * 128;
    __shared__ __attribute__((aligned(1024))) char s0[STAGE], s1[STAGE], s2[STAGE], s3[STAGE];
    const bool second = (int)blockIdx.x >= pp.nblk0;
    const i64h_fp8_codes_desc& p = pp.p[second ? 1 : 0];
    const int bid = second ? (int)blockIdx.x - pp.nblk0 : (int)blockIdx.x;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wid >> 1, wn = wid & 1;
    const int N = p.N, K = p.K, I = N / 2, nout = EPI == 1 ? I : N;
    constexpr int COLS = EPI == 1 ? FT_BN / 2 : FT_BN;
    const int n_tiles = (nout + COLS - 1) / COLS, n_pad = ft_pad_tiles(n_tiles);
    const int mt = bid / n_pad, nt = bid % n_pad;
    if (nt >= n_tiles) return;
    // (group, first row, rows) of row tile mt: lane i looks at group c0 + i; the grid is an upper bound
    int g = -1, row0 = 0, rows = 0;
    if (!p.group_offsets) {
        g = 0, row0 = mt * FT_BM, rows = min(FT_BM, (int)p.M - row0);
    } else {
        int base = 0;
        const int ng = p.num_groups;
        for (int c0 = 0; c0 < ng && g < 0; c0 += 64) {
            const int i = c0 + lane;
            int b = 0, e = 0;
            if (i < ng) { b = p.group_offsets[i]; e = p.group_offsets[i + 1]; }
            const int tiles = (e - b + FT_BM - 1) / FT_BM;
            int incl = tiles;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int t = __shfl_up(incl, o);
                if (lane >= o) incl += t;
            }
            const int excl = base + incl - tiles;
            const unsigned long long hit = __ballot(i < ng && mt >= excl && mt < excl + tiles);
            if (hit) {
                const int src = __ffsll(hit) - 1;
                g = c0 + src;
                row0 = __builtin_amdgcn_readlane(b, src) + (mt - __builtin_amdgcn_readlane(excl, src)) * FT_BM;
                rows = min(FT_BM, __builtin_amdgcn_readlane(e, src) - row0);
            }
            base += __builtin_amdgcn_readlane(incl, 63);
        }
    }
    if (g < 0) return;
    // EPI 2: lane j < 16 looks up what row wid + 4 j of the tile needs: position, cache page
    int qk_pos = 0, qk_pb = 0;
    if (EPI == 2) {
        const int64_t t = row0 + min(wid + 4 * (lane & 15), rows - 1);
        qk_pos = ta.positions[t];
        qk_pb = ta.block_table[(int64_t)ta.slot_ids[t] * ta.max_blocks_per_seq + qk_pos / ta.block];
    }
    // staging: 128-byte rows, the lane that fills chunk c of row r brings chunk c ^ (r & 7); a last step of 64 bytes brings 64 of what follows (the next row,
    // or nothing past the operand's end), which is not read
    const int64_t a_rows = p.a_src_row ? p.a_src_mod : p.M;
    const __amdgpu_buffer_rsrc_t bufA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.A), 0, (int)(uint32_t)(a_rows * K), 0x00020000);
    const __amdgpu_buffer_rsrc_t bufB = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.B + (int64_t)g * N * K), 0, (int)(uint32_t)((int64_t)N * K), 0x00020000);
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 16;
    const int KT = (K + 127) / 128, KF = K / 128;
    uint32_t oa[2], ob[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = (i * 4 + wid) * 8 + lr;
        int64_t arow = row0 + min(r, rows - 1);
        if (p.a_src_row) arow = p.a_src_row[arow] % p.a_src_mod;
        oa[i] = (uint32_t)(arow * K) + lc;
        // EPI 1: the wave's first 16 rows of weights are gate columns, its second 16 their up partners
        const int c = EPI == 1 ? min(nt * COLS + (r >> 5) * 16 + (r & 15), I - 1) + ((r >> 4) & 1 ? I : 0) : min(nt * COLS + r, N - 1);
        ob[i] = (uint32_t)((int64_t)c * K) + lc;
    }
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    constexpr std::integral_constant<int, 2> S2{};
    constexpr std::integral_constant<int, 3> S3{};
    auto stage = [&](auto set) -> char* {
        constexpr int S = decltype(set)::value;
        return S == 0 ? s0 : S == 1 ? s1 : S == 2 ? s2 : s3;
    };
    // (a step past the end asks for nothing: offsets past either operand; all of the offset is the lane's, so that it is checked against the operand's end)
    auto load = [&](int kt, auto set) {
        char* sm = stage(set);
        const uint32_t past = kt < KT ? 0u : 0xfffffff0u;
#pragma unroll
        for (int i = 0; i < 2; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(bufA, (__attribute__((address_space(3))) void*)(sm + (i * 4 + wid) * 1024), 16, (oa[i] + kt * 128) | past, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(bufB, (__attribute__((address_space(3))) void*)(sm + FT_BM * 128 + (i * 4 + wid) * 1024), 16, (ob[i] + kt * 128) | past, 0, 0, 0);
    };
    ft_v4f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = ft_v4f{0, 0, 0, 0};
    const int fr = lane & 15, fk = lane >> 4;
    uint4 a[2][2], w[2][2];  // the fragments of a step's two halves of 64 bytes: 16 bytes a lane, for two products of 32 each
    auto fragments = [&](auto set, auto half) {
        constexpr int H = decltype(half)::value;
        const char* sm = stage(set);
        const int ch = ((H * 4 + fk) ^ (fr & 7)) * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) a[H][i] = *(const uint4*)(sm + (wm * 32 + i * 16 + fr) * 128 + ch);
#pragma unroll
        for (int j = 0; j < 2; ++j) w[H][j] = *(const uint4*)(sm + (FT_BM + wn * 32 + j * 16 + fr) * 128 + ch);
    };
    auto lo = [](uint4 x) { return (long)(((unsigned long long)x.y << 32) | x.x); };
    auto hi = [](uint4 x) { return (long)(((unsigned long long)x.w << 32) | x.z); };
    auto multiply = [&](auto half) {
        constexpr int H = decltype(half)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(lo(w[H][j]), lo(a[H][i]), acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(hi(w[H][j]), hi(a[H][i]), acc[i][j], 0, 0, 0);
    };
    // this wave's loads of the next step are in LDS and its fragments in registers; then everybody's
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | (FT_NS - 2) * 4);      // vmcnt: the loads of the steps behind it, lgkmcnt 0
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // what the epilogue multiplies by, requested in front of the steps: this lane's rows' scales and places, its columns' scales
    const float* bs = p.b_scale + (int64_t)g * N;
    float as[2];
    int64_t crow[2];
    float4 ws[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int64_t r = row0 + min(wm * 32 + i * 16 + fr, rows - 1);
        as[i] = p.a_scale[p.a_src_row ? p.a_src_row[r] % p.a_src_mod : r];
        crow[i] = p.c_row_map ? p.c_row_map[r] : r;
        // (column counts are multiples of 16, of 32 for a pair)
        ws[i] = EPI == 1 ? *(const float4*)(bs + min(nt * COLS + wn * 16 + fk * 4, I - 4) + i * I) : *(const float4*)(bs + min(nt * COLS + wn * 32 + i * 16 + fk * 4, N - 4));
    }
    load(0, S0);
    load(1, S1);
    load(2, S2);
    load(3, S3);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (FT_NS - 1) * 4);
    asm volatile("s_barrier" ::: "memory");
    fragments(S0, S0);
    auto step = [&](int kt, auto cur, auto nxt) {
        fragments(cur, S1);
        multiply(S0);
        meet();
        load(kt + FT_NS, cur);
        fragments(nxt, S0);
        multiply(S1);
    };
    int kt = 0;
    for (; kt + 4 <= KF; kt += 4) {
        step(kt, S0, S1);
        step(kt + 1, S1, S2);
        step(kt + 2, S2, S3);
        step(kt + 3, S3, S0);
    }
    if (kt < KF) step(kt, S0, S1);
    if (kt + 1 < KF) step(kt + 1, S1, S2);
    if (kt + 2 < KF) step(kt + 2, S2, S3);
    if (KT > KF) multiply(S0);      // (64 bytes left: the first half of a step, whose fragments the step in front has read)
    __builtin_amdgcn_s_waitcnt(0x0f70);
    if constexpr (EPI == 2) {
        // the tile goes through LDS once so that a wave owns whole rows (lane = dim), the shape and operation order of the stand-alone row kernel
        __syncthreads();
        float* s_c = (float*)s0;
        static_assert(STAGE >= FT_BM * 64 * 4, "");
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = wm * 32 + i * 16 + fr;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int c = wn * 32 + j * 16 + fk * 4;
                *(float4*)(s_c + r * 64 + c) = make_float4(acc[i][j][0] * (as[i] * ws[j].x), acc[i][j][1] * (as[i] * ws[j].y), acc[i][j][2] * (as[i] * ws[j].z),
                                                           acc[i][j][3] * (as[i] * ws[j].w));
            }
        }
        __syncthreads();
        const int head = nt, nh = ta.nh, kvh = ta.kvh, hd = 64, half = 32;
        const bool is_q = head < nh, is_v = head >= nh + kvh;
        const float* nw = is_q ? ta.qw : ta.kw;
        const float qk_w = nw && !is_v ? nw[lane] : 1.0f;
        // four rows at a time: their chains of sums run side by side
#pragma unroll
        for (int j0 = 0; j0 < 16; j0 += 4) {
            if (wid + 4 * j0 >= rows) break;
            float x[4], cc[4], sn[4];
            int pos[4], pb[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int j = j0 + k, rj = min(wid + 4 * j, rows - 1);
                pos[k] = __builtin_amdgcn_readlane(qk_pos, j), pb[k] = __builtin_amdgcn_readlane(qk_pb, j);
                x[k] = s_c[rj * 64 + lane];
                const float* cs = ta.rope_tab + (int64_t)pos[k] * 64;
                cc[k] = cs[lane & 31], sn[k] = cs[32 + (lane & 31)];
            }
            if (!is_v) {
                float ss[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) ss[k] = wave_sum(__builtin_fmaf(x[k], x[k], 0.0f));
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float rr = nw ? rsqrtf(ss[k] / (float)hd + ta.qk_eps) : 1.0f;
                    const float self = nw ? x[k] * rr * qk_w : x[k];
                    const float partner = lane_xor(self, 32);
                    const float other = lane < half ? -partner : partner;
                    x[k] = self * cc[k] + other * sn[k];
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int rj = wid + 4 * (j0 + k);
                if (rj >= rows) break;
                const int64_t t = row0 + rj;
                const int64_t cache_row = ((int64_t)pb[k] * ta.block + pos[k] % ta.block) * kvh;  // in heads
                if (is_q) ta.q_out[(t * nh + head) * hd + lane] = x[k];
                else if (pb[k] >= 0) kv_store(is_v ? ta.v_cache : ta.k_cache, (cache_row + (head - nh - (is_v ? kvh : 0))) * hd + lane, x[k], ta.kv_dtype);
            }
        }
        return;
    }
    // the weights are the left operand: a lane holds four neighbouring columns of a row
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = wm * 32 + i * 16 + fr;
        if (r >= rows) continue;
        if (EPI == 1) {
            const int c = nt * COLS + wn * 16 + fk * 4;
            if (c >= I) continue;
            const float sg[4] = {ws[0].x, ws[0].y, ws[0].z, ws[0].w}, su[4] = {ws[1].x, ws[1].y, ws[1].z, ws[1].w};
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float gate = acc[i][0][k] * (as[i] * sg[k]), up = acc[i][1][k] * (as[i] * su[k]);
                v[k] = (gate / (1.0f + expf(-gate))) * up;
            }
            *(float4*)(p.C + crow[i] * I + c) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int c = nt * COLS + wn * 32 + j * 16 + fk * 4;
                if (c >= N) continue;
                float4 v = make_float4(acc[i][j][0] * (as[i] * ws[j].x), acc[i][j][1] * (as[i] * ws[j].y), acc[i][j][2] * (as[i] * ws[j].z), acc[i][j][3] * (as[i] * ws[j].w));
                if (p.c_add) {
                    const float4 h = *(const float4*)(p.c_add + crow[i] * N + c);
                    v = make_float4(h.x + v.x, h.y + v.y, h.z + v.z, h.w + v.w);
                }
                *(float4*)(p.C + crow[i] * N + c) = v;
            }
        }
    }
}

static int ft_check(const i64h_fp8_codes_desc* d, int epilogue, const char* who) {
    I64H_CHECK_ARG(d->M >= 0 && d->M < (1ll << 31) && d->N > 0 && d->K > 0 && d->K % 64 == 0, "%s: bad sizes (K=%d: a multiple of 64)", who, d->K);
    I64H_CHECK_ARG(d->N % (epilogue == 1 ? 32 : 16) == 0, "%s: N=%d must be whole blocks of 16 columns", who, d->N);
    I64H_CHECK_ARG(d->A && d->a_scale && d->B && d->b_scale, "%s: null operand", who);
    I64H_CHECK_ARG((((uintptr_t)d->A | (uintptr_t)d->B | (uintptr_t)d->C | (uintptr_t)d->c_add | (uintptr_t)d->b_scale) & 15) == 0, "%s: operands must be 16-byte aligned", who);
    I64H_CHECK_ARG(d->num_groups >= 1 && d->num_groups <= 4096 && (d->group_offsets != nullptr || d->num_groups == 1), "%s: bad grouping", who);
    I64H_CHECK_ARG(d->a_src_row == nullptr || d->a_src_mod > 0, "%s: a_src_row needs a_src_mod > 0", who);
    I64H_CHECK_ARG(d->c_add == nullptr || epilogue == 0, "%s: c_add goes with the plain epilogue", who);
    I64H_CHECK_ARG((d->a_src_row ? d->a_src_mod : d->M) * (int64_t)d->K < 0xffff0000ll && (int64_t)d->N * d->K < 0xffff0000ll, "%s: an operand beyond 32-bit offsets", who);
    return 0;
}
static int64_t ft_blocks(const i64h_fp8_codes_desc* d, int epilogue) {
    if (d->M == 0) return 0;
    const int cols = epilogue == 1 ? FT_BN / 2 : FT_BN, nout = epilogue == 1 ? d->N / 2 : d->N;
    return ((d->M + FT_BM - 1) / FT_BM + (d->group_offsets ? d->num_groups : 0)) * (int64_t)ft_pad_tiles((nout + cols - 1) / cols);
}

__global__ __launch_bounds__(256) void quantize_fp8_rows_pair_kernel(const float* __restrict__ x0, int64_t rows0, int K0, uint8_t* __restrict__ q0, float* __restrict__ sc0,
                                                                     const float* __restrict__ x1, int64_t rows1, int K1, uint8_t* __restrict__ q1, float* __restrict__ sc1) {
    // a wave a row, up to eight slices of four columns in its registers at a time (two reads of a longer row)
    const int lane = threadIdx.x & 63;
    int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool second = row >= (rows0 + 3) / 4 * 4;
    if (second) row -= (rows0 + 3) / 4 * 4;
    if (row >= (second ? rows1 : rows0)) return;
    const int K = second ? K1 : K0, nv = K / 4;
    const float4* xr = (const float4*)((second ? x1 : x0) + row * K);
    uint32_t* qr = (uint32_t*)((second ? q1 : q0) + row * K);
    auto amax = [](float m, float4 v) { return fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)))); };
    float4 v[8];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int i = lane + 64 * j;
        v[j] = i < nv ? xr[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) m = amax(m, v[j]);
    for (int i = lane + 512; i < nv; i += 64) m = amax(m, xr[i]);
    m = wave_max(m);
    const float s = fmaxf(m, 1e-12f) / 448.0f;
    if (lane == 0) (second ? sc1 : sc0)[row] = s;
    with_div_by(s, [&](auto dv) {
        auto q4 = [&](float4 x) -> uint32_t { return pack4_e4m3fn(clamp448(dv(x.x)), clamp448(dv(x.y)), clamp448(dv(x.z)), clamp448(dv(x.w))); };
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (lane + 64 * j < nv) qr[lane + 64 * j] = q4(v[j]);
        for (int i = lane + 512; i < nv; i += 64) qr[i] = q4(xr[i]);
    });
}

extern "C" {

int i64h_gemm_fp8_codes_pair(const i64h_fp8_codes_desc* a, const i64h_fp8_codes_desc* b, int32_t epilogue, void* stream) {
    I64H_CHECK_ARG(a != nullptr, "gemm_fp8_codes_pair: first problem missing");
    I64H_CHECK_ARG(epilogue == 0 || epilogue == 1, "gemm_fp8_codes_pair: epilogue %d", epilogue);
    if (ft_check(a, epilogue, "gemm_fp8_codes[0]") || (b && ft_check(b, epilogue, "gemm_fp8_codes[1]"))) return 1;
    I64H_CHECK_ARG(a->C && (!b || b->C), "gemm_fp8_codes_pair: null result");
    Fp8CodesPair pp;
    pp.p[0] = *a;
    pp.p[1] = b ? *b : *a;
    const int64_t n0 = ft_blocks(a, epilogue), n1 = b ? ft_blocks(b, epilogue) : 0;
    I64H_CHECK_ARG(n0 + n1 < (1ll << 31), "gemm_fp8_codes: grid too large");
    if (n0 + n1 == 0) return 0;
    pp.nblk0 = (int)n0;
    RowTailArgs ta;
    memset(&ta, 0, sizeof(ta));
    if (epilogue) hipLaunchKernelGGL(gemm_fp8_tile_kernel<1>, dim3((unsigned)(n0 + n1)), dim3(256), 0, (hipStream_t)stream, pp, ta);
    else hipLaunchKernelGGL(gemm_fp8_tile_kernel<0>, dim3((unsigned)(n0 + n1)), dim3(256), 0, (hipStream_t)stream, pp, ta);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_gemm_fp8_codes_qkv_rope_kv(const i64h_fp8_codes_desc* d, const float* q_norm_w, const float* k_norm_w, float qk_eps, const float* rope_tab,
                                    const int32_t* positions, const int32_t* slot_ids, const int32_t* block_table, int32_t max_blocks_per_seq, float* q_out,
                                    void* k_cache, void* v_cache, int32_t kv_dtype, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                    void* stream) {
    I64H_CHECK_ARG(d != nullptr, "gemm_fp8_codes_qkv_rope_kv: problem missing");
    if (ft_check(d, 2, "gemm_fp8_codes_qkv_rope_kv")) return 1;
    I64H_CHECK_ARG(d->group_offsets == nullptr && d->a_src_row == nullptr && d->c_row_map == nullptr && d->c_add == nullptr,
                   "gemm_fp8_codes_qkv_rope_kv: one group, no row maps, no residual");
    I64H_CHECK_ARG(head_dim == 64 && d->N == (num_heads + 2 * num_kv_heads) * 64,
                   "gemm_fp8_codes_qkv_rope_kv: head_dim %d / N %d unsupported (head_dim 64, N = (heads + 2 kv heads) * 64)", head_dim, d->N);
    I64H_CHECK_ARG(kv_dtype >= 0 && kv_dtype <= 4 && block_size > 0, "gemm_fp8_codes_qkv_rope_kv: bad kv dtype / block size");
    I64H_CHECK_ARG(positions && slot_ids && block_table && rope_tab && q_out && k_cache && v_cache, "gemm_fp8_codes_qkv_rope_kv: null argument");
    if (d->M == 0) return 0;
    RowTailArgs ta;
    memset(&ta, 0, sizeof(ta));
    ta.positions = positions; ta.slot_ids = slot_ids; ta.block_table = block_table; ta.max_blocks_per_seq = max_blocks_per_seq;
    ta.rope_tab = rope_tab; ta.qw = q_norm_w; ta.kw = k_norm_w; ta.qk_eps = qk_eps; ta.q_out = q_out; ta.k_cache = k_cache; ta.v_cache = v_cache;
    ta.kv_dtype = kv_dtype; ta.nh = num_heads; ta.kvh = num_kv_heads; ta.block = block_size;
    Fp8CodesPair pp;
    pp.p[0] = pp.p[1] = *d;
    const int64_t n0 = ft_blocks(d, 2);
    I64H_CHECK_ARG(n0 < (1ll << 31), "gemm_fp8_codes_qkv_rope_kv: grid too large");
    pp.nblk0 = (int)n0;
    hipLaunchKernelGGL(gemm_fp8_tile_kernel<2>, dim3((unsigned)n0), dim3(256), 0, (hipStream_t)stream, pp, ta);
    I64H_CHECK_LAUNCH();
    return 0;
}

int i64h_quantize_fp8_rows_pair(const float* x0, int64_t rows0, int32_t K0, uint8_t* q0, float* scale0, const float* x1, int64_t rows1, int32_t K1, uint8_t* q1,
                                float* scale1, void* stream) {
    I64H_CHECK_ARG(rows0 >= 0 && rows1 >= 0 && rows0 + rows1 < (1ll << 31) && K0 > 0 && K0 % 4 == 0 && (rows1 == 0 || (K1 > 0 && K1 % 4 == 0)), "quantize_fp8_rows_pair: bad sizes");
    I64H_CHECK_ARG((((uintptr_t)x0 | (uintptr_t)x1) & 15) == 0 && (((uintptr_t)q0 | (uintptr_t)q1) & 3) == 0, "quantize_fp8_rows_pair: alignment");
    const int64_t blocks = (rows0 + 3) / 4 + (rows1 + 3) / 4;
    if (blocks == 0) return 0;
    hipLaunchKernelGGL(quantize_fp8_rows_pair_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, x0, rows0, (int)K0, q0, scale0, x1, rows1, (int)K1, q1, scale1);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
