// Tied fp32 lm_head of a decode-sized step: logits[M, N] = A[M, K] @ B[N, K]^T with both operands fp32 (the reference computes
// F.linear(hidden.float(), embed.weight.float()), vllm_i64/models/complexity_deep/model.py:436-437), N = vocabulary.
//
// The f32 matrix-core instruction (v_mfma_f32_16x16x4_f32, 32 cycles for 4 deep) needs more matrix-core time for this product than
// its 131 MB of weights need to stream from HBM.  Here every fp32 value is cut into three bf16 terms by truncation
// (hi + mid + lo == the value, bit for bit: 8 + 8 + 8 significant bits), every bf16 x bf16 product is exact in fp32, and the six
// products whose weight is at least 2^-16 of the leading one (hi.hi, hi.mid, mid.hi, mid.mid, hi.lo, lo.hi) run on
// v_mfma_f32_16x16x32_bf16 (16 cycles for 32 deep): 96 instead of 256 matrix-core cycles per 32-deep step, fp32 accumulation.  The
// dropped products are below 2^-24 of the leading one, the rounding of one fp32 multiply.
// The activation rows (few, shared by every workgroup) are cut once by a small kernel into three bf16 planes, stored as the
// matrix-core fragments themselves; the weight rows, each used by one wave of one workgroup only, are cut in registers.
// Weight rows are K-major and the matrix-core operand wants lane = column: loading them in operand order makes every lane of a
// load instruction its own 16-byte request (64 requests per instruction, the address path's limit long before HBM's: measured
// 47-50 us whatever the prefetch depth).  So a wave loads weight rows in memory order and turns them into operand order through
// a private LDS strip.  A branch around a load makes the compiler wait for ALL loads in flight (it can no longer count them):
// every load here is unconditional, on clamped addresses.
#include <type_traits>

#include "i64h_common.h"

typedef float lm_v4f __attribute__((ext_vector_type(4)));
typedef uint32_t lm_v4u __attribute__((ext_vector_type(4)));
typedef __bf16 lm_v8b __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t lm_top(float x, float y) { return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u); }
__device__ __forceinline__ void lm_split_pair(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const float xr = x - __uint_as_float(__float_as_uint(x) & 0xffff0000u), yr = y - __uint_as_float(__float_as_uint(y) & 0xffff0000u);
    const float xl = xr - __uint_as_float(__float_as_uint(xr) & 0xffff0000u), yl = yr - __uint_as_float(__float_as_uint(yr) & 0xffff0000u);
    hi = lm_top(x, y);
    mid = lm_top(xr, yr);
    lo = lm_top(xl, yl);
}

// ---- K split over the waves of a workgroup -------------------------------------------------------------------------------------
// Wave w of a workgroup (64 rows x 64 vocabulary columns) contracts the w-th quarter of K for the WHOLE tile: its activation
// fragments come straight from L2 in matrix-core lane order (the split kernel writes them that way: one fragment = 1 KB of
// consecutive bytes), each used for four column fragments, so the activation planes never pass through LDS and the main loop has
// no workgroup barrier; its weight rows arrive in memory order (128-byte pieces, 8 lanes per row) and turn into operand order in
// a wave-private LDS strip.  The four partial tiles are summed through LDS at the end, in wave order.
#define LMK_LD 40  // strip row stride in floats (conflict-free for the operand-order ds_read_b128)

// planes in fragment order: [row tile][K step][p][row fragment i][lane (fr, fq)][8 bf16], element e of the lane = k 4 fq + e (e < 4),
// 16 + 4 fq + (e - 4) (e >= 4) of row 16 i + fr
__global__ __launch_bounds__(256) void lm_split_rows_frag_kernel(const float* __restrict__ A, const int32_t* __restrict__ a_rows, uint32_t* __restrict__ planes,
                                                                 int M, int K, int Kpad) {
    const int r = blockIdx.x;
    const int64_t src = r < M ? (a_rows ? a_rows[r] : r) : 0;
    const float2* x = (const float2*)(A + src * K);
    const int KTP = Kpad / 32;
    for (int i = threadIdx.x; i < Kpad / 2; i += 256) {
        uint32_t hi = 0, mid = 0, lo = 0;
        if (r < M && i < K / 2) {
            const float2 v = x[i];
            lm_split_pair(v.x, v.y, hi, mid, lo);
        }
        const int blk = i & 15, q = (blk & 7) >> 1, e2 = (blk & 1) + 2 * (blk >> 3);
        const int64_t frag = ((int64_t)(r >> 6) * KTP + (i >> 4)) * 12 + ((r & 63) >> 4);  // + 4 p
        const int64_t o = (frag * 64 + q * 16 + (r & 15)) * 4 + e2;
        planes[o] = hi;
        planes[o + 4 * 256] = mid;
        planes[o + 8 * 256] = lo;
    }
}

// MF: fragments of 16 rows that there are (few rows need neither the products nor the activation fragments of a 64-row tile, and the registers these leave hold more
// weights on their way); AHEAD: steps of weights in registers, beside the one in the strip.
// us, 32000 columns of 1024, weights from memory (131 MB: 28 at the copy rate), all rows as 64 | so: 1 to 16 rows 36.5 | 30.5, 17 to 32 rows 37 | 32.5.  (64 rows 40: their activation
// fragments are 196 MB from L2; cut weights held for two halves of the rows, with a step more on its way, spill: 51.)
template <int MF, int AHEAD>
__global__ __launch_bounds__(256, 2) void lm_head_bf16x3_ks_kernel(const uint32_t* __restrict__ planes, const float* __restrict__ B, float* __restrict__ C,
                                                                   int M, int N, int K, int Kpad) {
    constexpr int TILE = 16 * MF * 64, STRIPS = 4 * 64 * LMK_LD;      // floats: a wave's partial tile, the strips of all
    __shared__ __attribute__((aligned(16))) float smem[4 * TILE > STRIPS ? 4 * TILE : STRIPS];  // strips during the loop, the partial tiles after it
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int fr = lane & 15, fq = lane >> 4;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int KT = K / 32, KTP = Kpad / 32, S = KTP / 4;  // S steps per wave (Kpad is a multiple of 256: an even number)
    const int k_first = wid * S;
    float* strip = smem + wid * (64 * LMK_LD);
    // weight loads: instruction j takes rows 8 j .. 8 j + 7 of the tile, 128 contiguous bytes each (one K step)
    const int wr = lane >> 3, wc = (lane & 7) * 4;
    const float* Bt = B + (int64_t)n0 * K;
    uint32_t wrow[8];      // (bytes from the tile's first row)
#pragma unroll
    for (int j = 0; j < 8; ++j) wrow[j] = ((uint32_t)min(8 * j + wr, N - 1 - n0) * (uint32_t)K + wc) * 4u;
    const lm_v4u* ap = (const lm_v4u*)planes + ((int64_t)blockIdx.y * KTP * 12) * 64 + lane;  // fragment f = 4 p + i of step kt: ap[(kt * 12 + f) * 64]
    lm_v4f acc[MF][4];
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[i][c] = (lm_v4f){0.f, 0.f, 0.f, 0.f};
    lm_v4f g[AHEAD][8];
    lm_v4u af[2][3 * MF];
    // no branch around a load (the waits are counted): steps past the wave's share re-read its last step, steps past K read the
    // row's last step against zero planes
    auto wload = [&](int s, lm_v4f (&x)[8]) {
        const int kt = min(k_first + min(s, S - 1), KT - 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = *(const lm_v4f*)((const char*)(Bt + kt * 32) + wrow[j]);
    };
    auto aload = [&](int s, lm_v4u (&x)[3 * MF]) {
        const int64_t kt = k_first + min(s, S - 1);
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < MF; ++i) x[p * MF + i] = ap[(kt * 12 + 4 * p + i) * 64];
    };
    auto wstore = [&](const lm_v4f (&x)[8]) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j) *(lm_v4f*)&strip[(8 * j + wr) * LMK_LD + wc] = x[j];
        __builtin_amdgcn_wave_barrier();
    };
    auto multiply = [&](const lm_v4u (&x)[3 * MF]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const lm_v4f w0 = *(const lm_v4f*)&strip[(16 * c + fr) * LMK_LD + fq * 4];
            const lm_v4f w1 = *(const lm_v4f*)&strip[(16 * c + fr) * LMK_LD + 16 + fq * 4];
            lm_v4u bh, bm, bl;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t hi, mid, lo;
                lm_split_pair(e < 2 ? w0[2 * e] : w1[2 * e - 4], e < 2 ? w0[2 * e + 1] : w1[2 * e - 3], hi, mid, lo);
                bh[e] = hi, bm[e] = mid, bl[e] = lo;
            }
            const lm_v8b b1 = __builtin_bit_cast(lm_v8b, bh), b2 = __builtin_bit_cast(lm_v8b, bm), b3 = __builtin_bit_cast(lm_v8b, bl);
#pragma unroll
            for (int i = 0; i < MF; ++i) {
                const lm_v8b a1 = __builtin_bit_cast(lm_v8b, x[i]), a2 = __builtin_bit_cast(lm_v8b, x[MF + i]), a3 = __builtin_bit_cast(lm_v8b, x[2 * MF + i]);
                lm_v4f t = acc[i][c];
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a3, b1, t, 0, 0, 0);  // small terms first
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b3, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b2, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b1, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b2, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, t, 0, 0, 0);
                acc[i][c] = t;
            }
        }
    };
    // a step: its weights are in the strip, those of the next AHEAD in registers
    auto step = [&](int s, auto at) {
        constexpr int U = decltype(at)::value;
        // the scheduling barrier keeps the next steps' requests IN FRONT of this step's matrix-core instructions (left alone, the
        // scheduler sinks them behind the MFMAs, i.e. right in front of their use)
        aload(s + 1, af[(U + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(af[U & 1]);
        wstore(g[U % AHEAD]);      // step s + 1's weight rows replace step s's in the strip
        wload(s + 1 + AHEAD, g[U % AHEAD]);
    };
    wload(0, g[0]);
    aload(0, af[0]);
    wstore(g[0]);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) wload(1 + u, g[u]);
    constexpr std::integral_constant<int, 0> U0{};
    constexpr std::integral_constant<int, 1> U1{};
    constexpr std::integral_constant<int, 2> U2{};
    constexpr std::integral_constant<int, 3> U3{};
    int s = 0;
    for (; s + 4 <= S; s += 4) step(s, U0), step(s + 1, U1), step(s + 2, U2), step(s + 3, U3);
    if (s < S) step(s, U0), step(s + 1, U1);
    // the four partial tiles through LDS (the strips are dead: every wave is past its last read once the barrier is passed)
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int reg = 0; reg < 4; ++reg) smem[wid * TILE + (i * 16 + fq * 4 + reg) * 64 + c * 16 + fr] = acc[i][c][reg];
    __syncthreads();
    for (int e = tid; e < 16 * MF * 16; e += 256) {  // four consecutive columns per thread
        const int r = e >> 4, c4 = (e & 15) * 4;
        if (m0 + r >= M) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ((smem[r * 64 + c4 + j] + smem[TILE + r * 64 + c4 + j]) + smem[2 * TILE + r * 64 + c4 + j]) + smem[3 * TILE + r * 64 + c4 + j];
        float* cp = C + (int64_t)(m0 + r) * N + n0 + c4;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (n0 + c4 + j < N) cp[j] = v[j];
    }
}

static void lm_head_launch(const void* planes, const float* B, float* C, int64_t M, int32_t N, int32_t K, hipStream_t st) {
    const dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
    auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (const uint32_t*)planes, B, C, (int)M, (int)N, (int)K, (K + 255) / 256 * 256); };
    if (M <= 16) launch(lm_head_bf16x3_ks_kernel<1, 4>);
    else if (M <= 32) launch(lm_head_bf16x3_ks_kernel<2, 2>);
    else launch(lm_head_bf16x3_ks_kernel<4, 1>);
}

extern "C" {

// bytes of the workspace i64h_lm_head needs for M rows of K elements
int64_t i64h_lm_head_workspace_bytes(int64_t M, int32_t K) { return ((M + 63) / 64 * 64) * (int64_t)((K + 255) / 256 * 256) * 2 * 3; }

// C[M, N] = A[a_rows ? a_rows[r] : r, :K] @ B[N, K]^T, fp32 operands, on the bf16 matrix cores through the exact three-term
// split (six of the nine partial products).  K % 32 == 0; workspace: i64h_lm_head_workspace_bytes(M, K), 16-byte aligned.
int i64h_lm_head(const float* A, const int32_t* a_rows, const float* B, float* C, int64_t M, int32_t N, int32_t K, void* workspace, void* stream) {
    I64H_CHECK_ARG(M >= 0 && M < (1ll << 24) && N > 0 && K > 0 && K % 32 == 0, "lm_head: K=%d must be a multiple of 32", K);
    I64H_CHECK_ARG(workspace && ((uintptr_t)workspace | (uintptr_t)A | (uintptr_t)B) % 16 == 0, "lm_head: workspace missing or operands not 16-byte aligned");
    if (M == 0) return 0;
    const int Mpad = (int)((M + 63) / 64 * 64), Kpad = (K + 255) / 256 * 256;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(lm_split_rows_frag_kernel, dim3((unsigned)Mpad), dim3(256), 0, st, A, a_rows, (uint32_t*)workspace, (int)M, (int)K, Kpad);
    I64H_CHECK_LAUNCH();
    lm_head_launch(workspace, B, C, M, N, K, st);
    I64H_CHECK_LAUNCH();
    return 0;
}

// i64h_lm_head on activation planes that are already in the workspace (written by i64h_fused_residual_norm_lm for the rows 0 .. M - 1
// in order): the main launch only.
int i64h_lm_head_planes(const void* workspace, const float* B, float* C, int64_t M, int32_t N, int32_t K, void* stream) {
    I64H_CHECK_ARG(M >= 0 && M < (1ll << 24) && N > 0 && K > 0 && K % 32 == 0, "lm_head_planes: K=%d must be a multiple of 32", K);
    I64H_CHECK_ARG(workspace && ((uintptr_t)workspace | (uintptr_t)B) % 16 == 0, "lm_head_planes: workspace missing or operands not 16-byte aligned");
    if (M == 0) return 0;
    lm_head_launch(workspace, B, C, M, N, K, (hipStream_t)stream);
    I64H_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
