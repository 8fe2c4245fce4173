// Q4_0 / Q8_0 mat-mat for prompts on the matrix cores, BIT-EXACT with the reference's x86 AVX2 arm (the contract of mmvq.hip):
//
//   out[t][row] = residual[t][row] + vec_dot(W[row], act[t])
//
// Reference: ggml_vec_dot_q4_0_q8_0 (ggml-quants.c:2500-2523), ggml_vec_dot_q8_0_q8_0 (:3584-3605).  Per block of 32 values the AVX2 code has eight lanes; lane k is the integer dot product of
// values 4k .. 4k+3, converted to float, and extends its own fp32 chain by one fma per block in block order:  acc[k] = fma(d_x * d_y, (float) dot4, acc[k]).  The eight chains are folded at the end.
//
// What bounds it.  A block of one (row, token) pair is eight fma that may not be re-ordered or merged, plus one product of the scales: VALU issue, whatever computes the integer part.  That is
// v_mfma_f32_16x16x4_4b_f16 here: its K is exactly the four values of a lane, its four blocks are four lanes k of 16 rows x 16 tokens, its result is the converted float (integers of at most 128 * 128 * 4 = 2^16: exact in f16
// operands and fp32 sums), and it runs beside the fma of the product before it.  (v_mfma_f32_4x4x4_16b_f16, one lane k at a time, issues four times as often: with 32 fma 175 ns, 156 here.)
//
// A lane of a wave (row r, c) needs lanes k = c and c + 4 of its row: 16 contiguous bytes of a group of four blocks, which go from memory to its registers and are converted there, once for the TT token tiles that the wave
// owns.  The tokens' operands are converted once per workgroup, into LDS; a group has one barrier, loads are a group ahead, LDS reads a block (a single tile: two).  Few tokens: two waves share a row tile's lanes k, so that a
// block's serial chain is half as long.  Matrices that share their activations (q, k, v; up and gate) are one launch: its rounds fill better.
// Measured (Q4_0, us for 4096 x 4096 / 11008 x 4096, before / now): 16 tokens 34 / 25, 35 / 30; 32: 41 / 25, 44 / 36; 64: 60 / 34, 64 / 51; 128: 62 / 40, 110 / 89; 333: 114 / 75, 266 / 207; 512: 123 / 96 (179 TFLOP/s),
// 327 / 269; Q8_0 4096 x 4096 16 tokens 31 / 27, 333: 112 / 81, 11008 x 4096 16 tokens 33 / 31, 32: 41 / 36.  In a full round of 128 rows x 64 tokens the VALU issues in 86 % of the cycles.
#include "mmvq_args.h"
#include <hip/hip_ext.h>

#include <cstdlib>
#include <cstring>
#include <type_traits>

using q0_half4 = __attribute__((ext_vector_type(4))) _Float16;
using q0_half2 = __attribute__((ext_vector_type(2))) _Float16;
typedef uint32_t q0_u32x4 __attribute__((ext_vector_type(4)));
using q0_f32x4 = __attribute__((ext_vector_type(4))) float;
using q0_f32x16 = __attribute__((ext_vector_type(16))) float;

static __device__ __forceinline__ uint32_t q0_add(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(q0_half2, a) + __builtin_bit_cast(q0_half2, b)); }
static __device__ __forceinline__ uint32_t q0_fma(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(q0_half2, a), __builtin_bit_cast(q0_half2, b), __builtin_bit_cast(q0_half2, c)));
}
// four signed bytes -> four f16, in the order 0, 2, 1, 3: 0x6400 + u is 1024 + u (u = byte + 128), so one byte permutation and one packed addition per pair
static __device__ __forceinline__ uint2 q0_int8(uint32_t x) {
    const uint32_t u = x ^ 0x80808080u;
    return make_uint2(q0_add(__builtin_amdgcn_perm(0x64646464u, u, 0x04020400u), 0xE480E480u), q0_add(__builtin_amdgcn_perm(0x64646464u, u, 0x04030401u), 0xE480E480u));
}
// low / high nibbles of four bytes, minus 8, in the same order: 1024 + n, and 1024 + 16 n times 1 / 16
static __device__ __forceinline__ uint2 q0_low(uint32_t x, uint32_t magic) { return make_uint2(q0_add((x & 0x000F000Fu) | magic, 0xE408E408u), q0_add(((x >> 8) & 0x000F000Fu) | magic, 0xE408E408u)); }
static __device__ __forceinline__ uint2 q0_high(uint32_t x, uint32_t magic) {
    return make_uint2(q0_fma((x & 0x00F000F0u) | magic, 0x2C002C00u, 0xD480D480u), q0_fma(((x >> 8) & 0x00F000F0u) | magic, 0x2C002C00u, 0xD480D480u));
}
// the product of four lanes k at once: block c of the instruction is (token, lane c) of a against (row, lane c) of b
static __device__ __forceinline__ q0_f32x16 q0_mfma(uint2 a, uint2 b) {
    const q0_f32x16 z = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
    return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(q0_half4, a), __builtin_bit_cast(q0_half4, b), z, 0, 0, 0);
}
// workgroup barrier that waits for all but the last N of this wave's LDS operations (they end in order); loads stay in flight across it
template <int N> static __device__ __forceinline__ void q0_barrier() { asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" :: "n"(N) : "memory"); }
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t q0_rsrc(const void * p, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00027000); }

// WR row tiles a workgroup (one per wave; KS = 2: one per two waves, which share out the lanes k: 0 .. 3 and 4 .. 7), TT token tiles
template <int TYPE, int WR, int TT, int KS>
__global__ void __launch_bounds__(64 * WR * KS) k_mmq_q0(const mmvq_args g, const int row_blocks, const int tok_blocks) {
    if (pi_aborted(g.abort_w, 1)) return;
    constexpr bool Q8 = TYPE == PI_Q8_0;
    constexpr int NTHR = 64 * WR * KS, NH = 2 / KS, NK = 8 / KS, U = (TT * 256 + NTHR - 1) / NTHR;     // products of a tile, lanes k of a wave; staging: 16-byte operands a thread converts per group (a token's blocks (U) b .. of one pair of lanes k)
    constexpr int UB = U == 3 ? 4 : U;                                  // blocks of a thread: 1, 2 or all four
    constexpr int OPS = NTHR * UB * 16, BUF = OPS + NTHR * 4;           // LDS image of a group: operands [tile][block][64], scales [tile][block][16] (both with what the threads past them write)
    static_assert(UB <= 4 && NTHR * UB >= TT * 256 && NTHR >= TT * 64, "the workgroup stages a group in one go");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // the token blocks of one row block run on one XCD (workgroup n goes to XCD n % 8): its weights come from HBM once
    const int slot = blockIdx.x >> 3, rb = (blockIdx.x & 7) + 8 * (slot / tok_blocks), tb = slot % tok_blocks;
    if (rb >= row_blocks) return;
    const int si = (rb >= g.seg[1].wave0) + (rb >= g.seg[2].wave0);     // (wave0: the segment's first row block)
    const mmvq_seg & sg = g.seg[si];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, c = lane >> 4;
    const int ks = KS == 2 ? wave & 1 : 0, row0 = ((rb - sg.wave0) * WR + wave / KS) * 16, tok0 = tb * TT * 16, ng = g.nb;                            // ng: groups of four blocks
    const int first = min(row0, sg.M - 1);                              // rows and tokens past the end repeat the last one and are not stored
    const uint32_t my_row = (uint32_t) min(row0 + r, sg.M - 1) - (uint32_t) first;
    uint32_t magic = 0x64006400u;
    asm volatile("" : "+v"(magic));
    // ---- weights: lane (row r, c) needs lanes k = c and c + 4 of its row's blocks, which is 16 contiguous bytes of a group (Q8_0: two times 16): global -> registers, converted by the wave that uses them ----
    constexpr uint32_t A_GROUP = Q8 ? 128 : 64;
    const __amdgpu_buffer_rsrc_t wr = q0_rsrc(sg.p0 + (int64_t) first * ng * A_GROUP, 16u * ng * A_GROUP), dr = q0_rsrc(sg.p1 + (int64_t) first * ng * 8, 16u * ng * 8);
    const uint32_t w_off = my_row * ng * A_GROUP + 16 * c + (Q8 ? 64 * ks : 0), d_off = my_row * ng * 8;
    struct weights { q0_u32x4 q, q2; uint2 d; };
    auto load_w = [&](int gi, weights & W) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t) min(gi, ng - 1);
        W.q = __builtin_bit_cast(q0_u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, w_off, at * A_GROUP, 0));
        if constexpr (Q8 && KS == 1) W.q2 = __builtin_bit_cast(q0_u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + 64, at * A_GROUP, 0));
        W.d = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(dr, d_off, at * 8, 0));
    };
    // ---- activations: global -> registers -> f16 in operand order -> LDS ----
    const int s_unit = tid * UB, s_tile = min(s_unit >> 8, TT - 1), s_lane = UB == 4 ? tid & 63 : UB == 2 ? (tid >> 1) & 63 : (tid >> 2) & 63, s_b = s_unit & 3;
    const int toks = min(g.nt - tok0, TT * 16);
    const __amdgpu_buffer_rsrc_t yr = q0_rsrc(g.aq + (int64_t) tok0 * ng * 128, (uint32_t) toks * ng * 128), sr = q0_rsrc(g.ad + (int64_t) tok0 * ng * 8, (uint32_t) toks * ng * 8);
    const uint32_t y_off = (uint32_t) min(s_tile * 16 + (s_lane & 15), toks - 1) * ng * 128 + 16 * (s_lane >> 4) + 4 * s_b;
    const uint32_t s_off = (uint32_t) min(min(tid >> 6, TT - 1) * 16 + (tid & 15), toks - 1) * ng * 8 + 2 * ((tid >> 4) & 3);
    uint32_t y[2 * UB]; uint16_t ys;
    auto stage_load = [&](int gi) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t) min(gi, ng - 1) * 128;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if constexpr (UB == 4) {
                const q0_u32x4 v = __builtin_bit_cast(q0_u32x4, __builtin_amdgcn_raw_buffer_load_b128(yr, y_off + 64 * h, at, 0));
#pragma unroll
                for (int b = 0; b < 4; b++) y[h * 4 + b] = v[b];
            } else if constexpr (UB == 2) {
                const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(yr, y_off + 64 * h, at, 0));
                y[h * 2] = v.x; y[h * 2 + 1] = v.y;
            } else y[h] = __builtin_amdgcn_raw_buffer_load_b32(yr, y_off + 64 * h, at, 0);
        }
        ys = __builtin_amdgcn_raw_buffer_load_b16(sr, s_off, at / 16, 0);
    };
    auto stage_store = [&](uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < UB; b++) {
            const uint2 lo = q0_int8(y[b]), hi = q0_int8(y[UB + b]);
            *(uint4 *) (lds + buf + (((s_unit >> 8) * 4 + s_b + b) * 64 + s_lane) * 16) = make_uint4(lo.x, lo.y, hi.x, hi.y);      // (past the last tile: behind the operands)
        }
        *(float *) (lds + buf + OPS + tid * 4) = pi_h2f(ys);
    };
    // ---- a block is TT tiles x two products (lanes k = 0 .. 3, then 4 .. 7).  A step issues the next MFMA, then runs the sixteen fma of the MFMA before; operands of a tile are read a block ahead ----
    q0_f32x4 acc[TT][NK];
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int k = 0; k < NK; k++) acc[t][k] = q0_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    constexpr int AD = TT == 1 ? 2 : 1;                                 // blocks that operands are read ahead (one tile: a block is over before they would be there)
    uint2 a[AD * TT][NH]; float4 dy[AD * TT]; uint2 w[2][NH]; float dx[2];
    auto read_a = [&](int t, int b, uint32_t buf) __attribute__((always_inline)) {
        const uint8_t * at = lds + buf + ((t * 4 + b) * 64 + lane) * 16;
        if constexpr (KS == 2) a[b % AD * TT + t][0] = *(const uint2 *) (at + 8 * ks);
        else { const uint4 v = *(const uint4 *) at; a[b % AD * TT + t][0] = make_uint2(v.x, v.y); a[b % AD * TT + t][NH - 1] = make_uint2(v.z, v.w); }
    };
    auto read_dy = [&](int t, int b, uint32_t buf) __attribute__((always_inline)) { dy[b % AD * TT + t] = *(const float4 *) (lds + buf + OPS + ((t * 4 + b) * 16 + 4 * c) * 4); };
    auto build = [&](const weights & W, int b, int h) __attribute__((always_inline)) {      // block b's operand of lanes k = 4 h + c (KS = 2: 4 ks + c)
        uint2 & x = w[b & 1][h];
        if constexpr (Q8) x = q0_int8(h ? W.q2[b] : W.q[b]);
        else if constexpr (KS == 2) x = q0_low(W.q[b] >> (4 * ks), magic);
        else x = h ? q0_high(W.q[b], magic) : q0_low(W.q[b], magic);
        if (h == 0) dx[b & 1] = pi_h2f((uint16_t) ((b & 2 ? W.d.y : W.d.x) >> (16 * (b & 1))));
    };
    uint32_t buf = 0, buf1 = BUF, buf2 = 2 * BUF;
    q0_f32x16 v;
    // group gi in LDS image buf, its weights W; the next group's: buf1, Wn.  Three images: waves on either side of the group's one barrier read images gi - 1 and gi, and write gi + 1
    auto group = [&](int gi, weights & W, weights & Wn) __attribute__((always_inline)) {
        stage_store(buf1);
        stage_load(gi + 2);
        float p[4];
#pragma unroll
        for (int n = 0; n < 4 * NH * TT; n++) {
            const int b = n / (NH * TT), t = n / NH % TT, h = n % NH, b1 = (b + 1) & 3;
            const int s = b % AD * TT + t, s1 = t + 1 < TT ? s + 1 : b1 % AD * TT;       // slots of this tile and of the next one
            if (h == 0) { p[0] = dx[b & 1] * dy[s].x; p[1] = dx[b & 1] * dy[s].y; p[2] = dx[b & 1] * dy[s].z; p[3] = dx[b & 1] * dy[s].w; }
            if (n == NH * TT * (4 - AD) - 1) q0_barrier<2>();                       // (the image's writes are more than two LDS operations old)
            if (t == TT - 1 && h == 0) { build(b < 3 ? W : Wn, b1, 0); if (NH == 2) build(b < 3 ? W : Wn, b1, NH - 1); }      // the next block's operands
            const q0_f32x16 o = v;
            v = h + 1 < NH ? q0_mfma(a[s][NH - 1], w[b & 1][NH - 1]) : q0_mfma(a[s1][0], t + 1 < TT ? w[b & 1][0] : w[(b + 1) & 1][0]);
            if (h == 0) { read_a(t, (b + AD) & 3, b + AD < 4 ? buf : buf1); read_dy(t, (b + AD) & 3, b + AD < 4 ? buf : buf1); }          // (both products of this tile's operand have left)
            if (n == 4 * NH * TT - NH) load_w(gi + 2, W);                     // (its last block's operands are built)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][4 * h + k][i] = fmaf(p[i], o[4 * k + i], acc[t][4 * h + k][i]);
            __builtin_amdgcn_sched_barrier(0);
        }
        const uint32_t x = buf; buf = buf1; buf1 = buf2; buf2 = x;
    };
    weights W0, W1;
    stage_load(0);
    load_w(0, W0);
    stage_store(0);
    stage_load(1);
    load_w(1, W1);
    q0_barrier<0>();
#pragma unroll
    for (int t = 0; t < AD * TT; t++) { read_a(t % TT, t / TT, 0); read_dy(t % TT, t / TT, 0); }
    build(W0, 0, 0);
    if (NH == 2) build(W0, 0, NH - 1);
    v = q0_mfma(a[0][0], w[0][0]);
    int gi = 0;
    for (; gi + 1 < ng; gi += 2) { group(gi, W0, W1); group(gi + 1, W1, W0); }
    if (gi < ng) group(gi, W0, W1);
    // hsum_float_8: (a4+a0, a5+a1, a6+a2, a7+a3) -> (r0+r2, r1+r3) -> s0+s1
    float * X = (float *) lds + (wave / KS) * (TT * 16 * 64) + lane;    // KS = 2: the second wave's chains [tile][k][i][64]
    if constexpr (KS == 2) {
        __syncthreads();
        if (ks == 1)
#pragma unroll
            for (int e = 0; e < TT * 16; e++) X[e * 64] = acc[e / 16][e / 4 % 4][e & 3];
        __syncthreads();
        if (ks == 1) return;
    }
    const int row = row0 + r;
    if (row >= sg.M) return;
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tok = tok0 + t * 16 + 4 * c + i;
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) x[k] = k < NK ? acc[t][k < NK ? k : 0][i] : X[((t * 4 + (k & 3)) * 4 + i) * 64];
            const float s = ((x[0] + x[4]) + (x[2] + x[6])) + ((x[1] + x[5]) + (x[3] + x[7]));
            if (tok < g.nt) { const int64_t o = (int64_t) tok * sg.M + row; sg.out[o] = sg.res ? sg.res[o] + s : s; }
        }
}

// from seven tokens.  Measured, us k_mmvq_q0 / here: six tokens of 4096 x 4096 24 / 24, 11008 x 4096 30 / 32, 4096 x 11008 62 / 55, 2048 x 2048 12.5 / 13.9 (Q8_0 4096 x 4096 25 / 27); seven 27 / 24, 33 / 32, 70 / 55,
// 14.0 / 13.9 (Q8_0 30 / 27); nine, the second pass over the weights there, 34 / 24, 56 / 32, 92 / 54, 18.5 / 13.8 (Q8_0 38 / 27)
bool pi_mmq_q0_wants(int type, int n_tok) {
    static const int min_tok = getenv("PI_MMQ_Q0_MIN") ? atoi(getenv("PI_MMQ_Q0_MIN")) : 7;
    return (type == PI_Q4_0 || type == PI_Q8_0) && n_tok >= min_tok;
}

template <int TYPE, int WR, int TT, int KS>
static int launch_q0(mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    mmvq_args & g = L.g;
    constexpr int NTHR = 64 * WR * KS, U = (TT * 256 + NTHR - 1) / NTHR, UB = U == 3 ? 4 : U;
    constexpr size_t image = 3 * (size_t) (NTHR * UB * 16 + NTHR * 4), fold = KS == 2 ? (size_t) WR * TT * 4096 : 0, lds = image > fold ? image : fold;
    if (!g.aq) { PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_mmq_q0<TYPE, WR, TT, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); return 0; }      // pi_mmq_q0_reserve
    int rb = 0;
    for (int i = 0; i < MMVQ_MAX_SEG; i++) {
        if (i < L.nseg) { g.seg[i].wave0 = rb; rb += (g.seg[i].M + WR * 16 - 1) / (WR * 16); }
        else { g.seg[i] = g.seg[0]; g.seg[i].wave0 = 0x7fffffff; }
    }
    const int tb = (g.nt + TT * 16 - 1) / (TT * 16);
    const unsigned grid = (unsigned) ((rb + 7) / 8 * 8) * (unsigned) tb;
    if (ea) hipExtLaunchKernelGGL((k_mmq_q0<TYPE, WR, TT, KS>), dim3(grid), dim3(NTHR), lds, stream, ea, eb, 0, g, rb, tb);
    else    hipLaunchKernelGGL((k_mmq_q0<TYPE, WR, TT, KS>), dim3(grid), dim3(NTHR), lds, stream, g, rb, tb);
    PI_CHECK_LAUNCH();
    return 0;
}
template <int TYPE>
static int launch_q0_cfg(int cfg, mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    switch (cfg) {
        case 212: return launch_q0<TYPE, 2, 1, 2>(L, stream, ea, eb);
        case 412: return launch_q0<TYPE, 4, 1, 2>(L, stream, ea, eb);
        case 422: if constexpr (TYPE == PI_Q8_0) return launch_q0<TYPE, 4, 2, 2>(L, stream, ea, eb); else break;      // (Q4_0: 128 x 16 takes as long: 36.1 and 36.6 for 11008 x 4096 at 32 tokens)
        case 81: return launch_q0<TYPE, 8, 1, 1>(L, stream, ea, eb);
        case 83: return launch_q0<TYPE, 8, 3, 1>(L, stream, ea, eb);
        case 84: return launch_q0<TYPE, 8, 4, 1>(L, stream, ea, eb);
        case 82: return launch_q0<TYPE, 8, 2, 1>(L, stream, ea, eb);
    }
    pi_set_error("mmq_q0: configuration %d", cfg);
    return -1;
}
// Which tiles: the shortest estimate of  rounds of workgroups x time of a round, as in mmq_prompt.hip.  A round's time (us for 128 blocks, launch taken off, 4096 columns): rows x tokens of a workgroup 32 x 16 (two of them
// fit a CU; few tokens: a block is the shortest serial chain), 64 x 16 and x 32 (the same chain, and one round where the smallest tile needs more than one to a CU), 128 x 16, x 32, x 48, x 64 (the wider, the fewer
// instructions per tile).  The 64-row tiles against the others' best, us: Q8_0 11008 x 4096 at 9 / 16 / 24 / 32 tokens 29.4 / 31.2 / 36 / 36 and 35.7 / 36.3 / 46 / 48, 6144 x 4096 at 64 36.4 and 46.1; Q4_0 11008 x 4096 at
// 16 30.1 and 33.5, 4096 x 4096 at 48 30.4 and 33.5.  (Where they do not help, Q8_0 22016 and 32000 x 4096 at 16 tokens take 50.7 and 55; the kernel that
// converted its weights once per workgroup, in LDS, took 47.8 and 51: there a wave's conversions serve one tile of tokens.)
static int q0_choose(int type, const mmvq_launch & L) {
    struct tiles { int cfg, wr, tt, per_cu; float one, full; };
    static const tiles q4[] = { { 212, 2, 1, 2, 20.0f, 30.0f }, { 412, 4, 1, 1, 25.0f, 25.0f }, { 81, 8, 1, 1, 32.0f, 32.0f }, { 82, 8, 2, 1, 47.0f, 47.0f }, { 83, 8, 3, 1, 69.0f, 69.0f }, { 84, 8, 4, 1, 89.0f, 89.0f } };
    static const tiles q8[] = { { 212, 2, 1, 2, 23.0f, 30.5f }, { 412, 4, 1, 1, 27.0f, 27.0f }, { 422, 4, 2, 1, 33.0f, 33.0f }, { 81, 8, 1, 1, 41.0f, 41.0f }, { 82, 8, 2, 1, 54.0f, 54.0f }, { 83, 8, 3, 1, 74.0f, 74.0f }, { 84, 8, 4, 1, 95.0f, 95.0f } };
    const tiles * cfgs = type == PI_Q8_0 ? q8 : q4; const int n_cfgs = type == PI_Q8_0 ? 7 : 6;
    int best = 83; float best_t = 1e30f;
    for (int n = 0; n < n_cfgs; n++) {
        const tiles & c = cfgs[n];
        int64_t rb = 0;
        for (int i = 0; i < L.nseg; i++) rb += (L.g.seg[i].M + c.wr * 16 - 1) / (c.wr * 16);
        const int64_t wgs = rb * ((L.g.nt + c.tt * 16 - 1) / (c.tt * 16)), slots = (int64_t) pi_cu_count() * c.per_cu, whole = wgs / slots, rest = wgs % slots;
        // (up to three rounds the last one counts in full; behind more, workgroups of many rounds run past each other and about half a round is lost)
        const float t = whole >= 3 ? c.full * ((float) wgs / slots + 0.5f) : c.full * whole + (rest == 0 ? 0.0f : rest <= pi_cu_count() ? c.one : c.full);
        if (t < best_t) { best_t = t; best = c.cfg; }
    }
    return best;
}
// once per process and outside any stream capture (pi_op_mul_mat_reserve): the instances' dynamic LDS is more than a kernel gets by default
int pi_mmq_q0_reserve() {
    mmvq_launch L; memset(&L.g, 0, sizeof L.g);                        // g.aq == nullptr: the instances only set their attribute
    for (int cfg : { 212, 412, 422, 81, 82, 83, 84 })
        if ((cfg != 422 && launch_q0_cfg<PI_Q4_0>(cfg, L, nullptr, nullptr, nullptr) != 0) || launch_q0_cfg<PI_Q8_0>(cfg, L, nullptr, nullptr, nullptr) != 0) return -1;
    return 0;
}
// the whole pass in one launch (up to three matrices of one type; g.aq / g.ad at the first token, g.nt tokens)
int pi_mmq_q0_launch(int type, mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    if (pi_op_mul_mat_reserve() != 0) return -1;
    const int cfg = q0_choose(type, L);
    return type == PI_Q4_0 ? launch_q0_cfg<PI_Q4_0>(cfg, L, stream, ea, eb) : launch_q0_cfg<PI_Q8_0>(cfg, L, stream, ea, eb);
}
