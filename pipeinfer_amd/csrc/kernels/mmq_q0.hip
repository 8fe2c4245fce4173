// Q4_0 / Q8_0 mat-mat for prompts on the matrix cores, BIT-EXACT with the reference's x86 AVX2 arm (the contract of mmvq.hip):
//
//   out[t][row] = residual[t][row] + vec_dot(W[row], act[t])
//
// Reference: ggml_vec_dot_q4_0_q8_0 (ggml-quants.c:2500-2523), ggml_vec_dot_q8_0_q8_0 (:3584-3605).  Per block of 32 values the AVX2 code has eight lanes; lane k is the integer dot product of
// values 4k .. 4k+3, converted to float, and extends its own fp32 chain by one fma per block in block order:  acc[k] = fma(d_x * d_y, (float) dot4, acc[k]).  The eight chains are folded at the end.
//
// What bounds it.  A block of one (row, token) pair is eight fma that may not be re-ordered or merged, plus one product of the scales: 9 VALU operations per 32 multiply-adds, whatever computes the
// integer part.  On the VALU (k_mmvq_q0, 8 tokens per pass over the weights) the integer part costs another 16 (a dot4 and a conversion per lane), every pass reads all weights again and 8 x 16 bytes
// of LDS per block: 9 TFLOP/s (4096 x 4096; 40 us for 8 tokens, so 512 tokens take 2 500 us).  Here the integer part is ONE v_mfma_f32_4x4x4_16b_f16 per lane k for 16 rows x 16 tokens: its K is exactly the four values of a lane, its result is the
// converted float (integers of at most 128 * 128 * 4 = 2^16: exact in f16 operands and fp32 sums), and it runs beside the fma chains of the other lanes.
//
// Operands.  The instruction multiplies sixteen 4 x 4 blocks.  Block 4 rg + tg is rows 4 rg .. + 3 against tokens 4 tg .. + 3.  Without help each operand would have to be there four times (a row group
// in four blocks, a token group in four); instead A is loaded with FOUR lanes k side by side — block 4 rg + s of the register holds row group rg at lane k = s — and cbsz = 2 / abid = s broadcasts
// block s of each group of four, and B holds lane k = s in its s-th sixteen lanes, which blgp = 4 + s broadcasts.  One 16-byte LDS read per lane then feeds the eight MFMAs of a tile, and lane (rg, s, i)
// of A is one dword of the weight planes: its low nibbles are lane k = s, its high nibbles k = s + 4.
//
// Tiles.  A wave owns 16 rows x TT tiles of 16 tokens, 32 chains per tile and lane (TT = 2: 64 registers, so that four waves share a SIMD); a workgroup is WR x WT waves.  Groups of four blocks are
// converted to f16 once per workgroup, in operand order, into one of two LDS buffers while the other is multiplied; one barrier per group.  Measured (Q4_0, us for 4096 x 4096 / 11008 x 4096): 16 tokens 33 / 35, 32: 41 / 43, 64: 58 / 63, 128: 61 / 109, 512: 114 / 322 (144 TFLOP/s); Q8_0 within 5 % of that.
// Short of the 140 000 issue cycles of its fma chains and products (of 257 000 at 512 tokens) it waits for barriers and operand reads; two tiles of rows per wave (half the waves) took 132 us, register
// sets loaded further ahead changed nothing.
#include "mmvq_args.h"
#include <hip/hip_ext.h>

#include <cstdlib>
#include <cstring>
#include <type_traits>

using q0_half4 = __attribute__((ext_vector_type(4))) _Float16;
using q0_half2 = __attribute__((ext_vector_type(2))) _Float16;
typedef uint32_t q0_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t q0_u32x2 __attribute__((ext_vector_type(2)));
using q0_f32x4 = __attribute__((ext_vector_type(4))) float;

// four unsigned bytes -> four f16 of (byte - bias): 0x6400 + u is 1024 + u, so one byte permutation and one packed addition per pair; bias as the f16 bits of -(1024 + bias)
static __device__ __forceinline__ uint2 q0_expand(uint32_t u, uint32_t minus) {
    const q0_half2 m = __builtin_bit_cast(q0_half2, minus);
    const q0_half2 a = __builtin_bit_cast(q0_half2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + m, b = __builtin_bit_cast(q0_half2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + m;
    return make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
}
static __device__ __forceinline__ uint2 q0_int8(uint32_t x) { return q0_expand(x ^ 0x80808080u, 0xE480E480u); }                        // signed byte: u = byte + 128, -(1024 + 128)
static __device__ __forceinline__ uint2 q0_nibbles(uint32_t x) { return q0_expand(x & 0x0F0F0F0Fu, 0xE408E408u); }                     // low nibble - 8

#define Q0_WAVES 8
// KS = 2: the lanes k of a tile are split over two waves (even ones, odd ones), which meet in the last addition of the fold
template <int TYPE, int TT, int WR, int WT, int KS>
__global__ void __launch_bounds__(64 * Q0_WAVES, 4) k_mmq_q0(const mmvq_args g, const int row_blocks, const int tok_blocks) {
    if (pi_aborted(g.abort_w, 1)) return;
    static_assert(WR * WT * KS == Q0_WAVES, "eight waves");
    constexpr int MR = WR, MT = TT * WT, NT = MR + MT, NK = 8 / KS;    // tiles of the workgroup; lanes k of a wave
    static_assert(NT <= Q0_WAVES && MR * 16 + MT * 16 <= 64 * Q0_WAVES, "a wave stages one tile at most");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int TILES = NT * 4096, BUF = TILES + NT * 256;            // operands of the row tiles, then the token tiles; their scales as floats
    // the token blocks of one row block run on one XCD (workgroup n goes to XCD n % 8): its weights come from HBM once
    const int slot = blockIdx.x >> 3, rb = (blockIdx.x & 7) + 8 * (slot / tok_blocks), tb = slot % tok_blocks;
    if (rb >= row_blocks) return;
    const mmvq_seg & sg = g.seg[0];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / (WT * KS), wt = wave / KS % WT, ks = wave % KS;
    const int row0 = rb * MR * 16, tok0 = tb * MT * 16;
    const int ng = g.nb;                                               // groups of four blocks
    // staging: wave w converts tile w (row tiles first); rows and tokens past the end repeat the last one and are not stored
    const bool is_row = wave < MR, staging = wave < NT;
    const int s_row = min(row0 + wave * 16 + (lane >> 4) * 4 + (lane & 3), sg.M - 1), s_tok = min(tok0 + max(wave - MR, 0) * 16 + (lane & 15), g.nt - 1);
    constexpr int A_GROUP = TYPE == PI_Q4_0 ? 64 : 128;
    const uint8_t * src = is_row ? sg.p0 + (int64_t) s_row * ng * A_GROUP + 16 * ((lane >> 2) & 3) : g.aq + (int64_t) s_tok * ng * 128 + 16 * (lane >> 4);
    const int step = is_row ? A_GROUP : 128, second = is_row && TYPE == PI_Q4_0 ? 0 : 64;      // (nibbles: both lanes k of a dword are in it)
    const bool d_mine = tid < NT * 16;                                  // the scales: a thread per row, then a thread per token
    const uint8_t * d_src = tid < MR * 16 ? sg.p1 + (int64_t) min(row0 + tid, sg.M - 1) * ng * 8 : g.ad + (int64_t) min(tok0 + tid - MR * 16, g.nt - 1) * ng * 8;
    q0_u32x4 x0, x1; q0_u32x2 dv;
    // (every thread loads, whether it stages or not: where paths with different numbers of loads meet, the compiler waits for all of them)
    auto fetch = [&](int gi) {
        x0 = *(const q0_u32x4 *) (src + (int64_t) gi * step); x1 = *(const q0_u32x4 *) (src + (int64_t) gi * step + second);
        dv = *(const q0_u32x2 *) (d_src + (int64_t) gi * 8);
    };
    auto stage = [&](int buf) {
        uint8_t * base = lds + buf * BUF;
        if (staging)
#pragma unroll
            for (int b = 0; b < 4; b++) {
                uint2 lo, hi;
                if (TYPE == PI_Q4_0 && is_row) { lo = q0_nibbles(x0[b]); hi = q0_nibbles(x0[b] >> 4); }
                else { lo = q0_int8(x0[b]); hi = q0_int8(x1[b]); }
                *(uint4 *) (base + ((wave * 4 + b) * 64 + lane) * 16) = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        if (d_mine) {
            float * d = (float *) (base + TILES) + (tid >> 4) * 64 + (tid & 15);
            d[0] = pi_h2f((uint16_t) (dv[0] & 0xffff)); d[16] = pi_h2f((uint16_t) (dv[0] >> 16)); d[32] = pi_h2f((uint16_t) (dv[1] & 0xffff)); d[48] = pi_h2f((uint16_t) (dv[1] >> 16));
        }
    };
    q0_f32x4 acc[TT][NK];                                              // rows 4 (lane / 16) .. + 3 of token lane % 16
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int k = 0; k < NK; k++) acc[t][k] = q0_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint8_t * a_at = lds + (wr * 256 + lane) * 16, * b_at = lds + ((MR + wt * TT) * 256 + lane) * 16;
    const uint8_t * dx_at = lds + TILES + wr * 256 + (lane >> 4) * 16, * dy_at = lds + TILES + (MR + wt * TT) * 256 + (lane & 15) * 4;
    // the block's products for lanes k = S, S + ST, .. (and S + 4, ..): one MFMA, then the four fma of the product before it — in plain order each MFMA would be followed by idle cycles
    auto group = [&](auto s0, int buf) {
        constexpr int S0 = decltype(s0)::value, ST = KS;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint4 a4 = *(const uint4 *) (a_at + buf * BUF + b * 1024); const float4 dx = *(const float4 *) (dx_at + buf * BUF + b * 64);
            uint4 b4[TT]; float dy[TT];
#pragma unroll
            for (int t = 0; t < TT; t++) { b4[t] = *(const uint4 *) (b_at + buf * BUF + t * 4096 + b * 1024); dy[t] = *(const float *) (dy_at + buf * BUF + t * 256 + b * 64); }
            const q0_half4 al = __builtin_bit_cast(q0_half4, make_uint2(a4.x, a4.y)), ah = __builtin_bit_cast(q0_half4, make_uint2(a4.z, a4.w));
            const q0_f32x4 zero = q0_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            auto product = [&](int n) -> q0_f32x4 {                    // (n is a constant after unrolling)
                const int t = n / NK, k = n % NK, s = S0 + ST * (k % (NK / 2));
                const q0_half4 x = k < NK / 2 ? al : ah, y = __builtin_bit_cast(q0_half4, k < NK / 2 ? make_uint2(b4[t].x, b4[t].y) : make_uint2(b4[t].z, b4[t].w));
                switch (s) {
                    case 0:  return __builtin_amdgcn_mfma_f32_4x4x4f16(x, y, zero, 2, 0, 4);
                    case 1:  return __builtin_amdgcn_mfma_f32_4x4x4f16(x, y, zero, 2, 1, 5);
                    case 2:  return __builtin_amdgcn_mfma_f32_4x4x4f16(x, y, zero, 2, 2, 6);
                    default: return __builtin_amdgcn_mfma_f32_4x4x4f16(x, y, zero, 2, 3, 7);
                }
            };
            q0_f32x4 d = product(0);
            float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;
#pragma unroll
            for (int n = 0; n < TT * NK; n++) {
                const int t = n / NK, k = n % NK;
                if (k == 0) { p0 = dx.x * dy[t]; p1 = dx.y * dy[t]; p2 = dx.z * dy[t]; p3 = dx.w * dy[t]; }
                const q0_f32x4 v = d;
                if (n + 1 < TT * NK) d = product(n + 1);
                __builtin_amdgcn_sched_barrier(0);
                q0_f32x4 & c = acc[t][k];
                c[0] = fmaf(p0, v[0], c[0]); c[1] = fmaf(p1, v[1], c[1]); c[2] = fmaf(p2, v[2], c[2]); c[3] = fmaf(p3, v[3], c[3]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    fetch(0);
    stage(0);
    fetch(min(1, ng - 1));
    __syncthreads();
    for (int g0 = 0; g0 < ng; g0 += 2)
#pragma unroll
        for (int gd = 0; gd < 2; gd++) {
            if (g0 + gd >= ng) break;
            stage(gd ^ 1);                                             // (its readers finished before the last barrier; past the last group: values that nobody reads)
            fetch(min(g0 + gd + 2, ng - 1));
            if (KS == 1 || ks == 0) group(std::integral_constant<int, 0>{}, gd); else group(std::integral_constant<int, KS - 1>{}, gd);
            __syncthreads();
        }
    // hsum_float_8: (a4+a0, a5+a1, a6+a2, a7+a3) -> (r0+r2, r1+r3) -> s0+s1
    float * other = (float *) lds;                                     // KS = 2: the odd lanes' sums [row tile][lane][4]
    if constexpr (KS == 2) {
        static_assert(TT == 1 && WT == 1, "one token tile");
        if (ks == 1)
#pragma unroll
            for (int i = 0; i < 4; i++) other[(wr * 64 + lane) * 4 + i] = (acc[0][0][i] + acc[0][2][i]) + (acc[0][1][i] + acc[0][3][i]);      // ((a1 + a5) + (a3 + a7))
        __syncthreads();
        if (ks == 1) return;
    }
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const int tok = tok0 + (wt * TT + t) * 16 + (lane & 15), row = row0 + wr * 16 + (lane >> 4) * 4;
        const q0_f32x4 * a = acc[t];
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (KS == 2) v[i] = ((a[0][i] + a[2][i]) + (a[1][i] + a[3][i])) + other[(wr * 64 + lane) * 4 + i];
            else v[i] = ((a[0][i] + a[4][i]) + (a[2][i] + a[6][i])) + ((a[1][i] + a[5][i]) + (a[3][i] + a[7][i]));
        }
        if (tok >= g.nt) continue;
        const int64_t o = (int64_t) tok * sg.M + row;
        if ((sg.M & 3) == 0 && (((uintptr_t) sg.out | (uintptr_t) sg.res) & 15) == 0) {
            if (row >= sg.M) continue;
            if (sg.res) { const float4 x = *(const float4 *) (sg.res + o); v[0] = x.x + v[0]; v[1] = x.y + v[1]; v[2] = x.z + v[2]; v[3] = x.w + v[3]; }
            *(float4 *) (sg.out + o) = make_float4(v[0], v[1], v[2], v[3]);
        } else
#pragma unroll
            for (int i = 0; i < 4; i++) if (row + i < sg.M) sg.out[o + i] = sg.res ? sg.res[o + i] + v[i] : v[i];
    }
}

// from the first width that costs k_mmvq_q0 a second pass over the weights.  Measured, us there / here at 4096 x 4096, 11008 x 4096 and 4096 x 11008: 5 tokens 21 / 33, 27 / 35, 55 / 83;
// 8 tokens 29 / 33, 37 / 35, 82 / 83; 9 tokens two passes, about 44 / 33, 57 / 35, 120 / 84.  The second pass of nine tokens has one token: quick where the rows are few and long, and Q4_0 has more to expand here than Q8_0 (9 tokens of
// 2048 x 4096 30.0 / 31.9, 2048 x 11008 72.4 / 80.0, 1000 x 2048 17.6 / 17.7, 4096 x 4096 32.6 / 32.1; Q8_0 29.1 / 28.6, 73.6 / 71.4; 10 tokens of 2048 x 11008 88 / 80)
bool pi_mmq_q0_wants(int type, int n_tok, int64_t rows, int64_t k) {
    static const int min_tok = getenv("PI_MMQ_Q0_MIN") ? atoi(getenv("PI_MMQ_Q0_MIN")) : 9;
    if (type == PI_Q4_0 && n_tok == 9 && rows <= 2048 && k >= 4096) return false;
    return (type == PI_Q4_0 || type == PI_Q8_0) && n_tok >= min_tok;
}

template <int TYPE, int TT, int WR, int WT, int KS>
static int launch_q0(mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    mmvq_args & g = L.g;
    constexpr int MR = WR, MT = TT * WT;
    constexpr size_t lds = 2 * (size_t) (MR + MT) * (4096 + 256);
    if (!g.aq) { PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_mmq_q0<TYPE, TT, WR, WT, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); return 0; }      // pi_mmq_q0_reserve
    const int rb = (g.seg[0].M + MR * 16 - 1) / (MR * 16), tb = (g.nt + MT * 16 - 1) / (MT * 16);
    const unsigned grid = (unsigned) ((rb + 7) / 8 * 8) * (unsigned) tb;
    if (ea) hipExtLaunchKernelGGL((k_mmq_q0<TYPE, TT, WR, WT, KS>), dim3(grid), dim3(64 * Q0_WAVES), lds, stream, ea, eb, 0, g, rb, tb);
    else    hipLaunchKernelGGL((k_mmq_q0<TYPE, TT, WR, WT, KS>), dim3(grid), dim3(64 * Q0_WAVES), lds, stream, g, rb, tb);
    PI_CHECK_LAUNCH();
    return 0;
}
// 16 tokens at most: the lanes k over two waves (a tile's chains are the longest serial part of such a launch: 36 us on one wave, 33 on two); 32: one tile of tokens per wave; more: two, which share the
// operands of a row tile
template <int TYPE>
static int launch_q0_type(mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    const int nt = L.g.nt;
    if (nt <= 16) return launch_q0<TYPE, 1, 4, 1, 2>(L, stream, ea, eb);
    if (nt <= 32) return launch_q0<TYPE, 1, 4, 2, 1>(L, stream, ea, eb);
    return launch_q0<TYPE, 2, 4, 2, 1>(L, stream, ea, eb);
}
// once per process and outside any stream capture (pi_op_mul_mat_reserve): the instances' dynamic LDS is more than a kernel gets by default
int pi_mmq_q0_reserve() {
    mmvq_launch L; memset(&L.g, 0, sizeof L.g);                        // g.aq == nullptr: the instances only set their attribute
    for (int nt : { 16, 32, 64 }) {
        L.g.nt = nt;
        if (launch_q0_type<PI_Q4_0>(L, nullptr, nullptr, nullptr) != 0 || launch_q0_type<PI_Q8_0>(L, nullptr, nullptr, nullptr) != 0) return -1;
    }
    return 0;
}
// the whole pass in one launch (seg[0] only; g.aq / g.ad at the first token, g.nt tokens)
int pi_mmq_q0_launch(int type, mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    if (pi_op_mul_mat_reserve() != 0) return -1;
    return type == PI_Q4_0 ? launch_q0_type<PI_Q4_0>(L, stream, ea, eb) : launch_q0_type<PI_Q8_0>(L, stream, ea, eb);
}
