// Dense operators over bfloat16 weight matrices stored [rows][K] as the checkpoint has them (no re-ordering: a row is one contiguous run of K values).
//
//   out[t][r] = act(sum_k W[r][k] * in(x[t][k]) [+ bias[r]])          fp32 accumulation, fp32 in and out
//
// `exact` selects what enters the product: 0 (serving precision) rounds the activations to bfloat16 (nearest even), so a product of two bfloat16 values is exact in fp32 and only the
// order of the fp32 sum differs between the kernels below; 1 keeps the activations in fp32 (weights widen exactly), every multiply-add a true fp32 fma.
//
//   k_dense_rows   one wave per output row, K spread over the lanes with 16 / 8 / 2-byte weight loads, TT tokens held in registers: the mat-vec of single tokens (weights streamed once from HBM:
//                  6.7 TB/s at 32000 x 4096, 4.3 at 4096 x 4096, 4 us of launch below 1024 x 1024) and every width of the fp32 mode
//   k_dense_split  serving precision, 2 .. 32 tokens: 4 .. 32 rows x all tokens per workgroup on the matrix cores, K over its eight waves.  Bound by the weight stream (5.8 TB/s at 32000 x 4096 and 2
//                  tokens, 4.6 at 8) and by the address unit.  On the mat-vec every row reads all tokens' activations again, 2 T times its own bytes: 28 us for 4096 x 4096 at 8 tokens, 11 here
//   k_dense_tile   serving precision, more tokens: tiles of 64 .. 256 rows x 64 .. 128 tokens through LDS (dense_tile.h).  Small grids are bound by what one compute unit can have on its way from memory and by the
//                  latency of a step, large ones by the shared levels of memory: 850 TFLOP/s at 16384 x 4096 x 2048 tokens (128 x 128 tiles with a step's parts one after another: 710), 14 us for
//                  2048 x 2048 x 512 (17)
//   k_dense_async  the same from activations that are bfloat16 in memory (dense_async.h): what the engine's passes of more than 32 tokens take (matrices of 16384 rows and more: of more than 8); k_round_bf16 makes such activations where no kernel
//                  ahead writes them
//   k_embed        rows of the table gathered, widened and scaled
#include "ops_common.h"
#include "dense_tile.h"
#include "dense_async.h"
#include "kernel_timing.h"

#include <algorithm>
#include <type_traits>

typedef uint16_t dn_u16x8 __attribute__((ext_vector_type(8)));

static __device__ __forceinline__ float dn_widen(uint16_t b) { return __uint_as_float((uint32_t) b << 16); }
// nearest-even rounding of an fp32 value to bfloat16 precision, kept in an fp32 register
static __device__ __forceinline__ uint32_t dn_round_bits(float f) { const uint32_t u = __float_as_uint(f); return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16; }
static __device__ __forceinline__ float dn_round(float f) { return __uint_as_float(dn_round_bits(f) << 16); }

static __device__ __forceinline__ float dn_act(float v, int act) {
    switch (act) {
        case PI_ACT_SILU:     return v / (1.0f + expf(-v));
        case PI_ACT_SIGMOID:  return 1.0f / (1.0f + expf(-v));
        case PI_ACT_RELU_SQR: { const float r = fmaxf(v, 0.0f); return r * r; }
        case PI_ACT_TANH:     return tanhf(v);
        case PI_ACT_GELU_TANH: return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
        case PI_ACT_GELU_ERF: return 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
        default:              return v;
    }
}

// grid (token, 2048 values); vec: eight values of a thread in one 16-byte load (rows and output start 16-byte aligned), else one by one
__global__ void __launch_bounds__(256) k_embed(const uint16_t * __restrict__ table, int64_t width, int64_t n_rows, const int32_t * __restrict__ tokens, float scale, int vec, float * __restrict__ out, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int t = blockIdx.x;
    const int64_t row = tokens[t], i0 = (int64_t) blockIdx.y * 2048;
    if (pi_abort_late(gone, abort_w)) return;
    const bool ok = row >= 0 && row < n_rows;
    if (vec) {
        const int64_t i = i0 + 8 * threadIdx.x;
        if (i >= width) return;
        const dn_u16x8 a = *(const dn_u16x8 *) (table + (ok ? row : 0) * width + i);
        float4 o[2];
#pragma unroll
        for (int c = 0; c < 8; c++) ((float *) o)[c] = ok ? dn_widen(a[c]) * scale : 0.0f;
        float4 * dst = (float4 *) (out + (int64_t) t * width + i);
        dst[0] = o[0]; dst[1] = o[1];
        if (rd.h) *(dt_u32x4 *) (rd.h + t * rd.stride + i) = dt_pack8(*(const dt_f32x4 *) &o[0], *(const dt_f32x4 *) &o[1]);
        return;
    }
    for (int64_t i = i0 + threadIdx.x; i < min(width, i0 + 2048); i += 256) out[(int64_t) t * width + i] = ok ? dn_widen(table[row * width + i]) * scale : 0.0f;
}

// VW weights per lane and step (8: one 16-byte load, 4: 8 bytes, 1: any K and alignment)
template <int TT, int VW, bool EXACT>
__global__ void __launch_bounds__(256) k_dense_rows(const uint16_t * __restrict__ W, int64_t K, int64_t N, const float * __restrict__ X, int64_t xs, int T, float * __restrict__ Y, int64_t ys,
                                                    int act_a, int64_t rows_a, int act_b, const float * __restrict__ bias, int64_t seg_rows, int64_t seg_off, int seg_last, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t row = (int64_t) blockIdx.x * 4 + wave;
    if (row >= N) return;
    if (seg_rows > 0) X += min(row / seg_rows, (int64_t) seg_last) * seg_off;       // rows in segments of seg_rows (the last one takes the rest), every segment with an input of its own
    const int t0 = blockIdx.y * TT;
    float acc[TT];
#pragma unroll
    for (int i = 0; i < TT; i++) acc[i] = 0.0f;
    const uint16_t * w = W + row * K;
    if constexpr (TT == 1 && VW == 8) {
        // one token: of rows below 8 KB two steps of 512 values go out together (a step at a time 32000 x 1024 / 2048 took 15.1 / 25.8 us, now 13.4 / 23.5).  Longer rows keep single steps, which the compiler may run into
        // each other (4096 x 4096 9.1, with a step's loads held together 9.5; 32000 x 4096 48.9, in pairs 50.1; 5120 x 13824 27.1, in pairs 31.6)
        const float * x0 = X + (int64_t) t0 * xs;
        auto product = [&](const dn_u16x8 & v, const float4 & lo, const float4 & hi) __attribute__((always_inline)) {
            const float xf[8] = { lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w };
#pragma unroll
            for (int i = 0; i < 8; i++) acc[0] = fmaf(dn_widen(v[i]), EXACT ? xf[i] : dn_round(xf[i]), acc[0]);
        };
        int64_t done = 0;
        if (K < 4096) for (; done + 1024 <= K && (done == 0 || !(gone & 1)); done += 1024) {
            const int64_t k = done + lane * 8;
            dn_u16x8 wv[2]; float4 xv[2][2];
#pragma unroll
            for (int u = 0; u < 2; u++) { xv[u][0] = *(const float4 *) (x0 + k + 512 * u); xv[u][1] = *(const float4 *) (x0 + k + 512 * u + 4); wv[u] = *(const dn_u16x8 *) (w + k + 512 * u); }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 2; u++) product(wv[u], xv[u][0], xv[u][1]);
        }
        for (int64_t k = done + lane * 8; k < K && (k < 512 || !(gone & 1)); k += 512) {
            const float4 lo = *(const float4 *) (x0 + k), hi = *(const float4 *) (x0 + k + 4);
            product(*(const dn_u16x8 *) (w + k), lo, hi);
        }
    } else {
        if (pi_abort_late(gone, abort_w, 0)) return;
        for (int64_t k = (int64_t) lane * VW; k < K; k += 64 * VW) {
            float wf[VW];
            if constexpr (VW == 8) { const dn_u16x8 v = *(const dn_u16x8 *) (w + k); for (int i = 0; i < 8; i++) wf[i] = dn_widen(v[i]); }
            else if constexpr (VW == 4) { const uint2 v = *(const uint2 *) (w + k); wf[0] = __uint_as_float(v.x << 16); wf[1] = __uint_as_float(v.x & 0xffff0000u); wf[2] = __uint_as_float(v.y << 16); wf[3] = __uint_as_float(v.y & 0xffff0000u); }
            else wf[0] = dn_widen(w[k]);
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                if (t0 + tt >= T) break;
                const float * x = X + (int64_t) (t0 + tt) * xs + k;
                float xf[VW];
                if constexpr (VW >= 4) {
#pragma unroll
                    for (int i = 0; i < VW; i += 4) { const float4 v = *(const float4 *) (x + i); xf[i] = v.x; xf[i + 1] = v.y; xf[i + 2] = v.z; xf[i + 3] = v.w; }
                } else xf[0] = x[0];
#pragma unroll
                for (int i = 0; i < VW; i++) acc[tt] = fmaf(wf[i], EXACT ? xf[i] : dn_round(xf[i]), acc[tt]);
            }
        }
    }
    const int act = row < rows_a ? act_a : act_b;
    if (pi_abort_late(gone, abort_w, 0)) return;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        if (t0 + tt >= T) break;
        const float s = pi_lanes_sum<64>(acc[tt]);
        if (lane == 0) Y[(int64_t) (t0 + tt) * ys + row] = dn_act(bias ? s + bias[row] : s, act);
    }
}

// the value of the lane N further on in the row of 16 (what the last N lanes get is of no use)
template <int N>
static __device__ __forceinline__ uint32_t dn_from_lane(uint32_t v) { return (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, 0x100 + N, 0xf, 0xf, true); }
// one float4 of results (four rows of one token): bias, activation, store
static __device__ __forceinline__ void dn_store4(dt_f32x4 v4, int64_t row, int64_t N, int tok, float * __restrict__ Y, int64_t ys, int act_a, int64_t rows_a, int act_b, const float * __restrict__ bias) {
    float v[4] = { v4[0], v4[1], v4[2], v4[3] };
    if (bias || act_a != PI_ACT_NONE || act_b != PI_ACT_NONE)
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = dn_act(bias ? v4[r] + bias[min(row + r, N - 1)] : v4[r], row + r < rows_a ? act_a : act_b);
    float * dst = Y + (int64_t) tok * ys + row;
    if (row + 3 < N && (ys & 3) == 0 && (((uintptr_t) Y) & 15) == 0) *(float4 *) dst = make_float4(v[0], v[1], v[2], v[3]);
    else for (int r = 0; r < 4; r++) if (row + r < N) dst[r] = v[r];
}

// BN rows x BT tokens per workgroup (dense_tile.h).  Workgroup n runs on XCD n % 8: an XCD takes a contiguous run of tiles, eight blocks of rows wide and then along the tokens, so that the 64 tiles it
// works on at a time are 8 x 8 and share the rows and tokens that pass through its L2
template <int BN, int BT, int WN, int WT, int KG>
__global__ void __launch_bounds__(64 * WN * WT * KG, 2) k_dense_tile(const uint16_t * __restrict__ W, int64_t K, int64_t N, const float * __restrict__ X, int64_t xs, int T, float * __restrict__ Y, int64_t ys,
                                                       int act_a, int64_t rows_a, int act_b, const float * __restrict__ bias, int tok_blocks, int tiles, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 1)) return;
    __shared__ __attribute__((aligned(16))) uint8_t lds[DT_LDS_BYTES(BN, BT, KG)];
    const int tile = (int) (blockIdx.x & 7) * (int) (gridDim.x >> 3) + (int) (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int row_blocks = tiles / tok_blocks, grp = tile / (8 * tok_blocks), in_grp = tile % (8 * tok_blocks), gsz = min(8, row_blocks - 8 * grp);
    const int64_t n0 = (int64_t) (8 * grp + in_grp % gsz) * BN;
    const int t0 = (in_grp / gsz) * BT, tid = threadIdx.x % (64 * WN * WT), lane = tid & 63, wave = tid >> 6;
    dt_offs wo, xo;                                                    // the rows this thread stages, from the tile's first
#pragma unroll
    for (int i = 0; i < BN / (8 * WN * WT); i++) wo[i] = (uint32_t) ((min(n0 + (tid >> 3) + 8 * WN * WT * i, N - 1) - n0) * K);
#pragma unroll
    for (int i = 0; i < BT / (8 * WN * WT); i++) xo[i] = (uint32_t) ((min(t0 + (tid >> 3) + 8 * WN * WT * i, T - 1) - t0) * xs);
    dt_f32x4 acc[BN / WN / 16][BT / WT / 16];
    dt_tile<BN, BT, WN, WT, 2, KG, false>(W + n0 * K, wo, X + (int64_t) t0 * xs, xo, 0, [](float a, float) { return a; }, K, lds, acc);
    if (KG > 1 && threadIdx.x >= 64 * WN * WT) return;
#pragma unroll
    for (int b = 0; b < BT / WT / 16; b++) {
        const int tok = t0 + (wave % WT) * (BT / WT) + b * 16 + (lane & 15);
        if (tok >= T) continue;
#pragma unroll
        for (int a = 0; a < BN / WN / 16; a++) dn_store4(acc[a][b], n0 + (wave / WT) * (BN / WN) + a * 16 + (lane >> 4) * 4, N, tok, Y, ys, act_a, rows_a, act_b, bias);
    }
}

// 2 .. 32 tokens: up to RT x 16 rows (`rows`, a multiple of 4: the lanes of the others read the last one again, which costs no bytes) and TT x 16 tokens per workgroup, K split over its eight waves, which meet in LDS.  The weights are streamed once, straight from memory in the operand's lane layout: the
// four lanes of a row take 64 consecutive bytes of it per product, the activations come from L2 once per workgroup.  Rows in segments: as k_dense_rows, whole workgroups
// inside a segment (the host checks).
// XS: tokens that a product's sixteen columns stand for.  With 8 (4) the lanes of the other columns load the rest of the tokens' values, which a move across the lanes then brings to their columns: half
// (a quarter of) the loads of activations, which would otherwise be most of what the address unit works through (16 rows of weights are two loads a step, their sixteen columns of activations four).  us at 2 / 8 tokens, before: 4096 x 4096 9.4 / 11.1, now 8.3 / 10.4;
// 2048 x 5632 10.8 / 12.8, 8.2 / 11.4; 5120 x 13824 31.8 / 35.6, 26.1 / 32.7 (reading the weights alone takes 6.3 us for 4096 x 4096).
template <int RT, int TT, int XS>
__global__ void __launch_bounds__(512) k_dense_split(const uint16_t * __restrict__ W, int64_t K, int64_t N, const float * __restrict__ X, int64_t xs, int T, float * __restrict__ Y, int64_t ys,
                                                     int act_a, int64_t rows_a, int act_b, const float * __restrict__ bias, int64_t seg_rows, int64_t seg_off, int seg_last, int rows, const int32_t * __restrict__ abort_w) {
    static_assert(XS == 16 || TT == 1, "one group of columns where they share a token");
    const int gone = pi_abort_peek(abort_w);
    constexpr int KS = 8;
    __shared__ dt_f32x4 red[KS][RT * TT][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
    const int64_t n0 = (int64_t) blockIdx.x * rows;
    const int t0 = blockIdx.y * (16 * TT);
    if (seg_rows > 0) X += min(n0 / seg_rows, (int64_t) seg_last) * seg_off;
    const int64_t per = (K + 64 * KS - 1) / (64 * KS) * 64, k_begin = wave * per, k_end = min(K, k_begin + per);
    constexpr int NX = XS / 4;                                         // loads of activations per step and group of columns
    const int part = li / XS;                                          // of the step's values: this lane's
    const int x_at = XS == 16 ? kb * 8 : XS == 8 ? kb * 8 + part * 32 : kb * 8 + (part >> 1) * 32 + (part & 1) * 4;
    const uint16_t * wrow[RT]; const float * xrow[TT];
#pragma unroll
    for (int a = 0; a < RT; a++) wrow[a] = W + min(n0 + min(a * 16 + li, rows - 1), N - 1) * K + kb * 8;
#pragma unroll
    for (int b = 0; b < TT; b++) xrow[b] = X + (int64_t) min(t0 + b * 16 + li % XS, T - 1) * xs + x_at;
    dt_f32x4 acc[RT][TT];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < TT; b++) acc[a][b] = dt_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const dt_u32x4 zero4 = { 0, 0, 0, 0 }; const dt_f32x4 zerof = { 0.0f, 0.0f, 0.0f, 0.0f };
    constexpr int U = RT * TT == 1 ? 4 : RT * TT == 2 ? 2 : 1;                                            // steps of 64 whose loads go out together
    auto steps = [&](auto n_steps, int64_t k, bool ok0, bool ok1) __attribute__((always_inline)) {
        constexpr int NS = decltype(n_steps)::value;
        const bool okx = XS == 16 || (XS == 8 ? part : part >> 1) == 0 ? ok0 : ok1;     // (fewer columns: of this lane's own values)
        dt_u32x4 af[NS][RT][2]; dt_f32x4 xf[NS][TT][NX];
#pragma unroll
        for (int u = 0; u < NS; u++) {
            auto load_x = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int b = 0; b < TT; b++)
#pragma unroll
                    for (int i = 0; i < NX; i++) xf[u][b][i] = (i < 2 ? okx : ok1) ? *(const dt_f32x4 *) (xrow[b] + k + 64 * u + (i < 2 ? 0 : 24) + 4 * i) : zerof;
            };
            // (16 rows and 32 tokens, where the activations are most of it: the weights first.  4096 x 11008 at 17 / 32 tokens 36.1 / 50.2 us, the other way round 39.0 / 53.5; 32 rows 8192 x 4096 at 24 22.6 and 22.1)
            constexpr bool W_FIRST = RT == 1 && TT == 2;
            if constexpr (!W_FIRST) load_x();
#pragma unroll
            for (int a = 0; a < RT; a++) { af[u][a][0] = ok0 ? *(const dt_u32x4 *) (wrow[a] + k + 64 * u) : zero4; af[u][a][1] = ok1 ? *(const dt_u32x4 *) (wrow[a] + k + 64 * u + 32) : zero4; }
            if constexpr (W_FIRST) load_x();
        }
        __builtin_amdgcn_sched_barrier(0);                             // (all of them issued before the first product waits)
#pragma unroll
        for (int u = 0; u < NS; u++)
#pragma unroll
            for (int b = 0; b < TT; b++) {
                dt_u32x4 b0, b1;
                if constexpr (XS == 16) { b0 = dt_pack8(xf[u][b][0], xf[u][b][1]); b1 = dt_pack8(xf[u][b][2], xf[u][b][3]); }
                else if constexpr (XS == 8) {
                    b0 = dt_pack8(xf[u][b][0], xf[u][b][1]);
#pragma unroll
                    for (int i = 0; i < 4; i++) b1[i] = dn_from_lane<8>(b0[i]);
                } else {
                    const uint32_t p0 = dt_pack(xf[u][b][0][0], xf[u][b][0][1]), p1 = dt_pack(xf[u][b][0][2], xf[u][b][0][3]);
                    b0 = dt_u32x4{ p0, p1, dn_from_lane<4>(p0), dn_from_lane<4>(p1) };
                    b1 = dt_u32x4{ dn_from_lane<8>(p0), dn_from_lane<8>(p1), dn_from_lane<12>(p0), dn_from_lane<12>(p1) };
                }
#pragma unroll
                for (int a = 0; a < RT; a++) { acc[a][b] = dt_mfma(af[u][a][0], b0, acc[a][b]); acc[a][b] = dt_mfma(af[u][a][1], b1, acc[a][b]); }
            }
    };
    using one = std::integral_constant<int, 1>;
    // Where the waves' parts begin a multiple of 4 KB apart (K 16384), all of them and all rows ask the same memory channel at a time: there workgroups begin at steps of their own and go round
    // (4096 x 16384 at 2 / 8 / 16 tokens: 40.6 / 43.6 / 49.8 us, with this and the shared columns 23.3 / 31.3 / 44.6; at K 4096 and 8192 it gives nothing and the order stays)
    const int turns = k_begin < K ? (int) ((k_end - k_begin) / (64 * U)) : 0, turn = per % 2048 == 0 ? (int) (((uint64_t) ((blockIdx.x >> 3) * 0x9E3779B1u) * (uint32_t) turns) >> 32) : 0;
    // The abort word is asked for at the top and looked at behind the first round of loads: on its own the trip to memory was 0.2 us of every launch (and between loads and products it costs the larger forms 10 %)
    for (int i = turn; i < turns && (i == turn || !(gone & 1)); i++) steps(std::integral_constant<int, U>{}, k_begin + 64 * U * (int64_t) i, true, true);
    for (int i = 0; i < turn && !(gone & 1); i++) steps(std::integral_constant<int, U>{}, k_begin + 64 * U * (int64_t) i, true, true);
    int64_t k = k_begin + 64 * U * (int64_t) turns;
    if constexpr (U > 1) for (; k + 64 <= k_end; k += 64) steps(one{}, k, true, true);
    if (k < k_end) steps(one{}, k, k + kb * 8 < K, k + kb * 8 + 32 < K);       // (K % 8 == 0)
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < TT; b++) red[wave][a * TT + b][lane] = acc[a][b];
    __syncthreads();
    if (pi_abort_late(gone, abort_w, 0)) return;
    for (int i = tid; i < RT * TT * 64; i += 512) {
        const int tile = i >> 6, l = i & 63, tok = t0 + (tile % TT) * 16 + (l & 15);
        if (tok >= T) continue;
        dt_f32x4 v = red[0][tile][l];
#pragma unroll
        for (int w = 1; w < KS; w++) v += red[w][tile][l];
        const int own = (tile / TT) * 16 + (l >> 4) * 4;
        if (own < rows && n0 + own < N) dn_store4(v, n0 + own, N, tok, Y, ys, act_a, rows_a, act_b, bias);
    }
}

// Tiles as k_dense_tile's, activations in bfloat16 (dense_async.h).  Rows in segments: as k_dense_rows, tiles inside a segment (blocks_of: tiles of rows to a segment; the last one takes the rest)
template <int BN, int BT, int WN, int WT, int S>
__global__ void __launch_bounds__(64 * WN * WT, WN * WT == 8 && BN * BT >= 32768 ? 2 : 1) k_dense_async(const uint16_t * __restrict__ W, int64_t K, int64_t N, const uint16_t * __restrict__ X, int64_t xs, int T, float * __restrict__ Y,
                                                       int64_t ys, int act_a, int64_t rows_a, int act_b, const float * __restrict__ bias, int blocks_of, int64_t seg_rows, int64_t seg_off, int seg_last, int tok_blocks, int tiles,
                                                       const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 1)) return;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[DA_LDS_BYTES(BN, BT, S)];
    const int tile = (int) (blockIdx.x & 7) * (int) (gridDim.x >> 3) + (int) (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int row_blocks = tiles / tok_blocks, grp = tile / (8 * tok_blocks), in_grp = tile % (8 * tok_blocks), gsz = min(8, row_blocks - 8 * grp), block = 8 * grp + in_grp % gsz;
    const int seg = seg_rows > 0 ? min(block / blocks_of, seg_last) : 0;
    const int64_t n0 = seg_rows > 0 ? seg * seg_rows + (int64_t) (block - seg * blocks_of) * BN : (int64_t) block * BN, n_end = seg_rows > 0 && seg < seg_last ? (seg + 1) * seg_rows : N;
    const int t0 = (in_grp / gsz) * BT, wave = threadIdx.x >> 6;
    const bool vec = (ys & 3) == 0 && ((uintptr_t) Y & 15) == 0;
    dt_f32x4 acc[BN / WN / 16][BT / WT / 16];
    da_tile<BN, BT, WN, WT, S>(W + n0 * K, [&](int r) { return (uint32_t) (min((int64_t) r, n_end - 1 - n0) * K * 2); }, X + seg * seg_off + (int64_t) t0 * xs, [&](int r) { return (uint32_t) ((int64_t) min(r, T - 1 - t0) * xs * 2); },
                               (int) (K / 64), lds, acc);
    __syncthreads();                                                   // (the operands of every wave are read)
    constexpr int SHARE = DA_LDS_BYTES(BN, BT, S) / (WN * WT) & ~15;
    const int64_t row0 = n0 + (wave / WT) * (BN / WN); const int tok0 = t0 + (wave % WT) * (BT / WT);
    da_rows<BN / WN / 16, BT / WT / 16, SHARE>(acc, lds + wave * SHARE, [&](int t, int r, dt_f32x4 v) __attribute__((always_inline)) {
        const int64_t row = row0 + r; const int tok = tok0 + t;
        if (tok >= T || row >= n_end) return;
        if (bias)
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += bias[min(row + e, n_end - 1)];
        if (act_a != PI_ACT_NONE || act_b != PI_ACT_NONE) {
            const int act = row < rows_a ? act_a : act_b, act3 = row + 3 < rows_a ? act_a : act_b;      // (a group of four that both activations share: one by one)
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = dn_act(v[e], act == act3 ? act : row + e < rows_a ? act_a : act_b);
        }
        float * dst = Y + (int64_t) tok * ys + row;
        if (row + 3 < n_end && vec) *(dt_f32x4 *) dst = v;
        else for (int e = 0; e < 4; e++) if (row + e < n_end) dst[e] = v[e];
        if (rd.h && row >= rd.from && row < rd.from + rd.n) pi_round_store4(rd, tok, row - rd.from, v[0], v[1], v[2], v[3]);
    });
}

// rows of fp32 values as bfloat16, nearest even: grid (2048 values, row), eight of a thread (n % 8 == 0)
__global__ void __launch_bounds__(256) k_round_bf16(const float * __restrict__ x, int64_t xs, int64_t n, int vec, uint16_t * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int64_t i = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 8, t = blockIdx.y;
    if (i >= n) return;
    dt_f32x4 lo, hi;
    const float * r = x + t * xs + i;
    if (vec) { lo = *(const dt_f32x4 *) r; hi = *(const dt_f32x4 *) (r + 4); }
    else
#pragma unroll
        for (int e = 0; e < 4; e++) { lo[e] = r[e]; hi[e] = r[4 + e]; }
    if (pi_abort_late(gone, abort_w)) return;
    *(dt_u32x4 *) (out + t * os + i) = dt_pack8(lo, hi);
}

extern "C" int pi_op_embed(const pi_weight * w, const int32_t * tokens, int n_tok, float scale, float * out, void * stream) {
    if (!w || w->type != PI_BF16) { pi_set_error("pi_op_embed: the table must be a bfloat16 weight"); return -1; }
    if (n_tok <= 0) return 0;
    const int vec = w->ne0 % 8 == 0 && w->ne1 > 0 && (((uintptr_t) w->p0 | (uintptr_t) out) & 15) == 0;
    PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 6.0 * w->ne0 * n_tok, k_embed, dim3((unsigned) n_tok, (unsigned) ((w->ne0 + 2047) / 2048)), dim3(256), 0, (hipStream_t) stream, (const uint16_t *) w->p0, w->ne0, w->ne1, tokens, scale, vec, out,
                 vec ? pi_round_asked(0, w->ne0) : pi_round_dst{}, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

template <int VW, bool EXACT>
static void launch_rows(const pi_weight * w, const float * x, int64_t xs, int n_tok, float * out, int64_t os, int act_a, int64_t rows_a, int act_b, hipStream_t s, double bytes, const float * bias = nullptr, int64_t seg_rows = 0, int64_t seg_off = 0, int seg_last = 0) {
    const uint16_t * W = (const uint16_t *) w->p0;
    const unsigned gx = (unsigned) ((w->ne1 + 3) / 4);
    const int nt_acct = std::min(n_tok, PI_KT_MAXNT - 1);
    if (n_tok == 1)      PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, nt_acct, bytes, (k_dense_rows<1, VW, EXACT>), dim3(gx, 1), dim3(256), 0, s, W, w->ne0, w->ne1, x, xs, n_tok, out, os, act_a, rows_a, act_b, bias, seg_rows, seg_off, seg_last, pi_abort_word());
    else if (n_tok <= 4) PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, nt_acct, bytes, (k_dense_rows<4, VW, EXACT>), dim3(gx, 1), dim3(256), 0, s, W, w->ne0, w->ne1, x, xs, n_tok, out, os, act_a, rows_a, act_b, bias, seg_rows, seg_off, seg_last, pi_abort_word());
    else PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, nt_acct, bytes, (k_dense_rows<8, VW, EXACT>), dim3(gx, (unsigned) ((n_tok + 7) / 8)), dim3(256), 0, s, W, w->ne0, w->ne1, x, xs, n_tok, out, os, act_a, rows_a, act_b, bias, seg_rows, seg_off, seg_last, pi_abort_word());
}

// Rows per workgroup: the chip's 256 compute units take a workgroup each at a time, and a round of them lasts about as long as `base` + rows, the base being the activations (K 4096, us a round at 8 / 16 / 24 / 32 rows:
// 2 tokens 3.7 / 5.0 / 7.7 / 11.3, 8 tokens 5.7 / 7.6 / 9.8 / 12.2, 16 tokens 9.0 / 11.0 / 12.8 / 15, 32 tokens 16 / 17.2 / 19.4 / 24; K 2048 at 2 tokens - / 3.6 / 5.0 / 6.2).  So the split that needs the least,
// in steps of 4 rows, the larger one of two that need the same.  The addresses of rows of whole 8 KB meet, which is what a round of many of them at few tokens waits for (16384 x 4096 at 2 tokens: 32 rows 27.9, 16 rows
// 23.5; 32000 x 4096 51.1 and 44.7, but 32000 x 2048 25.5 and 28.7).
static int split_rows(int64_t n, int64_t k, int n_tok, int64_t seg_rows) {
    const int base = n_tok <= 4 ? 6 : n_tok <= 8 ? 13 : n_tok <= 16 ? 28 : 70;
    int best = 16; int64_t least = INT64_MAX;
    for (int r = 32; r >= 4; r -= 4) {
        const int64_t cost = ((n + r - 1) / r + 255) / 256 * (base + r + (n_tok <= 4 && k % 4096 == 0 && r > 16 ? (r - 16) / 2 : 0));
        if (cost < least && (seg_rows <= 0 || seg_rows % r == 0)) { least = cost; best = r; }
    }
    return best;
}
// Which kernel takes a pass of serving precision (aligned rows; measured against each other over 512 .. 32000 rows, K 1024 .. 4096, us):
//   1 token                the mat-vec (at 2 the split kernel is ahead everywhere: 2048 x 2048 4.6 and 5.5, 8192 x 4096 13.3 and 20.1, 32000 x 4096 45 and 70; equal below 1024 x 1024)
//   .. 32 tokens           k_dense_split (4096 x 4096 at 4 / 8 / 16 / 32 tokens: 8.8 / 10.4 / 14 / 21; the mat-vec 15 / 28 at 4 / 8, k_dense_tile 27 at 32); of 16384 rows and more only .. 8 tokens, where the tiles
//                          fill the chip and read the activations less often (32000 x 2048 at 24: 41 against 26)
//   more                   k_dense_tile
static bool dense_takes_split(int64_t rows, int n_tok) {
    return n_tok > 1 && n_tok <= (rows >= 16384 ? 8 : 32);
}
static void launch_split(const pi_weight * w, const float * x, int64_t xs, int n_tok, float * out, int64_t os, int act_a, int64_t rows_a, int act_b, hipStream_t s, double bytes, const float * bias, int64_t seg_rows = 0,
                         int64_t seg_off = 0, int seg_last = 0) {
    const int r = split_rows(w->ne1, w->ne0, n_tok, seg_rows);
    const bool two = r > 16;
#define DN_SPLIT(RT, TT, XS) PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, std::min(n_tok, PI_KT_MAXNT - 1), bytes, (k_dense_split<RT, TT, XS>), dim3((unsigned) ((w->ne1 + r - 1) / r), (unsigned) ((n_tok + 16 * TT - 1) / (16 * TT))), \
                                     dim3(512), 0, s, (const uint16_t *) w->p0, w->ne0, w->ne1, x, xs, n_tok, out, os, act_a, rows_a, act_b, bias, seg_rows, seg_off, seg_last, r, pi_abort_word())
    if (n_tok <= 4)       { if (two) DN_SPLIT(2, 1, 4); else DN_SPLIT(1, 1, 4); }
    else if (n_tok <= 8)  { if (two) DN_SPLIT(2, 1, 8); else DN_SPLIT(1, 1, 8); }
    else if (n_tok <= 16) { if (two) DN_SPLIT(2, 1, 16); else DN_SPLIT(1, 1, 16); }
    else                  { if (two) DN_SPLIT(2, 2, 16); else DN_SPLIT(1, 2, 16); }
#undef DN_SPLIT
}
// The tile that needs the least time, by rounds of 256 workgroups (one per compute unit; us a round at K 2048): 64 x 64 and 128 x 64 in two groups of waves that share K 14.2 and 23, 128 x 128 by eight waves 29.6,
// 256 x 128 by eight 47; of 128 x 128 by four waves two fit a compute unit and a last round that is not full costs less: 15 + 23.5 a round, from the second on.  Measured at 512 .. 32000 rows x 64 .. 2048 tokens; the crossings, K 2048:
// 2048 rows at 1000 tokens 128 x 64 19.9, 128 x 128 by eight 25.6, at 2048 32.7 (by four) and 29.6; 6144 at 1000 128 x 128 by four 48.0, by eight 54.3, 256 x 128 46.4, at 2048 80.6 / 85.1 / 84.4; K 4096: 4608 rows
// at 2048 132 / 139 / 136, 16384 at 512 118 / 124 / 89.5, at 2048 376 / 390 / 323
static void launch_tile(const pi_weight * w, const float * x, int64_t xs, int n_tok, float * out, int64_t os, int act_a, int64_t rows_a, int act_b, hipStream_t s, double bytes, const float * bias) {
    auto tiles = [&](int bn, int bt) { return (w->ne1 + bn - 1) / bn * ((n_tok + bt - 1) / bt); };
#define DN_TILE(BN, BT, WN, WT, KG) PI_KT_LAUNCH(PI_KT_MMQ, PI_BF16, std::min(n_tok, PI_KT_MAXNT - 1), bytes, (k_dense_tile<BN, BT, WN, WT, KG>), dim3((unsigned) ((tiles(BN, BT) + 7) / 8 * 8)), dim3(64 * WN * WT * KG), 0, s, \
                     (const uint16_t *) w->p0, w->ne0, w->ne1, x, xs, n_tok, out, os, act_a, rows_a, act_b, bias, (n_tok + BT - 1) / BT, (int) tiles(BN, BT), pi_abort_word())
    auto rounds = [&](int bn, int bt) { return (double) ((tiles(bn, bt) + 255) / 256); };
    const double cost[5] = { 14.2 * rounds(64, 64), 23.0 * rounds(128, 64), 29.6 * rounds(128, 128), 47.0 * rounds(256, 128), tiles(128, 128) <= 256 ? 1e30 : 15.0 + 23.5 * (double) tiles(128, 128) / 256 };
    switch ((int) (std::min_element(cost, cost + 5) - cost)) {
        case 0:  DN_TILE(64, 64, 2, 2, 2); break;
        case 1:  DN_TILE(128, 64, 2, 2, 2); break;
        case 2:  DN_TILE(128, 128, 4, 2, 1); break;
        case 3:  DN_TILE(256, 128, 4, 2, 1); break;
        default: DN_TILE(128, 128, 2, 2, 1);
    }
#undef DN_TILE
}

extern "C" int pi_op_dense(const pi_weight * w, const float * x, int64_t x_stride, int n_tok, float * out, int64_t out_stride, int act_a, int64_t rows_a, int act_b, int exact, void * stream) {
    return pi_op_dense_bias(w, nullptr, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, exact, stream);
}
extern "C" int pi_op_dense_bias(const pi_weight * w, const float * bias, const float * x, int64_t x_stride, int n_tok, float * out, int64_t out_stride, int act_a, int64_t rows_a, int act_b, int exact, void * stream) {
    if (!w || w->type != PI_BF16) { pi_set_error("pi_op_dense: the weight must be bfloat16"); return -1; }
    if (n_tok <= 0 || w->ne1 <= 0) return 0;
    if (x_stride < w->ne0 || out_stride < w->ne1) { pi_set_error("pi_op_dense: row strides (%lld, %lld) below the matrix's sizes (%lld, %lld)", (long long) x_stride, (long long) out_stride, (long long) w->ne0, (long long) w->ne1); return -1; }
    hipStream_t s = (hipStream_t) stream;
    const int64_t K = w->ne0;
    const double bytes = 2.0 * K * w->ne1 + 4.0 * n_tok * (K + w->ne1);
    const bool al16 = K % 8 == 0 && ((uintptr_t) w->p0 % 16) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0;
    const bool al8  = K % 4 == 0 && ((uintptr_t) w->p0 % 8) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0;
    if (!exact && al16 && n_tok > 1 && (dense_takes_split(w->ne1, n_tok) || (K < (1 << 22) && x_stride < (1 << 22)))) {      // (a tile's offsets in 32 bits)
        if (dense_takes_split(w->ne1, n_tok)) launch_split(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias);
        else launch_tile(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias);
        PI_CHECK_LAUNCH(); return 0;
    }
    if (al16 && K >= 512) { if (exact) launch_rows<8, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); else launch_rows<8, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); }
    else if (al8)         { if (exact) launch_rows<4, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); else launch_rows<4, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); }
    else                  { if (exact) launch_rows<1, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); else launch_rows<1, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, bias); }
    PI_CHECK_LAUNCH(); return 0;
}

extern "C" int pi_op_round_bf16(const float * x, int64_t x_stride, int64_t n, int n_tok, uint16_t * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (n % 8 || x_stride < n || out_stride < n || out_stride % 8 || ((uintptr_t) out % 16)) { pi_set_error("pi_op_round_bf16: rows of a multiple of 8 values, 16-byte aligned where they are written"); return -1; }
    const int vec = x_stride % 4 == 0 && ((uintptr_t) x % 16) == 0;
    for (int t = 0; t < n_tok; t += 65535)                             // (rows are the grid's second dimension)
        PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 6.0 * n * n_tok, k_round_bf16, dim3((unsigned) ((n + 2047) / 2048), (unsigned) std::min(65535, n_tok - t)), dim3(256), 0, (hipStream_t) stream, x + (int64_t) t * x_stride, x_stride, n, vec,
                     out + (int64_t) t * out_stride, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
// The tile that needs the least time, by rounds of 256 workgroups: 2.5 us + K / 2048 * rounds * the cost of one, in us at K 2048: 32 x 64 4.6, 64 x 64 7.2, 64 x 96 10, 64 x 128 10.5, 128 x 128 19.5, 128 x 192 26, 128 x 256 31,
// 256 x 256 58.  The numbers are those that choose best among all tiles at 300 sizes (512 .. 32000 rows, K 1024 .. 4096, 40 .. 2048 tokens, weights from memory): 0.2 % above the quickest tile of each on the mean, 3.8 % with 6.3 and 8.5
// for the two smaller ones and without 64 x 128.  Both sides of the crossings, us: 2048 x 2048 at 512 tokens 64 x 64 12.0, 64 x 128 15.3, at 1000 18.4 and 15.4; 2560 x 2048 at 512 64 x 96 12.6, 64 x 64 15.2; 3072 x 2048 at 1000
// 64 x 64 24.8, 128 x 128 21.7; 12288 x 4096 at 700 64 x 96 106, 128 x 192 83; 32000 x 2048 at 512 128 x 192 79, 256 x 256 61
static int async_tile_of(int64_t rows, int64_t K, int n_tok, int64_t seg_rows, int n_seg, int & row_blocks, int & tok_blocks, int & blocks_of) {
    static const struct { int bn, bt; double us; } shape[] = { { 32, 64, 4.6 }, { 64, 64, 7.2 }, { 64, 96, 10.0 }, { 64, 128, 10.5 }, { 128, 128, 19.5 }, { 128, 192, 26.0 }, { 128, 256, 31.0 }, { 256, 256, 58.0 } };
    int best = 0; double least = 1e30;
    for (int i = 0; i < 8; i++) {
        const int64_t seg_blocks = seg_rows > 0 ? (seg_rows + shape[i].bn - 1) / shape[i].bn : 0, blocks = seg_rows > 0 ? (n_seg - 1) * seg_blocks + (rows - (n_seg - 1) * seg_rows + shape[i].bn - 1) / shape[i].bn : (rows + shape[i].bn - 1) / shape[i].bn;
        const int64_t toks = (n_tok + shape[i].bt - 1) / shape[i].bt, tiles = blocks * toks;
        if (tiles > INT32_MAX / 2) continue;
        const double cost = 2.5 + (double) K / 2048 * (double) ((tiles + 255) / 256) * shape[i].us;
        if (cost < least) { least = cost; best = i; row_blocks = (int) blocks; tok_blocks = (int) toks; blocks_of = (int) seg_blocks; }
    }
    return best;
}
// whether a pass takes the products of bfloat16 activations: more tokens than the kernels that share K out take, whole steps of K, offsets inside a tile in 32 bits
extern "C" int pi_op_dense_rounded_ok(const pi_weight * w, int64_t x_stride, int n_tok) {
    return w && w->type == PI_BF16 && n_tok > 1 && !dense_takes_split(w->ne1, n_tok) && w->ne0 > 0 && w->ne0 % 64 == 0 && ((uintptr_t) w->p0 % 16) == 0 && w->ne0 < (1 << 22) && x_stride < (1 << 22) && w->ne1 <= INT32_MAX;
}
// x: bfloat16 rows.  n_seg > 1: rows of the matrix in segments of seg_rows, each with an input of its own, x + g * seg_off (pi_op_dense_segments), in one launch
extern "C" int pi_op_dense_rounded(const pi_weight * w, const float * bias, const uint16_t * x, int64_t x_stride, int64_t seg_rows, int64_t seg_off, int n_seg, int n_tok, float * out, int64_t out_stride, int act_a, int64_t rows_a,
                                   int act_b, void * stream) {
    if (!w || w->type != PI_BF16) { pi_set_error("pi_op_dense_rounded: the weight must be bfloat16"); return -1; }
    if (n_tok <= 0 || w->ne1 <= 0) return 0;
    if (n_seg < 1 || (n_seg > 1 && (seg_rows < 1 || (int64_t) (n_seg - 1) * seg_rows >= w->ne1 || seg_rows % 4))) { pi_set_error("pi_op_dense_rounded: %d segments of %lld rows do not fit %lld rows", n_seg, (long long) seg_rows, (long long) w->ne1); return -1; }
    if (n_seg == 1) seg_rows = seg_off = 0;
    if (x_stride < (int64_t) (n_seg - 1) * seg_off + w->ne0 || out_stride < w->ne1) { pi_set_error("pi_op_dense_rounded: row strides (%lld, %lld) below the sizes (%lld, %lld)", (long long) x_stride, (long long) out_stride, (long long) w->ne0, (long long) w->ne1); return -1; }
    if (w->ne0 % 64 || ((uintptr_t) w->p0 % 16) || ((uintptr_t) x % 16) || x_stride % 8 || seg_off % 8 || seg_off < 0 || w->ne0 >= (1 << 22) || x_stride >= (1 << 22) || w->ne1 > INT32_MAX) {
        pi_set_error("pi_op_dense_rounded: rows of whole steps of 64 values, 16-byte aligned, of less than 2^22 values"); return -1;
    }
    hipStream_t s = (hipStream_t) stream;
    int row_blocks = 0, tok_blocks = 0, blocks_of = 0;
    const int which = async_tile_of(w->ne1, w->ne0, n_tok, seg_rows, n_seg, row_blocks, tok_blocks, blocks_of), tiles = row_blocks * tok_blocks;
    const double bytes = 2.0 * w->ne0 * w->ne1 + 2.0 * n_tok * n_seg * w->ne0 + 4.0 * n_tok * w->ne1;
    pi_round_dst rd = pi_round_take();
    if (rd.h && (rd.from % 4 || rd.n % 4 || rd.from < 0 || rd.from + rd.n > w->ne1 || rd.stride % 4)) { pi_set_error("pi_op_dense_rounded: rounded columns [%lld, + %lld) of %lld rows", (long long) rd.from, (long long) rd.n, (long long) w->ne1); return -1; }
#define DN_ASYNC(BN, BT, WN, WT, S) PI_KT_LAUNCH(PI_KT_MMQ, PI_BF16, std::min(n_tok, PI_KT_MAXNT - 1), bytes, (k_dense_async<BN, BT, WN, WT, S>), dim3((unsigned) ((tiles + 7) / 8 * 8)), dim3(64 * WN * WT), 0, s, \
                     (const uint16_t *) w->p0, w->ne0, w->ne1, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, bias, blocks_of, seg_rows, seg_off, n_seg - 1, tok_blocks, tiles, rd, pi_abort_word())
    switch (which) {
        case 0:  DN_ASYNC(32, 64, 2, 2, 4); break;
        case 1:  DN_ASYNC(64, 64, 2, 2, 4); break;                       // (eight waves of 16 x 32: 1 .. 13 % more, 5 on the mean)
        case 2:  DN_ASYNC(64, 96, 2, 2, 4); break;
        case 3:  DN_ASYNC(64, 128, 2, 4, 4); break;
        case 4:  DN_ASYNC(128, 128, 4, 2, 4); break;
        case 5:  DN_ASYNC(128, 192, 2, 4, 3); break;
        case 6:  DN_ASYNC(128, 256, 2, 4, 3); break;
        default: DN_ASYNC(256, 256, 4, 2, 2);
    }
#undef DN_ASYNC
    PI_CHECK_LAUNCH(); return 0;
}

// one matrix whose rows fall into segments that each read an input of their own: rows [g * seg_rows, (g + 1) * seg_rows) read x + g * seg_off (g < n_seg - 1; the last segment takes the remaining
// rows).  Few tokens (the mat-vec kernel): ONE launch; wider passes take a matrix-core launch per segment
extern "C" int pi_op_dense_segments(const pi_weight * w, const float * x, int64_t x_stride, int64_t seg_rows, int64_t seg_off, int n_seg, int n_tok, float * out, int64_t out_stride, int act_a, int64_t rows_a,
                                    int act_b, int exact, void * stream) {
    if (!w || w->type != PI_BF16) { pi_set_error("pi_op_dense: the weight must be bfloat16"); return -1; }
    if (n_tok <= 0 || w->ne1 <= 0) return 0;
    if (n_seg < 1 || seg_rows < 1 || (int64_t) (n_seg - 1) * seg_rows >= w->ne1) { pi_set_error("pi_op_dense_segments: %d segments of %lld rows do not fit %lld rows", n_seg, (long long) seg_rows, (long long) w->ne1); return -1; }
    const int64_t K = w->ne0;
    if (x_stride < (int64_t) (n_seg - 1) * seg_off + K || out_stride < w->ne1) { pi_set_error("pi_op_dense_segments: row strides below the sizes"); return -1; }
    const bool al16 = K % 8 == 0 && ((uintptr_t) w->p0 % 16) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0 && seg_off % 4 == 0;
    if (!exact && al16 && dense_takes_split(w->ne1, n_tok) && seg_rows % 32 == 0) {
        launch_split(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, (hipStream_t) stream, 2.0 * K * w->ne1 + 4.0 * n_tok * (n_seg * K + w->ne1), nullptr, seg_rows, seg_off, n_seg - 1);
        PI_CHECK_LAUNCH(); return 0;
    }
    if (exact || !al16 || n_tok < 16) {                                // (up to 15 tokens of segments that no split fits one launch of mat-vecs: 5 segments of 1000 rows, K 4096, 15 tokens 51 us, a launch each 55)
        const bool al8 = K % 4 == 0 && ((uintptr_t) w->p0 % 8) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0 && seg_off % 4 == 0;
        const double bytes = 2.0 * K * w->ne1 + 4.0 * n_tok * (n_seg * K + w->ne1);
        hipStream_t s = (hipStream_t) stream;
        if (al16 && K >= 512) { if (exact) launch_rows<8, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); else launch_rows<8, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); }
        else if (al8)         { if (exact) launch_rows<4, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); else launch_rows<4, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); }
        else                  { if (exact) launch_rows<1, true>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); else launch_rows<1, false>(w, x, x_stride, n_tok, out, out_stride, act_a, rows_a, act_b, s, bytes, nullptr, seg_rows, seg_off, n_seg - 1); }
        PI_CHECK_LAUNCH(); return 0;
    }
    for (int g = 0; g < n_seg; g++) {                                  // a view of the segment's rows
        pi_weight view = *w;
        const int64_t r0 = (int64_t) g * seg_rows;
        view.p0 = w->p0 + (size_t) r0 * K * 2; view.ne1 = g == n_seg - 1 ? w->ne1 - r0 : seg_rows;
        const int64_t ra = std::max<int64_t>(0, std::min<int64_t>(view.ne1, rows_a - r0));
        if (pi_op_dense(&view, x + g * seg_off, x_stride, n_tok, out + r0, out_stride, act_a, ra, act_b, exact, stream) != 0) return -1;
    }
    return 0;
}
