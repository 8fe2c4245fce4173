// Matrix-core tiles of the bfloat16 products, shared by the dense operators (dense.hip) and the routed experts (hybrid.hip).
//
//   D[token][row] += sum_k W[row][k] * bf16(X[token][k])         W bfloat16, X fp32 rounded to nearest even while it is staged, fp32 sums (v_mfma_f32_16x16x32_bf16)
//
// A workgroup of WN x WT waves owns BN rows x BT tokens.  64 values of K at a time are staged through LDS as bfloat16, in two buffers: while a buffer is multiplied, the other is filled from
// registers.  KG groups of waves share K out (every group stages and multiplies a part of its own, the sums meet at the end): where a matrix has few tiles a workgroup's steps follow each other with
// little to hide their latency behind.  Loads are issued two steps ahead of that, into two sets of registers.  A row of a buffer is 128 bytes, eight 16-byte chunks; chunk c of row r sits at
// place c ^ (r % 8): the sixteen rows an operand read touches, and the eight chunks of a row a staging write touches, then fall into different banks.
// What a step costs is the sum of what its waves do one after another, not any one unit's time (128 x 128 x 64 by four waves: matrix cores 36 % busy, LDS 36 %, address unit 57 %).  So the loads, the writes and the
// operand reads stand between the products, the barrier stands in the middle of a step's products, and loads take a scalar address that moves on and a 32-bit offset that stays: 14 vector instructions a step besides the
// 32 products, where clamping, masking and adding up addresses took 95.  us for 2048 x 2048 at 512 tokens 17.0, now 14.2; 4096 x 4096 at 2048 tokens (with 256 x 128 tiles) 111, now 82.
#pragma once
#include "ops_common.h"
#include <type_traits>

typedef __bf16 dt_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 dt_bf16x2 __attribute__((ext_vector_type(2)));
typedef float dt_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dt_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t dt_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dt_offs __attribute__((ext_vector_type(4)));          // offsets of up to four rows from a first one, in elements (an array of pointers would not stay in registers); rows of X that are gathered from a wide range take 64 bits each
typedef uint64_t dt_offs64 __attribute__((ext_vector_type(4)));

// a pointer to global memory that is the same in all lanes
typedef const __attribute__((address_space(1))) char dt_global;
static __device__ __forceinline__ dt_global * dt_uniform(const void * p) {
    const uint64_t v = (uint64_t) p;
    return (dt_global *) (((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (v >> 32)) << 32) | (uint32_t) __builtin_amdgcn_readfirstlane((int) v));
}
template <class V> static __device__ __forceinline__ V dt_load(dt_global * p) { return *(const __attribute__((address_space(1))) V *) p; }
// two fp32 values as bfloat16, nearest even (v_cvt_pk_bf16_f32)
static __device__ __forceinline__ uint32_t dt_pack(float a, float b) { const dt_bf16x2 v = { (__bf16) a, (__bf16) b }; return __builtin_bit_cast(uint32_t, v); }
static __device__ __forceinline__ dt_u32x4 dt_pack8(dt_f32x4 a, dt_f32x4 b) { return dt_u32x4{ dt_pack(a[0], a[1]), dt_pack(a[2], a[3]), dt_pack(b[0], b[1]), dt_pack(b[2], b[3]) }; }
static __device__ __forceinline__ dt_f32x4 dt_mfma(dt_u32x4 a, dt_u32x4 b, dt_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dt_bf16x8, a), __builtin_bit_cast(dt_bf16x8, b), c, 0, 0, 0); }

// a barrier behind this wave's reads and writes of LDS: the loads that are on their way stay so
static __device__ __forceinline__ void dt_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
#define DT_LDS_BYTES(BN, BT, KG) ((KG) * 2 * ((BN) + (BT)) * 128)
#define DT_LDS_BYTES_PL(BN, BT, PL) (2 * ((BN) + (PL) * (BT)) * 128)

// w + wo[i] / x + xo[i]: the rows this thread stages, numbers tid / 8 + (threads / 8) i of the tile; w and x are the same in all lanes (16-byte aligned, wo and dt_offs xo below 2^30; rows past the end repeat a valid one and are not stored); K % 8 == 0.
// PL = 3: X is not rounded but taken apart into three bfloat16 values that add up to it, three products instead of one: the products are exact, as an fp32 one of the two factors is.
// PAIR: an X value is join(x[k], x[k + pair_off]) of two fp32 values (the two halves of a gated hidden layer).  On return lane l of wave (wn, wt) holds in acc[a][b] the rows
// wn BN / WN + 16 a + 4 (l / 16) .. + 3 of token wt BT / WT + 16 b + l % 16.
template <int BN, int BT, int WN, int WT, int D, int KG, bool PAIR, int PL = 1, class Offs, class Join>
static __device__ __forceinline__ void dt_tile(const uint16_t * __restrict__ w, dt_offs wo, const float * __restrict__ x, Offs xo, int64_t pair_off, Join join, int64_t K, uint8_t * lds,
                                               dt_f32x4 (&acc)[BN / WN / 16][BT / WT / 16]) {
    static_assert(PL == 1 || KG == 1, "one group of waves where X is in three parts");
    static_assert(D == 2, "two register sets and two buffers: a step's are known when the code is compiled");
    constexpr int TH = 64 * WN * WT, SR = TH / 8;                      // threads of a group; rows they stage at a time
    constexpr int NW = BN / SR, NX = BT / SR, RT = BN / WN / 16, TT = BT / WT / 16, BUF = (BN + PL * BT) * 128;
    const int tid = threadIdx.x % TH, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4, kg = KG > 1 ? threadIdx.x / TH : 0;
    uint8_t * const all = lds;
    lds += kg * (2 * BUF);
    const int wn = wave / WT, wt = wave % WT, sr = tid >> 3, sc = tid & 7;
    // A thread loads 16 bytes of a row of W (its chunk sc) and twice 16 bytes of a row of X (values 4 sc and 32 + 4 sc): the eight threads of a row take a whole 128-byte line with each load.  (32 consecutive
    // bytes of X per thread touch every line twice: the address unit was busy 85 % of the time with that, at 32 bytes a cycle.)
    const int place = sr * 128 + ((sc ^ (sr & 7)) << 4);               // (rows a whole number of eights apart: the same place in their own)
    const int place_x = sr * 128 + (((sc >> 1) ^ (sr & 7)) << 4) + (sc & 1) * 8;      // (chunk 4 + sc / 2: the place with bit 6 turned over)
    // where this thread's loads begin, in bytes from w and x, which are the same for the whole workgroup: a load then takes a scalar address and one of these, and a step costs no address arithmetic
    dt_global * const wg = dt_uniform(w), * const xg = dt_uniform(x);
    uint32_t ow[NW]; std::conditional_t<std::is_same_v<Offs, dt_offs>, uint32_t, uint64_t> ox[NX];
#pragma unroll
    for (int i = 0; i < NW; i++) ow[i] = (wo[i] + sc * 8) * 2;
#pragma unroll
    for (int i = 0; i < NX; i++) ox[i] = (xo[i] + sc * 4) * 4;
    dt_u32x4 wset[D][NW]; dt_f32x4 xset[D][NX][2], yset[D][PAIR ? NX : 1][2];
    dt_u32x4 af[2][RT], bf[2][TT];
    const int steps = ((int) ((K + 63) / 64) + KG - 1) / KG;          // (of every group of waves: what a group has past the end of K is zeros)
    const int64_t kg0 = (int64_t) 64 * steps * __builtin_amdgcn_readfirstlane(kg);
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < TT; b++) acc[a][b] = dt_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // WHOLE: every group of waves has whole steps; otherwise loads past the end of K take the last values again, and zeros are staged for them
    auto walk = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        // (q of Q: a share of the rows, so that the loads and the writes of a step stand between its products.  A step past the end is the last one again, and nobody reads it)
        auto fetch = [&](int set, int i, int q, int Q) __attribute__((always_inline)) {
            const int64_t k0 = kg0 + 64 * (int64_t) (WHOLE ? min(i, steps - 1) : i);
            int64_t bw = 2 * k0, bx = 4 * k0, bx1 = 4 * k0 + 128;
            if constexpr (!WHOLE) {
                bw = 2 * (min(k0 + sc * 8, K - 8) - sc * 8);
                bx = 4 * (min(k0 + sc * 4, K - 4) - sc * 4); bx1 = 4 * (min(k0 + 32 + sc * 4, K - 4) - sc * 4);
            }
            dt_global * wk = wg + bw, * xk = xg + bx, * xk1 = xg + bx1;
#pragma unroll
            for (int r = 0; r < NW; r++) if (r * Q / NW == q) wset[set][r] = dt_load<dt_u32x4>(wk + ow[r]);
#pragma unroll
            for (int r = 0; r < NX; r++) if (r * Q / NX == q) {
                xset[set][r][0] = dt_load<dt_f32x4>(xk + ox[r]); xset[set][r][1] = dt_load<dt_f32x4>(xk1 + ox[r]);
                if constexpr (PAIR) { yset[set][r][0] = dt_load<dt_f32x4>(xk + 4 * pair_off + ox[r]); yset[set][r][1] = dt_load<dt_f32x4>(xk1 + 4 * pair_off + ox[r]); }
            }
        };
        auto stage = [&](int set, int buf, int i, int q, int Q) __attribute__((always_inline)) {
            const int64_t k0 = kg0 + 64 * (int64_t) i;
            const bool okw = WHOLE || k0 + sc * 8 < K, okx[2] = { WHOLE || k0 + sc * 4 < K, WHOLE || k0 + 32 + sc * 4 < K };      // (K % 8 == 0: four values are inside or outside as a whole)
            uint8_t * base = lds + buf * BUF;
#pragma unroll
            for (int r = 0; r < NW; r++) if (r * Q / NW == q) *(dt_u32x4 *) (base + place + r * (SR * 128)) = okw ? wset[set][r] : dt_u32x4{ 0, 0, 0, 0 };
#pragma unroll
            for (int r = 0; r < NX; r++) if (r * Q / NX == q)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    dt_f32x4 a = xset[set][r][h];
                    if constexpr (PAIR) {
#pragma unroll
                        for (int e = 0; e < 4; e++) a[e] = join(a[e], yset[set][r][h][e]);
                    }
                    a = okx[h] ? a : dt_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
                    for (int p = 0; p < PL; p++) {
                        const dt_u32x2 b = { dt_pack(a[0], a[1]), dt_pack(a[2], a[3]) };
                        *(dt_u32x2 *) (base + (BN + p * BT) * 128 + r * (SR * 128) + (h ? place_x ^ 64 : place_x)) = b;
                        if constexpr (PL > 1) a -= dt_f32x4{ __uint_as_float(b[0] << 16), __uint_as_float(b[0] & 0xffff0000u), __uint_as_float(b[1] << 16), __uint_as_float(b[1] & 0xffff0000u) };
                    }
                }
        };
        const int f_at[2] = { (kb ^ (li & 7)) << 4, ((4 + kb) ^ (li & 7)) << 4 };
        const uint8_t * const wl = lds + (wn * (BN / WN) + li) * 128, * const xl = lds + BN * 128 + (wt * (BT / WT) + li) * 128;
        auto operands = [&](int ks, int buf, int q, int Q) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < TT; b++) if (b * Q / (TT + RT) == q) bf[ks][b] = *(const dt_u32x4 *) (xl + buf * BUF + b * 2048 + f_at[ks]);
#pragma unroll
            for (int a = 0; a < RT; a++) if ((TT + a) * Q / (TT + RT) == q) af[ks][a] = *(const dt_u32x4 *) (wl + buf * BUF + a * 2048 + f_at[ks]);
        };
        constexpr int H = PL == 1 ? RT / 2 : 1, Q = PL == 1 ? RT + H : 1;      // groups of products behind and in front of a step's barrier
        // step i (buffer i % 2) is multiplied while step i + 1 goes from its registers to the other buffer and step i + 3 takes its place there.  In front of a step's barrier stand the products of its first half, those
        // of half the second, every write, every load and the reads of the second half; behind it the rest of the products and the reads of the next step's first half: a wave that waits has work on its way
        auto step = [&](auto dc, int i) __attribute__((always_inline)) {
            constexpr int d = decltype(dc)::value;
            if constexpr (PL == 1) {
#pragma unroll
                for (int g = 0; g < 2 * RT; g++) {
                    const int ks = g / RT, a = g % RT;
#pragma unroll
                    for (int b = 0; b < TT; b++) acc[a][b] = dt_mfma(af[ks][a], bf[ks][b], acc[a][b]);
                    if (g < RT) operands(1, d, g, RT);
                    if (g < Q) { stage(1 - d, 1 - d, i + 1, g, Q); fetch(1 - d, i + 3, g, Q); }
                    if (g == Q - 1) dt_barrier();
                    if (g >= Q) operands(0, 1 - d, g - Q, H);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                stage(1 - d, 1 - d, i + 1, 0, 1);
                fetch(1 - d, i + 3, 0, 1);
                const uint8_t * wb = wl + d * BUF, * xb = xl + d * BUF;
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    dt_u32x4 a1[RT], b1[TT];
#pragma unroll
                    for (int a = 0; a < RT; a++) a1[a] = *(const dt_u32x4 *) (wb + a * 2048 + f_at[ks]);
#pragma unroll
                    for (int p = 0; p < PL; p++) {
#pragma unroll
                        for (int b = 0; b < TT; b++) b1[b] = *(const dt_u32x4 *) (xb + p * BT * 128 + b * 2048 + f_at[ks]);
#pragma unroll
                        for (int a = 0; a < RT; a++)
#pragma unroll
                            for (int b = 0; b < TT; b++) acc[a][b] = dt_mfma(a1[a], b1[b], acc[a][b]);
                    }
                }
                dt_barrier();
            }
        };
        fetch(0, 0, 0, 1);
        stage(0, 0, 0, 0, 1);
#pragma unroll
        for (int d = 1; d <= D; d++)
#pragma unroll
            for (int q = 0; q < Q; q++) { fetch(d % D, d, q, Q); __builtin_amdgcn_sched_barrier(0); }      // (in the order of the steps', whose wait counts hold for these as well)
        dt_barrier();
        if constexpr (PL == 1) operands(0, 0, 0, 1);
        // (no way out between the two steps of a round: where paths with different loads on their way meet, the compiler waits for the younger ones too)
        int i = 0;
        for (; i + 2 <= steps; i += 2) { step(std::integral_constant<int, 0>{}, i); step(std::integral_constant<int, 1>{}, i + 1); }
        if (i < steps) step(std::integral_constant<int, 0>{}, i);
    };
    if (K % (64 * KG) == 0) walk(std::true_type{});
    else walk(std::false_type{});
    if constexpr (KG > 1) {                                            // the groups meet in LDS; the first one has the sum
        __syncthreads();                                               // (the last operands, read ahead, are of no use)
        dt_f32x4 * part = (dt_f32x4 *) all;                            // [group - 1][wave][tile][lane]
        static_assert((KG - 1) * WN * WT * RT * TT * 1024 <= KG * 2 * BUF, "the partial sums fit");
        if (kg > 0)
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int b = 0; b < TT; b++) part[(((kg - 1) * (WN * WT) + wave) * RT * TT + a * TT + b) * 64 + lane] = acc[a][b];
        __syncthreads();
        if (kg == 0)
#pragma unroll
            for (int o = 0; o < KG - 1; o++)
#pragma unroll
                for (int a = 0; a < RT; a++)
#pragma unroll
                    for (int b = 0; b < TT; b++) acc[a][b] += part[((o * (WN * WT) + wave) * RT * TT + a * TT + b) * 64 + lane];
    }
}
