// Matrix-core tiles of the bfloat16 products, shared by the dense operators (dense.hip) and the routed experts (hybrid.hip).
//
//   D[token][row] += sum_k W[row][k] * bf16(X[token][k])         W bfloat16, X fp32 rounded to nearest even while it is staged, fp32 sums (v_mfma_f32_16x16x32_bf16)
//
// A workgroup of four waves (WN x WT) owns BN rows x BT tokens.  64 values of K at a time are staged through LDS as bfloat16, in two buffers: while a buffer is multiplied, the other is filled from
// registers.  KG groups of four waves share K out (every group stages and multiplies a part of its own, the sums meet at the end): where a matrix has few tiles a workgroup's steps follow each other with
// little to hide their latency behind.  Loads are issued D steps ahead of that, into D sets of registers.  A row of a buffer is 128 bytes, eight 16-byte chunks; chunk c of row r sits at
// place c ^ (r % 8): the sixteen rows an operand read touches, and the eight chunks of a row a staging write touches, then fall into different banks.
#pragma once
#include "ops_common.h"

typedef __bf16 dt_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 dt_bf16x2 __attribute__((ext_vector_type(2)));
typedef float dt_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dt_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t dt_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dt_offs __attribute__((ext_vector_type(4)));          // offsets of up to four rows from a first one, in elements (an array of pointers would not stay in registers); rows of X that are gathered from a wide range take 64 bits each
typedef uint64_t dt_offs64 __attribute__((ext_vector_type(4)));

// two fp32 values as bfloat16, nearest even (v_cvt_pk_bf16_f32)
static __device__ __forceinline__ uint32_t dt_pack(float a, float b) { const dt_bf16x2 v = { (__bf16) a, (__bf16) b }; return __builtin_bit_cast(uint32_t, v); }
static __device__ __forceinline__ dt_u32x4 dt_pack8(dt_f32x4 a, dt_f32x4 b) { return dt_u32x4{ dt_pack(a[0], a[1]), dt_pack(a[2], a[3]), dt_pack(b[0], b[1]), dt_pack(b[2], b[3]) }; }
static __device__ __forceinline__ dt_f32x4 dt_mfma(dt_u32x4 a, dt_u32x4 b, dt_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dt_bf16x8, a), __builtin_bit_cast(dt_bf16x8, b), c, 0, 0, 0); }

#define DT_LDS_BYTES(BN, BT, KG) ((KG) * 2 * ((BN) + (BT)) * 128)
#define DT_LDS_BYTES_PL(BN, BT, PL) (2 * ((BN) + (PL) * (BT)) * 128)

// w + wo[i] / x + xo[i]: the rows this thread stages, numbers tid / 8 + 32 i of the tile (16-byte aligned; rows past the end repeat a valid one and are not stored); K % 8 == 0.
// PL = 3: X is not rounded but taken apart into three bfloat16 values that add up to it, three products instead of one: the products are exact, as an fp32 one of the two factors is.
// PAIR: an X value is join(x[k], x[k + pair_off]) of two fp32 values (the two halves of a gated hidden layer).  On return lane l of wave (wn, wt) holds in acc[a][b] the rows
// wn BN / WN + 16 a + 4 (l / 16) .. + 3 of token wt BT / WT + 16 b + l % 16.
template <int BN, int BT, int WN, int WT, int D, int KG, bool PAIR, int PL = 1, class Offs, class Join>
static __device__ __forceinline__ void dt_tile(const uint16_t * __restrict__ w, dt_offs wo, const float * __restrict__ x, Offs xo, int64_t pair_off, Join join, int64_t K, uint8_t * lds,
                                               dt_f32x4 (&acc)[BN / WN / 16][BT / WT / 16]) {
    static_assert(PL == 1 || KG == 1, "one group of waves where X is in three parts");
    static_assert(D % 2 == 0, "an even number of register sets: a step's buffer is known when the code is compiled");
    constexpr int NW = BN / 32, NX = BT / 32, RT = BN / WN / 16, TT = BT / WT / 16, BUF = (BN + PL * BT) * 128;
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4, kg = KG > 1 ? threadIdx.x >> 8 : 0;
    uint8_t * const all = lds;
    lds += kg * (2 * BUF);
    const int wn = wave / WT, wt = wave % WT, sr = tid >> 3, sc = tid & 7;
    // A thread loads 16 bytes of a row of W (its chunk sc) and twice 16 bytes of a row of X (values 4 sc and 32 + 4 sc): the eight threads of a row take a whole 128-byte line with each load.  (32 consecutive
    // bytes of X per thread touch every line twice: the address unit was busy 85 % of the time with that, at 32 bytes a cycle.)
    const int place = sr * 128 + ((sc ^ (sr & 7)) << 4);               // (rows 32 apart: the same place in their own 4 KB)
    const int place_x = sr * 128 + (((sc >> 1) ^ (sr & 7)) << 4) + (sc & 1) * 8;      // (chunk 4 + sc / 2: the place with bit 6 turned over)
    dt_u32x4 wset[D][NW]; dt_f32x4 xset[D][NX][2], yset[D][PAIR ? NX : 1][2];
    const dt_u32x4 zero4 = { 0, 0, 0, 0 }; const dt_f32x4 zerof = { 0.0f, 0.0f, 0.0f, 0.0f };
    const int64_t k_last = K - 8;
    auto fetch = [&](dt_u32x4 (&wreg)[NW], dt_f32x4 (&xreg)[NX][2], dt_f32x4 (&yreg)[PAIR ? NX : 1][2], int64_t k0) {
        const int64_t k = min(k0 + sc * 8, k_last);                    // (past the end: the last values again, made zero when they are staged)
        const int64_t ka = min(k0 + sc * 4, k_last + 4), kb4 = min(k0 + 32 + sc * 4, k_last + 4);
#pragma unroll
        for (int i = 0; i < NW; i++) wreg[i] = *(const dt_u32x4 *) (w + wo[i] + k);
#pragma unroll
        for (int i = 0; i < NX; i++) {
            xreg[i][0] = *(const dt_f32x4 *) (x + xo[i] + ka); xreg[i][1] = *(const dt_f32x4 *) (x + xo[i] + kb4);
            if constexpr (PAIR) { yreg[i][0] = *(const dt_f32x4 *) (x + xo[i] + pair_off + ka); yreg[i][1] = *(const dt_f32x4 *) (x + xo[i] + pair_off + kb4); }
        }
    };
    auto stage = [&](dt_u32x4 (&wreg)[NW], dt_f32x4 (&xreg)[NX][2], dt_f32x4 (&yreg)[PAIR ? NX : 1][2], int buf, int64_t k0) {
        if (k0 + 64 > K) {                                             // (K % 8 == 0: four values are inside or outside as a whole)
            if (k0 + sc * 8 > k_last)
#pragma unroll
                for (int i = 0; i < NW; i++) wreg[i] = zero4;
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (k0 + 32 * h + sc * 4 >= K)
#pragma unroll
                    for (int i = 0; i < NX; i++) {
                        xreg[i][h] = zerof;
                        if constexpr (PAIR) yreg[i][h] = zerof;
                    }
        }
        uint8_t * base = lds + buf * BUF;
#pragma unroll
        for (int i = 0; i < NW; i++) *(dt_u32x4 *) (base + place + i * 4096) = wreg[i];
#pragma unroll
        for (int i = 0; i < NX; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                dt_f32x4 a = xreg[i][h];
                if constexpr (PAIR) {
#pragma unroll
                    for (int e = 0; e < 4; e++) a[e] = join(a[e], yreg[i][h][e]);
                }
#pragma unroll
                for (int p = 0; p < PL; p++) {
                    const dt_u32x2 b = { dt_pack(a[0], a[1]), dt_pack(a[2], a[3]) };
                    *(dt_u32x2 *) (base + (BN + p * BT) * 128 + i * 4096 + (h ? place_x ^ 64 : place_x)) = b;
                    if constexpr (PL > 1) a -= dt_f32x4{ __uint_as_float(b[0] << 16), __uint_as_float(b[0] & 0xffff0000u), __uint_as_float(b[1] << 16), __uint_as_float(b[1] & 0xffff0000u) };
                }
            }
    };
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < TT; b++) acc[a][b] = dt_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // step i (buffer i % 2) is multiplied while step i + 1 goes from its registers to the other buffer and step i + 1 + D takes its place there
    const int steps = ((int) ((K + 63) / 64) + KG - 1) / KG;          // (of every group of waves: what a group has past the end of K is zeros)
    const int64_t kg0 = (int64_t) 64 * steps * kg;
    fetch(wset[0], xset[0], yset[0], kg0);
    stage(wset[0], xset[0], yset[0], 0, kg0);
#pragma unroll
    for (int d = 1; d <= D; d++) fetch(wset[d % D], xset[d % D], yset[d % D], kg0 + 64 * d);      // (a step past the end reads the last values again)
    __syncthreads();
    for (int i0 = 0; i0 < steps; i0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int i = i0 + d;
            if (i >= steps) break;
            const int nx = (d + 1) % D;
            // (no conditions here: where paths with different numbers of loads meet, the compiler waits for all of them.  Past the last step the other buffer gets values that nobody reads)
            stage(wset[nx], xset[nx], yset[nx], (d + 1) & 1, kg0 + 64 * (i + 1));
            fetch(wset[nx], xset[nx], yset[nx], kg0 + 64 * (i + 1 + D));
            const uint8_t * wb = lds + (d & 1) * BUF + (wn * (BN / WN) + li) * 128, * xb = lds + (d & 1) * BUF + BN * 128 + (wt * (BT / WT) + li) * 128;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const int at = ((ks * 4 + kb) ^ (li & 7)) << 4;
                dt_u32x4 af[RT], bf[TT];
#pragma unroll
                for (int a = 0; a < RT; a++) af[a] = *(const dt_u32x4 *) (wb + a * 2048 + at);
#pragma unroll
                for (int p = 0; p < PL; p++) {
#pragma unroll
                    for (int b = 0; b < TT; b++) bf[b] = *(const dt_u32x4 *) (xb + p * BT * 128 + b * 2048 + at);
#pragma unroll
                    for (int a = 0; a < RT; a++)
#pragma unroll
                        for (int b = 0; b < TT; b++) acc[a][b] = dt_mfma(af[a], bf[b], acc[a][b]);
                }
            }
            __syncthreads();
        }
    }
    if constexpr (KG > 1) {                                            // the groups meet in LDS; the first one has the sum
        dt_f32x4 * part = (dt_f32x4 *) all;                            // [group - 1][wave][tile][lane]
        static_assert((KG - 1) * 4 * RT * TT * 1024 <= KG * 2 * BUF, "the partial sums fit");
        if (kg > 0)
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int b = 0; b < TT; b++) part[(((kg - 1) * 4 + wave) * RT * TT + a * TT + b) * 64 + lane] = acc[a][b];
        __syncthreads();
        if (kg == 0)
#pragma unroll
            for (int o = 0; o < KG - 1; o++)
#pragma unroll
                for (int a = 0; a < RT; a++)
#pragma unroll
                    for (int b = 0; b < TT; b++) acc[a][b] += part[((o * 4 + wave) * RT * TT + a * TT + b) * 64 + lane];
    }
}
