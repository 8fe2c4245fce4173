// Matrix-core tiles of the bfloat16 products whose activations are bfloat16 already: both operands go from memory to LDS without a register between.
//
//   D[token][row] += sum_k W[row][k] * X[token][k]          W and X bfloat16, fp32 sums (v_mfma_f32_16x16x32_bf16)
//
// A workgroup of WN x WT waves owns BN rows x BT tokens.  64 values of K are a stage of (BN + BT) 128-byte rows; S stages are on their way or in use at a time (global_load_lds_dwordx4: a wave's load fills 1 KB of LDS in the
// order of its lanes, so the lanes' addresses carry the swizzle: chunk c of row r sits at place c ^ (r % 8), as in dense_tile.h).  What bounds the tiles that stage through registers (dense_tile.h) is how little a compute unit
// can have on its way: two steps' loads and the fp32 activations, twice the bytes, fill the registers.  Here it is up to 96 KB.  us on weights that are not in a cache, tiles of dense_tile.h / these: 2048 x 2048 at 512 tokens
// 13.4 / 9.2, 4096 x 4096 at 296 33.9 / 19.5, at 2048 79 / 56, 8192 x 2048 at 512 31.8 / 22.9, 32000 x 2048 at 333 89.6 / 59.5, 16384 x 4096 at 2048 305 / 207 (1330 TFLOP/s); fp32 activations staged the same way 10 - 60 % slower than
// bfloat16 ones everywhere.  Small grids are bound by the 64 bytes a clock that a compute unit takes from its L1 and by the first stage's trip to memory.
//
// The loads are written in assembly because the compiler, which cannot tell one stage of LDS from another, would wait for all of them ahead of every operand read.  They have no destination register; the waits are counted here.
#pragma once
#include "ops_common.h"
#include "dense_tile.h"
#include <type_traits>

static __device__ __forceinline__ void da_load(uint32_t lds, uint32_t offset, uint64_t base) {       // lds and base the same in all lanes (a write of m0 is one wait state ahead of its use)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
// all but the youngest N of this wave's loads have arrived, and its operand reads are done; then every wave's
template <int N> static __device__ __forceinline__ void da_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

// What lane l of a wave holds behind da_tile, four rows of sixteen tokens at a time, goes through the wave's own share of LDS, so that a store covers a token's RW rows (a store of four rows of sixteen tokens writes 64 bytes in
// sixteen places) and what is done to a value on its way stands in the code once, not once per register: with silu and sigmoid 16384 x 4096 at 2048 tokens took 329 us, 207 without.  put(token, row, four values) of the wave's part.
template <int RT, int TT, int BYTES, class Put>
static __device__ __forceinline__ void da_rows(dt_f32x4 (&acc)[RT][TT], uint8_t * share, Put put) {
    constexpr int RW = 16 * RT, ROW = RW + 4, NB = BYTES / (16 * ROW * 4) < TT ? BYTES / (16 * ROW * 4) : TT, LPT = RW / 4, TPI = 64 / LPT;
    static_assert(NB > 0, "sixteen tokens fit");
    const int lane = threadIdx.x & 63, li = lane & 15, kb = lane >> 4;
    float * const own = (float *) share;
#pragma unroll
    for (int b0 = 0; b0 < TT; b0 += NB) {
#pragma unroll
        for (int b = b0; b < b0 + NB && b < TT; b++)
#pragma unroll
            for (int a = 0; a < RT; a++) *(dt_f32x4 *) (own + ((b - b0) * 16 + li) * ROW + a * 16 + kb * 4) = acc[a][b];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int n = 16 * (TT - b0 < NB ? TT - b0 : NB);
#pragma unroll 1
        for (int t = lane / LPT; t < n; t += TPI) put(b0 * 16 + t, (lane % LPT) * 4, *(const dt_f32x4 *) (own + t * ROW + (lane % LPT) * 4));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

#define DA_LDS_BYTES(BN, BT, S) ((S) * ((BN) + (BT)) * 128)

// w, x: the same in all lanes, 16-byte aligned.  w_row(r), x_row(r): where row r of the tile begins, in bytes from w / x, below 2^32 (rows past the end repeat a valid one and are not stored).  steps = K / 64.
// On return lane l of wave (wn, wt) holds in acc[a][b] the rows wn BN / WN + 16 a + 4 (l / 16) .. + 3 of token wt BT / WT + 16 b + l % 16.
template <int BN, int BT, int WN, int WT, int S, class WRow, class XRow>
static __device__ __forceinline__ void da_tile(const uint16_t * __restrict__ w, WRow w_row, const uint16_t * __restrict__ x, XRow x_row, int steps, uint8_t * lds, dt_f32x4 (&acc)[BN / WN / 16][BT / WT / 16]) {
    constexpr int NW = WN * WT, LW = BN / 8 / NW, LX = BT / 8 / NW, L = LW + LX, RT = BN / WN / 16, TT = BT / WT / 16, STAGE = (BN + BT) * 128;
    static_assert(LW * 8 * NW == BN && LX * 8 * NW == BT, "a wave's loads are whole rows of one operand");
    static_assert(S >= 2 && L * (S - 1) < 64, "the wait counter holds what is on its way");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kb = lane >> 4, wn = wave / WT, wt = wave % WT;
    uint32_t ow[LW], ox[LX];
#pragma unroll
    for (int j = 0; j < LW; j++) { const int r = (wave + NW * j) * 8 + (lane >> 3); ow[j] = w_row(r) + (((lane & 7) ^ (r & 7)) << 4); }
#pragma unroll
    for (int j = 0; j < LX; j++) { const int r = (wave + NW * j) * 8 + (lane >> 3); ox[j] = x_row(r) + (((lane & 7) ^ (r & 7)) << 4); }
    uint64_t wp = (uint64_t) dt_uniform(w), xp = (uint64_t) dt_uniform(x);
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) lds, lw = lds0 + wave * 1024, lx = lds0 + BN * 128 + wave * 1024;
    // stage at byte `at` of LDS <- the next 64 values of K (q of Q: a share of the loads)
    auto fetch = [&](int at, int q, int Q) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LW; j++) if (j * Q / L == q) da_load(lw + at + j * NW * 1024, ow[j], wp);
#pragma unroll
        for (int j = 0; j < LX; j++) if ((LW + j) * Q / L == q) da_load(lx + at + j * NW * 1024, ox[j], xp);
        if (q == Q - 1) { wp += 128; xp += 128; }
    };
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < TT; b++) acc[a][b] = dt_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    dt_u32x4 af[2][RT], bf[2][TT];
    const int f_at[2] = { (kb ^ (li & 7)) << 4, ((4 + kb) ^ (li & 7)) << 4 };
    const uint8_t * const wl = lds + (wn * (BN / WN) + li) * 128, * const xl = lds + BN * 128 + (wt * (BT / WT) + li) * 128;
    auto operands = [&](int ks, int at, int q, int Q) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < TT; b++) if (b * Q / (TT + RT) == q) bf[ks][b] = *(const dt_u32x4 *) (xl + at + b * 2048 + f_at[ks]);
#pragma unroll
        for (int a = 0; a < RT; a++) if ((TT + a) * Q / (TT + RT) == q) af[ks][a] = *(const dt_u32x4 *) (wl + at + a * 2048 + f_at[ks]);
    };
    // A step: the products of the first half of its 64 values (operands read before) while the second half's are read; the next stage has arrived and nobody reads this one any more (the barrier); the second half's products while the
    // next stage's first operands are read and this stage's place is filled again.  LEFT: stages behind the next one that may still be on their way
    auto step = [&](int at, int next, auto left, auto more) __attribute__((always_inline)) {
        constexpr int LEFT = decltype(left)::value; constexpr bool MORE = decltype(more)::value;
#pragma unroll
        for (int a = 0; a < RT; a++) {
            operands(1, at, a, RT);
#pragma unroll
            for (int b = 0; b < TT; b++) acc[a][b] = dt_mfma(af[0][a], bf[0][b], acc[a][b]);
            __builtin_amdgcn_sched_barrier(0);
        }
        da_barrier<LEFT * L>();
#pragma unroll
        for (int a = 0; a < RT; a++) {
            operands(0, next, a, RT);                                  // (behind the last step: of no use, but inside the workgroup's LDS)
            if constexpr (MORE) fetch(at, a, RT);
#pragma unroll
            for (int b = 0; b < TT; b++) acc[a][b] = dt_mfma(af[1][a], bf[1][b], acc[a][b]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto behind = [](int at) __attribute__((always_inline)) { return at + STAGE == S * STAGE ? 0 : at + STAGE; };
    int at = 0;
    if (steps >= S) {
#pragma unroll
        for (int p = 0; p < S; p++) fetch(p * STAGE, 0, 1);
        da_barrier<(S - 1) * L>();
        operands(0, 0, 0, 1);
        for (int i = 0; i + S < steps; i++) { const int next = behind(at); step(at, next, std::integral_constant<int, S - 2>{}, std::true_type{}); at = next; }
        auto drain = [&](auto self, auto m) __attribute__((always_inline)) -> void {      // m steps left, all of their stages on their way
            constexpr int M = decltype(m)::value;
            const int next = behind(at);
            step(at, next, std::integral_constant<int, (M >= 2 ? M - 2 : 0)>{}, std::false_type{});
            at = next;
            if constexpr (M > 1) self(self, std::integral_constant<int, M - 1>{});
        };
        drain(drain, std::integral_constant<int, S>{});
    } else {
        for (int p = 0; p < steps; p++) fetch(p * STAGE, 0, 1);
        da_barrier<0>();
        operands(0, 0, 0, 1);
        for (int i = 0; i < steps; i++) { const int next = behind(at); step(at, next, std::integral_constant<int, 0>{}, std::false_type{}); at = next; }
    }
}
