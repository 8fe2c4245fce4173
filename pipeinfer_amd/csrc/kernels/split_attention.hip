// Attention of a prompt whose keys and values are up-projections of a latent, on the bfloat16 matrix cores, to fp32's precision.
//
// What bounds k_prompt_attention there is the fp32 matrix rate (157 TFLOP/s) and that nothing else goes to a SIMD's vector unit meanwhile.  Here queries, keys, values and weights are taken apart into three bfloat16 values each
// that add up to the fp32 one (8 + 8 + 8 bits of 24: nothing is lost), and a product is the six of their products that are not below 2^-24 of it, sums in fp32: six times the work at sixteen times the rate, and the vector unit is
// free beside it.  Keys and values are taken apart once, where they are written out (k_latent_split), in the order in which a wave's lanes read them as operands: a load is 1 KB in one piece, there is no LDS between and no
// barrier until the waves' sums meet.  Only the weights are taken apart in the loop.
// Measured, us (k_latent_expand + k_prompt_attention / these): 2048 tokens, 32 heads of 128, rank 512 425 / 260 (the parts 60, the attention 200: 1030 TFLOP/s of bfloat16 products); 512 tokens, 16 heads of 128 48 / 37; 1000 tokens, 16 heads
// of 128 + 64 127 / 78; 1500 of 64 + 32, rank 256 112 / 79; 64 tokens of 64 18.2 / 15.5; 33 tokens of 4000 cells 245 / 137.  Error against 64 bits (2-norm) at the same sizes 4.7e-7 / 3.8e-7, 4.6e-7 / 3.8e-7, 5.1e-7 / 3.9e-7,
// 3.7e-7 / 2.8e-7, 2.9e-7 / 2.4e-7, 5.0e-7 / 3.7e-7: a run's products with the values are summed for themselves, and what joins the sums of all cells is rounded once a run.
//   k_latent_split     the keys and values of the pass's cells from their latents (as k_latent_expand: exact products), and the keys' part that all heads share
//   k_split_attention  16 QU queries of a head to a workgroup; a wave owns every fourth run of 32 cells.  Scores transposed (rows = cells), so that what a lane holds - eight cells of one query - is the operand of the product
//                      with the values
#include "prompt_attention.h"
#include "dense_async.h"
#include "kernel_timing.h"

#include <algorithm>
#include <cmath>

#define SA_MAX_RANK 512                                                /* a run's latents fill 96 KB of LDS */

typedef __bf16 sa_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t sa_u32x4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ float sa_low(uint32_t x) { return __uint_as_float(x << 16); }
static __device__ __forceinline__ float sa_high(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }
// two values in three parts: nearest even, then what that leaves, twice
static __device__ __forceinline__ void sa_split(float a, float b, uint32_t & h, uint32_t & m, uint32_t & l) {
    h = dt_pack(a, b); a -= sa_low(h); b -= sa_high(h);
    m = dt_pack(a, b); a -= sa_low(m); b -= sa_high(m);
    l = dt_pack(a, b);
}
// eight values as three operands.  Infinities and NaNs are their first part alone, and what would round to an infinity is cut off instead
static __device__ __forceinline__ void sa_split8(const float (&x)[8], sa_u32x4 (&p)[3]) {
    uint32_t big = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) big = max(big, __float_as_uint(x[e]) & 0x7fffffffu);
#pragma unroll
    for (int i = 0; i < 4; i++) { uint32_t h, m, l; sa_split(x[2 * i], x[2 * i + 1], h, m, l); p[0][i] = h; p[1][i] = m; p[2][i] = l; }
    if (__builtin_expect(__any(big >= 0x7f7f8000u), 0)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t part[3] = { 0, 0, 0 };
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float v = x[2 * i + k];
                const uint32_t bits = __float_as_uint(v), mag = bits & 0x7fffffffu;
                uint32_t h = bits >> 16, m = 0, l = 0;
                if (mag > 0x7f800000u) h |= 0x40;
                else if (mag < 0x7f800000u) {
                    if (mag < 0x7f7f8000u) h = pi_round_one(v);
                    const float r = v - __uint_as_float(h << 16);
                    m = pi_round_one(r);
                    l = pi_round_one(r - __uint_as_float(m << 16));
                }
                part[0] |= h << (16 * k); part[1] |= m << (16 * k); part[2] |= l << (16 * k);
            }
#pragma unroll
            for (int q = 0; q < 3; q++) p[q][i] = part[q];
        }
    }
}
static __device__ __forceinline__ float sa_value(const sa_u32x4 (&p)[3], int e) {
    return e & 1 ? sa_high(p[0][e >> 1]) + (sa_high(p[1][e >> 1]) + sa_high(p[2][e >> 1])) : sa_low(p[0][e >> 1]) + (sa_low(p[1][e >> 1]) + sa_low(p[2][e >> 1]));
}
typedef float sa_f32x16 __attribute__((ext_vector_type(16)));
static __device__ __forceinline__ sa_f32x16 sa_mfma(sa_u32x4 a, sa_u32x4 b, sa_f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sa_bf16x8, a), __builtin_bit_cast(sa_bf16x8, b), c, 0, 0, 0); }
static __device__ __forceinline__ sa_f32x16 sa_zero() { return sa_f32x16{ 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f }; }

// An operand is 64 lanes x 16 bytes.  In units of operands, a run being 32 cells from cell0 on:
//   own keys     [head][run][step of 16 values][part]                        lane l: cell l % 32, values 8 (l / 32) .. + 7
//   shared keys  [run][step][part]                                           the same
//   values       [head][run][32 outputs][16 cells][part]                     lane l: output l % 32, cells 4 (l / 32) .. + 3 and 8 more of the sixteen
// Tiles of 256 rows of the two matrices x the 32 cells of a run; a workgroup takes tiles that follow each other, run by run.  A run's latents stand in LDS in three parts, as operands; a wave's 64 rows of a matrix come from memory
// to a part of LDS that is the wave's own (two stages of 64 values; dense_async.h has the loads), so that waves wait for their own loads alone.  The sums leave as operands from the registers they are in: keys after four
// exchanges between the halves of the wave, values as they are, their product being the other way round
#define SL_STAGE 8192
__global__ void __launch_bounds__(256, 1) k_latent_split(const float * __restrict__ cache, int64_t width, int rank, const uint16_t * __restrict__ wuk, int nk, const uint16_t * __restrict__ wuv, int nv, int dim_bits, int rot, int vdim_bits,
                                                         int cell0, int cell1, int live_max, const int32_t * __restrict__ dyn, sa_u32x4 * __restrict__ ko, sa_u32x4 * __restrict__ ro, sa_u32x4 * __restrict__ vo, int runs,
                                                         const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ __attribute__((aligned(1024))) uint8_t lds[SA_MAX_RANK * 192 + 8 * SL_STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, g = lane >> 5;
    if (dyn) { if (live_max > 0 && dyn[1] > live_max) return; cell1 = min(cell1, dyn[1]); }
    if (pi_abort_late(gone, abort_w, 5)) return;
    const int live = (max(cell1 - cell0, 0) + 31) / 32, k_blocks = (nk + 255) / 256, blocks = k_blocks + (nv + 255) / 256, steps = rank / 64;
    // From three tiles a workgroup on the same whole number to each but the last: the 32 of an XCD then stand at a few blocks of the matrices, whose rows they share in its L2.  In equal fractions they drift apart by a tile each at odd numbers
    // of runs (us, fractions / whole: 32 heads of 128, rank 512, 63 runs 96.6 / 68.2, 125 runs 172.9 / 110.5, even numbers alike); below, whole numbers leave compute units idle (1.5 tiles: up to 1.2 times as long)
    const int64_t all = (int64_t) live * blocks, wgs = gridDim.x, share = (all + wgs - 1) / wgs;
    const bool whole = all >= 3 * wgs;
    const int first = (int) (whole ? min(all, share * blockIdx.x) : all * blockIdx.x / wgs), last = (int) (whole ? min(all, share * (blockIdx.x + 1)) : all * (blockIdx.x + 1) / wgs);
    if (first >= last) return;
    sa_u32x4 * const xs = (sa_u32x4 *) lds;                            // [step of 16][part][64]
    uint8_t * const mine = lds + rank * 192 + wave * (2 * SL_STAGE);
    const uint32_t mine_at = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) mine;
    // the stage to be asked for next: step f_step of tile f_tile (past the last tile: that one again, so that the counts hold)
    int f_tile = first, f_step = 0, f_slot = 0;
    uint32_t f_off[8]; uint64_t f_base = 0;
    auto aim = [&]() __attribute__((always_inline)) {
        const int block = f_tile % blocks;
        const bool is_v = block >= k_blocks;
        const int n0 = (is_v ? block - k_blocks : block) * 256 + wave * 64, N = is_v ? nv : nk;
        f_base = (uint64_t) dt_uniform(is_v ? wuv : wuk);
#pragma unroll
        for (int j = 0; j < 8; j++) { const int r = j * 8 + (lane >> 3); f_off[j] = (uint32_t) min(n0 + r, N - 1) * (uint32_t) (rank * 2) + (((lane & 7) ^ (r & 7)) << 4); }
    };
    auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; j++) da_load(mine_at + f_slot * SL_STAGE + j * 1024, f_off[j], f_base + f_step * 128);
        f_slot ^= 1;
        if (++f_step == steps) { f_step = 0; f_tile = min(f_tile + 1, last - 1); aim(); }
    };
    aim();
    fetch(); fetch();
    sa_u32x4 w[2][4][2], x[2][2][3];                                   // [odd stage][step of 16][rows 0 .. 31, 32 .. 63]; [half of a stage][step of 16][part]
    int r_slot = 0;                                                    // the stage that is read next
    auto rows = [&](auto set) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int a = 0; a < 2; a++) w[decltype(set)::value][kk][a] = *(const sa_u32x4 *) (mine + r_slot * SL_STAGE + (32 * a + n) * 128 + (((2 * kk + g) ^ (n & 7)) << 4));
        r_slot ^= 1;
    };
    auto latents = [&](auto half, int step) __attribute__((always_inline)) {
        constexpr int H = decltype(half)::value;
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int p = 0; p < 3; p++) x[H][kk][p] = xs[((4 * step + 2 * H + kk) * 3 + p) * 64 + lane];
    };
    using zero = std::integral_constant<int, 0>; using one = std::integral_constant<int, 1>;
    int stored = 0;                                                    // stages for which a whole tile's twelve stores stand between the loads
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    rows(zero{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fetch();
    for (int tile = first; tile < last; ) {
        const int run = tile / blocks, end = min(last, (run + 1) * blocks), c0 = cell0 + run * 32;
        // the run's latents
        const float * const row = cache + (int64_t) min(c0 + n, cell1 - 1) * width + 8 * g;
        pa_f32x4 y0[SA_MAX_RANK / 64][2];
#pragma unroll
        for (int i = 0; i < SA_MAX_RANK / 64; i++) {                   // (all of them on their way together; a wave's steps past the end: the last one once more)
            const int ks = min(wave + 4 * i, rank / 16 - 1);
            y0[i][0] = *(const pa_f32x4 *) (row + 16 * ks); y0[i][1] = *(const pa_f32x4 *) (row + 16 * ks + 4);
        }
        __syncthreads();                                               // (the last run's are read)
#pragma unroll
        for (int i = 0; i < SA_MAX_RANK / 64; i++) {
            const int ks = wave + 4 * i;
            if (ks >= rank / 16) break;
            float y[8]; sa_u32x4 p[3];
#pragma unroll
            for (int e = 0; e < 8; e++) y[e] = y0[i][e >> 2][e & 3];
            sa_split8(y, p);
#pragma unroll
            for (int q = 0; q < 3; q++) xs[(ks * 3 + q) * 64 + lane] = p[q];
        }
        if (rot > 0 && tile % blocks == 0)                             // the keys' part that the heads share
            for (int ks = wave; ks < rot / 16; ks += 4) {
                float y[8]; sa_u32x4 p[3];
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = row[rank + 16 * ks + e];
                sa_split8(y, p);
#pragma unroll
                for (int q = 0; q < 3; q++) ro[(((int64_t) run * (rot / 16) + ks) * 3 + q) * 64 + lane] = p[q];
            }
        __syncthreads();
        latents(zero{}, 0);
        for (; tile < end; tile++) {                                   // (behind a run's last tile the first latents were read once more: now the next run's are)
            const int block = tile % blocks;
            const bool is_v = block >= k_blocks;
            sa_f32x16 acc[2] = { sa_zero(), sa_zero() };
            // A stage, its rows in registers: the next stage's have to be in LDS and go to registers beside the first half's products; then their place is asked for again
            auto stage = [&](auto set, auto value, int i) __attribute__((always_inline)) {
                constexpr int SET = decltype(set)::value;
                auto products = [&](auto half) __attribute__((always_inline)) {
                    constexpr int H = decltype(half)::value;
#pragma unroll
                    for (int kk = 0; kk < 2; kk++)
#pragma unroll
                        for (int p = 2; p >= 0; p--)
#pragma unroll
                            for (int a = 0; a < 2; a++) acc[a] = decltype(value)::value ? sa_mfma(x[H][kk][p], w[SET][2 * H + kk][a], acc[a]) : sa_mfma(w[SET][2 * H + kk][a], x[H][kk][p], acc[a]);
                };
                if (stored > 0) { asm volatile("s_waitcnt vmcnt(20) lgkmcnt(0)" ::: "memory"); stored--; }
                else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
                latents(one{}, i);
                rows(std::integral_constant<int, 1 - SET>{});
                __builtin_amdgcn_sched_barrier(0);                     // (all of them ahead of the products, which hide them)
                products(zero{});
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                fetch();
                latents(zero{}, i + 1 < steps ? i + 1 : 0);
                __builtin_amdgcn_sched_barrier(0);
                products(one{});
                __builtin_amdgcn_sched_barrier(0);
            };
            const int n0 = (is_v ? block - k_blocks : block) * 256 + wave * 64, N = is_v ? nv : nk;
            if (!is_v) {
#pragma unroll 1
                for (int i = 0; i < steps; i += 2) { stage(zero{}, std::false_type{}, i); stage(one{}, std::false_type{}, i + 1); }
            } else {
#pragma unroll 1
                for (int i = 0; i < steps; i += 2) { stage(zero{}, std::true_type{}, i); stage(one{}, std::true_type{}, i + 1); }
            }
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const int row0 = n0 + 32 * a, head = row0 >> (is_v ? vdim_bits : dim_bits), in = row0 - (head << (is_v ? vdim_bits : dim_bits));
                if (row0 >= N) continue;
                // sixteen rows of a head's 32: a step of its keys.  32 rows: its values of sixteen cells, twice
                sa_u32x4 * to = is_v ? vo + (((int64_t) head * runs + run) * (1 << (vdim_bits - 4)) + in / 16) * 192 : ko + (((int64_t) head * runs + run) * (1 << (dim_bits - 4)) + in / 16) * 192;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    float y[8]; sa_u32x4 p[3];
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const float lo = acc[a][8 * k + c], hi = acc[a][8 * k + 4 + c];
                        if (is_v) { y[c] = lo; y[4 + c] = hi; }
                        else {                                         // rows 8 b + 4 g + c of the lane's cell: the other half's of the same eight
                            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(lo), __float_as_int(hi), false, false);
                            y[c] = __int_as_float(r[0]); y[4 + c] = __int_as_float(r[1]);
                        }
                    }
                    sa_split8(y, p);
#pragma unroll
                    for (int q = 0; q < 3; q++) to[(k * 3 + q) * 64 + lane] = p[q];
                }
            }
            stored = n0 + 32 < N ? 2 : 0;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// the six products of two values in three parts, the small ones first
#define SA_A { 2, 1, 0, 1, 0, 0 }
#define SA_B { 0, 1, 2, 0, 1, 0 }

// KO, KR: steps of 16 values of a head's own keys and of the shared part; NJ: steps of 32 outputs; PARTS: waves that share the cells of 32 queries (the others have queries of their own).  Lane l of a wave holds, with n = l % 32 and
// g = l / 32: of query n the values 16 i + 8 g .. + 7 of step i, the scores of the cells 8 b + 4 g + c of a run (number 4 b + c), and the sums of the outputs 32 j + 8 b + 4 g + c.
// A run is 6 (KO + KR + 2 NJ) products of 32 clocks, some 350 vector instructions beside half of them (a vector instruction between two products is free up to six), and 60 that nothing stands beside
template <int KO, int KR, int NJ, int PARTS>
__global__ void __launch_bounds__(256, 1) k_split_attention(const pa_args A, const sa_u32x4 * __restrict__ kf, const sa_u32x4 * __restrict__ rf, const sa_u32x4 * __restrict__ vf, int runs, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int KS = KO + KR, VW = 32 * NJ, ROW = VW + 4, KB = KS % 4 == 0 ? 4 : 3, VB = KS > 8 ? 2 : NJ, STEP = 32 * PARTS, QUERIES = 32 * (4 / PARTS);      // KB, VB: steps whose keys, values are on their way
    constexpr int QLDS = 4 / PARTS * KS * 3072, MEET = 4 * 32 * ROW * 4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[QLDS > MEET ? QLDS : MEET];
    __shared__ float meet_m[4][32], meet_l[4][32];
    __shared__ int meet_odd[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, g = lane >> 5, part = wave % PARTS, group = wave / PARTS;
    const int h = blockIdx.x, t0 = (int) (gridDim.y - 1 - blockIdx.y) * QUERIES + 32 * group;        // (the last tokens, which see the most, first)
    const int words = (A.n_kv + 31) / 32, my_t = min(t0 + n, A.n_tok - 1);
    const sa_u32x4 * const kh = kf + (int64_t) h * runs * (KO * 192), * const vh = vf + (int64_t) h * runs * (NJ * 384);
    // Everything that a wave asks memory for ahead of its walk is on its way together: the mask of its first 64 runs, the queries, how many cells are live, the sink
    int base = A.cell0 + 32 * part, c_end = A.cell1;
    unsigned long long todo = 0;
    auto look = [&]() __attribute__((always_inline)) -> uint32_t {      // what the queries see of run `lane` of 64 (the words are there, whatever c_end is)
        const int c = base + STEP * lane;
        uint32_t any = 0;
        if (c < A.n_kv) {
            const uint32_t * at = A.mask + (c >> 5);
#pragma unroll 16
            for (int t = 0; t < 32; t++) any |= at[(int64_t) min(t0 + t, A.n_tok - 1) * words];
        }
        return any;
    };
    auto seen = [&](int c) __attribute__((always_inline)) -> uint32_t { return c_end - c >= 32 ? 0xffffffffu : (1u << max(c_end - c, 0)) - 1u; };
    constexpr int MINE = (KS + PARTS - 1) / PARTS;                     // operands of the queries that this wave takes apart
    pa_f32x4 x[MINE][2];
    const float * const qr = A.q + (int64_t) my_t * A.qs + (int64_t) h * (16 * KS) + 8 * g;
#pragma unroll
    for (int m = 0; m < MINE; m++) {
        const int i = min(part + PARTS * m, KS - 1);                   // (past the end: the last one once more)
        x[m][0] = *(const pa_f32x4 *) (qr + 16 * i); x[m][1] = *(const pa_f32x4 *) (qr + 16 * i + 4);
    }
    const float sk = A.sink ? A.sink[h] : 0.0f;
    const int live = A.dyn ? A.dyn[1] : A.n_kv;
    const uint32_t first_look = look();
    // the queries go to LDS, where each of the waves that share them takes some of the operands apart
    sa_u32x4 * const own = (sa_u32x4 *) lds + group * (KS * 192);
#pragma unroll
    for (int m = 0; m < MINE; m++) {
        pa_f32x4 * to = (pa_f32x4 *) own + min(part + PARTS * m, KS - 1) * 192 + lane;
        to[0] = x[m][0]; to[64] = x[m][1];
    }
    c_end = min(min(live, A.n_kv), A.cell1);
    if (A.live_max > 0 && min(live, A.n_kv) > A.live_max) return;
    if (pi_aborted_together(gone, abort_w, 5)) return;
    todo = __ballot((first_look & seen(base + STEP * lane)) != 0);
    // the runs of this wave that hold a cell which one of its queries sees, one after the other (-1: no more): 64 of them looked at at a time
    auto next = [&]() __attribute__((always_inline)) -> int {
        while (!todo) {
            base += 64 * STEP;
            if (base >= c_end) return -1;
            todo = __ballot((look() & seen(base + STEP * lane)) != 0);
        }
        const int c = base + STEP * (__ffsll(todo) - 1);
        todo &= todo - 1;
        return c;
    };
    const uint32_t mrow = (uint32_t) my_t * (uint32_t) words;
    auto key = [&](int c, int i, int p) __attribute__((always_inline)) -> sa_u32x4 {
        const int run = (c - A.cell0) >> 5;
        return i < KO ? kh[((int64_t) run * KO + i) * 192 + p * 64 + lane] : rf[((int64_t) run * KR + (i - KO)) * 192 + p * 64 + lane];
    };
    auto value = [&](int c, int j, int k, int p) __attribute__((always_inline)) -> sa_u32x4 { return vh[((int64_t) ((c - A.cell0) >> 5) * (2 * NJ) + 2 * j + k) * 192 + p * 64 + lane]; };
    sa_u32x4 k[KB][3], v[VB][2][3];
    uint32_t word = 0, word1 = 0;
    auto load_k = [&](int c, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 3; p++) k[i % KB][p] = key(c, i, p);
    };
    auto load_v = [&](int c, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int p = 0; p < 3; p++) v[j % VB][y][p] = value(c, j, y, p);
    };
    int c0 = base < c_end ? next() : -1, c1 = c0 >= 0 ? next() : -1, cn = c1 >= 0 ? c1 : c0;       // (cn behind the last run: of no use, but there)
    if (c0 >= 0) {
        word = A.mask[mrow + (uint32_t) (c0 >> 5)]; word1 = A.mask[mrow + (uint32_t) (cn >> 5)];
#pragma unroll
        for (int i = 0; i < KB; i++) load_k(c0, i);
    }
    sa_u32x4 q[KS][3];
#pragma unroll 1
    for (int i = part; i < KS; i += PARTS) {                           // times the scale, the shared part's turned by the token's position
        pa_f32x4 * at = (pa_f32x4 *) own + i * 192 + lane;
        const pa_f32x4 a = at[0], b = at[64];
        float y[8]; sa_u32x4 p[3];
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = e < 4 ? a[e & 3] : b[e & 3];
        if (KR > 0 && i >= KO) {
            const int pos = min(A.pos[my_t], A.n_pos - 1);
            const float * qt = A.q + (int64_t) my_t * A.qs + (int64_t) h * (16 * KS) + 16 * KO;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const pi_turn r = pi_turn_of(16 * (i - KO) + 8 * g + e, 8 * KR, A.pairing);
                const float2 t2 = A.cs[(int64_t) pos * (8 * KR) + r.angle];
                const float other = qt[r.mate];
                y[e] = r.lead ? y[e] * t2.x - other * t2.y : y[e] * t2.x + other * t2.y;
            }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] *= A.scale;
        sa_split8(y, p);
#pragma unroll
        for (int c = 0; c < 3; c++) own[(i * 3 + c) * 64 + lane] = p[c];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KS; i++)
#pragma unroll
        for (int c = 0; c < 3; c++) q[i][c] = own[(i * 3 + c) * 64 + lane];
    sa_f32x16 acc[NJ], s;
    float m_run, l_run;
    auto clear = [&]() __attribute__((always_inline)) {
        m_run = -INFINITY; l_run = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[j] = sa_zero();
    };
    // cells that a query does not see score minus infinity
    auto cover = [&](uint32_t vis) __attribute__((always_inline)) {
        const uint32_t mine = vis >> (4 * g);
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = mine >> (8 * (i >> 2) + (i & 3)) & 1u ? s[i] : -INFINITY;
    };
    // the maximum that the weights are relative to (k_prompt_attention: it may lag)
    auto raise = [&](float lag) __attribute__((always_inline)) {
        float top = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
        for (int i = 3; i < 15; i += 2) top = fmaxf(fmaxf(top, s[i]), s[i + 1]);
        top = fmaxf(top, s[15]);
        top = fmaxf(top, pi_partner<32>(top));
        if (__any(top > m_run + lag)) {
            const float m_new = top > m_run + lag ? top : m_run;
            const float f = m_run == m_new ? 1.0f : expf(m_run - m_new);                      // (nothing seen yet: expf(-inf) = 0)
            l_run *= f; m_run = m_new;
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[j] *= f;
        }
    };
    // The walk: while a run's scores become weights on the vector unit, the next run's scores are made on the matrix cores; then the products with the values
    clear();
    if (c0 >= 0) {
        const float lag = A.state ? 0.0f : 8.0f;
        sa_f32x16 s1[2];
        // scores of run c, whose first steps' keys are there; run `then`'s follow.  (beside(i): a share of what the vector unit does meanwhile, behind every product; SHARE: vector instructions of one)
        auto scores = [&](int c, int then, auto share, auto beside) __attribute__((always_inline)) {
            s1[0] = sa_zero(); s1[1] = sa_zero();
#pragma unroll
            for (int i = 0; i < KS; i++) {
#pragma unroll
                for (int w = 0; w < 6; w++) {
                    constexpr int KP[6] = SA_A, QP[6] = SA_B;
                    s1[w & 1] = sa_mfma(k[i % KB][KP[w]], q[i][QP[w]], s1[w & 1]);
                    beside(6 * i + w);
                    if (w & 1) {
                        if (w == 5) load_k(i + KB < KS ? c : then, (i + KB) % KS);
                        if constexpr (decltype(share)::value > 0)
#pragma unroll
                            for (int y = 0; y < 2; y++) { __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); __builtin_amdgcn_sched_group_barrier(0x2, decltype(share)::value, 0); }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        };
#pragma unroll
        for (int j = 0; j < VB; j++) load_v(c0, j);
        scores(c0, cn, std::integral_constant<int, 0>{}, [](int) {});
        auto run = [&](auto more, int then) __attribute__((always_inline)) {
            constexpr bool MORE = decltype(more)::value;
            const uint32_t vis = word & seen(c0);
            word = word1;
            s = s1[0] + s1[1];
            if (MORE) word1 = A.mask[mrow + (uint32_t) (then >> 5)];
            if (!__all(vis == 0xffffffffu)) cover(vis);
            raise(lag);
            __builtin_amdgcn_sched_barrier(0);
            sa_u32x4 w[2][3];
            // eight pairs of scores of a lane, three tasks for each: a weight, the other, both in three parts
            const float from = m_run == -INFINITY ? 0.0f : m_run;      // (scores of minus infinity alone: no weight, not a NaN)
            float sum = 0.0f;
            auto task = [&](int i) __attribute__((always_inline)) {
                const int d = i / 3;
                if (i % 3 < 2) { const float e = pi_exp_below(s[2 * d + i % 3] - from); s[2 * d + i % 3] = e; sum += e; }
                else { uint32_t hi, mid, lo; sa_split(s[2 * d], s[2 * d + 1], hi, mid, lo); w[d >> 2][0][d & 3] = hi; w[d >> 2][1][d & 3] = mid; w[d >> 2][2][d & 3] = lo; }
            };
            if constexpr (MORE) scores(cn, then, std::integral_constant<int, (300 + 6 * KS - 1) / (6 * KS)>{}, [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int y = 0; y < 24; y++) if (y * 6 * KS / 24 == i) task(y);
            });
            else
#pragma unroll
                for (int y = 0; y < 24; y++) task(y);
            l_run += sum;
            __builtin_amdgcn_sched_barrier(0);
            // a run's products for themselves, then to the sums: one rounding of these a run
            sa_f32x16 t[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j += 2) {
                t[j] = sa_zero(); t[j + 1] = sa_zero();
#pragma unroll
                for (int i = 0; i < 6; i++) {
                    constexpr int VP[6] = SA_A, WP[6] = SA_B;
#pragma unroll
                    for (int z = 0; z < 2; z++)
#pragma unroll
                        for (int y = 0; y < 2; y++) t[j + y] = sa_mfma(v[(j + y) % VB][z][VP[i]], w[z][WP[i]], t[j + y]);
                }
                if (j > 0) { acc[j - 2] += t[j - 2]; acc[j - 1] += t[j - 1]; }
#pragma unroll
                for (int y = 0; y < 2; y++) { if (j + y + VB < NJ) load_v(c0, j + y + VB); else if (MORE) load_v(cn, j + y + VB - NJ); }
#pragma unroll
                for (int i = 0; i < 24; i++) { __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); __builtin_amdgcn_sched_group_barrier(0x2, 3, 0); __builtin_amdgcn_sched_group_barrier(0x20, 1, 0); }
                __builtin_amdgcn_sched_barrier(0);
            }
            acc[NJ - 2] += t[NJ - 2]; acc[NJ - 1] += t[NJ - 1];
            __builtin_amdgcn_sched_barrier(0);
        };
        if (c1 >= 0) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x0f70);                        // vmcnt(0): where paths with different loads on their way meet, the compiler waits for the younger ones too, in every round
            __builtin_amdgcn_sched_barrier(0);
            do {
                const int c2 = next(), cm = c2 >= 0 ? c2 : c1;
                run(std::true_type{}, cm);
                c0 = c1; c1 = c2; cn = cm;
            } while (c1 >= 0);
        }
        run(std::false_type{}, c0);
    }
    // Values that are no numbers and sums out of range: as in k_prompt_attention.  The second walk is in fp32, from the values put together again.  (What a cell that nobody sees holds has met weights of zero, and is looked at here)
    uint32_t big = 0;
    int odd = 0, careful = 0;
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int c = 0; c < 16; c++) big = max(big, __float_as_uint(acc[j][c]) & 0x7fffffffu);
    if (__any(big >= 0x71800000u)) {
        careful = 1;
        clear();
        base = A.cell0 + 32 * part - 64 * STEP; todo = 0;
#pragma unroll 1
        for (int c = next(); c >= 0; c = next()) {
            const uint32_t vis = A.mask[mrow + (uint32_t) (c >> 5)] & seen(c);
            s = sa_zero();
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const sa_u32x4 y[3] = { key(c, i, 0), key(c, i, 1), key(c, i, 2) };
#pragma unroll
                for (int e = 0; e < 8; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(sa_value(y, e), sa_value(q[i], e), s, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            cover(vis);
            raise(0.0f);
            const float from = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
            for (int i = 0; i < 16; i++) { s[i] = pi_exp_below(s[i] - from); l_run += s[i]; }
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int z = 0; z < 2; z++) {                          // an infinity or a NaN among the values must not meet the zero weight of a query that does not see it: it joins at the end
                    const sa_u32x4 y[3] = { value(c, j, z, 0), value(c, j, z, 1), value(c, j, z, 2) };
                    float o[8]; bool bad = false;
#pragma unroll
                    for (int e = 0; e < 8; e++) { o[e] = sa_value(y, e); const bool b = (__float_as_uint(o[e]) & 0x7fffffffu) >= 0x7f800000u; bad |= b; o[e] = b ? 0.0f : o[e]; }
                    if (__any(bad)) odd = 1;
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(o[e], s[8 * z + e], acc[j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    }
    l_run += pi_partner<32>(l_run);
    if (lane == 0) meet_odd[wave] = odd | careful << 1;
    if (g == 0) { meet_m[wave][n] = m_run; meet_l[wave][n] = l_run; }
    // the waves of a group meet: sixteen threads per token, four outputs of every 64 each
    float (* const meet)[32][ROW] = (float (*)[32][ROW]) lds;
    constexpr int NV = VW / 64;
    __syncthreads();                                                   // (the queries are read)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int b = 0; b < 4; b++) *(pa_f32x4 *) &meet[wave][n][32 * j + 8 * b + 4 * g] = pa_f32x4{ acc[j][4 * b], acc[j][4 * b + 1], acc[j][4 * b + 2], acc[j][4 * b + 3] };
    __syncthreads();
    const int v0 = (tid & 15) * 4, w0 = group * PARTS;
#pragma unroll 1
    for (int r = tid / 16 % (4 * PARTS); r < 32; r += 4 * PARTS) {
        const int t = t0 + r;
        if (t >= A.n_tok) continue;
        float gates[NV][4];
        if (A.gate && A.gate_width > 1)
#pragma unroll
            for (int j = 0; j < NV; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) gates[j][e] = A.gate[(int64_t) t * A.gs + (int64_t) h * VW + v0 + 64 * j + e];
        int flags = 0;
        float * st = A.state ? A.state + ((int64_t) t * A.heads + h) * (VW + 2) : nullptr;
        float M = st && !A.first ? st[VW] : -INFINITY, L = 0.0f;
        const float m_before = M;
        pa_f32x4 o[NV];
#pragma unroll
        for (int w = 0; w < PARTS; w++) { M = fmaxf(M, meet_m[w0 + w][r]); flags |= meet_odd[w0 + w]; }
        if ((flags & 2) && !st)                                        // beside sums that weights of at most 1 are to keep in range: what the others' scores may have reached
#pragma unroll
            for (int w = 0; w < PARTS; w++) M = fmaxf(M, meet_m[w0 + w][r] + (meet_odd[w0 + w] & 2 ? 0.0f : 8.0f));
#pragma unroll
        for (int j = 0; j < NV; j++) o[j] = pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
        if (st && !A.first && m_before != -INFINITY) {
            const float f = expf(m_before - M);
            L = st[VW + 1] * f;
            if (f > 0.0f)
#pragma unroll
                for (int j = 0; j < NV; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[j][e] = st[v0 + 64 * j + e] * f;
        }
#pragma unroll
        for (int w = 0; w < PARTS; w++) {
            const float mw = meet_m[w0 + w][r], f = mw == -INFINITY ? 0.0f : expf(mw - M);
            L = fmaf(meet_l[w0 + w][r], f, L);
            if (mw != -INFINITY)
#pragma unroll
                for (int j = 0; j < NV; j++) o[j] += *(const pa_f32x4 *) &meet[w0 + w][r][v0 + 64 * j] * f;
        }
        if (flags & 1) {                                               // the infinities and NaNs of the cells that this token sees (each its first part alone)
            for (int cell = A.cell0; cell < c_end; cell++) {
                if (!(A.mask[(int64_t) t * words + (cell >> 5)] >> (cell & 31) & 1u)) continue;
                const int c = cell - A.cell0, slot = (c >> 3 & 1) * 4 + (c & 3), half = c >> 2 & 1;
#pragma unroll
                for (int j = 0; j < NV; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int vv = v0 + 64 * j + e;
                        const uint32_t two = vh[((int64_t) (c >> 5) * (2 * NJ) + (vv >> 5) * 2 + (c >> 4 & 1)) * 192 + half * 32 + (vv & 31)][slot >> 1];
                        const float y = slot & 1 ? sa_high(two) : sa_low(two);
                        if ((__float_as_uint(y) & 0x7fffffffu) >= 0x7f800000u) o[j][e] += y;
                    }
            }
        }
        if (!A.last) {
#pragma unroll
            for (int j = 0; j < NV; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) st[v0 + 64 * j + e] = o[j][e];
            if (v0 == 0) { st[VW] = M; st[VW + 1] = L; }
            continue;
        }
        const float ms = A.sink ? fmaxf(M, sk) : M, f = M == -INFINITY ? 0.0f : expf(M - ms);
        const bool none = M == -INFINITY;
        float mult = f / fmaf(L, f, A.sink ? expf(sk - ms) : 0.0f);
        if (A.gate && A.gate_width == 1) {
            float gt = A.gate[(int64_t) t * A.gs + h];
            if (A.gate_act == PI_ACT_SIGMOID) gt = 1.0f / (1.0f + expf(-gt));
            mult *= gt;
        }
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int vv = v0 + 64 * j;
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                y[e] = none ? 0.0f : o[j][e] * mult;
                if (A.gate && A.gate_width > 1) {
                    float gt = gates[j][e];
                    if (A.gate_act == PI_ACT_SIGMOID) gt = 1.0f / (1.0f + expf(-gt));
                    y[e] *= gt;
                }
            }
            if (!A.rd.only) {
                float * dst = A.out + (int64_t) t * A.os + (int64_t) h * VW + vv;
#pragma unroll
                for (int e = 0; e < 4; e++) dst[e] = y[e];
            }
            if (A.rd.h) pi_round_store4(A.rd, t, (int64_t) h * VW + vv, y[0], y[1], y[2], y[3]);
        }
    }
}

size_t sa_cell_floats(int heads, int dim, int rot, int vdim) { return (size_t) 3 * ((size_t) heads * (dim + vdim) + rot) / 2; }
bool sa_sizes(int dim, int rot, int vdim, int rank) { return rank > 0 && rank % 128 == 0 && rank <= SA_MAX_RANK && (dim == 64 || dim == 128) && (rot == 0 || rot == dim / 2) && (vdim == 64 || vdim == 128); }
bool sa_takes(const pa_args & a, int rank) {
    return sa_sizes(a.dim1, a.dim2, a.vdim, rank) && a.n_tok >= PA_LATENT_TOKENS && a.qs % 4 == 0 && ((uintptr_t) a.q & 15) == 0 && (int64_t) a.n_tok * ((a.n_kv + 31) / 32) < (1ll << 32);
}
// What a prompt takes, us: keys and values as they are (k_latent_expand + k_prompt_attention: two workgroups of 32 queries to a compute unit), in parts by four waves that share the cells of 32 queries, in parts by a wave for
// every 32 queries (a workgroup 128).  The last reads keys and values once for 128 queries and has no sums to join; the others have four times the workgroups.  The start, the latents' products, keys and values written and read, rounds of
// workgroups, and the walk: runs of cells x steps of a run, of all workgroups over the chip or of one over all cells, the longer one and a share of the other.  The constants are those that are nearest to 3500 sizes (six shapes of heads, 4 .. 192
// of them, 12 .. 2048 tokens, 12 .. 16000 cells): 14 .. 19 % off on the mean
enum { SA_PLAIN, SA_FOUR, SA_ONE };
static double sa_us(int form, const pa_args & a, int rank, int live) {
    static const struct { double start, latents, values, round, longer, shorter; int queries, cells, slots; } F[3] = {
        { 0.908, 5.74, 772, 18.2, 0.334, 0.353, 32, 128, 512 }, { 7.7, 5.02, 1520, 9.41, 0.153, 0.0183, 32, 128, 256 }, { 6.04, 3.87, 1520, 16.3, 0.133, 0.0434, 128, 32, 256 } };
    const auto & f = F[form];
    live = std::max(live, a.n_tok);
    const double values = 1e-9 * live * a.heads * (a.dim1 + a.vdim), groups = (double) a.heads * ((a.n_tok + f.queries - 1) / f.queries), seen = live - a.n_tok + 0.5 * (a.n_tok + f.queries);
    const double steps = form == SA_PLAIN ? (a.dim1 + 15) / 16 + (a.dim2 + 15) / 16 + 4 * ((a.vdim + 63) / 64) : (a.dim1 + a.dim2 + a.vdim) / 16;
    const double all = groups * seen / f.slots / f.cells * steps, one = (double) live / f.cells * steps;
    return f.start + f.latents * values * rank + f.values * values + f.round * std::ceil(groups / f.slots) + f.longer * std::max(all, one) + f.shorter * std::min(all, one);
}
// Four waves or one to 32 queries: by what they take with the pass's own cells alone and with all that there may be (how many are live is not known here).  us, four / one: 32 heads of 128, rank 512, 512 tokens alone 55 / 75, 1024 113 / 117, 2048
// 301 / 251; 128 heads, 128 tokens alone 44 / 47, 256 83 / 66, 512 180 / 138
static bool sa_many(const pa_args & a, int rank) { return sa_us(SA_ONE, a, rank, a.n_tok) / sa_us(SA_FOUR, a, rank, a.n_tok) + sa_us(SA_ONE, a, rank, a.n_kv) / sa_us(SA_FOUR, a, rank, a.n_kv) < 2; }
// In parts where that takes clearly less by the estimates, at both ends.  Few cells of more heads than a round of workgroups holds lose (us, as they are / in parts: 128 heads of 128, rank 512, 136 tokens alone 61 / 69; 64 heads of 64,
// rank 128, 300 tokens alone 34 / 40).  Of 8896 triples of a pass, cells live and cells there may be, times of the choice over those as they are: mean 0.80 (0.77 the quickest form each time), 1.00 at the 99th percent, at most 1.21
bool sa_pays(const pa_args & a, int rank, int live_max) {
    const int form = sa_many(a, rank) ? SA_ONE : SA_FOUR;
    return sa_us(form, a, rank, a.n_tok) <= 0.89 * sa_us(SA_PLAIN, a, rank, a.n_tok) && sa_us(form, a, rank, live_max) <= 0.89 * sa_us(SA_PLAIN, a, rank, live_max);
}
// scratch: 1.5 floats for every value of the cells [cell0, cell1) (sa_cell_floats), 16-byte aligned; cell0 a multiple of 64
void sa_launch(const pa_args & a, const float * cache, int rank, const pi_weight * wuk, const pi_weight * wuv, float * scratch, double bytes, hipStream_t s) {
    const int runs = (a.cell1 - a.cell0 + 63) / 64 * 2, tiles = (a.cell1 - a.cell0 + 31) / 32 * (int) ((wuk->ne1 + 255) / 256 + (wuv->ne1 + 255) / 256);
    sa_u32x4 * kf = (sa_u32x4 *) scratch, * vf = kf + (size_t) a.heads * runs * (a.dim1 / 16) * 192, * rf = vf + (size_t) a.heads * runs * (a.vdim / 16) * 192;
    PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, PI_KT_MAXNT - 1, 2.0 * rank * (wuk->ne1 + wuv->ne1) + 4.0 * std::min(a.cell1 - a.cell0, a.n_kv) * (double) (a.k2_row + 1.5 * (wuk->ne1 + wuv->ne1)), k_latent_split, dim3((unsigned) std::min(tiles, 256)), dim3(256), 0, s,
                 cache, a.k2_row, rank, (const uint16_t *) wuk->p0, (int) wuk->ne1, (const uint16_t *) wuv->p0, (int) wuv->ne1, a.dim1 == 64 ? 6 : 7, a.dim2, a.vdim == 64 ? 6 : 7, a.cell0, a.cell1, a.live_max, a.dyn, kf, rf, vf, runs, pi_abort_word());
    const int nta = std::min(a.n_tok, PI_KT_MAXNT - 1);
    const bool many = sa_many(a, rank);
#define SA_GO(KO, KR, NJ, P) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_split_attention<KO, KR, NJ, P>), dim3((unsigned) a.heads, (unsigned) ((a.n_tok + 128 / P - 1) / (128 / P))), dim3(256), 0, s, a, kf, rf, vf, runs, pi_abort_word())
#define SA_NJ(KO, KR) do { if (a.vdim == 64) { if (many) SA_GO(KO, KR, 2, 1); else SA_GO(KO, KR, 2, 4); } else if (many) SA_GO(KO, KR, 4, 1); else SA_GO(KO, KR, 4, 4); } while (0)
    if (a.dim1 == 64) { if (a.dim2) SA_NJ(4, 2); else SA_NJ(4, 0); }
    else if (a.dim2) SA_NJ(8, 4);
    else SA_NJ(8, 0);
#undef SA_NJ
#undef SA_GO
}
