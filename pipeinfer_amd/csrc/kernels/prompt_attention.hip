// Attention of a prompt: 32 tokens x one head per workgroup, scores and sums on the fp32 matrix cores.
//
// What bounds it: the fp32 matrix products (v_mfma_f32_16x16x4_f32: 157 TFLOP/s on the whole chip; 79 reached at 2048 tokens x 32 heads of 128) and the vector instructions, one after the other: while such a
// product runs, nothing else goes to its SIMD's vector unit, of whichever wave (2048 tokens: 830000 clocks, 530000 of products, 125000 of 240 vector instructions per tile of 16 cells x 32 tokens; with 460 of them 930000;
// tiles through LDS instead of registers, or the weights between the next tile's products: no less).  So a tile's vector work is kept small: weights relative to a maximum that may lag (below), cells that a token does
// not see as scores of minus infinity and only where there are some, an exponential for this range alone, no look at single values.  The kernels that give every token a workgroup (k_latent_scores, k_chunk_attention) are right for single
// tokens; with a prompt they read every key and value once per token and pay 2 rank instead of dim + vdim multiply-adds per pair of token and cell where the keys are up-projections of a latent.  Whole calls: 2048 tokens, 32 heads of 128, rank 512: 6.9 ms -> 0.44; 1000 tokens, 16 heads of 192: 1.11 ms -> 0.11;
// 1000 tokens of 16 differential heads over a window of 256: 526 us -> 70; 333 tokens of 16 heads of 64: 382 us -> 19.
//   k_latent_expand   the keys and values of the pass's cells written out once: an fp32 latent in three bfloat16 parts times the bfloat16 matrix on the matrix cores, exact products (dense_tile.h)
//   k_prompt_attention  a wave owns 32 queries (two operand tiles, so a key is read for both) and every fourth run of 32 cells; no barrier until the four waves' sums meet at the end.  The scores are
//                     computed transposed (rows = cells): what a lane then holds - four cells of one query - is already the operand of the product with the values, nothing crosses lanes but the maximum.
#include "prompt_attention.h"
#include "dense_tile.h"
#include "kernel_timing.h"

#include <algorithm>

typedef int pa_i32x4 __attribute__((ext_vector_type(4)));

// tiles of 128 rows of the two matrices x 64 cells; an XCD takes a contiguous run of tiles, eight blocks of rows wide and then along the cells (k_dense_tile)
__global__ void __launch_bounds__(256, 2) k_latent_expand(const float * __restrict__ cache, int64_t width, int64_t rank, const uint16_t * __restrict__ wuk, int64_t nk, const uint16_t * __restrict__ wuv, int64_t nv, int cell0, int cell1,
                                                          int live_max, const int32_t * __restrict__ dyn, float * __restrict__ ko, float * __restrict__ vo, int cell_blocks, int tiles, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 5)) return;
    __shared__ __attribute__((aligned(16))) uint8_t lds[DT_LDS_BYTES_PL(128, 64, 3)];
    const int tile = (int) (blockIdx.x & 7) * (int) (gridDim.x >> 3) + (int) (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int row_blocks = tiles / cell_blocks, grp = tile / (8 * cell_blocks), in_grp = tile % (8 * cell_blocks), gsz = min(8, row_blocks - 8 * grp);
    const int k_blocks = (int) ((nk + 127) / 128), block = 8 * grp + in_grp % gsz;
    const bool is_v = block >= k_blocks;
    const uint16_t * W = is_v ? wuv : wuk;
    const int64_t N = is_v ? nv : nk, n0 = (int64_t) (is_v ? block - k_blocks : block) * 128;
    if (dyn) { if (live_max > 0 && dyn[1] > live_max) return; cell1 = min(cell1, dyn[1]); }
    const int t0 = cell0 + (in_grp / gsz) * 64, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (t0 >= cell1) return;                                          // (cells of the context that hold nothing yet)
    dt_offs wo, xo;
#pragma unroll
    for (int i = 0; i < 4; i++) wo[i] = (uint32_t) ((min(n0 + (tid >> 3) + 32 * i, N - 1) - n0) * rank);
#pragma unroll
    for (int i = 0; i < 2; i++) xo[i] = (uint32_t) ((min(t0 + (tid >> 3) + 32 * i, cell1 - 1) - t0) * width);
    dt_f32x4 acc[4][2];
    dt_tile<128, 64, 2, 2, 2, 1, false, 3>(W + n0 * rank, wo, cache + (int64_t) t0 * width, xo, 0, [](float a, float) { return a; }, rank, lds, acc);
    float * out = is_v ? vo : ko;
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int cell = t0 + (wave & 1) * 32 + b * 16 + (lane & 15);
        if (cell >= cell1) continue;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int64_t n = n0 + (wave >> 1) * 64 + a * 16 + (lane >> 4) * 4;
            if (n < N) *(dt_f32x4 *) (out + (int64_t) (cell - cell0) * N + n) = acc[a][b];      // (N % 4 == 0)
        }
    }
}

// lane l: which of the 32 cells from c0 + step * l on lie at position `first` or behind it, or ahead of `keep` (the whole wave calls; two runs of 32 cells per load, so that a load is two lines of memory)
static __device__ __forceinline__ uint32_t pa_near(const int32_t * __restrict__ cell_pos, int c0, int step, int c_end, int first, int keep, int lane) {
    uint32_t near = 0;
#pragma unroll 8
    for (int i = 0; i < 32; i++) {
        const int cp = cell_pos[min(c0 + step * (2 * i + (lane >> 5)) + (lane & 31), c_end - 1)];
        const unsigned long long both = __ballot(cp >= first || cp < keep);
        if (lane >> 1 == i) near = (uint32_t) (lane & 1 ? both >> 32 : both);
    }
    return near;
}

// NK: steps of 16 key values (dim1 and dim2 rounded up each), NV: steps of 64 outputs.  Lane l of a wave holds, with n = l % 16 and g = l / 16: query 16 u + n (u = 0, 1), its key values 16 i + 4 g + c, the scores and
// weights of the cells 4 g + c of a tile of 16, and of the sums the outputs 4 NV (4 g + c) + j.  N1 > 0: whole steps only (dim1 = 16 N1, dim2 = 16 (NK - N1), vdim = 64 NV) and 32-bit offsets, so that a row's
// loads differ by constants: with an address apiece the registers held no more than one load at a time (2048 tokens, 32 heads of 128: 546 us, 495 this way), and the queries and
// the outputs have no test per value (32 tokens alone in a cache, 16 heads of 128 over 4: 20.2 us, 14.8 this way; a workgroup per token 15.7)
template <int NK, int N1, int NV, int MAPS>
__global__ void __launch_bounds__(256, N1 == 0 && NK + 4 * NV > 16 ? 1 : 2) k_prompt_attention(const pa_args A, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 5)) return;
    constexpr int NJ = 4 * NV, VW = 64 * NV, PARTS = 4 / MAPS;
    __shared__ __attribute__((aligned(16))) float meet[4][16][VW];
    __shared__ float meet_m[4][32], meet_l[4][32];
    __shared__ int meet_odd[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4, map = wave % MAPS, part = wave / MAPS;
    const int h = blockIdx.x, t0 = (int) (gridDim.y - 1 - blockIdx.y) * 32;       // (the last tokens, which see the most, first)
    const int n_kv = min(A.dyn ? A.dyn[1] : A.n_kv, A.n_kv), c_end = min(n_kv, A.cell1), words = (A.n_kv + 31) / 32;
    if (A.live_max > 0 && n_kv > A.live_max) return;
    const int dim1 = N1 > 0 ? 16 * N1 : A.dim1, dim2 = N1 > 0 ? 16 * (NK - N1) : A.dim2, vdim = N1 > 0 ? VW : A.vdim, n1 = (dim1 + 15) / 16;
    const float * k1 = A.k1 + (int64_t) (h / A.per_kv) * A.k1_head + map * dim1, * vb = A.v + (int64_t) (h / A.per_kv) * A.v_head;
    constexpr bool SHARED = N1 > 0 && N1 < NK;                         // keys of a latent: soft-max, the mask alone, no soft cap (pa_launch); the branches for the rest cost <12, 8, 2> 24 bytes of scratch a lane, 112.6 us instead of 109.7 for 1000 tokens
    const bool soft = SHARED || A.weights != PI_WEIGHTS_SIGMOID;
    pa_f32x4 q[2][NK], acc[2][NJ];
    float m_run[2] = { -INFINITY, -INFINITY }, l_run[2] = { 0.0f, 0.0f };
    int first_pos[2], odd = 0;
    uint32_t mrow[2];                                                  // (where its mask begins: pa_takes)
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int t = min(t0 + 16 * u + n, A.n_tok - 1), p = A.pos ? A.pos[t] : 0;
        mrow[u] = (uint32_t) t * (uint32_t) words;
        first_pos[u] = A.chunk <= 0 ? 0 : A.mask_kind == PI_MASK_WINDOW ? p - A.chunk + 1 : p / A.chunk * A.chunk;
        const float * qr = A.q + (int64_t) t * A.qs + (int64_t) (h * MAPS + map) * (dim1 + dim2);
#pragma unroll
        for (int i = 0; i < NK; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int d = (i < n1 ? i : i - n1) * 16 + 4 * g + c;
                float x = 0.0f;                                       // (values past the end: the keys there repeat others)
                if (i < n1) { if (d < dim1) x = qr[d]; }
                else if (d < dim2) {
                    const pi_turn r = pi_turn_of(d, dim2 / 2, A.pairing);
                    const float2 t2 = A.cs[(int64_t) min(p, A.n_pos - 1) * (dim2 / 2) + r.angle];
                    const float own = qr[dim1 + d], other = qr[dim1 + r.mate];
                    x = r.lead ? own * t2.x - other * t2.y : own * t2.x + other * t2.y;
                }
                q[u][i][c] = x;
                if (i >= n1) __builtin_amdgcn_sched_barrier(0);        // (one pair at a time)
            }
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[u][j] = pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    }
    const float bias = A.hbias ? A.hbias[h] : 0.0f;
    // Contexts whose walk is long: a lane looks at a run of 32 cells, the wave at 64 of its runs at a time, and only those are walked that hold a cell which one of the tokens may see (32 tokens in a window of 256 of 60000
    // cells: 160 us a workgroup per token, 630 with every run walked, 77 so; up to 64 runs of a wave the walk itself is as quick)
    const int start = (A.cell0 & ~31) + 32 * __builtin_amdgcn_readfirstlane(part);
    const bool far = c_end - start > 64 * 32 * PARTS;
    int first_min = 0;
    if (far) {
        first_min = min(first_pos[0], first_pos[1]);
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) first_min = min(first_min, __shfl_xor(first_min, o, 64));
        first_min = __builtin_amdgcn_readfirstlane(first_min);
    }
    // (a lane's rows from the tile's first on: the first that a tile reads is the scalar unit's)
    const uint32_t row1 = (uint32_t) A.k1_row * 4u, row2 = (uint32_t) A.k2_row * 4u, rowv = (uint32_t) A.v_row * 4u, lane1 = n * row1 + 16u * g, lane2 = n * row2 + 16u * g, lanev = 4u * g * rowv + 4u * (uint32_t) (NJ * n);
    // Values that are no numbers are looked for in the sums, behind the walk: where one is not finite, or so large (2^100) that a maximum which lags could have made it so, or the waves' sums together, the wave walks again with a look at
    // every value and weights of at most 1.  (Sums that the next launch adds to are relative to the maximum from the start)
    int careful = 0;
    for (; ; careful = 1) {
    const float lag = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(careful || A.state ? 0.0f : 8.0f)));
    unsigned long long todo = 0;
    for (int c0 = start; c0 < c_end; c0 += 32 * PARTS) {
        if (far) {
            const int at = (c0 - start) / (32 * PARTS) & 63;
            if (at == 0) {
                const int c = c0 + 32 * PARTS * lane;
                uint32_t any = 0;
                if (c < c_end) {
#pragma unroll 8
                    for (int t = 0; t < 32; t++) any |= A.mask[(int64_t) min(t0 + t, A.n_tok - 1) * words + (c >> 5)];
                }
                if (!SHARED && A.cell_pos) any &= pa_near(A.cell_pos, c0, 32 * PARTS, c_end, first_min, A.keep_first, lane);
                todo = __ballot(any != 0);
            }
            if (~todo) {
                const unsigned long long rest = todo >> at;
                const int skip = rest ? __ffsll(rest) - 1 : 63 - at;
                c0 += 32 * PARTS * skip;
                if (!rest) continue;
            }
        }
        uint32_t vis[2];
        const uint32_t in = (c_end - c0 >= 32 ? 0xffffffffu : (1u << (c_end - c0)) - 1u) & (c0 < A.cell0 ? 0xffffffffu << (A.cell0 - c0) : 0xffffffffu);
#pragma unroll
        for (int u = 0; u < 2; u++) vis[u] = A.mask[mrow[u] + (uint32_t) (c0 >> 5)] & in;
        if (!SHARED && A.cell_pos) {                   // a lane looks at eight cells, the four of a query put them together
            uint32_t near[2] = { 0u, 0u };
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const int cp = A.cell_pos[min(c0 + 8 * g + b, c_end - 1)];
#pragma unroll
                for (int u = 0; u < 2; u++) near[u] |= (cp >= first_pos[u] || cp < A.keep_first ? 1u : 0u) << (8 * g + b);
            }
#pragma unroll
            for (int u = 0; u < 2; u++) { near[u] |= __shfl_xor(near[u], 16, 64); near[u] |= __shfl_xor(near[u], 32, 64); vis[u] &= near[u]; }
        }
        int any = (int) (vis[0] | vis[1]);                            // the cells that any of the tokens sees; what the others hold is not read
        pi_butterfly<8>([&](auto o) { any |= pi_partner<decltype(o)::value>(any); });
        const uint32_t some = (uint32_t) __builtin_amdgcn_readfirstlane(any);
        const bool whole0 = __all(((vis[0] & vis[1]) & 0xffffu) == 0xffffu), whole1 = __all((vis[0] & vis[1]) >> 16 == 0xffffu);
#pragma unroll 1
        for (int half = 0; half < 2; half++) {
            const uint32_t here = (some >> (16 * half)) & 0xffffu;
            if (!here) continue;
            const int cb = c0 + 16 * half, spare = __ffs(here) - 1;
            const int ck = cb + (here >> n & 1u ? n : spare);
            pa_f32x4 kf[NK], vf[4][NV];
            if constexpr (N1 > 0) {
                const bool own = here >> n & 1u;
                const uint32_t o1 = (uint32_t) (cb - A.cell0) * row1 + (own ? lane1 : spare * row1 + 16u * g), o2 = N1 < NK ? (uint32_t) cb * row2 + (own ? lane2 : spare * row2 + 16u * g) : 0u;
#pragma unroll
                for (int i = 0; i < NK; i++) kf[i] = i < N1 ? *(const pa_f32x4 *) ((const char *) k1 + o1 + 64 * i) : *(const pa_f32x4 *) ((const char *) A.k2 + o2 + 64 * (i - N1));
            } else {
                const float * kr1 = k1 + (int64_t) (ck - A.cell0) * A.k1_row, * kr2 = A.k2 + (int64_t) ck * A.k2_row;
#pragma unroll
                for (int i = 0; i < NK; i++) {
                    const int d = (i < n1 ? i : i - n1) * 16 + 4 * g;
                    kf[i] = i < n1 || dim2 == 0 ? *(const pa_f32x4 *) (kr1 + min(d, dim1 - 4)) : *(const pa_f32x4 *) (kr2 + min(d, dim2 - 4));
                }
            }
            auto values = [&]() {
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    if constexpr (N1 > 0) {
                        const uint32_t o = (uint32_t) (cb - A.cell0) * rowv + (here >> (4 * g) & (1u << c) ? lanev + c * rowv : spare * rowv + 4u * (uint32_t) (NJ * n));
#pragma unroll
                        for (int j = 0; j < NV; j++) vf[c][j] = *(const pa_f32x4 *) ((const char *) vb + o + 16 * j);
                    } else {
                        const float * vr = vb + (int64_t) (cb + (here >> (4 * g + c) & 1u ? 4 * g + c : spare) - A.cell0) * A.v_row;
#pragma unroll
                        for (int j = 0; j < NV; j++) vf[c][j] = *(const pa_f32x4 *) (vr + min(NJ * n + 4 * j, vdim - 4));
                    }
                }
            };
            constexpr bool LATE = NK + 4 * NV > 16;                   // (the registers do not hold the keys and the values of a tile at a time)
            if constexpr (!LATE) values();
            if constexpr (N1 > 0) __builtin_amdgcn_sched_barrier(0);  // (all of them on their way before the first product)
            pa_f32x4 s[2] = { pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }, pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f } };
#pragma unroll
            for (int i = 0; i < NK; i++)
#pragma unroll
                for (int c = 0; c < 4; c++) { s[0] = pa_mfma(kf[i][c], q[0][i][c], s[0]); s[1] = pa_mfma(kf[i][c], q[1][i][c], s[1]); }
            if constexpr (LATE) { __builtin_amdgcn_sched_barrier(0); values(); }
            // Scores to weights (whole: every token sees every cell; else a cell that a token does not see scores minus infinity).  The maximum that a query's weights are relative to follows the scores' only when these pass
            // it by 8 (weights up to e^8 are as good in fp32 as long as no sum nears its range: below): of 128 tiles of a wave some 75 hold a new maximum of one of its 32 queries, and each of them cost all the sums their factor
#pragma unroll
            for (int u = 0; u < 2; u++) {
#pragma unroll
                for (int c = 0; c < 4; c++) s[u][c] = fmaf(s[u][c], A.scale, bias);
                if (!SHARED && soft && A.softcap > 0.0f) {
#pragma unroll
                    for (int c = 0; c < 4; c++) s[u][c] = A.softcap * tanhf(s[u][c] / A.softcap);
                }
                if (!(half ? whole1 : whole0)) {
                    const uint32_t mine = vis[u] >> (16 * half + 4 * g);
#pragma unroll
                    for (int c = 0; c < 4; c++) s[u][c] = mine >> c & 1u ? s[u][c] : -INFINITY;
                }
                if (soft) {
                    float top = fmaxf(fmaxf(s[u][0], s[u][1]), fmaxf(s[u][2], s[u][3]));
                    top = fmaxf(top, pi_partner<16>(top)); top = fmaxf(top, pi_partner<32>(top));
                    if (__any(top > m_run[u] + lag)) {
                        const float m_new = top > m_run[u] + lag ? top : m_run[u];
                        const float f = m_run[u] == m_new ? 1.0f : expf(m_run[u] - m_new);    // (nothing seen yet: expf(-inf) = 0)
                        l_run[u] *= f; m_run[u] = m_new;
#pragma unroll
                        for (int j = 0; j < NJ; j++) acc[u][j] *= f;
                    }
                    const float from = m_run[u] == -INFINITY ? 0.0f : m_run[u];               // (scores of minus infinity alone: no weight, not a NaN)
                    float sum = 0.0f;
#pragma unroll
                    for (int c = 0; c < 4; c++) { const float e = pi_exp_below(s[u][c] - from); s[u][c] = e; sum += e; }
                    l_run[u] += sum;                                                          // (a lane's own cells; the four of a query meet at the end)
                } else
#pragma unroll
                    for (int c = 0; c < 4; c++) s[u][c] = 1.0f / (1.0f + expf(-s[u][c]));
            }
            if (careful) {                                            // an infinity or a NaN among the values must not meet the zero weight of a token that does not see it: it joins at the end
                uint32_t big = 0;
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) big = max(big, __float_as_uint(vf[c][j >> 2][j & 3]) & 0x7fffffffu);
                if (__any(big >= 0x7f800000u)) {
                    odd = 1;
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int j = 0; j < NJ; j++) if ((__float_as_uint(vf[c][j >> 2][j & 3]) & 0x7fffffffu) >= 0x7f800000u) vf[c][j >> 2][j & 3] = 0.0f;
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int j = 0; j < NJ; j++) { acc[0][j] = pa_mfma(vf[c][j >> 2][j & 3], s[0][c], acc[0][j]); acc[1][j] = pa_mfma(vf[c][j >> 2][j & 3], s[1][c], acc[1][j]); }
        }
    }
    if (careful) break;
    uint32_t big = 0;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int c = 0; c < 4; c++) big = max(big, __float_as_uint(acc[u][j][c]) & 0x7fffffffu);
    if (!__any(big >= 0x71800000u)) break;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        m_run[u] = -INFINITY; l_run[u] = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[u][j] = pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    }
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        l_run[u] += __shfl_xor(l_run[u], 16, 64); l_run[u] += __shfl_xor(l_run[u], 32, 64);
        if (lane == 0) meet_odd[wave] = odd | careful << 1;
        if (g == 0) { meet_m[wave][16 * u + n] = m_run[u]; meet_l[wave][16 * u + n] = l_run[u]; }
    }
    // the waves meet, 16 tokens at a time: sixteen threads per token, four outputs of every 64 each
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (u) __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int j = 0; j < NV; j++) *(pa_f32x4 *) &meet[wave][n][NJ * (4 * g + c) + 4 * j] = pa_f32x4{ acc[u][4 * j][c], acc[u][4 * j + 1][c], acc[u][4 * j + 2][c], acc[u][4 * j + 3][c] };
        __syncthreads();
        const int r = tid >> 4, t = t0 + 16 * u + r, v0 = (tid & 15) * 4, again = (meet_odd[0] | meet_odd[1] | meet_odd[2] | meet_odd[3]) & 2;
        pa_f32x4 o[MAPS][NV]; float M[MAPS], L[MAPS];
        float * st = A.state ? A.state + ((int64_t) min(t, A.n_tok - 1) * A.heads + h) * (vdim + 2) : nullptr;
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            M[mp] = st && !A.first ? st[vdim] : -INFINITY; L[mp] = 0.0f;
            const float m_before = M[mp];
            if (soft) {
#pragma unroll
                for (int w = 0; w < PARTS; w++) M[mp] = fmaxf(M[mp], meet_m[w * MAPS + mp][16 * u + r]);
                if (again && !st)                                     // beside sums that weights of at most 1 are to keep in range: what the others' scores may have reached
#pragma unroll
                    for (int w = 0; w < PARTS; w++) M[mp] = fmaxf(M[mp], meet_m[w * MAPS + mp][16 * u + r] + (meet_odd[w * MAPS + mp] & 2 ? 0.0f : 8.0f));
            }
#pragma unroll
            for (int j = 0; j < NV; j++) o[mp][j] = pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
            if (st && !A.first) {
                const float f = !soft ? 1.0f : m_before == -INFINITY ? 0.0f : expf(m_before - M[mp]);
                L[mp] = st[vdim + 1] * f;
                if (f > 0.0f)
#pragma unroll
                    for (int j = 0; j < NV; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) if (v0 + 64 * j + e < vdim) o[mp][j][e] = st[v0 + 64 * j + e] * f;
            }
#pragma unroll
            for (int w = 0; w < PARTS; w++) {
                const int ww = w * MAPS + mp;
                const float mw = meet_m[ww][16 * u + r], f = !soft ? 1.0f : mw == -INFINITY ? 0.0f : expf(mw - M[mp]);
                L[mp] = fmaf(meet_l[ww][16 * u + r], f, L[mp]);
                if (!soft || mw != -INFINITY)
#pragma unroll
                    for (int j = 0; j < NV; j++) o[mp][j] += *(const pa_f32x4 *) &meet[ww][r][v0 + 64 * j] * f;
            }
        }
        if (t >= A.n_tok) continue;
        if ((meet_odd[0] | meet_odd[1] | meet_odd[2] | meet_odd[3]) & 1) {  // the infinities and NaNs of the cells that this token sees
            const int p = A.pos ? A.pos[t] : 0, fp = A.chunk <= 0 ? 0 : A.mask_kind == PI_MASK_WINDOW ? p - A.chunk + 1 : p / A.chunk * A.chunk;
            for (int cell = A.cell0; cell < c_end; cell++) {
                if (!(A.mask[(int64_t) t * words + (cell >> 5)] >> (cell & 31) & 1u)) continue;
                if (A.cell_pos && A.cell_pos[cell] < fp && A.cell_pos[cell] >= A.keep_first) continue;
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    const pa_f32x4 x = *(const pa_f32x4 *) (vb + (int64_t) (cell - A.cell0) * A.v_row + min(v0 + 64 * j, vdim - 4));
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if ((__float_as_uint(x[e]) & 0x7fffffffu) >= 0x7f800000u)
#pragma unroll
                            for (int mp = 0; mp < MAPS; mp++) o[mp][j][e] += x[e];
                }
            }
        }
        if (!A.last) {
#pragma unroll
            for (int j = 0; j < NV; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) if (v0 + 64 * j + e < vdim) st[v0 + 64 * j + e] = o[0][j][e];
            if (v0 == 0) { st[vdim] = M[0]; st[vdim + 1] = L[0]; }
            continue;
        }
        if (soft) {
            const bool has_sink = A.sink || A.weights == PI_WEIGHTS_SOFTMAX_SINK;
            const float sk = A.sink ? A.sink[h] : 0.0f;
#pragma unroll
            for (int mp = 0; mp < MAPS; mp++) {
                const float ms = has_sink ? fmaxf(M[mp], sk) : M[mp];
                const float f = M[mp] == -INFINITY ? 0.0f : expf(M[mp] - ms), den = fmaf(L[mp], f, has_sink ? expf(sk - ms) : 0.0f);
                const float inv = f / den;
#pragma unroll
                for (int j = 0; j < NV; j++) o[mp][j] = M[mp] == -INFINITY ? pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f } : o[mp][j] * inv;
            }
        }
        float mult = A.out_mult;
        if constexpr (MAPS == 2) {                                    // the difference of the two maps, normed
            float ss = 0.0f;
#pragma unroll
            for (int j = 0; j < NV; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) if (v0 + 64 * j + e < vdim) { const float x = o[0][j][e] - A.lam * o[1][j][e]; o[0][j][e] = x; ss = fmaf(x, x, ss); }
#pragma unroll
            for (int s = 1; s < 16; s <<= 1) ss += __shfl_xor(ss, s, 64);
            mult = A.out_mult / sqrtf(ss / (float) vdim + A.eps);
        } else if (A.gate && A.gate_width == 1) {
            float gt = A.gate[(int64_t) t * A.gs + h];
            if (A.gate_act == PI_ACT_SIGMOID) gt = 1.0f / (1.0f + expf(-gt));
            mult *= gt;
        }
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int v = v0 + 64 * j;
            if (v >= vdim) continue;                                  // (vdim % 4 == 0)
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[e] = o[0][j][e] * mult;
                if (MAPS == 1 && A.gate && A.gate_width > 1) {
                    float gt = A.gate[(int64_t) t * A.gs + (int64_t) h * vdim + v + e];
                    if (A.gate_act == PI_ACT_SIGMOID) gt = 1.0f / (1.0f + expf(-gt));
                    x[e] *= gt;
                }
            }
            if (!A.rd.only) {
                float * dst = A.out + (int64_t) t * A.os + (int64_t) h * vdim + v;
#pragma unroll
                for (int e = 0; e < 4; e++) dst[e] = x[e];
            }
            if (A.rd.h) pi_round_store4(A.rd, t, (int64_t) h * vdim + v, x[0], x[1], x[2], x[3]);
        }
    }
}

static int pa_steps(const pa_args & a) { return (a.dim1 + 15) / 16 + (a.dim2 + 15) / 16; }
bool pa_takes(const pa_args & a, int maps, int min_tokens) {
    auto four = [](int64_t n) { return (n & 3) == 0; };
    return a.n_tok >= min_tokens && pa_steps(a) <= 12 && a.vdim <= 128 && a.dim1 >= 4 && a.vdim >= 4 && four(a.dim1) && four(a.dim2) && four(a.vdim) && four(a.k1_row) && four(a.k1_head) && four(a.k2_row) && four(a.v_row) &&
           four(a.v_head) && ((uintptr_t) a.k1 & 15) == 0 && ((uintptr_t) a.k2 & 15) == 0 && ((uintptr_t) a.v & 15) == 0 && (maps == 1 || a.dim2 == 0) && (int64_t) a.n_tok * ((a.n_kv + 31) / 32) < (1ll << 32);
}
template <int NK, int N1, int NV>
static void pa_go(const pa_args & a, int maps, double bytes, hipStream_t s) {
    const dim3 grid((unsigned) a.heads, (unsigned) ((a.n_tok + 31) / 32));
    const int nta = std::min(a.n_tok, PI_KT_MAXNT - 1);
    if constexpr (N1 == 0 || N1 == NK)                                 // (two maps: no part that the heads share)
        if (maps == 2) { PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_prompt_attention<NK, N1, NV, 2>), grid, dim3(256), 0, s, a, pi_abort_word()); return; }
    PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_prompt_attention<NK, N1, NV, 1>), grid, dim3(256), 0, s, a, pi_abort_word());
}
void pa_launch(const pa_args & a, int maps, double bytes, hipStream_t s) {
    const int nk = pa_steps(a), n1 = a.dim1 / 16;
    const int64_t most = (int64_t) 1 << 30;                            // floats within 32-bit byte offsets
    const bool latent = !a.cell_pos && a.softcap <= 0.0f && a.weights != PI_WEIGHTS_SIGMOID;
    const bool whole = a.dim1 % 16 == 0 && a.dim2 % 16 == 0 && (a.vdim == 64 || a.vdim == 128) && (a.cell1 - a.cell0) * a.k1_row < most && (a.cell1 - a.cell0) * a.v_row < most && a.cell1 * a.k2_row < most;
#define PA_NK(NV) do { if (whole && nk == 4 && n1 == 4) pa_go<4, 4, NV>(a, maps, bytes, s); else if (whole && nk == 8 && n1 == 8) pa_go<8, 8, NV>(a, maps, bytes, s); \
                       else if (whole && latent && nk == 6 && n1 == 4) pa_go<6, 4, NV>(a, maps, bytes, s); else if (whole && latent && nk == 12 && n1 == 8) pa_go<12, 8, NV>(a, maps, bytes, s); \
                       else if (nk <= 4) pa_go<4, 0, NV>(a, maps, bytes, s); else if (nk <= 8) pa_go<8, 0, NV>(a, maps, bytes, s); else pa_go<12, 0, NV>(a, maps, bytes, s); } while (0)
    if (a.vdim <= 64) PA_NK(1); else PA_NK(2);
#undef PA_NK
}
void pa_expand(const float * cache, int64_t width, int rank, const pi_weight * wuk, const pi_weight * wuv, int cell0, int cell1, int n_kv, int live_max, const int32_t * dyn, float * k, float * v, hipStream_t s) {
    const int cell_blocks = (cell1 - cell0 + 63) / 64, tiles = cell_blocks * (int) ((wuk->ne1 + 127) / 128 + (wuv->ne1 + 127) / 128);
    PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, PI_KT_MAXNT - 1, 2.0 * rank * (wuk->ne1 + wuv->ne1) + 4.0 * std::min(cell1 - cell0, n_kv) * (double) (width + wuk->ne1 + wuv->ne1), k_latent_expand, dim3((unsigned) ((tiles + 7) / 8 * 8)), dim3(256), 0, s,
                 cache, width, (int64_t) rank, (const uint16_t *) wuk->p0, wuk->ne1, (const uint16_t *) wuv->p0, wuv->ne1, cell0, cell1, live_max, dyn, k, v, cell_blocks, tiles, pi_abort_word());
}

// ---- a few tokens ---------------------------------------------------------------------------------------------------------------------------------------------------
// grid (token, key head; split).  A workgroup per token that stages keys, then scores them, then stages values, waits for memory at every one of these (29 us for 4 tokens of 16 differential heads in a window of 256
// of 700 cells); here the keys and values of 32 cells are on their way together, the scores of the key head's query heads are one tile of a matrix product, and so is every 16 outputs of theirs.  With the merge of the
// splits, us: 4 tokens of 16 differential heads over 4 key heads in a window of 256 of 700 cells 34 -> 12.8; 8 tokens of 32 sigmoid heads in chunks of 64 of 350 cells 24 -> 8.9.
// Lane layout as above, rows = query heads: scores of row n and the cells 4 g + c, sums of row n and the outputs 16 NV wave + NV (4 g + r) + j
// FAR: splits of many runs of 32 cells: a lane looks at a run, the wave at 64 of them at a time (us for tokens in a window of 256 of 4000 cells, a context of 65536, 32 sigmoid heads: 35 with every run walked, 19 so; 16 tokens of 16 key heads in chunks of
// 512 of 60000 cells: 108 with a workgroup per token, 149, 36)
template <int NK, int NV, int MAPS, bool FAR>
__global__ void __launch_bounds__(256) k_few_attention(const pa_args A, int n_cs, int split_cells, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int V = 64 * NV, STEPS = MAPS == 2 ? NK : NK / 2;       // one map: two waves share a tile's key values
    typedef float vec __attribute__((ext_vector_type(NV)));
    __shared__ __attribute__((aligned(16))) float ps[MAPS][16][36], half[2][16][20];
    __shared__ float top[MAPS][2][16], sum[MAPS][2][16];
    const int G = A.heads / A.per_kv, t = blockIdx.x / G, kvh = blockIdx.x % G, cs = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4, ct = wave & 1, wm = wave >> 1;
    const int n_kv = min(A.dyn ? A.dyn[1] : A.n_kv, A.n_kv), words = (A.n_kv + 31) / 32, c_end = min(n_kv, (cs + 1) * split_cells);
    const int h = kvh * A.per_kv + min(n, A.per_kv - 1), p = A.pos[t], map = MAPS == 2 ? wm : 0, step0 = MAPS == 2 ? 0 : wm * STEPS;
    const int first = A.chunk <= 0 ? 0 : A.mask_kind == PI_MASK_WINDOW ? p - A.chunk + 1 : p / A.chunk * A.chunk;
    const bool soft = A.weights != PI_WEIGHTS_SIGMOID;
    const float * qr = A.q + (int64_t) t * A.qs + (int64_t) (h * MAPS + map) * (16 * NK), * kb = A.k1 + (int64_t) kvh * A.k1_head + map * (16 * NK), * vb = A.v + (int64_t) kvh * A.v_head;
    const float bias = A.hbias ? A.hbias[h] : 0.0f;
    pa_f32x4 qf[STEPS], acc[MAPS][NV];
#pragma unroll
    for (int i = 0; i < STEPS; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) qf[i][c] = qr[16 * (step0 + i) + 4 * g + c];
    float m_run[MAPS], l_run[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        m_run[mp] = -INFINITY; l_run[mp] = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; j++) acc[mp][j] = pa_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    }
    bool any = false;
    const int start = cs * split_cells;
    uint32_t seen = 0;
    for (int c0 = start; c0 < c_end; c0 += 32) {
        uint32_t vis;
        if constexpr (FAR) {
            const int at = (c0 - start) >> 5 & 63;
            if (at == 0) {
                const int c = c0 + 32 * lane;
                seen = c < c_end ? A.mask[(int64_t) t * words + (c >> 5)] : 0u;
                if (c_end - c < 32 && c < c_end) seen &= (1u << (c_end - c)) - 1u;
                seen &= pa_near(A.cell_pos, c0, 32, c_end, first, A.keep_first, lane);
            }
            const unsigned long long rest = __ballot(seen != 0) >> at;
            const int skip = rest ? __ffsll(rest) - 1 : 63 - at;
            c0 += 32 * skip;
            if (!rest) continue;
            vis = (uint32_t) __builtin_amdgcn_readlane((int) seen, at + skip);
        } else {
            const int mc = c0 + (lane & 31);
            bool see = false;
            if (mc < c_end) { const int cp = A.cell_pos[mc]; see = (A.mask[(int64_t) t * words + (c0 >> 5)] >> (lane & 31) & 1u) && (cp >= first || cp < A.keep_first); }
            vis = (uint32_t) __ballot(see);
        }
        if (gone & 1) break;                                          // (a cancelled run: its keys and values are not read)
        if (!vis) continue;
        pa_f32x4 kf[STEPS]; vec vf[2][4];
        {
            const float * kr = kb + (int64_t) min(c0 + 16 * ct + n, c_end - 1) * A.k1_row + 16 * step0 + 4 * g;
#pragma unroll
            for (int i = 0; i < STEPS; i++) kf[i] = *(const pa_f32x4 *) (kr + 16 * i);
        }
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
            for (int c = 0; c < 4; c++) vf[jt][c] = *(const vec *) (vb + (int64_t) min(c0 + 16 * jt + 4 * g + c, c_end - 1) * A.v_row + 16 * NV * wave + NV * n);
        __builtin_amdgcn_sched_barrier(0);
        pa_f32x4 s = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < STEPS; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) s = pa_mfma(kf[i][c], qf[i][c], s);
        if (any) __syncthreads();                                     // (the last round's weights are no longer read)
        if constexpr (MAPS == 1) {
            if (wm) *(pa_f32x4 *) &half[ct][n][4 * g] = s;
            __syncthreads();
            if (!wm) s += *(const pa_f32x4 *) &half[ct][n][4 * g];
        }
        const bool scores = MAPS == 2 || !wm;
        const uint32_t mine = vis >> (16 * ct + 4 * g);
        float m = -INFINITY;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float x = s[c] * A.scale + bias;
            if (soft && A.softcap > 0.0f) x = A.softcap * tanhf(x / A.softcap);
            s[c] = x;
            if (mine >> c & 1u) m = fmaxf(m, x);
        }
        if (soft) {
            m = fmaxf(m, __shfl_xor(m, 16, 64)); m = fmaxf(m, __shfl_xor(m, 32, 64));
            if (scores && g == 0) top[map][ct][n] = m;
            __syncthreads();
        }
        float m_new[MAPS], f[MAPS], from[MAPS];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            m_new[mp] = soft ? fmaxf(m_run[mp], fmaxf(top[mp][0][n], top[mp][1][n])) : 0.0f;
            f[mp] = !soft || m_run[mp] == m_new[mp] ? 1.0f : expf(m_run[mp] - m_new[mp]);
            m_run[mp] = m_new[mp];
            from[mp] = m_new[mp] == -INFINITY ? 0.0f : m_new[mp];     // (scores of minus infinity alone: no weight, not a NaN)
        }
        if (scores) {
            float l = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; c++) { const float e = !(mine >> c & 1u) ? 0.0f : soft ? expf(s[c] - from[map]) : 1.0f / (1.0f + expf(-s[c])); s[c] = e; l += e; }
            l += __shfl_xor(l, 16, 64); l += __shfl_xor(l, 32, 64);
            if (g == 0) sum[map][ct][n] = l;
            *(pa_f32x4 *) &ps[map][n][16 * ct + 4 * g] = s;
        }
        __syncthreads();
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
            for (int c = 0; c < 4; c++) if (!(vis >> (16 * jt + 4 * g + c) & 1u)) vf[jt][c] = vec(0.0f);        // (a cell that the token does not see may hold anything)
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            l_run[mp] = fmaf(l_run[mp], f[mp], sum[mp][0][n] + sum[mp][1][n]);
#pragma unroll
            for (int j = 0; j < NV; j++) acc[mp][j] *= f[mp];
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                const pa_f32x4 w = *(const pa_f32x4 *) &ps[mp][n][16 * jt + 4 * g];
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int j = 0; j < NV; j++) { float x; if constexpr (NV == 1) x = vf[jt][c][0]; else x = vf[jt][c][j]; acc[mp][j] = pa_mfma(x, w[c], acc[mp][j]); }
            }
        }
        any = true;
    }
    if (pi_abort_late(gone, abort_w, 5) || n >= A.per_kv) return;
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        float * pr = A.state + (((int64_t) (t * A.heads + h) * MAPS + mp) * n_cs + cs) * (V + 2);
        if (wave == 0 && g == 0) { pr[V] = any ? m_run[mp] : -INFINITY; pr[V + 1] = l_run[mp]; }
        if (any)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < NV; j++) pr[16 * NV * wave + NV * (4 * g + r) + j] = acc[mp][j][r];
    }
}
int pa_few_split(const pa_args & a, int maps, size_t scratch_floats, int * split_cells) {
    auto four = [](int64_t n) { return (n & 3) == 0; };
    if (a.n_tok >= PA_CACHE_TOKENS || a.n_kv <= 64 || !a.state || a.per_kv > 16 || (a.dim1 != 64 && a.dim1 != 128) || (a.vdim != 64 && a.vdim != 128) || !four(a.k1_row) || !four(a.k1_head) || !four(a.v_row) || !four(a.v_head) ||
        (((uintptr_t) a.k1 | (uintptr_t) a.v) & 15)) return 0;
    const int most = std::max(1, std::min(PA_FEW_SPLITS, 8192 / (a.n_tok * (a.heads / a.per_kv))));      // (more workgroups than that only wait for each other: 31 tokens of 16 key heads, 64 live cells of 1024: 16.1 us with a workgroup per token, 20.3 with 32 splits, 13.7 with 16; 16 tokens,
                                                                                                          // 200 cells of 4096: 15.4, with half as many workgroups 19.4)
    const int chunks = (a.n_kv + 31) / 32, per = (chunks + most - 1) / most, n_cs = (chunks + per - 1) / per;
    if ((size_t) a.n_tok * a.heads * maps * n_cs * (a.vdim + 2) > scratch_floats) return 0;
    *split_cells = 32 * per;
    return n_cs;
}
void pa_few_launch(const pa_args & a, int maps, int n_cs, int split_cells, double bytes, hipStream_t s) {
    const dim3 grid((unsigned) (a.n_tok * (a.heads / a.per_kv)), (unsigned) n_cs);
    const int nta = std::min(a.n_tok, PI_KT_MAXNT - 1);
#define FEW_GO2(NK, NV, MAPS, FAR) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_few_attention<NK, NV, MAPS, FAR>), grid, dim3(256), 0, s, a, n_cs, split_cells, pi_abort_word())
#define FEW_GO(NK, NV) do { if (maps == 2) { if (far) FEW_GO2(NK, NV, 2, true); else FEW_GO2(NK, NV, 2, false); } else { if (far) FEW_GO2(NK, NV, 1, true); else FEW_GO2(NK, NV, 1, false); } } while (0)
    const bool far = split_cells > 256;                                // (up to eight runs the walk is as quick)
    if (a.dim1 == 64) { if (a.vdim == 64) FEW_GO(4, 1); else FEW_GO(4, 2); } else { if (a.vdim == 64) FEW_GO(8, 1); else FEW_GO(8, 2); }
#undef FEW_GO2
#undef FEW_GO
}
