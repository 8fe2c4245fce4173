// Prompt passes of K-quant weights (Q3_K, Q4_K, Q5_K, Q6_K) on the matrix cores: a whole pass of any number of tokens in one launch (two types: whatever the caller gives a launch, 64 tokens), BIT-EXACT with the reference's x86 AVX2 arm (the contract of mmvq.hip).
//
//   out[t][row] = residual[t][row] + vec_dot(W[row], act[t])
//
// The arithmetic is mmq_mfma.hip's: per 256-block the eight integer lane sums come from v_mfma_f32_16x16x32_f16 (scale x weight as f16 against the activations as f16: exact), and each extends its own fp32
// chain by one fma per block in block order, on the VALU; Q4_K's mins have four chains of their own, Q5_K's one (a product and an addition), Q3_K and Q6_K none.  Q4_K's four chains of mins are one
// v_mfma_f32_16x16x4_4b_f16 where a wave has all of them: block c of the instruction is K-slice c.
//
// What bounds it.  A tile of 16 rows x 16 tokens and one 256-block is 48 fma that may not be merged (32 for Q3_K, Q6_K), 4 - 16 products of the scales and its share of the weights' operands (9 instructions per lane k and
// row group in Q4_K, 21 in Q6_K): VALU issue.  So a wave keeps CH chunks of 16 tokens (every operand it builds serves CH tiles) and, where the registers do not do for all eight lanes k of CH chunks, two waves share them
// out (S = 2).  The steps go on across blocks without a gap: the next MFMA, the fragments AR products ahead, a part of the next operand, then the four fma of the MFMA before; loads are a block ahead (activations) and more
// (weights), a block has one barrier, and loads take a scalar offset (buffer loads: no address arithmetic).  The kernel before walked 32 tokens in two chunks or 64 in four per launch and drained every load in flight at
// the barrier of every block.  Measured (us for 128 tokens, before / now): Q4_K 8192 x 8192 91 / 45, 57344 x 8192 424 / 320, 8192 x 28672 279 / 162; Q6_K 8192 x 28672 303 / 212, 32000 x 8192 310 / 242; Q5_K 8192 x 8192
// 88 / 56; Q3_K 80 / 48.  Of 45 us 5 are the launch; in the others the VALU issues in 75 % of the cycles.  Taking out the global loads, the barrier or the fragments' reads one at a time changes nothing of the 45 and 2 - 8 % of
// the 320.
// Q6_K's K-slices pair halves of two fragment lanes.  They are put together where the image is written: read as two halves 256 bytes apart they met in the LDS banks (41 % of the LDS' cycles, which was busy for 66 % of the launch), and
// of the weights' operands 27 instructions were needed where the upper bits come in place and one fma takes the offset along (21).  Measured together (us, before / now): 8192 x 28672 columns 181 / 166, 32000 x 8192 205 / 196,
// 8192 x 8192 at 64 tokens 37.4 / 35.4.  Its two products of a tile apart by a step (the second takes the first as its sum): 163, 194 and 36.7: not kept.
// Where one wave has all of Q4_K's lanes k (S = 1) a launch is many rounds of workgroups that read their weights from HBM: a block is 1.2 us there, no longer than such a load takes, so the loads run two blocks ahead, with a
// third set of registers for the weights and the image written a block earlier, from the same registers.  Measured (us, 57344 x 8192, one block / two blocks ahead): 128 tokens 289 / 272, 64 tokens 170 / 162; short rows
// lose (MP_FAR_BLOCKS).  The other types and S = 2 lose (registers, steps of half the length): Q3_K 276 / 294, Q5_K 333 / 336, Q6_K 32000 x 8192 192 / 197.
#include "mmvq_args.h"
#include <hip/hip_ext.h>

#include <cstdlib>
#include <cstring>
#include <type_traits>

using mp_half8 = __attribute__((ext_vector_type(8))) _Float16;
using mp_half4 = __attribute__((ext_vector_type(4))) _Float16;
using mp_half2 = __attribute__((ext_vector_type(2))) _Float16;
using mp_f32x4 = __attribute__((ext_vector_type(4))) float;
using mp_f32x16 = __attribute__((ext_vector_type(16))) float;
using mp_f32x2 = __attribute__((ext_vector_type(2))) float;
typedef uint32_t mp_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mp_u32x2 __attribute__((ext_vector_type(2)));

static __device__ __forceinline__ mp_half2 mp_h2(uint32_t u) { return __builtin_bit_cast(mp_half2, u); }
static __device__ __forceinline__ uint32_t mp_bits(mp_half2 v) { return __builtin_bit_cast(uint32_t, v); }
static __device__ __forceinline__ uint32_t mp_fma(uint32_t a, uint32_t b, uint32_t c) { return mp_bits(__builtin_elementwise_fma(mp_h2(a), mp_h2(b), mp_h2(c))); }
static __device__ __forceinline__ uint32_t mp_mul(uint32_t a, uint32_t b) { return mp_bits(mp_h2(a) * mp_h2(b)); }
static __device__ __forceinline__ uint32_t mp_add(uint32_t a, uint32_t b) { return mp_bits(mp_h2(a) + mp_h2(b)); }
// (f16 -> f32 as instructions of their own: folded into a mixed-precision product the scale would be read as f16 in every use)
static __device__ __forceinline__ mp_f32x2 mp_pair(uint32_t dd) { mp_f32x2 v = { pi_h2f((uint16_t) (dd & 0xffff)), pi_h2f((uint16_t) (dd >> 16)) }; asm volatile("" : "+v"(v)); return v; }
static __device__ __forceinline__ mp_f32x4 mp_mfma(uint4 a, uint4 b, mp_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mp_half8, a), __builtin_bit_cast(mp_half8, b), c, 0, 0, 0);
}
static __device__ __forceinline__ mp_f32x4 mp_mfma_k16(uint2 a, uint2 b, mp_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(mp_half4, a), __builtin_bit_cast(mp_half4, b), c, 0, 0, 0);
}
// four products of K = 4 at once: block c is (token, K-slice c) of a against (row, K-slice c) of b
static __device__ __forceinline__ mp_f32x16 mp_mfma_4b(uint2 a, uint2 b) {
    const mp_f32x16 z = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
    return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(mp_half4, a), __builtin_bit_cast(mp_half4, b), z, 0, 0, 0);
}
// workgroup barrier that waits for all but the last N of this wave's LDS operations (they end in order); loads of later blocks stay in flight across it
template <int N> static __device__ __forceinline__ void mp_barrier() { asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" :: "n"(N) : "memory"); }
// loads through a buffer descriptor: the lane's offset stays in one register, the block's is a scalar, so that a step of the loop adds nothing to addresses
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t mp_rsrc(const void * p, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00027000); }
static __device__ __forceinline__ mp_u32x4 mp_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off) { return __builtin_bit_cast(mp_u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0)); }
static __device__ __forceinline__ mp_u32x2 mp_load8(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off) { return __builtin_bit_cast(mp_u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0)); }
static __device__ __forceinline__ uint32_t mp_load4(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b32(r, lane_off, off, 0); }

// S waves share a row group's accumulator lanes: lane kk of wave s is lane k = s * 8 / S + kk of the reference
template <int TYPE, int KS> struct mp_w { uint32_t dd, rec, rec2, q[KS], h[TYPE == PI_Q4_K ? 1 : KS]; };       // a lane's share of one block

template <int TYPE, int S, int RG, int CH, bool NEAR>
static __device__ __forceinline__ void mmq_prompt_body(const mmvq_args & g, const int group_end, const int group0, const int tb) {
    constexpr bool Q5 = TYPE == PI_Q5_K, Q6 = TYPE == PI_Q6_K, Q3 = TYPE == PI_Q3_K, Q4 = TYPE == PI_Q4_K;
    constexpr uint32_t TILE = Q6 ? PI_MQ_TILE_Q6 : Q5 ? PI_MQ_TILE_Q5 : Q3 ? PI_MQ_TILE_Q3 : PI_MQ_TILE, QOFF = Q6 ? 1600 : (Q5 || Q3) ? 832 : 320, QPART = Q3 ? 512 : 1024;
    constexpr bool FAR = Q4 && S == 1 && !NEAR;        // loads run two blocks ahead
    constexpr int KS = 8 / S, CS = Q4 ? 4 / S : 1, NTHR = 64 * S * RG, NL = CH * 512 / NTHR, IMG = CH * 8192 + NTHR * 8;      // IMG: LDS image of one block: fragments of CH chunks, then their aux (and what the threads past it write)
    static_assert(S == 1 || S == 2, "one or two waves a row group");
    static_assert((512 % NTHR == 0) && CH * 128 <= NTHR, "whole strips of 16-byte units; eight bytes of aux a thread");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rgl = wave / S, s = wave % S, r = lane & 15, gq = lane >> 4;
    const int raw = group0 + rgl;
    const bool active = raw < group_end;
    const int rg = active ? raw : group_end - 1;
    const int si = (rg >= g.seg[1].wave0) + (rg >= g.seg[2].wave0);
    const mmvq_seg & sg = g.seg[si];
    const int64_t row0 = (int64_t) (rg - sg.wave0) * 16;
    const int nb = g.nb, nt = g.nt, nch = (nt + 15) >> 4, ch0 = tb * CH;
    uint32_t magic = 0x64006400u;
    asm volatile("" : "+v"(magic));
    const __amdgpu_buffer_rsrc_t wr = mp_rsrc(sg.mq + (size_t) (rg - sg.wave0) * nb * TILE, (uint32_t) nb * TILE);
    const uint32_t dd_off = 4 * r, rec_off = 64 + (Q6 ? 8 : 4) * lane, q_off = QOFF + 16 * (Q3 ? 2 * r + (gq >> 1) : lane) + (S == 2 ? QPART * s : 0), h_off = (Q6 ? 576 + 64 * r + 32 * (gq >> 1) : 320 + 32 * r) + (S == 2 ? 16 * s : 0);
    auto load_w = [&](int b, mp_w<TYPE, KS> & W) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t) (b < nb ? b : nb - 1) * TILE;                  // (clamped, not skipped: no branch between a load and its use)
        W.dd = mp_load4(wr, dd_off, at);
        if constexpr (Q6) { const mp_u32x2 v = mp_load8(wr, rec_off, at); W.rec = v[0]; W.rec2 = v[1]; } else W.rec = mp_load4(wr, rec_off, at);
#pragma unroll
        for (int p = 0; p < 2 / S; p++) {
            const mp_u32x4 v = mp_load16(wr, q_off + QPART * p, at);
#pragma unroll
            for (int i = 0; i < 4; i++) W.q[4 * p + i] = v[i];
            if constexpr (!Q4) {
                const mp_u32x4 u = mp_load16(wr, h_off + 16 * p, at);
#pragma unroll
                for (int i = 0; i < 4; i++) W.h[4 * p + i] = u[i];
            }
        }
    };
    // activations: block b's image, global -> registers -> LDS.  Chunks past the pass's last one repeat it and are not stored
    mp_u32x4 st[NL];
    mp_u32x2 sa;
    const int chunks = nch - ch0 < CH ? nch - ch0 : CH;
    const __amdgpu_buffer_rsrc_t fr_r = mp_rsrc(g.frag + (size_t) ch0 * nb * 8192, (uint32_t) chunks * nb * 8192), ax_r = mp_rsrc(g.aux + (size_t) ch0 * nb * 1024, (uint32_t) chunks * nb * 1024);
    const uint32_t a_off = ((tid >> 7) < chunks ? tid >> 7 : chunks - 1) * (nb * 1024) + (tid & 127) * 8;
    auto stage_load = [&](int b, mp_u32x4 * st, mp_u32x2 & sa) __attribute__((always_inline)) {
        const int bb = b < nb ? b : nb - 1;
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int ch = i * NTHR / 512, c = ch < chunks ? ch : chunks - 1;
            st[i] = mp_load16(fr_r, (tid & 511) * 16, (uint32_t) (c * nb + bb) * 8192 + i * NTHR % 512 * 16);
        }
        sa = mp_load8(ax_r, a_off, bb * 1024);
    };
    const uint32_t q6_at = (tid >> 6) * 1024 + (r + 32 * (gq >> 1)) * 16 + 8 * (gq & 1);
    auto stage_store = [&](uint8_t * img, const mp_u32x4 * st, mp_u32x2 sa) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            if constexpr (Q6) {                        // K-slice (n, hh) pairs 32-groups hh and hh + 2 of half n: the halves of two fragment lanes change places, and read_a reads 16 bytes like the others
                uint8_t * at = img + i * NTHR * 16 + q6_at;
                *(mp_u32x2 *) at = mp_u32x2{ st[i][0], st[i][1] };
                *(mp_u32x2 *) (at + 256) = mp_u32x2{ st[i][2], st[i][3] };
            } else *(mp_u32x4 *) (img + (i * NTHR + tid) * 16) = st[i];
        }
        *(mp_u32x2 *) (img + CH * 8192 + tid * 8) = sa;
    };
    float acc[CH][KS][4], accm[CH][CS][4];
#pragma unroll
    for (int ch = 0; ch < CH; ch++) {
#pragma unroll
        for (int kk = 0; kk < KS; kk++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[ch][kk][i] = 0.0f;
#pragma unroll
        for (int cc = 0; cc < CS; cc++)
#pragma unroll
            for (int i = 0; i < 4; i++) accm[ch][cc][i] = 0.0f;
    }
    // ---- a block is PS products (accumulator lanes, then mins) times CH chunks.  A step issues the next MFMA, reads from LDS what a later one needs, builds a part of the next product's weight operand and runs the four fma
    //      of the MFMA before: the steps go on across blocks, so that neither the matrix cores nor the VALU wait for the other's latency. ----
    constexpr bool MINS = Q4 || Q5;
    constexpr int PC = Q4 && S == 2 ? 2 : MINS ? 1 : 0, PS = KS + PC;      // products of the mins: Q4_K's four chains are one (S = 1) or two (S = 2, two chains a wave); Q5_K one
    constexpr int NM = KS * CH, AR = CH == 4 ? 4 : NM / 2 < 8 ? NM / 2 : 8;            // fragments are read AR products ahead; never from the next image before the barrier
    static_assert(NM % AR == 0, "a block starts with the first slot");
    uint4 af[AR], bw[2], bw2[Q6 ? 2 : 1];              // operands: af[fragment % AR], bw[product & 1]
    uint2 am[CH], bm[CS];
    float4 dy[CH];
    float d[CH][4], nd[CH][4];
    uint32_t sc[4];                                    // the block's scales as pairs of f16: Q4_K / Q5_K S1, S2, C1, C2; Q6_K SLa, SHa, SLb, SHb; Q3_K SA, SB
    uint32_t c6[2];                                    // Q6_K: -1536 times the second sub-block's scales
    const uint32_t q6_sh = 4 + 2 * (gq & 1);
    float dx, dminx;
    auto read_a = [&](int m, uint32_t img) __attribute__((always_inline)) {              // fragment m = kk * CH + chunk of an image
        const uint8_t * fr = lds + img + m % CH * 8192 + (s * KS + m / CH) * 1024;
        af[m % AR] = *(const uint4 *) (fr + lane * 16);
    };
    auto read_aux = [&](int ch, uint32_t img) __attribute__((always_inline)) {
        const uint8_t * aux = lds + img + CH * 8192 + ch * 1024;
        if constexpr (MINS) am[ch] = *(const uint2 *) (aux + 64 + lane * 8);
        dy[ch] = *(const float4 *) (aux + 16 * gq);
    };
    auto scales = [&](const mp_w<TYPE, KS> & W, int half) __attribute__((always_inline)) {      // half: lanes k >= 4 use the second scale of a 32-group (Q3_K, Q6_K)
        if constexpr (MINS) {
            sc[0] = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, 0x04000400u), 0xE400E400u);
            sc[1] = mp_fma(__builtin_amdgcn_perm(0x64646464u, W.rec, 0x04010401u), 0x2C002C00u, 0xD400D400u);
            sc[2] = mp_mul(sc[0], 0xE400E400u); sc[3] = mp_mul(sc[1], 0xE400E400u);
        } else {
            const uint32_t selA = 0x04000400u + (uint32_t) half * 0x00010001u, selB = selA + 0x00020002u;
            if constexpr (Q6) {
                sc[0] = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, selA), 0xE400E400u); sc[1] = mp_fma(__builtin_amdgcn_perm(0x64646464u, W.rec2, selA), 0x4C004C00u, 0xF408F408u);
                sc[2] = mp_fma(__builtin_amdgcn_perm(0x64646464u, W.rec, selB), 0x2C002C00u, 0xD400D400u); sc[3] = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec2, selB), 0xE408E408u);
                c6[0] = mp_mul(sc[2], 0xE600E600u); c6[1] = mp_mul(sc[3], 0xE600E600u);
            } else {
                sc[0] = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, selA), 0xE420E420u); sc[1] = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, selB), 0xE420E420u);
            }
        }
    };
    // dword i of lane kk's operand: weights (i0, i2), (i1, i3) of the first sub-block of the K-slice, then of the second
    auto build = [&](const mp_w<TYPE, KS> & W, int kk, int i) __attribute__((always_inline)) {
        const int sh = 8 * (i & 1), hi = i >> 1;
        const uint32_t q = W.q[kk] >> sh;
        uint32_t o, o2 = 0;
        if constexpr (MINS) {
            uint32_t f = 0;
            if constexpr (Q5) { const uint32_t u = W.h[kk] >> (2 * gq + sh); f = hi ? (u & 0x00020002u) << 7 : (u & 0x00010001u) << 4; }
            o = mp_fma((q & (hi ? 0x00F000F0u : 0x000F000Fu)) | magic | f, sc[hi], sc[2 + hi]);
        } else if constexpr (Q6) {
            const uint32_t h = sh ? W.h[kk] >> q6_sh : W.h[kk] << (8 - q6_sh);         // (the two upper bits where they belong)
            if (hi) {                                  // 16 times the weight plus 1536: one fma a part
                const uint32_t w = (q & 0x00F000F0u) | magic | (h & 0x03000300u);
                o = mp_fma(w, sc[3], c6[1]); o2 = mp_fma(w, sc[2], c6[0]);
            } else {                                   // (1056 times the larger part would pass 65504)
                const uint32_t w = mp_add((q & 0x000F000Fu) | magic | (h & 0x00300030u), 0xE420E420u);
                o = mp_mul(w, sc[1]); o2 = mp_mul(w, sc[0]);
            }
        } else {
            const uint32_t lo2 = W.q[kk] >> (4 * (gq & 1)), hm = W.h[kk] >> (2 * gq);      // (shared by the four dwords)
            const uint32_t u = hi ? ((lo2 >> 2) & 0x03030303u) | ((hm & 0x02020202u) << 1) : (lo2 & 0x03030303u) | ((hm & 0x01010101u) << 2);
            o = mp_mul(mp_add(((u >> sh) & 0x00FF00FFu) | magic, 0xE404E404u), sc[hi]);
        }
        uint4 & x = bw[kk & 1];
        if (i == 0) x.x = o; else if (i == 1) x.y = o; else if (i == 2) x.z = o; else x.w = o;
        if constexpr (Q6) { uint4 & y = bw2[kk & 1]; if (i == 0) y.x = o2; else if (i == 1) y.y = o2; else if (i == 2) y.z = o2; else y.w = o2; }
    };
    struct result { mp_f32x4 v; mp_f32x16 m; };        // (m: all four chains of mins, S = 1)
    auto product = [&](int p, int ch) __attribute__((always_inline)) -> result {        // (constants after unrolling)
        const mp_f32x4 z = { 0.0f, 0.0f, 0.0f, 0.0f };
        result c;
        if (p >= KS) {
            if constexpr (Q4 && S == 1) c.m = mp_mfma_4b(am[ch], bm[0]);
            else if constexpr (MINS) c.v = mp_mfma_k16(am[ch], bm[p >= KS ? p - KS : 0], z);
            return c;
        }
        const uint4 a = af[(p * CH + ch) % AR];
        if constexpr (Q6) c.v = mp_mfma(a, bw2[p & 1], mp_mfma(a, bw[p & 1], z));
        else c.v = mp_mfma(a, bw[p & 1], z);
        return c;
    };
    mp_w<TYPE, KS> W0, W1, W2;
    result c;
    // block b: image `img`, weights W; the next block's: img1, Wn.  Its one barrier is in its middle: image img1, written ahead of it, may then be read.
    // Three images: waves on either side of a barrier read images b - 1 and b, and write b + 1 (b - 2's readers left it before the barrier of b - 1).
    // Two blocks ahead, block b writes image b + 2 at its end: the readers of b - 1, which was there, left it before the barrier of b
    uint32_t img = 0, img1 = IMG, img2 = 2 * IMG;
    auto block = [&](int b, mp_w<TYPE, KS> & W, mp_w<TYPE, KS> & Wn) __attribute__((always_inline)) {
        if constexpr (!FAR) { stage_store(lds + img1, st, sa); stage_load(b + 2, st, sa); }
#pragma unroll
        for (int n = 0; n < PS * CH; n++) {
            const int p = n / CH, ch = n % CH;
            if (p == 0) {
                const float y[4] = { dy[ch].x, dy[ch].y, dy[ch].z, dy[ch].w };
#pragma unroll
                for (int i = 0; i < 4; i++) { d[ch][i] = y[i] * dx; if constexpr (MINS) nd[ch][i] = -y[i] * dminx; }
            }
            if (n == NM - AR) mp_barrier<4>();                                      // (at least four reads were issued behind the image's writes)
            // the parts of the next product's operand that belong to this step
            if (S == 1 && !MINS && p == 3 && ch == 0) scales(W, 1);
            if (p + 1 == PS && ch == 0) { scales(Wn, s * KS >> 2); const mp_f32x2 dp = mp_pair(Wn.dd); dx = dp.x; dminx = dp.y; }
            if (MINS && p == KS - 1 && ch == 0) {
                const uint32_t M0 = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, 0x04020402u), 0xE400E400u), M1 = mp_add(__builtin_amdgcn_perm(0x64646464u, W.rec, 0x04030403u), 0xE400E400u);
                if constexpr (Q5 || S == 1) bm[0] = make_uint2(M0, M1);
                else
#pragma unroll
                    for (int cc = 0; cc < CS; cc++) { const bool o = gq == s * CS + cc; bm[cc] = make_uint2(o ? M0 : 0u, o ? M1 : 0u); }      // chain c: K-slice c's mins
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i * CH / 4 == ch) {
                    if (p + 1 < KS) build(W, p + 1 < KS ? p + 1 : 0, i);
                    else if (p + 1 == PS) build(Wn, 0, i);
                }
            if (n == (PS - 1) * CH) {                                                   // (W's last use is behind us)
                if constexpr (FAR) { stage_store(lds + img2, st, sa); stage_load(b + 3, st, sa); }
                load_w(b + (FAR ? 3 : 2), W);
            }
            const result o = c;
            const mp_f32x4 v = o.v;
            c = n + 1 < PS * CH ? product((n + 1) / CH, (n + 1) % CH) : product(0, 0);
            if (n < NM) { if (n + AR < NM) read_a(n + AR, img); else read_a(n + AR - NM, img1); }      // (the MFMA of this step's product has read its fragment)
            if (p == PS - 1) read_aux(ch, img1);
            __builtin_amdgcn_sched_barrier(0);
            if (p < KS) {
#pragma unroll
                for (int i = 0; i < 4; i++) acc[ch][p < KS ? p : 0][i] = fmaf(d[ch][i], v[i], acc[ch][p < KS ? p : 0][i]);
            } else if constexpr (Q4 && S == 1) {
#pragma unroll
                for (int cc = 0; cc < 4; cc++)
#pragma unroll
                    for (int i = 0; i < 4; i++) accm[ch][cc][i] = fmaf(nd[ch][i], o.m[4 * cc + i], accm[ch][cc][i]);
            } else if constexpr (Q4) {
#pragma unroll
                for (int i = 0; i < 4; i++) accm[ch][p >= KS ? p - KS : 0][i] = fmaf(nd[ch][i], v[i], accm[ch][p >= KS ? p - KS : 0][i]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) { const float prod = nd[ch][i] * v[i]; accm[ch][0][i] = accm[ch][0][i] + prod; }       // (S = 2: wave 1's copy of Q5_K's one chain is not read)
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const uint32_t t = img; img = img1; img1 = img2; img2 = t;
    };
    if constexpr (FAR) {
        mp_u32x4 st0[NL], st1[NL];
        mp_u32x2 sa0, sa1;
        stage_load(0, st0, sa0);
        load_w(0, W0);
        stage_load(1, st1, sa1);
        load_w(1, W1);
        stage_load(2, st, sa);
        load_w(2, W2);
        stage_store(lds, st0, sa0);
        stage_store(lds + IMG, st1, sa1);
    } else {
        stage_load(0, st, sa);
        load_w(0, W0);
        stage_store(lds, st, sa);
        stage_load(1, st, sa);
        load_w(1, W1);
    }
    mp_barrier<0>();
#pragma unroll
    for (int m = 0; m < AR; m++) read_a(m, 0);
#pragma unroll
    for (int ch = 0; ch < CH; ch++) read_aux(ch, 0);
    scales(W0, s * KS >> 2);
    { const mp_f32x2 dp = mp_pair(W0.dd); dx = dp.x; dminx = dp.y; }
#pragma unroll
    for (int i = 0; i < 4; i++) build(W0, 0, i);
    c = product(0, 0);
    int b = 0;
    if constexpr (FAR) {
        __builtin_amdgcn_s_waitcnt(0x0f70);            // vmcnt(0): the loop's waits count the loads of its own order alone
        for (; b + 2 < nb; b += 3) { block(b, W0, W1); block(b + 1, W1, W2); block(b + 2, W2, W0); }
        if (b < nb) { block(b, W0, W1); if (b + 1 < nb) block(b + 1, W1, W2); }
    } else {
        for (; b + 1 < nb; b += 2) { block(b, W0, W1); block(b + 1, W1, W0); }
        if (b < nb) block(b, W0, W1);
    }
    // ---- fold: hsum_float_8 = ((a0 + a4) + (a2 + a6)) + ((a1 + a5) + (a3 + a7)), mins ((m0 + m2) + (m1 + m3)) ----
    constexpr int XN = KS + CS;                                                        // S = 2: a wave's chains of the chunks that the other one finishes (ch % 2 == its s), [chunk / 2][i][XN][64]
    float * X = (float *) lds + (size_t) wave * ((CH + 1) / 2 * 4 * XN * 64);
    if constexpr (S == 2) {
        __syncthreads();
#pragma unroll
        for (int ch = 0; ch < CH; ch++)
            if ((ch & 1) != s)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float * x = X + ((ch >> 1) * 4 + i) * XN * 64 + lane;
#pragma unroll
                    for (int kk = 0; kk < KS; kk++) x[kk * 64] = acc[ch][kk][i];
#pragma unroll
                    for (int cc = 0; cc < CS; cc++) x[(KS + cc) * 64] = accm[ch][cc][i];
                }
        __syncthreads();
    }
    if (!active) return;
    const float * Y = (const float *) lds + (size_t) (wave ^ 1) * ((CH + 1) / 2 * 4 * XN * 64);
    const int el = (int) __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), er = el & 15;      // (the lane, asked for again: its registers are the loop's)
    const int64_t row = row0 + er;
    const bool mine = row < sg.M;
#pragma unroll
    for (int ch = 0; ch < CH; ch++) {
        if (S == 2 && (ch & 1) != s) continue;
        const int t0 = (ch0 + ch) * 16 + 4 * (el >> 4);
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float a[8], m[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
            if constexpr (S == 2) {
                const float * y = Y + ((ch >> 1) * 4 + i) * XN * 64 + el;
#pragma unroll
                for (int kk = 0; kk < KS; kk++) { const float o = y[kk * 64]; a[kk] = s == 0 ? acc[ch][kk][i] : o; a[KS + kk] = s == 0 ? o : acc[ch][kk][i]; }
                if constexpr (Q4) for (int cc = 0; cc < CS; cc++) { const float o = y[(KS + cc) * 64]; m[cc] = s == 0 ? accm[ch][cc][i] : o; m[CS + cc] = s == 0 ? o : accm[ch][cc][i]; }
                if constexpr (Q5) m[0] = s == 0 ? accm[ch][0][i] : y[KS * 64];
            } else {
#pragma unroll
                for (int kk = 0; kk < 8; kk++) a[kk] = acc[ch][kk][i];
#pragma unroll
                for (int cc = 0; cc < CS; cc++) m[cc] = accm[ch][cc][i];
            }
            v[i] = ((a[0] + a[4]) + (a[2] + a[6])) + ((a[1] + a[5]) + (a[3] + a[7]));
            if constexpr (Q4) v[i] = v[i] + ((m[0] + m[2]) + (m[1] + m[3]));
            if constexpr (Q5) v[i] = v[i] + m[0];
        }
        if (sg.store == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (mine && t0 + i < nt) { const int64_t o = (int64_t) (t0 + i) * sg.M + row; sg.out[o] = sg.res ? sg.res[o] + v[i] : v[i]; }
        } else if (sg.store == 3) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (mine && t0 + i < nt) sg.dst16[(int64_t) pi_cell_of(g.dyn, g.kv_head, g.tok0 + t0 + i) * sg.stride16 + row] = pi_f2h(v[i]);
        } else {
            // RoPE of rows 2j, 2j + 1 of a head, on neighbouring lanes (M is even); the rounding points of k_rope_kv
            const int j = (int) (row % g.hd) >> 1;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float mate = pi_partner<1>(v[i]);
                if (mine && t0 + i < nt) {
                    const int tok = g.tok0 + t0 + i;
                    const float2 cs = *(const float2 *) (g.rope_cs + ((int64_t) g.pos[tok] * (g.hd / 2) + j) * 2);
                    const float y = (er & 1) ? mate * cs.y + v[i] * cs.x : v[i] * cs.x - mate * cs.y;
                    sg.dst16[(int64_t) (sg.store == 2 ? pi_cell_of(g.dyn, g.kv_head, tok) : tok) * sg.stride16 + row] = pi_f2h(y);
                }
            }
        }
    }
}

// workgroup n runs on XCD n % 8: the token blocks of a row block go to one XCD one behind the other, so that its weights come from HBM once.
// SB, RGB: waves per row group and row groups of the second type's workgroups.  They are few and come last, so the launch ends with one of them: where the first type keeps one wave to a row group the second takes two
// (a Q6_K tile costs a wave 1.6 times a Q4_K one; 8192 + 1024 rows of Q4_K with 1024 of Q6_K, 8192 columns, 64 tokens: 57.6 us with one wave to all row groups, now 41.4; Q5_K 50 and 41.1)
template <int TA, int TB, int S, int RG, int CH, int SB = S, int RGB = RG, bool NEAR = false>
__global__ void __launch_bounds__(64 * S * RG) k_mmq_prompt(const mmvq_args g, const int groups_a, const int groups_all, const int blocks_a, const int row_blocks, const int tok_blocks) {
    static_assert(S * RG == SB * RGB, "workgroups of one size");
    if (pi_aborted(g.abort_w, 1)) return;
    const int slot = blockIdx.x >> 3, rb = (blockIdx.x & 7) + 8 * (slot / tok_blocks), tb = slot % tok_blocks;
    if (rb >= row_blocks) return;
    if constexpr (TA != TB) {
        if (rb >= blocks_a) { mmq_prompt_body<TB, SB, RGB, CH, NEAR>(g, groups_all, groups_a + (rb - blocks_a) * RGB, tb); return; }
    }
    mmq_prompt_body<TA, S, RG, CH, NEAR>(g, groups_a, rb * RG, tb);
}

template <int TA, int TB, int S, int RG, int CH, int SB = S, int RGB = RG, bool NEAR = false>
static int prompt_go(const mmvq_args & g, int groups_a, int groups_all, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    constexpr size_t image = 3 * ((size_t) CH * 8192 + 64 * S * RG * 8), fold = S == 2 || SB == 2 ? (size_t) S * RG * ((CH + 1) / 2) * 4 * 6 * 256 : 0, lds = image > fold ? image : fold;
    const auto kernel = k_mmq_prompt<TA, TB, S, RG, CH, SB, RGB, NEAR>;
    if (!g.frag) { PI_CHECK_HIP(hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); return 0; }       // pi_op_mul_mat_reserve
    const int blocks_a = (groups_a + RG - 1) / RG, row_blocks = blocks_a + (groups_all - groups_a + RGB - 1) / RGB, tok_blocks = (g.nt + CH * 16 - 1) / (CH * 16);
    const unsigned grid = (unsigned) ((row_blocks + 7) / 8 * 8) * (unsigned) tok_blocks;
    if (ea) hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(64 * S * RG), lds, stream, ea, eb, 0, g, groups_a, groups_all, blocks_a, row_blocks, tok_blocks);
    else    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * S * RG), lds, stream, g, groups_a, groups_all, blocks_a, row_blocks, tok_blocks);
    PI_CHECK_LAUNCH();
    return 0;
}
// Loads two blocks ahead from rows of eight blocks on: a row asks for three blocks behind its end instead of two, and three have to be there before its first product.  us one block / two blocks ahead, weights
// from memory: 28672 rows x 64 tokens K 512 13.6 / 14.0, 768 15.8 / 17.1, 1536 24.1 / 24.3, 2048 29.3 / 28.6, 4096 50.0 / 48.6, 8192 88.4 / 83.1; x 128 tokens 768 27.3 / 29.6, 1536 41.8 / 42.3, 2048 51.6 / 50.0, 8192 161 / 152; 57344 x 300
// 768 105 / 114, 2048 198 / 200, 8192 679 / 673
#define MP_FAR_BLOCKS 8
template <int TA, int TB, bool NEAR>
static int prompt_182(const mmvq_args & g, int groups_a, int groups_all, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    if constexpr (TA != TB) return prompt_go<TA, TB, 1, 8, 2, 2, 4, NEAR>(g, groups_a, groups_all, stream, ea, eb); else return prompt_go<TA, TB, 1, 8, 2, 1, 8, NEAR>(g, groups_a, groups_all, stream, ea, eb);
}
template <int TA, int TB>
static int prompt_cfg(int cfg, const mmvq_args & g, int groups_a, int groups_all, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    switch (cfg) {                                             // S, RG, CH
        case 242: return prompt_go<TA, TB, 2, 4, 2>(g, groups_a, groups_all, stream, ea, eb);
        case 243: return prompt_go<TA, TB, 2, 4, 3>(g, groups_a, groups_all, stream, ea, eb);
        case 244: return prompt_go<TA, TB, 2, 4, 4>(g, groups_a, groups_all, stream, ea, eb);
        case 222: return prompt_go<TA, TB, 2, 2, 2>(g, groups_a, groups_all, stream, ea, eb);
        case 182:
            if constexpr (TA == PI_Q4_K) if (g.nb < MP_FAR_BLOCKS) { const int rc = prompt_182<TA, TB, true>(g, groups_a, groups_all, stream, ea, eb); if (g.frag || rc != 0) return rc; }      // (reserving: both)
            return prompt_182<TA, TB, false>(g, groups_a, groups_all, stream, ea, eb);
    }
    pi_set_error("mmq_prompt: configuration %d", cfg);
    return -1;
}
static const int prompt_cfgs[] = { 242, 243, 244, 222, 182 };
static int prompt_types(int type_a, int type_b, int cfg, const mmvq_args & g, int groups_a, int groups_all, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    if (type_a == PI_Q4_K && type_b == PI_Q5_K) return prompt_cfg<PI_Q4_K, PI_Q5_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
    if (type_a == PI_Q4_K && type_b == PI_Q6_K) return prompt_cfg<PI_Q4_K, PI_Q6_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
    if (type_a == PI_Q3_K) return prompt_cfg<PI_Q3_K, PI_Q3_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
    if (type_a == PI_Q4_K) return prompt_cfg<PI_Q4_K, PI_Q4_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
    if (type_a == PI_Q5_K) return prompt_cfg<PI_Q5_K, PI_Q5_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
    return prompt_cfg<PI_Q6_K, PI_Q6_K>(cfg, g, groups_a, groups_all, stream, ea, eb);
}
// once per process and outside any stream capture (pi_op_mul_mat_reserve): the instances' dynamic LDS is more than a kernel gets by default
int pi_mmq_prompt_reserve() {
    mmvq_args g; memset(&g, 0, sizeof g);                      // g.frag == nullptr: the instances only set their attribute
    const int types[][2] = { { PI_Q3_K, PI_Q3_K }, { PI_Q4_K, PI_Q4_K }, { PI_Q5_K, PI_Q5_K }, { PI_Q6_K, PI_Q6_K }, { PI_Q4_K, PI_Q5_K }, { PI_Q4_K, PI_Q6_K } };
    for (const auto & t : types) for (int cfg : prompt_cfgs) if (prompt_types(t[0], t[1], cfg, g, 0, 0, nullptr, nullptr, nullptr) != 0) return -1;
    return 0;
}
// from 17 tokens (two chunks); up to 32 only where the launch has row groups enough.  Measured, us per launch of up to 32 tokens, k_mmq_kq's two chunks / here: Q4_K 1024 x 8192 24.3 / 25.7, 3072 x 8192 25.3 / 26.4,
// 4096 x 4096 15.2 / 15.7, 8192 x 8192 30.7 / 28.6, 57344 x 8192 109.7 / 94.5; Q6_K 2048 x 5632 20.5 / 21.1, 4096 x 11008 42.4 / 38.1, 8192 x 8192 39.3 / 32.0; from 33 tokens everything is faster here (48 tokens: Q4_K
// 2048 x 2048 15.1 / 10.2, 1024 x 8192 41.6 / 26.1, 57344 x 8192 191 / 180; Q6_K 1024 x 8192 42.3 / 28.5)
bool pi_mmq_prompt_wants(int type, int n_tok, int64_t rows) {
    if (!pi_mmq_supported(type) || n_tok < pi_mmq_min_nt()) return false;            // (below that the quantisers write no operand planes)
    if (n_tok > 32) return true;
    return n_tok > 16 && (rows + 15) / 16 * 256 / pi_cu_count() >= (type == PI_Q6_K ? 256 : 384);
}
// Which tiles: the shortest estimate of  rounds of workgroups x time of a round.  A round's time (us for 32 blocks, launch taken off; 8192 columns, measured per type on a full round) is about the same for all sizes:
// what differs is how many tiles a wave's operand serves (4 chunks: least work per tile) against how well the launch fills its rounds.  [Q3_K, Q4_K, Q5_K, Q6_K]; two of the four-wave workgroups fit a CU.
// Two types: the second one's workgroups come last, and what a round of them takes longer is added at the end
static int prompt_choose(int type_a, int type_b, int groups_a, int groups_b, int chunks) {
    struct tiles { int cfg, rg, ch, per_cu; float one, full; };
    static const tiles cfgs[4][5] = {
        { { 222, 2, 2, 2, 24.0f, 36.0f }, { 242, 4, 2, 1, 28.0f, 28.0f }, { 243, 4, 3, 1, 35.0f, 35.0f }, { 244, 4, 4, 1, 43.5f, 43.5f }, { 182, 8, 2, 1, 48.7f, 48.7f } },
        { { 222, 2, 2, 2, 22.5f, 35.0f }, { 242, 4, 2, 1, 26.0f, 26.0f }, { 243, 4, 3, 1, 35.5f, 35.5f }, { 244, 4, 4, 1, 43.0f, 43.0f }, { 182, 8, 2, 1, 39.8f, 39.8f } },
        { { 222, 2, 2, 2, 26.0f, 39.0f }, { 242, 4, 2, 1, 33.0f, 33.0f }, { 243, 4, 3, 1, 40.0f, 40.0f }, { 244, 4, 4, 1, 51.0f, 51.0f }, { 182, 8, 2, 1, 51.0f, 51.0f } },
        { { 222, 2, 2, 2, 27.0f, 42.0f }, { 242, 4, 2, 1, 37.0f, 37.0f }, { 243, 4, 3, 1, 46.0f, 46.0f }, { 244, 4, 4, 1, 56.7f, 56.7f }, { 182, 8, 2, 1, 64.5f, 64.5f } },
    };
    auto of = [](int type) { return cfgs[type == PI_Q3_K ? 0 : type == PI_Q4_K ? 1 : type == PI_Q5_K ? 2 : 3]; };
    int best = 244; float best_t = 1e30f;
    for (int i = 0; i < 5; i++) {
        const tiles & c = of(type_a)[i], & d = of(type_b)[groups_b > 0 && c.cfg == 182 ? 1 : i];          // (182: the second type's are 242, see the kernel)
        const int64_t wgs = (int64_t) ((groups_a + c.rg - 1) / c.rg + (groups_b + d.rg - 1) / d.rg) * ((chunks + c.ch - 1) / c.ch), slots = (int64_t) pi_cu_count() * c.per_cu, whole = wgs / slots, rest = wgs % slots;
        // (up to three rounds the last one counts in full; behind more, workgroups of many rounds run past each other and about half a round is lost)
        float t = whole >= 3 ? c.full * ((float) wgs / slots + 0.5f) : c.full * whole + (rest == 0 ? 0.0f : rest <= pi_cu_count() ? c.one : c.full);
        if (groups_b > 0 && d.full > c.full) t += d.full - c.full;
        if (t < best_t) { best_t = t; best = c.cfg; }
    }
    return best;
}
// the whole pass in one launch: segments [0, n_a) of type_a, the others of type_b (Q4_K followed by Q5_K or Q6_K; n_a == nseg: one type); g.frag / g.aux / g.nt set
int pi_mmq_prompt_launch(int type_a, int type_b, int n_a, mmvq_launch & L, hipStream_t stream, hipEvent_t ea, hipEvent_t eb) {
    if (pi_op_mul_mat_reserve() != 0) return -1;
    mmvq_args & g = L.g;
    int groups = 0, groups_a = 0;
    for (int i = 0; i < MMVQ_MAX_SEG; i++) {
        if (i < L.nseg) { g.seg[i].wave0 = groups; groups += (g.seg[i].M + 15) / 16; if (i < n_a) groups_a = groups; }
        else { g.seg[i] = g.seg[0]; g.seg[i].wave0 = 0x7fffffff; }
    }
    if (n_a >= L.nseg) type_b = type_a;
    return prompt_types(type_a, type_b, prompt_choose(type_a, type_b, groups_a, groups - groups_a, (g.nt + 15) / 16), g, groups_a, groups, stream, ea, eb);
}
