// Operators of blocks whose norm comes AFTER the sum (x <- R(alpha x + ls * sublayer(x)) * w) and of recurrent mixers whose state decays per key channel:
//
//   k_embed_pair         token row * scale + a row of a second table (a hashed pair embedding: the host names the row of every token)
//   k_rms_post           the end of a sublayer in one launch: [the mean of two RMS-normed branch outputs ->] layer scale -> + alpha x -> RMS norm [-> a second RMS norm for what reads x next]
//   k_token_shift(_walk) m_s = h + (h_prev - h) * mu_s for several s at once; h_prev of a sequence's first token of the pass comes from (and its last token goes to) the sequence's state
//   k_channel_recurrence per head a [dim][vdim] state, per token and key channel a decay.  Two rules:
//                          delta   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q        (the read-out sees the token's own write)
//                          bonus   o = (S + diag(b) k v^T)^T q;  S <- diag(g) S + k v^T                         (the read-out sees the token through the bonus only)
//                        decays arrive raw and are formed here (exp(-exp(raw + bias)) or exp(-exp(A_h) softplus(raw + bias))), q / k can be made unit vectors here, beta is sigmoid(raw)
//   k_head_norm_gate     every head's output divided by its root mean square, * weight (shared by the heads or one per head), * gate (as is, sigmoid or silu of it)
//
// Everything is fp32 in both precisions of the engine.
#include "ops_common.h"
#include "kernel_timing.h"

#include <algorithm>
#include <cmath>

#define CM_FRESH (1 << 30)

typedef uint16_t cm_u16x8 __attribute__((ext_vector_type(8)));
static __device__ __forceinline__ float cm_widen(uint16_t b) { return __uint_as_float((uint32_t) b << 16); }
static __device__ __forceinline__ float cm_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }
static __device__ __forceinline__ float cm_softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }        // (beyond 20 the two agree to the last bit of fp32)
static __device__ __forceinline__ float cm_block_sum(float v, float * red) {          // sum over the block's threads (every thread gets it); red: 4 floats, reusable after the call
    v = pi_lanes_sum<64>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.0f;
    for (int i = 0; i < (int) (blockDim.x >> 6); i++) s += red[i];
    return s;
}

// ---- embedding: token row * scale + a row of a second table ---------------------------------------------------------------------------------------------
// grid (token, 2048 values): eight values of a thread in one 16-byte load of each table (vec: rows and output start 16-byte aligned).  A thread that walked the row in 2-byte loads made a trip to memory at every one of
// them: 18 us for 8 tokens of width 4096, now 4.3
__global__ void __launch_bounds__(256) k_embed_pair(const uint16_t * __restrict__ table, int64_t width, int64_t n_rows, const int32_t * __restrict__ tokens, float scale, const uint16_t * __restrict__ table2, int64_t n_rows2,
                             const int32_t * __restrict__ rows2, int vec, float * __restrict__ out, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int t = blockIdx.x;
    const int64_t row = tokens[t], row2 = rows2[t], i0 = (int64_t) blockIdx.y * 2048;
    if (pi_abort_late(gone, abort_w)) return;
    const bool ok = row >= 0 && row < n_rows, ok2 = row2 >= 0 && row2 < n_rows2;
    if (vec) {
        const int64_t i = i0 + 8 * threadIdx.x;
        if (i >= width) return;
        const cm_u16x8 a = *(const cm_u16x8 *) (table + (ok ? row : 0) * width + i), b = *(const cm_u16x8 *) (table2 + (ok2 ? row2 : 0) * width + i);
        float4 o[2];
#pragma unroll
        for (int c = 0; c < 8; c++) ((float *) o)[c] = (ok ? cm_widen(a[c]) * scale : 0.0f) + (ok2 ? cm_widen(b[c]) : 0.0f);
        float4 * dst = (float4 *) (out + (int64_t) t * width + i);
        dst[0] = o[0]; dst[1] = o[1];
        if (rd.h) *(uint4 *) (rd.h + t * rd.stride + i) = make_uint4(pi_round_pair(o[0].x, o[0].y), pi_round_pair(o[0].z, o[0].w), pi_round_pair(o[1].x, o[1].y), pi_round_pair(o[1].z, o[1].w));
        return;
    }
    for (int64_t i = i0 + threadIdx.x; i < min(width, i0 + 2048); i += 256)
        out[(int64_t) t * width + i] = (ok ? cm_widen(table[row * width + i]) * scale : 0.0f) + (ok2 ? cm_widen(table2[row2 * width + i]) : 0.0f);
}
extern "C" int pi_op_embed_pair(const pi_weight * w, const int32_t * tokens, int n_tok, float scale, const pi_weight * w2, const int32_t * rows2, float * out, void * stream) {
    if (!w || w->type != PI_BF16 || !w2 || w2->type != PI_BF16 || w->ne0 != w2->ne0) { pi_set_error("pi_op_embed_pair: two bfloat16 tables of the same width are required"); return -1; }
    if (n_tok <= 0) return 0;
    const int vec = w->ne0 % 8 == 0 && w->ne1 > 0 && w2->ne1 > 0 && (((uintptr_t) w->p0 | (uintptr_t) w2->p0 | (uintptr_t) out) & 15) == 0;
    PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 8.0 * w->ne0 * n_tok, k_embed_pair, dim3((unsigned) n_tok, (unsigned) ((w->ne0 + 2047) / 2048)), dim3(256), 0, (hipStream_t) stream, (const uint16_t *) w->p0, w->ne0, w->ne1, tokens, scale,
                 (const uint16_t *) w2->p0, w2->ne1, rows2, vec, out, vec ? pi_round_asked(0, w->ne0) : pi_round_dst{}, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// ---- the end of a sublayer whose norm comes after the sum ------------------------------------------------------------------------------------------------
// per token row:  m = b ? mb * (R(a) * wa + R(b) * wb) : a;   v = alpha * x + ls * m;   out = R(v) * w;   (w_next)  out_next = R(out) * w_next.   R(y) = y / sqrt(mean(y^2) + eps).
// A thread keeps its NPT values of every row in registers; out may be x.  PRE: every input (rows and weight vectors) is loaded before the first block sum, so that the launch makes ONE
// trip to memory instead of one per stage (rows up to 4096 wide; wider rows would not fit the registers and load stage by stage).
template <int NPT, bool PRE>
__global__ void __launch_bounds__(256) k_rms_post(const float * __restrict__ a, int64_t as, const float * __restrict__ wa, const float * __restrict__ b, int64_t bs, const float * __restrict__ wb, float mb,
                                                  const float * __restrict__ ls, const float * __restrict__ x, int64_t xs, float alpha, const float * __restrict__ w, float eps, int n,
                                                  float * __restrict__ out, int64_t os, const float * __restrict__ w_next, float * __restrict__ out_next, int64_t ons, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ float red[4];
    const int t = blockIdx.x, tid = threadIdx.x;
    float m[NPT], v[NPT];
    float pwa[PRE ? NPT : 1], pwb[PRE ? NPT : 1], pls[PRE ? NPT : 1], px[PRE ? NPT : 1], pw[PRE ? NPT : 1], pwn[PRE ? NPT : 1];
#pragma unroll
    for (int j = 0; j < NPT; j++) {
        const int i = j * 256 + tid;
        m[j] = i < n ? a[(int64_t) t * as + i] : 0.0f;
        v[j] = b && i < n ? b[(int64_t) t * bs + i] : 0.0f;
        if (PRE) {
            pwa[j] = b && i < n ? wa[i] : 0.0f; pwb[j] = b && i < n ? wb[i] : 0.0f;
            pls[j] = ls && i < n ? ls[i] : 1.0f; px[j] = i < n ? x[(int64_t) t * xs + i] : 0.0f; pw[j] = i < n ? w[i] : 0.0f; pwn[j] = w_next && i < n ? w_next[i] : 0.0f;
        }
    }
    if (b) {
        float sa = 0.0f, sb = 0.0f;
#pragma unroll
        for (int j = 0; j < NPT; j++) { sa = fmaf(m[j], m[j], sa); sb = fmaf(v[j], v[j], sb); }
        sa = cm_block_sum(sa, red); sb = cm_block_sum(sb, red);
        const float ia = 1.0f / sqrtf(sa / (float) n + eps), ib = 1.0f / sqrtf(sb / (float) n + eps);
#pragma unroll
        for (int j = 0; j < NPT; j++) { const int i = j * 256 + tid; if (i < n) m[j] = mb * (m[j] * ia * (PRE ? pwa[j] : wa[i]) + v[j] * ib * (PRE ? pwb[j] : wb[i])); }
    }
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NPT; j++) {
        const int i = j * 256 + tid;
        v[j] = i < n ? fmaf(alpha, PRE ? px[j] : x[(int64_t) t * xs + i], (PRE ? pls[j] : ls ? ls[i] : 1.0f) * m[j]) : 0.0f;
        ss = fmaf(v[j], v[j], ss);
    }
    ss = cm_block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) n + eps);
    if (pi_abort_late(gone, abort_w)) return;
    float s2 = 0.0f;
#pragma unroll
    for (int j = 0; j < NPT; j++) { const int i = j * 256 + tid; if (i < n) { v[j] = v[j] * inv * (PRE ? pw[j] : w[i]); out[(int64_t) t * os + i] = v[j]; s2 = fmaf(v[j], v[j], s2); } }
    if (!w_next) {
        if (rd.h)
#pragma unroll
            for (int j = 0; j < NPT; j++) { const int i = j * 256 + tid; if (i < n) rd.h[t * rd.stride + i] = pi_round_one(v[j]); }
        return;
    }
    s2 = cm_block_sum(s2, red);
    const float inv2 = 1.0f / sqrtf(s2 / (float) n + eps);
#pragma unroll
    for (int j = 0; j < NPT; j++) { const int i = j * 256 + tid; if (i < n) {
        const float y = v[j] * inv2 * (PRE ? pwn[j] : w_next[i]);
        if (!rd.only) out_next[(int64_t) t * ons + i] = y;
        if (rd.h) rd.h[t * rd.stride + i] = pi_round_one(y);
    } }
}
// The same in loads of 16 bytes, for rows whose places and lengths allow them: a thread has NV times four values.  A row of a step is bound by its one trip to memory and by how many loads a thread has on it, many rows by memory.
// Every sum has a place of its own in LDS: a barrier each.  us of one norm / with two inputs and a second norm, before -> now: one row of 2048 3.6 / 5.7 -> 2.2 / 3.2, eight rows of 4096 5.5 / 8.5 -> 3.2 / 4.8, 333 of 2048 4.4 / 7.0 ->
// 3.1 / 5.1, 2048 of 4096 19.6 / 34 -> 15.6 / 26, one of 8192 11.4 / 20.0 -> 2.6 / 5.2, 2048 of 8192 50 / 112 -> 31 / 75
template <int NV, int NT>
__global__ void __launch_bounds__(NT) k_rms_post4(const float * __restrict__ a, int64_t as, const float * __restrict__ wa, const float * __restrict__ b, int64_t bs, const float * __restrict__ wb, float mb,
                                                  const float * __restrict__ ls, const float * __restrict__ x, int64_t xs, float alpha, const float * __restrict__ w, float eps, int n,
                                                  float * __restrict__ out, int64_t os, const float * __restrict__ w_next, float * __restrict__ out_next, int64_t ons, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ float red[4][16];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = (int) (blockDim.x >> 6);
    float4 m[NV], v[NV], pwa[NV], pwb[NV], pls[NV], px[NV], pw[NV], pwn[NV];
    const float4 none = make_float4(0.0f, 0.0f, 0.0f, 0.0f), one = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
#pragma unroll
    for (int j = 0; j < NV; j++) {                                     // (behind the row's end: its last values, which count for nothing)
        const int i = min(4 * (j * (int) blockDim.x + tid), n - 4);
        m[j] = *(const float4 *) (a + (int64_t) t * as + i); px[j] = *(const float4 *) (x + (int64_t) t * xs + i); pw[j] = *(const float4 *) (w + i);
        v[j] = none; pwa[j] = none; pwb[j] = none; pwn[j] = none; pls[j] = one;
        if (b) { v[j] = *(const float4 *) (b + (int64_t) t * bs + i); pwa[j] = *(const float4 *) (wa + i); pwb[j] = *(const float4 *) (wb + i); }
        if (ls) pls[j] = *(const float4 *) (ls + i);
        if (w_next) pwn[j] = *(const float4 *) (w_next + i);
    }
    auto in = [&](int j) { return 4 * (j * (int) blockDim.x + tid) < n; };
    auto square = [&](const float4 & y, float s) { return fmaf(y.w, y.w, fmaf(y.z, y.z, fmaf(y.y, y.y, fmaf(y.x, y.x, s)))); };
    auto leave = [&](int k, float s) __attribute__((always_inline)) { s = pi_lanes_sum<64>(s); if (lane == 0) red[k][wave] = s; };
    auto whole = [&](int k) __attribute__((always_inline)) { float s = (lane & 15) < nw ? red[k][lane & 15] : 0.0f; pi_butterfly<8>([&](auto o) { s += pi_partner<decltype(o)::value>(s); }); return 1.0f / sqrtf(s / (float) n + eps); };
    if (b) {
        float sa = 0.0f, sb = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; j++) if (in(j)) { sa = square(m[j], sa); sb = square(v[j], sb); }
        leave(0, sa); leave(1, sb);
        __syncthreads();
        const float ia = whole(0), ib = whole(1);
#pragma unroll
        for (int j = 0; j < NV; j++)
            m[j] = make_float4(mb * (m[j].x * ia * pwa[j].x + v[j].x * ib * pwb[j].x), mb * (m[j].y * ia * pwa[j].y + v[j].y * ib * pwb[j].y), mb * (m[j].z * ia * pwa[j].z + v[j].z * ib * pwb[j].z), mb * (m[j].w * ia * pwa[j].w + v[j].w * ib * pwb[j].w));
    }
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        v[j] = make_float4(fmaf(alpha, px[j].x, pls[j].x * m[j].x), fmaf(alpha, px[j].y, pls[j].y * m[j].y), fmaf(alpha, px[j].z, pls[j].z * m[j].z), fmaf(alpha, px[j].w, pls[j].w * m[j].w));
        if (in(j)) ss = square(v[j], ss);
    }
    leave(2, ss);
    __syncthreads();
    const float inv = whole(2);
    if (pi_abort_late(gone, abort_w)) return;
    float s2 = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        v[j] = make_float4(v[j].x * inv * pw[j].x, v[j].y * inv * pw[j].y, v[j].z * inv * pw[j].z, v[j].w * inv * pw[j].w);
        if (in(j)) { *(float4 *) (out + (int64_t) t * os + 4 * (j * (int) blockDim.x + tid)) = v[j]; s2 = square(v[j], s2); }
    }
    if (!w_next) {
        if (rd.h)
#pragma unroll
            for (int j = 0; j < NV; j++) if (in(j)) pi_round_store4(rd, t, 4 * (j * (int) blockDim.x + tid), v[j].x, v[j].y, v[j].z, v[j].w);
        return;
    }
    leave(3, s2);
    __syncthreads();
    const float inv2 = whole(3);
#pragma unroll
    for (int j = 0; j < NV; j++) if (in(j)) {
        const int i = 4 * (j * (int) blockDim.x + tid);
        const float4 y = make_float4(v[j].x * inv2 * pwn[j].x, v[j].y * inv2 * pwn[j].y, v[j].z * inv2 * pwn[j].z, v[j].w * inv2 * pwn[j].w);
        if (!rd.only) *(float4 *) (out_next + (int64_t) t * ons + i) = y;
        if (rd.h) pi_round_store4(rd, t, i, y.x, y.y, y.z, y.w);
    }
}
extern "C" int pi_op_rms_post(const float * a, int64_t a_stride, const float * wa, const float * b, int64_t b_stride, const float * wb, float mean_mult, const float * layer_scale, const float * x, int64_t x_stride,
                              float alpha, const float * w, float eps, int n, int n_tok, float * out, int64_t out_stride, const float * w_next, float * out_next, int64_t out_next_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (n > 256 * 32) { pi_set_error("pi_op_rms_post: rows of %d values (at most %d)", n, 256 * 32); return -1; }
    if (b && (!wa || !wb)) { pi_set_error("pi_op_rms_post: two inputs need the weights of their norms"); return -1; }
    if (w_next && !out_next) { pi_set_error("pi_op_rms_post: a second norm needs a place for its result"); return -1; }
    const double bytes = 4.0 * n * n_tok * (3.0 + (b ? 1 : 0) + (w_next ? 1 : 0));
    const pi_round_dst rd = pi_round_asked(0, n);                      // (of the second norm where there is one)
    const uintptr_t at = (uintptr_t) a | (uintptr_t) wa | (uintptr_t) b | (uintptr_t) wb | (uintptr_t) layer_scale | (uintptr_t) x | (uintptr_t) w | (uintptr_t) out | (uintptr_t) w_next | (uintptr_t) out_next;
    const int64_t apart = a_stride | (b ? b_stride : 0) | x_stride | out_stride | (w_next ? out_next_stride : 0) | (rd.h ? rd.stride : 0) | n;
    // workgroups of 256 up to what a thread's registers hold, beyond of 1024 (of 1024 from the start: eight rows of 4096 and two norms 5.0 us, 4.8 so, 2048 rows 28.6 and 26.4)
    if ((at & 15) == 0 && ((uintptr_t) rd.h & 7) == 0 && (apart & 3) == 0) {
        const int threads = std::min(n > 4096 ? 1024 : 256, (n / 4 + 63) / 64 * 64);
#define RP_GO4(N, T) PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, bytes, (k_rms_post4<N, T>), dim3((unsigned) n_tok), dim3((unsigned) threads), 0, (hipStream_t) stream, a, a_stride, wa, b, b_stride, wb, mean_mult, layer_scale, x, x_stride, alpha, w, eps, n, \
                                  out, out_stride, w_next, out_next, out_next_stride, rd, pi_abort_word())
        if (n <= 1024) RP_GO4(1, 256); else if (n <= 2048) RP_GO4(2, 256); else if (n <= 4096) RP_GO4(4, 256); else RP_GO4(2, 1024);
#undef RP_GO4
        PI_CHECK_LAUNCH(); return 0;
    }
#define RP_GO(N, P) PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, bytes, (k_rms_post<N, P>), dim3((unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, a, a_stride, wa, b, b_stride, wb, mean_mult, layer_scale, x, x_stride, alpha, w, eps, n, \
                              out, out_stride, w_next, out_next, out_next_stride, rd, pi_abort_word())
    if (n <= 256 * 2) RP_GO(2, true); else if (n <= 256 * 4) RP_GO(4, true); else if (n <= 256 * 8) RP_GO(8, true); else if (n <= 256 * 16) RP_GO(16, true); else RP_GO(32, false);
#undef RP_GO
    PI_CHECK_LAUNCH(); return 0;
}

// ---- token shift: every mix of a token with the token before it ------------------------------------------------------------------------------------------------
// out[t][s][i] = h[t][i] + (prev[i] - h[t][i]) * mu[s][i], s < n_mix; prev = h[t - 1] inside a sequence's run, the sequence's state (zeros on a fresh slot) at the run's first token.
// rec as for the recurrences; state: [slots][n].  grid (token, blocks of 256 values)
__global__ void __launch_bounds__(256) k_token_shift(const float * __restrict__ h, int64_t hs, int n, const float * __restrict__ mu, int n_mix, const float * __restrict__ state, const int32_t * __restrict__ rec,
                                                     float * __restrict__ out, int64_t os, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    if (i >= n) return;
    const int word = rec[t], slot = word & ~CM_FRESH;
    const bool inside = t > 0 && (rec[t - 1] & ~CM_FRESH) == slot;
    const float cur = h[(int64_t) t * hs + i];
    const float prev = inside ? h[(int64_t) (t - 1) * hs + i] : (word & CM_FRESH) ? 0.0f : state[(int64_t) slot * n + i];
    const float d = prev - cur;
    for (int s = 0; s < n_mix; s++) {
        const float y = fmaf(d, mu[(int64_t) s * n + i], cur);
        if (!rd.only) out[(int64_t) t * os + (int64_t) s * n + i] = y;
        if (rd.h) rd.h[t * rd.stride + (int64_t) s * n + i] = pi_round_one(y);
    }
}
// a run's last token becomes the sequence's state (its own launch: the run's first token reads the state in the launch above)
__global__ void __launch_bounds__(256) k_token_shift_state(const float * __restrict__ h, int64_t hs, int n, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    const int slot = rec[t] & ~CM_FRESH;
    if (i >= n || (t + 1 < n_tok && (rec[t + 1] & ~CM_FRESH) == slot)) return;
    state[(int64_t) slot * n + i] = h[(int64_t) t * hs + i];
}
// short passes in ONE launch: the thread of a run's first token walks the run for its value and leaves the state, so nothing it writes is read by another thread
__global__ void __launch_bounds__(256) k_token_shift_walk(const float * __restrict__ h, int64_t hs, int n, const float * __restrict__ mu, int n_mix, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok,
                                                          float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int t = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    const int word = rec[t], slot = word & ~CM_FRESH;
    if (i >= n || (t > 0 && (rec[t - 1] & ~CM_FRESH) == slot)) return;
    if (pi_abort_late(gone, abort_w)) return;                          // (behind the slot words)
    float prev = (word & CM_FRESH) ? 0.0f : state[(int64_t) slot * n + i];
    for (int tt = t; tt < n_tok && (rec[tt] & ~CM_FRESH) == slot; tt++) {
        const float cur = h[(int64_t) tt * hs + i], d = prev - cur;
        for (int s = 0; s < n_mix; s++) out[(int64_t) tt * os + (int64_t) s * n + i] = fmaf(d, mu[(int64_t) s * n + i], cur);
        prev = cur;
    }
    state[(int64_t) slot * n + i] = prev;
}
#define TS_WALK_MAX_TOKENS 32
extern "C" int pi_op_token_shift(const float * h, int64_t h_stride, int n, const float * mu_dev, int n_mix, float * state_dev, const int32_t * rec_dev, int n_tok, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (n_mix < 1 || out_stride < (int64_t) n_mix * n) { pi_set_error("pi_op_token_shift: %d mixes of %d values do not fit rows %lld floats apart", n_mix, n, (long long) out_stride); return -1; }
    if (out == h) { pi_set_error("pi_op_token_shift: the output may not overwrite the input (the next token reads it)"); return -1; }
    hipStream_t s = (hipStream_t) stream;
    const dim3 grid((unsigned) n_tok, (unsigned) ((n + 255) / 256));
    const double bytes = 4.0 * n * n_tok * (1.0 + n_mix) + 4.0 * n * n_mix;
    if (n_tok <= TS_WALK_MAX_TOKENS) {
        PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, bytes, k_token_shift_walk, grid, dim3(256), 0, s, h, h_stride, n, mu_dev, n_mix, state_dev, rec_dev, n_tok, out, out_stride, pi_abort_word());
        PI_CHECK_LAUNCH(); return 0;
    }
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, bytes, k_token_shift, grid, dim3(256), 0, s, h, h_stride, n, mu_dev, n_mix, state_dev, rec_dev, out, out_stride, pi_round_asked(0, (int64_t) n_mix * n), pi_abort_word());
    PI_CHECK_LAUNCH();
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 8.0 * n, k_token_shift_state, grid, dim3(256), 0, s, h, h_stride, n, state_dev, rec_dev, n_tok, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// ---- recurrences with a decay per key channel ------------------------------------------------------------------------------------------------------------------
// Workgroup (head, block of value columns, piece of the pass): thread (column j, part sp of R) keeps S[i][j] for its DPT rows i in registers and walks the piece's tokens in order; q, k,
// the decays and v of CR_TB tokens at a time are staged (and finished: decays formed, unit vectors, sigmoid) in LDS.  A value column never meets another: o_j, u_j and S[:, j]
// depend on column j alone, so the only exchange is the sum over the R parts of a column (neighbouring lanes).
//   delta:  S <- g S;  a = S^T k, c = S^T q (one pass over the registers);  u = beta (v - a);  o = c + u (k . q);  S <- S + k u
//   bonus:  c = S^T q;  o = c + v (sum_i q_i b_i k_i);  S <- g S + k v
// A pass of up to CR_TB tokens (or keys too wide for the scan's tile) is ONE launch, mode 0: a piece is a sequence's whole run, S comes from and goes back to HBM.  Longer passes cut
// every run into pieces of CR_PIECE tokens that run side by side, because a column's step is affine in the column, s <- A_t s + b_t v_j with A_t the same for every column:
//   mode 1  every piece but a run's last, with extra columns: L_p = the state the piece builds from ZERO, and T_p = A_n .. A_1.  Delta rule: dim extra columns, column c of T_p is what the
//           piece makes of the unit vector e_c with v = 0 — the same walk over a column that starts as e_c.  Bonus rule: A_t is diagonal, ONE extra column that starts as all ones ends as
//           the diagonal of T_p.  Both into scratch [piece][head][dim][vdim + extra]
//   k_channel_state_scan / _diag  per run, piece by piece: S_in(p + 1) = T_p S_in(p) + L_p, S_in(0) = the slot's state (or zero); scratch[p][..][0 .. vdim) <- S_in(p)
//   mode 2  every piece from its true S_in(p): outputs; a run's last piece leaves the slot's new state
#define CR_TB 32                                  // tokens staged in LDS at a time
#define CR_PIECE 64                               // most tokens of a piece of a long pass (the launcher picks 32 or 64: longer pieces leave the scan fewer to chain, shorter ones put more side by side)
#define CR_MAXRUNS 256
#define CR_SCAN_MAXDIM 128                        // widest key whose transition matrix the scan keeps in LDS
// the pass's runs in order (a run: the consecutive tokens of one slot): every thread looks at its own tokens for a run's first one, the few found are ranked by position.  first[r] in `sorted`
static __device__ __forceinline__ int cr_mark(const int32_t * __restrict__ rec, int t) { return t == 0 || (rec[t] & ~CM_FRESH) != (rec[t - 1] & ~CM_FRESH); }
// (mark: a caller's own for token threadIdx.x, asked for ahead of loads of its own, which would be waited for with it)
static __device__ __forceinline__ int cr_runs(const int32_t * __restrict__ rec, int n_tok, int * bnd, int * sorted, int * nb, int mark = -1) {
    if (threadIdx.x == 0) *nb = 0;
    __syncthreads();
    for (int t = threadIdx.x; t < n_tok; t += blockDim.x)
        if (mark >= 0 && t == (int) threadIdx.x ? mark : cr_mark(rec, t)) { const int at = atomicAdd(nb, 1); if (at < CR_MAXRUNS) bnd[at] = t; }
    __syncthreads();
    const int n = min(*nb, CR_MAXRUNS);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        int rank = 0;
        for (int o = 0; o < n; o++) rank += bnd[o] < bnd[i];
        sorted[rank] = bnd[i];
    }
    __syncthreads();
    return n;
}
// (amdgpu_waves_per_eu(1, 2): at most two workgroups fit a compute unit's LDS anyway, so the registers of the other waves a SIMD could hold are free for a token's reads)
template <int DPT, int RULE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) k_channel_recurrence(const float * __restrict__ q, int64_t qs, const float * __restrict__ k, int64_t ks, const float * __restrict__ v, int64_t vs,
                                                            const float * __restrict__ draw, int64_t ds, int decay_mode, const float * __restrict__ dbias, const float * __restrict__ a_log,
                                                            const float * __restrict__ braw, int64_t bs, const float * __restrict__ bonus, int qk_unit, float q_mult,
                                                            int heads, int hpg, int dim, int vdim, int R, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, int mode, int tb, int piece,
                                                            float * __restrict__ scratch, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    extern __shared__ float lds[];                // q [CR_TB][dp] | k [CR_TB][dp] | g [CR_TB][dp] | v [CR_TB][cols];  a row is R parts of DPT values, DPT + 4 floats apart (the parts of one wave-wide read then fall into different banks), dp = R * (DPT + 4); rows end in zeros so that the token loop needs no bounds
    __shared__ int seg[4], bnd[CR_MAXRUNS], sorted[CR_MAXRUNS], nbnd;      // seg: first token, length, slot word of this workgroup's piece, whether it is its run's last
    __shared__ float beta_t[CR_TB], dot_t[CR_TB];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
    const int n_runs = n_tok == 1 ? 1 : cr_runs(rec, n_tok, bnd, sorted, &nbnd);      // (a single token is its own run: no search, no barrier)
    if (n_tok == 1) { if (tid == 0) { seg[0] = 0; seg[1] = blockIdx.z == 0 ? 1 : 0; seg[2] = rec[0]; seg[3] = 1; } }
    else if (tid == 0) {                          // piece number blockIdx.z of the pass (mode 0: pieces are whole runs)
        const int lseg = mode ? piece : 0, want = blockIdx.z;
        int ord = 0;
        seg[1] = 0; seg[2] = -1;
        for (int r = 0; r < n_runs; r++) {
            const int t = sorted[r], e = r + 1 < n_runs ? sorted[r + 1] : n_tok;
            const int nsub = lseg > 0 ? (e - t + lseg - 1) / lseg : 1;
            if (want < ord + nsub) {
                const int pc = want - ord;
                seg[0] = lseg > 0 ? t + pc * lseg : t; seg[1] = lseg > 0 ? min(lseg, e - seg[0]) : e - t; seg[2] = rec[t]; seg[3] = pc == nsub - 1;
                break;
            }
            ord += nsub;
        }
    }
    __syncthreads();
    const int first = seg[0], len = seg[1], word = seg[2], last = seg[3];
    if (pi_abort_late(gone, abort_w)) return;
    if (len == 0 || word < 0 || (mode == 1 && last)) return;
    const int slot = word & ~CM_FRESH;
    const int cols = blockDim.x / R;
    const int ext = RULE == 0 ? dim : 1;                              // extra columns of mode 1
    const int ncol = mode == 1 ? vdim + ext : vdim, sw = vdim + ext;   // columns this launch walks; row stride of a piece's block in scratch
    const int j = blockIdx.y * cols + tid / R, sp = tid % R;
    const bool col_ok = j < ncol;
    const int hq = h / hpg;                                            // the q / k head this head reads
    float * S_hbm = state + ((int64_t) slot * heads + h) * dim * vdim;
    float * S_scr = scratch ? scratch + ((int64_t) blockIdx.z * heads + h) * dim * sw : nullptr;
    float S[DPT];
#pragma unroll
    for (int ii = 0; ii < DPT; ii++) {
        const int i = sp * DPT + ii;
        float s0 = 0.0f;
        if (col_ok && i < dim) {
            if (mode == 1) s0 = j >= vdim && (RULE == 1 || i == j - vdim) ? 1.0f : 0.0f;
            else if (mode == 2) s0 = S_scr[(int64_t) i * sw + j];
            else if (!(word & CM_FRESH)) s0 = S_hbm[(int64_t) i * vdim + j];
        }
        S[ii] = s0;
    }
    const int dp = R * (DPT + 4);
    float * qt = lds, * kt = qt + tb * dp, * gt = kt + tb * dp, * vt = gt + tb * dp;        // tb <= CR_TB tokens at a time (fewer where the keys are very wide)
    const float ah = decay_mode == 2 ? expf(a_log[h]) : 0.0f;
    for (int t0 = 0; t0 < len; t0 += tb) {
        const int nt = min(tb, len - t0);
        __syncthreads();
        for (int idx = tid; idx < nt * R * DPT; idx += blockDim.x) {
            const int tt = idx / (R * DPT), i = idx % (R * DPT);
            const int64_t tok = first + t0 + tt;
            float qv = 0.0f, kv = 0.0f, d = 0.0f;
            if (i < dim) {
                qv = q[tok * qs + (int64_t) hq * dim + i];
                kv = k[tok * ks + (int64_t) hq * dim + i];
                d = draw[tok * ds + (int64_t) h * dim + i];
                if (decay_mode == 1) d = expf(-expf(d + (dbias ? dbias[h * dim + i] : 0.0f)));
                else if (decay_mode == 2) d = expf(-ah * cm_softplus(d + (dbias ? dbias[h * dim + i] : 0.0f)));
            }
            const int at = tt * dp + i / DPT * (DPT + 4) + i % DPT;
            qt[at] = qv; kt[at] = kv; gt[at] = d;
        }
        if (tid < nt) beta_t[tid] = braw ? cm_sigmoid(braw[(int64_t) (first + t0 + tid) * bs + h]) : 1.0f;
        for (int idx = tid; idx < nt * cols; idx += blockDim.x) {
            const int tt = idx / cols, jj = blockIdx.y * cols + idx % cols;
            vt[idx] = jj < vdim ? v[(int64_t) (first + t0 + tt) * vs + (int64_t) h * vdim + jj] : 0.0f;       // (the extra columns of mode 1 carry v = 0)
        }
        __syncthreads();
        for (int tt = wave; tt < nt; tt += nw) {                          // a wave per token: unit vectors, then the token's scalar (k . q, or sum q b k)
            float * qr = qt + tt * dp, * kr = kt + tt * dp;
            auto at = [&](int i) { return i / DPT * (DPT + 4) + i % DPT; };
            if (qk_unit) {
                float sq = 0.0f, sk = 0.0f;
                for (int i = lane; i < dim; i += 64) { sq = fmaf(qr[at(i)], qr[at(i)], sq); sk = fmaf(kr[at(i)], kr[at(i)], sk); }
                const float iq = q_mult / sqrtf(pi_lanes_sum<64>(sq) + 1e-6f), ik = 1.0f / sqrtf(pi_lanes_sum<64>(sk) + 1e-6f);
                for (int i = lane; i < dim; i += 64) { qr[at(i)] *= iq; kr[at(i)] *= ik; }
            } else if (q_mult != 1.0f) for (int i = lane; i < dim; i += 64) qr[at(i)] *= q_mult;
            float d = 0.0f;
            for (int i = lane; i < dim; i += 64) d = fmaf(RULE == 1 && bonus ? qr[at(i)] * bonus[h * dim + i] : qr[at(i)], kr[at(i)], d);      // (a lane re-reads only what it wrote itself)
            d = pi_lanes_sum<64>(d);
            if (lane == 0) dot_t[tt] = d;
        }
        __syncthreads();
        for (int tt = 0; tt < nt; tt++) {
            const float vj = vt[tt * cols + tid / R];
            const float * kr = kt + tt * dp + sp * (DPT + 4), * qr = qt + tt * dp + sp * (DPT + 4), * gr = gt + tt * dp + sp * (DPT + 4);
            float a = 0.0f, c = 0.0f, o;
            float4 k4[DPT / 4], q4[DPT / 4], g4[DPT / 4];                 // 16-byte LDS reads, no bounds (rows beyond dim: k = q = g = 0, their S stays 0): all of a token's reads go out before the first use
#pragma unroll
            for (int ii = 0; ii < DPT / 4; ii++) { k4[ii] = *(const float4 *) (kr + 4 * ii); q4[ii] = *(const float4 *) (qr + 4 * ii); g4[ii] = *(const float4 *) (gr + 4 * ii); }
            float a2 = 0.0f, c2 = 0.0f;                                   // (two chains each: half the depth of the dependent sums)
#pragma unroll
            for (int ii = 0; ii < DPT / 4; ii++) {
                const float4 kv = k4[ii], qv = q4[ii], gv = g4[ii];
                float * Sq = S + 4 * ii;
                if (RULE == 0) {
                    Sq[0] *= gv.x; Sq[1] *= gv.y; Sq[2] *= gv.z; Sq[3] *= gv.w;
                    a = fmaf(Sq[0], kv.x, a); a2 = fmaf(Sq[1], kv.y, a2); a = fmaf(Sq[2], kv.z, a); a2 = fmaf(Sq[3], kv.w, a2);
                }
                c = fmaf(Sq[0], qv.x, c); c2 = fmaf(Sq[1], qv.y, c2); c = fmaf(Sq[2], qv.z, c); c2 = fmaf(Sq[3], qv.w, c2);
                if (RULE == 1) { Sq[0] *= gv.x; Sq[1] *= gv.y; Sq[2] *= gv.z; Sq[3] *= gv.w; }
            }
            a += a2; c += c2;
            if (R == 2) { if (RULE == 0) a += pi_partner<1>(a); c += pi_partner<1>(c); }
            else if (R == 4) { if (RULE == 0) { a += pi_partner<2>(a); a += pi_partner<1>(a); } c += pi_partner<2>(c); c += pi_partner<1>(c); }
            else for (int d = R >> 1; d > 0; d >>= 1) { if (RULE == 0) a += __shfl_xor(a, d, PI_WAVE); c += __shfl_xor(c, d, PI_WAVE); }
            const float u = RULE == 0 ? beta_t[tt] * (vj - a) : vj;       // what the token writes under its key
            o = fmaf(u, dot_t[tt], c);
#pragma unroll
            for (int ii = 0; ii < DPT / 4; ii++) { S[4 * ii] = fmaf(k4[ii].x, u, S[4 * ii]); S[4 * ii + 1] = fmaf(k4[ii].y, u, S[4 * ii + 1]); S[4 * ii + 2] = fmaf(k4[ii].z, u, S[4 * ii + 2]); S[4 * ii + 3] = fmaf(k4[ii].w, u, S[4 * ii + 3]); }
            if (mode != 1 && col_ok && sp == 0) out[(int64_t) (first + t0 + tt) * os + (int64_t) h * vdim + j] = o;
        }
    }
    if (!col_ok) return;
    if (mode == 1) {
#pragma unroll
        for (int ii = 0; ii < DPT; ii++) { const int i = sp * DPT + ii; if (i < dim) S_scr[(int64_t) i * sw + j] = S[ii]; }
    } else if (last) {
#pragma unroll
        for (int ii = 0; ii < DPT; ii++) { const int i = sp * DPT + ii; if (i < dim) S_hbm[(int64_t) i * vdim + j] = S[ii]; }
    }
}

// The same for a step: a few tokens, most of them a run of their own.  What bounds it: a state is read and written once (16.8 MB of eight sequences, 6.7 us at a copy's rate), and the trips to memory in front of that.  So nothing goes
// through LDS but the sums over the rows, which the four waves share: a wave finds its run by a ballot, every operand of its first token leaves beside the state, the unit vectors' lengths and the token's scalar are added up by
// every wave for itself.  Workgroup (head, 32 columns of values, run); thread (four columns, rows rg + 8 NW m), states in runs of 128 bytes; a token is one barrier.
// Keys of 32 values: one wave (NW = 1), no LDS and no barrier.  What every wave repeats is most of such a token, and where workgroups fill the chip four waves paid for it four times: 64 heads of 32 x 256 under the delta rule, eight runs
// of four tokens, 35.3 by k_channel_recurrence, 49.2 by four waves, 15.7 by one; 32 tokens of one run, 128 heads of 32 x 128, 74 / 60 / 37; one token of 32 heads of 32 x 64 11.5 / 3.8 / 3.5.
// Measured, us (k_channel_recurrence / this), 32 heads of 128 x 128 under the delta rule: one token 14.5 / 4.8, eight of a sequence each 19.8 / 8.3, eight of one 35.6 / 13.7, 32 of one 109 / 46; 64 heads of 64 x 64 under the bonus rule
// 11.8 / 3.7, 15.6 / 6.1, 24.5 / 8.6, 67.8 / 23.5.  (There a token's operands were staged for 32, with four barriers and a search by one thread ahead of them, and a state came in runs of 64 bytes.)
#define CS_TOKENS CR_TB                           // (a run's first tokens are found among a wave's lanes; longer passes go in pieces)
template <int NR, int RULE, int NW>
__global__ void __launch_bounds__(64 * NW) k_channel_step(const float * __restrict__ q, int64_t qs, const float * __restrict__ k, int64_t ks, const float * __restrict__ v, int64_t vs,
                                                      const float * __restrict__ draw, int64_t ds, int decay_mode, const float * __restrict__ dbias, const float * __restrict__ a_log,
                                                      const float * __restrict__ braw, int64_t bs, const float * __restrict__ bonus, int qk_unit, float q_mult,
                                                      int heads, int hpg, int vdim, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok,
                                                      float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int STEP = 8 * NW, DIM = STEP * NR, NL = (DIM + 63) / 64;
    __shared__ __attribute__((aligned(16))) float meet[2][NW][2][NW > 1 ? 32 : 1];    // [token % 2][wave][with the keys, with the queries][column]
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), quad = tid & 7, rg = tid >> 3, col = blockIdx.y * 32 + quad * 4, hq = h / hpg;
    // run number blockIdx.z
    const int own = rec[min(lane, n_tok - 1)], before = rec[max(min(lane, n_tok - 1) - 1, 0)];
    const float ah = decay_mode == 2 ? expf(a_log[h]) : 0.0f;
    uint64_t starts = __ballot(lane < n_tok && (lane == 0 || (own & ~CM_FRESH) != (before & ~CM_FRESH)));
    for (int r = 0; r < (int) blockIdx.z; r++) starts &= starts - 1;
    if (!starts) return;
    const int first = __ffsll((unsigned long long) starts) - 1, rest = __ffsll((unsigned long long) (starts & (starts - 1))), end = rest ? rest - 1 : n_tok, word = __builtin_amdgcn_readlane(own, first);
    if (word < 0) return;
    float * const S_hbm = state + ((int64_t) (word & ~CM_FRESH) * heads + h) * DIM * vdim + (int64_t) rg * vdim + col;
    float4 S[NR];
    if (word & CM_FRESH) {
#pragma unroll
        for (int m = 0; m < NR; m++) S[m] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
#pragma unroll
        for (int m = 0; m < NR; m++) S[m] = *(const float4 *) (S_hbm + (int64_t) STEP * m * vdim);
    }
    struct token { float q[NR], k[NR], d[NR], lq[NL], lk[NL], lb[NL], beta; float4 v; };
    float bias[NR];
#pragma unroll
    for (int m = 0; m < NR; m++) bias[m] = dbias ? dbias[h * DIM + rg + STEP * m] : 0.0f;
    auto ask = [&](token & T, int t) __attribute__((always_inline)) {
        const float * qr = q + (int64_t) t * qs + (int64_t) hq * DIM, * kr = k + (int64_t) t * ks + (int64_t) hq * DIM, * dr = draw + (int64_t) t * ds + (int64_t) h * DIM;
#pragma unroll
        for (int m = 0; m < NR; m++) { T.q[m] = qr[rg + STEP * m]; T.k[m] = kr[rg + STEP * m]; T.d[m] = dr[rg + STEP * m]; }
#pragma unroll
        for (int x = 0; x < NL; x++) {
            const int i = min(lane + 64 * x, DIM - 1);
            T.lq[x] = qr[i]; T.lk[x] = kr[i]; T.lb[x] = RULE == 1 && bonus ? bonus[h * DIM + i] : 1.0f;
        }
        T.beta = braw ? braw[(int64_t) t * bs + h] : 0.0f;
        T.v = *(const float4 *) (v + (int64_t) t * vs + (int64_t) h * vdim + col);
    };
    token T;
    ask(T, first);
    if (pi_abort_late(gone, abort_w)) return;
    for (int t = first; t < end; t++) {
        // lengths, then the token's scalar (k . q, or sum q b k)
        float iq = q_mult, ik = 1.0f, dot = 0.0f;
        if (qk_unit) {
            float sq = 0.0f, sk = 0.0f;
#pragma unroll
            for (int x = 0; x < NL; x++) if (DIM % 64 == 0 || lane < DIM) { sq = fmaf(T.lq[x], T.lq[x], sq); sk = fmaf(T.lk[x], T.lk[x], sk); }
            pi_butterfly<32>([&](auto o) { constexpr int O = decltype(o)::value; sq += pi_partner<O>(sq); sk += pi_partner<O>(sk); });
            iq = q_mult / sqrtf(sq + 1e-6f); ik = 1.0f / sqrtf(sk + 1e-6f);
        }
#pragma unroll
        for (int x = 0; x < NL; x++) if (DIM % 64 == 0 || lane < DIM) dot = fmaf(T.lq[x] * iq * T.lb[x], T.lk[x] * ik, dot);
        dot = pi_lanes_sum<64>(dot);
        float kk[NR], a[4] = { 0.0f, 0.0f, 0.0f, 0.0f }, c[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
        const float beta = braw ? cm_sigmoid(T.beta) : 1.0f;
        const float4 vv = T.v;
#pragma unroll
        for (int m = 0; m < NR; m++) {
            float g = T.d[m];
            if (decay_mode == 1) g = expf(-expf(g + bias[m]));
            else if (decay_mode == 2) g = expf(-ah * cm_softplus(g + bias[m]));
            const float qq = T.q[m] * iq;
            kk[m] = T.k[m] * ik;
            if (RULE == 0) {
                S[m].x *= g; S[m].y *= g; S[m].z *= g; S[m].w *= g;
                a[0] = fmaf(S[m].x, kk[m], a[0]); a[1] = fmaf(S[m].y, kk[m], a[1]); a[2] = fmaf(S[m].z, kk[m], a[2]); a[3] = fmaf(S[m].w, kk[m], a[3]);
            }
            c[0] = fmaf(S[m].x, qq, c[0]); c[1] = fmaf(S[m].y, qq, c[1]); c[2] = fmaf(S[m].z, qq, c[2]); c[3] = fmaf(S[m].w, qq, c[3]);
            if (RULE == 1) { S[m].x *= g; S[m].y *= g; S[m].z *= g; S[m].w *= g; }
        }
        if (t + 1 < end) ask(T, t + 1);
        // over the wave's eight rows: lanes 8 apart
#pragma unroll
        for (int x = 0; x < 4; x++) {
            if (RULE == 0) { a[x] += pi_partner<8>(a[x]); a[x] += pi_partner<16>(a[x]); a[x] += pi_partner<32>(a[x]); }
            c[x] += pi_partner<8>(c[x]); c[x] += pi_partner<16>(c[x]); c[x] += pi_partner<32>(c[x]);
        }
        // of all rows: what the four waves left (a wave alone has it in every lane)
        float (* const M)[2][NW > 1 ? 32 : 1] = meet[t & 1];
        if constexpr (NW > 1) {
            if (lane < 8) {
                if (RULE == 0) *(float4 *) &M[wave][0][quad * 4] = make_float4(a[0], a[1], a[2], a[3]);
                *(float4 *) &M[wave][1][quad * 4] = make_float4(c[0], c[1], c[2], c[3]);
            }
            __syncthreads();
        }
        auto met = [&](int which, const float * own) __attribute__((always_inline)) {
            if constexpr (NW > 1) {
                const float4 w0 = *(const float4 *) &M[0][which][quad * 4], w1 = *(const float4 *) &M[1][which][quad * 4], w2 = *(const float4 *) &M[2][which][quad * 4], w3 = *(const float4 *) &M[3][which][quad * 4];
                return make_float4((w0.x + w1.x) + (w2.x + w3.x), (w0.y + w1.y) + (w2.y + w3.y), (w0.z + w1.z) + (w2.z + w3.z), (w0.w + w1.w) + (w2.w + w3.w));
            } else return make_float4(own[0], own[1], own[2], own[3]);
        };
        float4 u = vv;                                                  // what the token writes under its key
        if (RULE == 0) { const float4 wa = met(0, a); u.x = beta * (vv.x - wa.x); u.y = beta * (vv.y - wa.y); u.z = beta * (vv.z - wa.z); u.w = beta * (vv.w - wa.w); }
#pragma unroll
        for (int m = 0; m < NR; m++) { S[m].x = fmaf(kk[m], u.x, S[m].x); S[m].y = fmaf(kk[m], u.y, S[m].y); S[m].z = fmaf(kk[m], u.z, S[m].z); S[m].w = fmaf(kk[m], u.w, S[m].w); }
        if (tid < 8) {
            const float4 wc = met(1, c);
            *(float4 *) (out + (int64_t) t * os + (int64_t) h * vdim + col) = make_float4(fmaf(u.x, dot, wc.x), fmaf(u.y, dot, wc.y), fmaf(u.z, dot, wc.z), fmaf(u.w, dot, wc.w));
        }
    }
#pragma unroll
    for (int m = 0; m < NR; m++) *(float4 *) (S_hbm + (int64_t) STEP * m * vdim) = S[m];
}

// grid (head, blocks of CR_SCAN_COLS value columns, run): per piece p of the run, in order: scratch[p] holds [L_p | T_p] coming in and S_in(p) (in L_p's place) going out.
// A workgroup keeps its columns of S in LDS (two buffers) and T_p transposed ([c][i], so that a thread's rows are neighbours); a thread owns a tile of 8 rows x 4 columns: per column c of T_p
// three 16-byte LDS reads feed 32 multiply-adds.
template <int CR_SCAN_COLS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) k_channel_state_scan(int heads, int dim, int vdim, int piece, const float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok,
                                                                                                     float * __restrict__ scratch, const int32_t * __restrict__ abort_w) {
    if (pi_aborted_together(pi_abort_peek(abort_w), abort_w)) return;
    extern __shared__ float lds[];                // T^T [dim][tp] | S [2][dim][CR_SCAN_COLS]
    __shared__ int seg[3], bnd[CR_MAXRUNS], sorted[CR_MAXRUNS], nbnd;      // slot word, first piece ordinal, pieces of the run (0: no such run)
    const int tid = threadIdx.x, h = blockIdx.x, j0 = blockIdx.y * CR_SCAN_COLS;
    const int n_runs = cr_runs(rec, n_tok, bnd, sorted, &nbnd);
    if (tid == 0) {
        int ord = 0;
        seg[0] = -1; seg[2] = 0;
        for (int r = 0; r < n_runs; r++) {
            const int t = sorted[r], e = r + 1 < n_runs ? sorted[r + 1] : n_tok;
            const int ns = (e - t + piece - 1) / piece;
            if (r == (int) blockIdx.z) { seg[0] = rec[t]; seg[1] = ord; seg[2] = ns; break; }
            ord += ns;
        }
    }
    __syncthreads();
    const int word = seg[0], sub0 = seg[1], nsub = seg[2];
    if (nsub == 0 || word < 0) return;
    const int slot = word & ~CM_FRESH, sw = vdim + dim, tp = (dim + 3) / 4 * 4 + 4;       // (rows of T^T start 16-byte aligned)
    float * Tt = lds, * Sb = Tt + dim * tp;
    constexpr int CG = CR_SCAN_COLS / 4;                               // column groups of 4
    const int jg = tid % CG, part = tid / CG, jl = jg * 4, pstep = 8 * (256 / CG);      // row parts of 8 rows
    const float * S0 = state + ((int64_t) slot * heads + h) * dim * vdim;
    for (int idx = tid; idx < dim * CR_SCAN_COLS; idx += 256) {
        const int i = idx / CR_SCAN_COLS, jj = j0 + idx % CR_SCAN_COLS;
        Sb[idx] = (jj < vdim && !(word & CM_FRESH)) ? S0[(int64_t) i * vdim + jj] : 0.0f;
    }
    int cur = 0;
    for (int p = 0; p < nsub; p++) {
        float * blk = scratch + ((int64_t) (sub0 + p) * heads + h) * dim * sw;
        const bool more = p + 1 < nsub;
        __syncthreads();                                               // (S of this piece is complete, T of the last one is no longer read)
        if (more) for (int idx = tid; idx < dim * dim; idx += 256) { const int i = idx / dim, c = idx % dim; Tt[c * tp + i] = blk[(int64_t) i * sw + vdim + c]; }
        __syncthreads();
        const float * Sc = Sb + cur * dim * CR_SCAN_COLS;
        float * Sn = Sb + (cur ^ 1) * dim * CR_SCAN_COLS;
        for (int i0 = part * 8; i0 < dim; i0 += pstep) {
            float acc[8][4];
#pragma unroll
            for (int r = 0; r < 8; r++)
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const bool ok = i0 + r < dim && j0 + jl + u < vdim;
                    acc[r][u] = (more && ok) ? blk[(int64_t) (i0 + r) * sw + j0 + jl + u] : 0.0f;                                     // L_p, read before S_in(p) takes its place
                    if (ok) blk[(int64_t) (i0 + r) * sw + j0 + jl + u] = Sc[(i0 + r) * CR_SCAN_COLS + jl + u];
                }
            if (!more) continue;
            for (int c = 0; c < dim; c++) {
                const float4 sv = *(const float4 *) (Sc + c * CR_SCAN_COLS + jl);
                const float4 ta = *(const float4 *) (Tt + c * tp + i0), tb = *(const float4 *) (Tt + c * tp + i0 + 4);      // (rows beyond dim read the pad or the next row of T^T: their sums are dropped)
                const float tv[8] = { ta.x, ta.y, ta.z, ta.w, tb.x, tb.y, tb.z, tb.w };
#pragma unroll
                for (int r = 0; r < 8; r++) { acc[r][0] = fmaf(tv[r], sv.x, acc[r][0]); acc[r][1] = fmaf(tv[r], sv.y, acc[r][1]); acc[r][2] = fmaf(tv[r], sv.z, acc[r][2]); acc[r][3] = fmaf(tv[r], sv.w, acc[r][3]); }
            }
#pragma unroll
            for (int r = 0; r < 8; r++) if (i0 + r < dim) *(float4 *) (Sn + (i0 + r) * CR_SCAN_COLS + jl) = make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
        }
        cur ^= 1;
    }
}

// the same chain where T_p is diagonal (bonus rule): scratch[p] holds [L_p | diag T_p] ([dim][vdim + 1]).  grid (head, blocks over dim * vdim, run): eight pieces' loads in flight, the chain in registers
__global__ void __launch_bounds__(256) k_channel_state_scan_diag(int heads, int dim, int vdim, int piece, const float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, float * __restrict__ scratch,
                                                                 const int32_t * __restrict__ abort_w) {
    if (pi_aborted_together(pi_abort_peek(abort_w), abort_w)) return;
    __shared__ int seg[3], bnd[CR_MAXRUNS], sorted[CR_MAXRUNS], nbnd;
    const int tid = threadIdx.x, h = blockIdx.x;
    const int n_runs = cr_runs(rec, n_tok, bnd, sorted, &nbnd);
    if (tid == 0) {
        int ord = 0;
        seg[0] = -1; seg[2] = 0;
        for (int r = 0; r < n_runs; r++) {
            const int t = sorted[r], e = r + 1 < n_runs ? sorted[r + 1] : n_tok;
            const int ns = (e - t + piece - 1) / piece;
            if (r == (int) blockIdx.z) { seg[0] = rec[t]; seg[1] = ord; seg[2] = ns; break; }
            ord += ns;
        }
    }
    __syncthreads();
    const int word = seg[0], sub0 = seg[1], nsub = seg[2];
    if (nsub == 0 || word < 0) return;
    const int64_t per = (int64_t) dim * vdim, idx = (int64_t) blockIdx.y * 256 + tid;
    if (idx >= per) return;
    const int i = (int) (idx / vdim), j = (int) (idx % vdim), sw = vdim + 1;
    float run = (word & CM_FRESH) ? 0.0f : state[((int64_t) (word & ~CM_FRESH) * heads + h) * per + idx];
    for (int p0 = 0; p0 < nsub; p0 += 8) {
        float lp[8], tp[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float * blk = scratch + ((int64_t) (sub0 + p0 + u) * heads + h) * dim * sw + (int64_t) i * sw;
            const bool more = p0 + u < nsub - 1;
            lp[u] = more ? blk[j] : 0.0f; tp[u] = more ? blk[vdim] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (p0 + u < nsub) {
                scratch[((int64_t) (sub0 + p0 + u) * heads + h) * dim * sw + (int64_t) i * sw + j] = run;
                run = fmaf(tp[u], run, lp[u]);
            }
    }
}

// ---- long passes on the fp32 matrix cores -----------------------------------------------------------------------------------------------------------------------
// What bounds the walks above: a token's chain (two dependent sums over the key, then the state) at one column per R lanes, and for the delta rule a dim x dim transition matrix per piece, built by as many extra
// columns and chained by a scan of its own.  Written for a piece of 32 tokens at a time, with G_t the decays' product from the piece's start (v_mfma_f32_16x16x4_f32 throughout):
//   (I + A) U = beta (V - W S_in),  W_t = G_t k_t,  A[t][j] = beta_t sum_i k_t k_j (g_{j+1} .. g_t)_i for j < t      (bonus rule: U = V)
//   O = Q' S_in + P U,  Q'_t = G_t q_t,  P[t][j] = sum_i q_t k_j (g_{j+1} .. g_t)_i for j <= t                     (bonus rule: products up to t - 1, the bonus on the diagonal)
//   S_out = G_32 S_in + K' U,  K'_j = k_j (g_{j+1} .. g_32)
//   k_channel_pieces  per (head, piece), side by side: everything that does not know S_in, T = (I + A)^-1 applied to beta V and beta W.  Decays are products of factors only, never quotients: two tokens' decays meet at
//                     the border between them - of the piece's two tiles of 16, or of two halves of a square inside one, down to single tokens (a decay of 1e-30 per token is as good as any other).  Unit keys and
//                     beta <= 1 bound T's entries by 1; keys as they come (qk_unit = 0) of the delta rule stay with the walks.  Bound by a workgroup's run through its phases: of 18 us (delta rule, 128 x 128) loads and
//                     the search for its run take 4, the decays' logarithms 4, the squares 3.5.  A column's walk down the tile with eight threads took 8, the loads one after the other 7: 25 us with both
//   k_channel_walk    per (head, 16 value columns, run): takes the run's pieces in order, the state in the registers of four waves (a quarter of the rows each) - a product's result is laid out as the next one's
//                     operand; the waves' parts of T beta (V - W S_in) meet in LDS.  Helping waves bring the pieces through LDS, two ahead in registers, add up and write the outputs: one barrier a piece.  Of a
//                     piece's 3100 clocks (delta rule, 128 x 128) 1630 are products, the rest the exchange and waits for LDS, and the 54 KB that a workgroup loads per piece take nearly as long.  One wave with the
//                     whole state, loads and all: 10000.  An infinity or a NaN in a piece would meet zeros of tokens before it: such a piece is walked token by token
// 333 tokens of one sequence, pieces + walk, us: delta rule, 16 heads of 128 x 128: 82 with those, 39 now (walked token by token: 2 x 271 + scan 331); bonus rule, 32 heads of 64 x 64: 42, 24 (2 x 129 + scan 22).
// 2048 tokens, delta rule, 32 heads: 466, 200
#define CP_TB 32
#define CP_PIECE_THREADS 512
typedef float cm_f32x4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ cm_f32x4 cm_mfma(float a, float b, cm_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
static __device__ __forceinline__ cm_f32x4 cm_mfma4(cm_f32x4 a, cm_f32x4 b, cm_f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; i++) c = cm_mfma(a[i], b[i], c);
    return c;
}
// a piece's block in scratch, in floats: operands as the lanes hold them, [tile][lane][4]:  Q' [2][dim / 16], K' [dim / 16][2], -T beta W [2][dim / 16], P [3], G_32 [dim], a flag, U: T beta V (bonus rule: V) [2][vdim / 16]
// (flagged: q, k, g as rows [32][dim] in the first three places, beta [32] and the scalar of the token's own write [32] in P's)
struct cp_layout { int q, k, w, p, g, flag, u, total; };
static __host__ __device__ __forceinline__ cp_layout cp_of(int dim, int vdim) {
    cp_layout l;
    l.q = 0; l.k = CP_TB * dim; l.w = 2 * CP_TB * dim; l.p = 3 * CP_TB * dim; l.g = l.p + 768; l.flag = l.g + dim; l.u = l.flag + 4; l.total = l.u + CP_TB * vdim;
    return l;
}
template <int DI, int RULE>
__global__ void __launch_bounds__(CP_PIECE_THREADS) k_channel_pieces(const float * __restrict__ q, int64_t qs, const float * __restrict__ k, int64_t ks, const float * __restrict__ v, int64_t vs, const float * __restrict__ draw, int64_t ds,
                                                        int decay_mode, const float * __restrict__ dbias, const float * __restrict__ a_log, const float * __restrict__ braw, int64_t bs, const float * __restrict__ bonus,
                                                        int qk_unit, float q_mult, int heads, int hpg, int vdim, const int32_t * __restrict__ rec, int n_tok, float * __restrict__ scratch, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int DIM = 16 * DI, PITCH = DIM + 4, TH = CP_PIECE_THREADS, NW = TH / 64, PER = CP_TB * DIM / TH;
    __shared__ __attribute__((aligned(16))) float qt[CP_TB * PITCH], kt[CP_TB * PITCH], gt[CP_TB * PITCH], Am[CP_TB][36], Pm[CP_TB][36], Tm[CP_TB][36], whole[2][DIM], ones[DIM];
    __shared__ float beta[CP_TB], dot[CP_TB];
    __shared__ int seg[3], bnd[CR_MAXRUNS], sorted[CR_MAXRUNS], nbnd;
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4, nvt = vdim / 16;
    // every load of the piece on its way before the first is waited for, and ahead of the search for the runs: for the piece that a pass of one run has here (another one's are loaded behind the search)
    float qv[PER], kv[PER], dv[PER], bv = 0.0f;
    cm_f32x4 x0[2];                                                   // the values of the wave's first tile, as the product over them takes them
    auto values = [&](cm_f32x4 * x, int vt, int first, int last) {
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
            for (int r = 0; r < 4; r++) x[jt][r] = v[(int64_t) min(first + 16 * jt + 4 * g + r, last) * vs + (int64_t) h * vdim + 16 * vt + n];
    };
    auto fetch = [&](int first, int last) {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int idx = tid + u * TH, i = idx % DIM;
            const int64_t tok = min(first + idx / DIM, last);
            qv[u] = q[tok * qs + (int64_t) (h / hpg) * DIM + i]; kv[u] = k[tok * ks + (int64_t) (h / hpg) * DIM + i]; dv[u] = draw[tok * ds + (int64_t) h * DIM + i];
        }
        values(x0, min(wave, nvt - 1), first, last);
        if (tid < CP_TB && braw) bv = braw[(int64_t) min(first + tid, last) * bs + h];
    };
    const int mark = tid < n_tok ? cr_mark(rec, tid) : 0;
    const int guess = min((int) blockIdx.y * CP_TB, n_tok - 1);
    fetch(guess, n_tok - 1);
    const float ah = decay_mode == 2 ? expf(a_log[h]) : 0.0f, db = decay_mode != 0 && dbias ? dbias[h * DIM + tid % DIM] : 0.0f;      // (TH is a multiple of DIM: one channel per thread)
    const int n_runs = cr_runs(rec, n_tok, bnd, sorted, &nbnd, mark);
    if (tid == 0) {
        int ord = 0;
        seg[1] = 0;
        for (int r = 0; r < n_runs; r++) {
            const int t = sorted[r], e = r + 1 < n_runs ? sorted[r + 1] : n_tok, nsub = (e - t + CP_TB - 1) / CP_TB, pc = (int) blockIdx.y - ord;
            if (pc < nsub) { seg[0] = t + pc * CP_TB; seg[1] = min(CP_TB, e - seg[0]); seg[2] = rec[t]; break; }
            ord += nsub;
        }
    }
    for (int idx = tid; idx < CP_TB * 36; idx += TH) { (&Am[0][0])[idx] = 0.0f; (&Pm[0][0])[idx] = 0.0f; (&Tm[0][0])[idx] = 0.0f; }
    if (tid < DIM) ones[tid] = 1.0f;
    __syncthreads();
    const int first = seg[0], len = seg[1];
    if (len == 0 || seg[2] < 0) return;
    if (pi_abort_late(gone, abort_w)) return;
    const int last = first + len - 1;
    if (first != guess) fetch(first, last);
    const cp_layout L = cp_of(DIM, vdim);
    float * blk = scratch + ((int64_t) blockIdx.y * heads + h) * L.total;
    uint32_t big = 0;
    auto seen = [&](float x) { big = max(big, __float_as_uint(x) & 0x7fffffffu); };
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int idx = tid + u * TH, t = idx / DIM, i = idx % DIM;
        if (t >= len) { qv[u] = 0.0f; kv[u] = 0.0f; }
        qt[t * PITCH + i] = qv[u]; kt[t * PITCH + i] = kv[u]; gt[t * PITCH + i] = dv[u];
        seen(qv[u]); seen(kv[u]);
    }
#pragma unroll 1
    for (int u = 0; u < PER; u++) {                                    // (not unrolled, like the squares below: a workgroup runs through the code once, and what it runs through has to be fetched)
        const int t = (tid + u * TH) / DIM;
        float * at = gt + t * PITCH + tid % DIM, d = *at;
        if (decay_mode == 1) d = expf(-expf(d + db));
        else if (decay_mode == 2) d = expf(-ah * cm_softplus(d + db));
        if (t >= len) d = 1.0f;
        *at = d;
        seen(d);
    }
    if (tid < CP_TB) { bv = tid >= len ? 0.0f : braw ? cm_sigmoid(bv) : 1.0f; beta[tid] = bv; seen(bv); }
#pragma unroll
    for (int i = 0; i < 8; i++) {                                      // (behind the piece's end there may be another run's values: the products take the last one of this)
        if (first + 16 * (i >> 2) + 4 * g + (i & 3) > last) x0[i >> 2][i & 3] = 0.0f;
        seen(x0[i >> 2][i & 3]);
    }
    for (int vt = wave + NW; vt < nvt; vt += NW) {
        cm_f32x4 x[2];
        values(x, vt, first, last);
#pragma unroll
        for (int i = 0; i < 8; i++) seen(x[i >> 2][i & 3]);
    }
    const bool odd = __syncthreads_or(big >= 0x7f800000u);
    {   // unit vectors, and the scalar of the token's own write: sixteen lanes per token
        const int t = tid >> 4;
        float * qr = qt + t * PITCH + n, * kr = kt + t * PITCH + n, y[DI], z[DI], iq = q_mult, ik = 1.0f, d = 0.0f;
#pragma unroll
        for (int i = 0; i < DI; i++) { y[i] = qr[16 * i]; z[i] = kr[16 * i]; }
        if (qk_unit) {
            float sq = 0.0f, sk = 0.0f;
#pragma unroll
            for (int i = 0; i < DI; i++) { sq = fmaf(y[i], y[i], sq); sk = fmaf(z[i], z[i], sk); }
            iq = q_mult / sqrtf(pi_lanes_sum<16>(sq) + 1e-6f); ik = 1.0f / sqrtf(pi_lanes_sum<16>(sk) + 1e-6f);
        }
#pragma unroll
        for (int i = 0; i < DI; i++) {
            y[i] *= iq; z[i] *= ik;
            if (qk_unit || q_mult != 1.0f) { qr[16 * i] = y[i]; kr[16 * i] = z[i]; }
            d = fmaf(RULE == 1 && bonus ? y[i] * bonus[h * DIM + n + 16 * i] : y[i], z[i], d);
        }
        d = pi_lanes_sum<16>(d);
        if (n == 0) dot[t] = d;
    }
    __syncthreads();
    if (tid == 0) *(int *) (blk + L.flag) = odd ? 1 : 0;
    if (odd) {
        for (int idx = tid; idx < CP_TB * DIM; idx += TH) { const int at = idx / DIM * PITCH + idx % DIM; blk[L.q + idx] = qt[at]; blk[L.k + idx] = kt[at]; blk[L.w + idx] = gt[at]; }
        if (tid < CP_TB) { blk[L.p + tid] = beta[tid]; blk[L.p + CP_TB + tid] = dot[tid]; }
        return;
    }
    {   // the tiles on the diagonal, cut into squares below it whose sides are 8, 4, 2 and 1 (a wave for each size and tile): a square's rows and columns are decayed to the border between them, its rows from there,
        // its columns up to there - a token is one or the other, so one product of its decays serves both.  Of a 16 x 16 product the squares of its size are kept
        const int t0 = wave >> 2 << 4, hs = 8 >> (wave & 3), top = (n & -2 * hs) + hs;
        const bool row = (n & hs) != 0;
        const int from = row ? top : n + 1, to = row ? (RULE == 1 ? n : n + 1) : top;       // the decays [from, to) of the tile (bonus rule: a row takes the state ahead of its own decay)
        const float * qr = qt + (t0 + n) * PITCH + 4 * g, * kr = kt + (t0 + n) * PITCH + 4 * g;
        cm_f32x4 a = { 0.0f, 0.0f, 0.0f, 0.0f }, p = { 0.0f, 0.0f, 0.0f, 0.0f };
        auto square = [&](auto most) {
            const float * gr[decltype(most)::value];
#pragma unroll
            for (int u = 0; u < decltype(most)::value; u++) gr[u] = (from + u < to ? gt + (t0 + from + u) * PITCH : ones) + 4 * g;
#pragma unroll 1
            for (int s = 0; s < DI; s++) {
                cm_f32x4 f = *(const cm_f32x4 *) (gr[0] + 16 * s);
#pragma unroll
                for (int u = 1; u < decltype(most)::value; u++) f *= *(const cm_f32x4 *) (gr[u] + 16 * s);
                const cm_f32x4 kf = *(const cm_f32x4 *) (kr + 16 * s) * f, qf = *(const cm_f32x4 *) (qr + 16 * s) * f;
                if (RULE == 0) a = cm_mfma4(kf, kf, a);
                p = cm_mfma4(qf, kf, p);
            }
        };
        if (hs == 8) square(std::integral_constant<int, 8>{});
        else if (hs == 4) square(std::integral_constant<int, 4>{});
        else if (hs == 2) square(std::integral_constant<int, 2>{});
        else square(std::integral_constant<int, 1>{});
#pragma unroll
        for (int r = 0; r < 4; r++) {                                  // (row 4 g + r, column n)
            const int t = 4 * g + r;
            if ((t & hs) && !row && (t & -2 * hs) == (n & -2 * hs)) { if (RULE == 0) Am[t0 + t][t0 + n] = a[r]; Pm[t0 + t][t0 + n] = p[r]; }
        }
        if (hs == 1 && g == 0) Pm[t0 + n][t0 + n] = dot[t0 + n];
    }
    __syncthreads();
    if (tid < 2 * DIM) {                                               // a thread per channel and tile: gt <- k to the tile's start, qt <- q to it (both decayed), kt <- k to the tile's end
        const int i = tid % DIM, t0 = tid / DIM << 4;
        float gv[16], w = 1.0f;
#pragma unroll
        for (int t = 0; t < 16; t++) gv[t] = gt[(t0 + t) * PITCH + i];
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int at = (t0 + t) * PITCH + i;
            if (RULE == 1) qt[at] *= w;
            w *= gv[t];
            if (RULE == 0) { qt[at] *= w; gt[at] = kt[at] * w; }
        }
        whole[t0 >> 4][i] = w;
        w = 1.0f;
#pragma unroll
        for (int t = 15; t >= 0; t--) { kt[(t0 + t) * PITCH + i] *= w; w *= gv[t]; }
    }
    __syncthreads();
    if (wave < 2 && (RULE == 0 || wave == 1)) {                       // the tile below them
        const float * rows = wave == 0 ? gt : qt;
        cm_f32x4 a = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int s = 0; s < DI; s++) a = cm_mfma4(*(const cm_f32x4 *) &rows[(16 + n) * PITCH + 16 * s + 4 * g], *(const cm_f32x4 *) &kt[n * PITCH + 16 * s + 4 * g], a);
#pragma unroll
        for (int r = 0; r < 4; r++) (wave == 0 ? Am : Pm)[16 + 4 * g + r][n] = a[r];
    }
    __syncthreads();
    if constexpr (RULE == 1) {
        for (int vt = wave; vt < nvt; vt += NW) {
            if (vt != wave) values(x0, vt, first, last);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) *(cm_f32x4 *) (blk + L.u + ((mt * nvt + vt) * 64 + lane) * 4) = x0[mt];      // (behind the end: met by keys of zero)
        }
    }
    if constexpr (RULE == 0) {
        for (int idx = tid; idx < CP_TB * CP_TB; idx += TH) Am[idx >> 5][idx & 31] *= beta[idx >> 5];
        __syncthreads();
        if (tid < 32) {                                                // T on the diagonal: a thread per column, forward substitution
            const int t0 = tid & 16, c = tid & 15;
            float x[16];
#pragma unroll
            for (int t = 0; t < 16; t++) {
                float y = t == c ? 1.0f : 0.0f;
#pragma unroll
                for (int j = 0; j < t; j++) y = fmaf(-Am[t0 + t][t0 + j], x[j], y);
                x[t] = y;
                Tm[t0 + t][t0 + c] = y;
            }
        }
        __syncthreads();
        const int t = tid >> 4 & 15, c = tid & 15;                     // below it: -T_11 (A_10 T_00)
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; j++) m = fmaf(Am[16 + t][j], Tm[j][c], m);
        if (tid < 256) Am[t][16 + c] = m;
        __syncthreads();
        m = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; j++) m = fmaf(Tm[16 + t][16 + j], Am[j][16 + c], m);
        if (tid < 256) Tm[16 + t][c] = -m;
        __syncthreads();
        for (int s = wave; s < DI; s += NW) {                           // -(T beta W), transposed: a lane's four rows are four channels of one token
            const int i = 16 * s + n;
            const float w0 = whole[0][i];
            cm_f32x4 a[2] = { { 0.0f, 0.0f, 0.0f, 0.0f }, { 0.0f, 0.0f, 0.0f, 0.0f } };
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                cm_f32x4 w;
#pragma unroll
                for (int r = 0; r < 4; r++) { const int j = 16 * jt + 4 * g + r; w[r] = -beta[j] * gt[j * PITCH + i] * (jt ? w0 : 1.0f); }
#pragma unroll
                for (int mt = jt; mt < 2; mt++) a[mt] = cm_mfma4(w, *(const cm_f32x4 *) &Tm[16 * mt + n][16 * jt + 4 * g], a[mt]);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++) *(cm_f32x4 *) (blk + L.w + ((mt * DI + s) * 64 + lane) * 4) = a[mt];
        }
        for (int vt = wave; vt < nvt; vt += NW) {
            if (vt != wave) values(x0, vt, first, last);
            cm_f32x4 a[2] = { { 0.0f, 0.0f, 0.0f, 0.0f }, { 0.0f, 0.0f, 0.0f, 0.0f } };
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                cm_f32x4 x;
#pragma unroll
                for (int r = 0; r < 4; r++) { const int j = 16 * jt + 4 * g + r; x[r] = beta[j] * x0[jt][r]; }       // (beta = 0 behind the end)
#pragma unroll
                for (int mt = jt; mt < 2; mt++) a[mt] = cm_mfma4(*(const cm_f32x4 *) &Tm[16 * mt + n][16 * jt + 4 * g], x, a[mt]);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++) *(cm_f32x4 *) (blk + L.u + ((mt * nvt + vt) * 64 + lane) * 4) = a[mt];
        }
    }
    for (int idx = tid; idx < 2 * DI * 64; idx += TH) {
        const int tile = idx >> 6, ln = idx & 15, lg = idx >> 4 & 3;
        const int t = 16 * (tile / DI) + ln, i = 16 * (tile % DI) + 4 * lg;
        cm_f32x4 x = *(const cm_f32x4 *) &qt[t * PITCH + i];
        if (tile / DI) x *= *(const cm_f32x4 *) &whole[0][i];
        *(cm_f32x4 *) (blk + L.q + idx * 4) = x;
        const int c = 16 * (tile >> 1) + ln, j = 16 * (tile & 1) + 4 * lg;
        cm_f32x4 y;
#pragma unroll
        for (int r = 0; r < 4; r++) y[r] = kt[(j + r) * PITCH + c] * (tile & 1 ? 1.0f : whole[1][c]);
        *(cm_f32x4 *) (blk + L.k + idx * 4) = y;
    }
    if (wave < 3) *(cm_f32x4 *) (blk + L.p + tid * 4) = *(const cm_f32x4 *) &Pm[(wave ? 16 : 0) + n][(wave == 2 ? 16 : 0) + 4 * g];
    for (int i = tid; i < DIM; i += TH) blk[L.g + i] = whole[0][i] * whole[1][i];
}

// the walk's waves: CP_WAVES walk, each with DI / CP_WAVES sixteens of the state's rows, and CP_HELP help.  Helpers of the delta rule: 8 (its pieces are half as large again; 4: 40.1 us for pieces and walk of 16 heads of
// 128 x 128, 333 tokens; 8: 39.3); of the bonus rule 4 (one sequence of 333 tokens, 32 heads of 64 x 64: 24.1, with 8 22.4; eight of 42: 27.4, with 8 32.9, where workgroups come and go)
#define CP_WAVES(DI) ((DI) < 4 ? (DI) : 4)
#define CP_HELP(RULE) ((RULE) == 0 ? 8 : 4)
// memory accesses stay on their side (loads of two pieces mixed would have the wait for the first wait for both)
static __device__ __forceinline__ void cp_keep_order() { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }
template <int DI, int RULE> struct cp_stage {                          // a piece in LDS, tiles of 256 floats: Q', K', -T beta W (delta rule), P and what follows it, U of the value columns
    static constexpr int NT = (RULE == 0 ? 6 : 4) * DI, P = NT * 256, G = P + 768, FLAG = G + 16 * DI, U = P + 1024, TILES = NT + 6, FLOATS = TILES * 256;
    static constexpr int NW = CP_WAVES(DI), PARTS = NW * 512, OUT = NW * 512, LDS = 4 * (2 * FLOATS + (RULE == 0 ? 2 * PARTS : 0) + 2 * OUT);
};
template <int DI, int RULE>
__global__ void __launch_bounds__(64 * (CP_WAVES(DI) + CP_HELP(RULE)), 1) k_channel_walk(const float * __restrict__ v, int64_t vs, int heads, int vdim, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok,
                                                                                   const float * __restrict__ scratch, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    typedef cp_stage<DI, RULE> ST;
    constexpr int DIM = 16 * DI, NW = ST::NW, MT = DI / NW, HELP = CP_HELP(RULE);
    extern __shared__ __attribute__((aligned(16))) float walk_lds[];
    __shared__ int bnd[CR_MAXRUNS], sorted[CR_MAXRUNS], nbnd;
    __shared__ float one[2][NW][2][16];
    float * const stage = walk_lds, * const op = stage + 2 * ST::FLOATS, * const us = op + 2 * ST::OUT;      // two buffers of each
    const int h = blockIdx.x, vt = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4, c = 16 * vt + n, m0 = wave * MT;
    const int n_runs = cr_runs(rec, n_tok, bnd, sorted, &nbnd);
    if ((int) blockIdx.z >= n_runs) return;
    int ord = 0;
    for (int r = 0; r < (int) blockIdx.z; r++) ord += ((r + 1 < n_runs ? sorted[r + 1] : n_tok) - sorted[r] + CP_TB - 1) / CP_TB;
    const int start = sorted[blockIdx.z], end = (int) blockIdx.z + 1 < n_runs ? sorted[blockIdx.z + 1] : n_tok, word = rec[start], np = (end - start + CP_TB - 1) / CP_TB;
    if (word < 0) return;
    if (pi_abort_late(gone, abort_w)) return;
    const cp_layout L = cp_of(DIM, vdim);
    const int nvt = vdim / 16;
    const float * blk0 = scratch + ((int64_t) ord * heads + h) * L.total;
    const int64_t step = (int64_t) heads * L.total;
    if (wave >= NW) {                                                  // a helper: pieces through LDS, two ahead in registers, and the outputs of the piece before
        const int hw = wave - NW, ht = tid - 64 * NW;
        constexpr int CH = (ST::TILES + HELP - 1) / HELP;
        int from[CH];                                                  // (the tail repeats the last tile)
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const int t = min(hw + HELP * j, ST::TILES - 1);
            from[j] = (t < 4 * DI || RULE == 0 && t < 6 * DI ? 256 * t : t < ST::NT + 4 ? L.p + 256 * (t - ST::NT) : L.u + ((t - ST::NT - 4) * nvt + vt) * 256) + 4 * lane;
        }
        cm_f32x4 A[CH], B[CH];
        auto load = [&](cm_f32x4 * x, int p) {
            const float * b = blk0 + min(p, np - 1) * step;
#pragma unroll
            for (int j = 0; j < CH; j++) x[j] = *(const cm_f32x4 *) (b + from[j]);
        };
        auto pass = [&](const cm_f32x4 * x, int p) {
            float * to = stage + (p & 1) * ST::FLOATS + 4 * lane;
#pragma unroll
            for (int j = 0; j < CH; j++) *(cm_f32x4 *) (to + min(hw + HELP * j, ST::TILES - 1) * 256) = x[j];
        };
        bool due = false;                                              // whether the piece before left outputs to be added
        auto put = [&](int p) {                                        // the waves' parts, added in their order
#pragma unroll
            for (int i = 0; i < 8 / HELP; i++) {                    // (row t, column ht & 15 of what the products left: 4 g + r = t & 15)
                const int t = (ht >> 4) + 4 * HELP * i, at = start + p * CP_TB + t;
                const float * o = op + (p & 1) * ST::OUT + (t >> 4) * 256 + (t >> 2 & 3) * 64 + (ht & 15) * 4 + (t & 3);
                float y = *o;
#pragma unroll
                for (int w = 1; w < NW; w++) y += o[w * 512];
                if (at < end) out[(int64_t) at * os + (int64_t) h * vdim + 16 * vt + (ht & 15)] = y;
            }
        };
        auto turn = [&](cm_f32x4 * x, int p) {                         // x: piece p + 1, and then p + 3
            const bool odd = __float_as_int(stage[(p & 1) * ST::FLOATS + ST::FLAG]) != 0;
            pass(x, p + 1);
            cp_keep_order();
            load(x, p + 3);
            cp_keep_order();
            if (odd) for (int t = 0; t < min(CP_TB, end - start - p * CP_TB); t++) __syncthreads();
            __syncthreads();
            if (due) put(p - 1);
            due = !odd;
        };
        load(A, 0);
        pass(A, 0);
        cp_keep_order();
        load(B, 1);
        cp_keep_order();
        load(A, 2);
        cp_keep_order();
        __syncthreads();
        for (int p = 0; p < np; p += 2) {
            turn(B, p);
            if (p + 1 >= np) break;
            turn(A, p + 1);
        }
        __syncthreads();
        if (due) put(np - 1);
        return;
    }
    float * S_hbm = state + ((int64_t) (word & ~CM_FRESH) * heads + h) * DIM * vdim + c;
    cm_f32x4 S[MT];                                                   // rows 16 (m0 + m) + 4 g + r of column c: as a product leaves them, and as the next one takes them
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) S[m][r] = word & CM_FRESH ? 0.0f : S_hbm[(int64_t) (16 * (m0 + m) + 4 * g + r) * vdim];
    __builtin_amdgcn_s_setprio(1);
    __syncthreads();
    // a piece's operands are in registers when it begins: what its first products have read is read again behind the barrier, for the next piece, the rest behind its last products
    cm_f32x4 W[RULE == 0 ? 2 * MT : 1], Q[2 * MT], K[2 * MT], G[MT], V[2];
    float P[3][4 / NW];
    int flag;
    auto first = [&](int p) {
        const float * x = stage + (p & 1) * ST::FLOATS + 4 * lane;
        flag = __float_as_int(stage[(p & 1) * ST::FLOATS + ST::FLAG]);
        if constexpr (RULE == 0)
#pragma unroll
            for (int m = 0; m < 2; m++)
#pragma unroll
                for (int i = 0; i < MT; i++) W[m * MT + i] = *(const cm_f32x4 *) (x + (4 * DI + m * DI + m0 + i) * 256);
#pragma unroll
        for (int m = 0; m < 2; m++) V[m] = *(const cm_f32x4 *) (x + ST::U + m * 256);
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int i = 0; i < MT; i++) Q[m * MT + i] = *(const cm_f32x4 *) (x + (m * DI + m0 + i) * 256);
    };
    auto second = [&](int p) {
        const float * x = stage + (p & 1) * ST::FLOATS;
#pragma unroll
        for (int m = 0; m < MT; m++) G[m] = *(const cm_f32x4 *) (x + ST::G + 16 * (m0 + m) + 4 * g);
#pragma unroll
        for (int i = 0; i < 2 * MT; i++) K[i] = *(const cm_f32x4 *) (x + (2 * DI + 2 * m0 + i) * 256 + 4 * lane);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int e = 0; e < 4 / NW; e++) P[i][e] = x[ST::P + i * 256 + 4 * lane + wave + NW * e];
    };
    first(0); second(0);
    for (int p = 0; p < np; p++) {
        const bool odd = __builtin_amdgcn_readfirstlane(flag) != 0;
        cm_f32x4 U[2], O[2] = { { 0.0f, 0.0f, 0.0f, 0.0f }, { 0.0f, 0.0f, 0.0f, 0.0f } };
        if (odd) {                                                     // token by token
            const float * blk = blk0 + p * step;
            const int at = start + p * CP_TB, len = min(CP_TB, end - at);
            for (int t = 0; t < len; t++) {
                cm_f32x4 kv[MT];
                float a = 0.0f, o = 0.0f;
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const int i = t * DIM + 16 * (m0 + m) + 4 * g;
                    kv[m] = *(const cm_f32x4 *) (blk + L.k + i);
                    const cm_f32x4 qv = *(const cm_f32x4 *) (blk + L.q + i), gv = *(const cm_f32x4 *) (blk + L.w + i);
                    if (RULE == 0) S[m] *= gv;
#pragma unroll
                    for (int r = 0; r < 4; r++) { a = fmaf(S[m][r], kv[m][r], a); o = fmaf(S[m][r], qv[r], o); }
                    if (RULE == 1) S[m] *= gv;
                }
                a += __shfl_xor(a, 16, 64); a += __shfl_xor(a, 32, 64); o += __shfl_xor(o, 16, 64); o += __shfl_xor(o, 32, 64);
                if (g == 0) { one[t & 1][wave][0][n] = a; one[t & 1][wave][1][n] = o; }
                __syncthreads();
                a = one[t & 1][0][0][n]; o = one[t & 1][0][1][n];
#pragma unroll
                for (int w = 1; w < NW; w++) { a += one[t & 1][w][0][n]; o += one[t & 1][w][1][n]; }
                const float y = v[(int64_t) (at + t) * vs + (int64_t) h * vdim + c], u = RULE == 0 ? blk[L.p + t] * (y - a) : y;
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int r = 0; r < 4; r++) S[m][r] = fmaf(kv[m][r], u, S[m][r]);
                if (tid < 16) out[(int64_t) (at + t) * os + (int64_t) h * vdim + c] = fmaf(u, blk[L.p + CP_TB + t], o);
            }
        } else {
            U[0] = V[0]; U[1] = V[1];
            if constexpr (RULE == 0) {
                if (wave) U[0] = U[1] = cm_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };       // (T beta V goes in once)
#pragma unroll
                for (int s = 0; s < MT; s++)
#pragma unroll
                    for (int i = 0; i < 4; i++) { U[0] = cm_mfma(W[s][i], S[s][i], U[0]); U[1] = cm_mfma(W[MT + s][i], S[s][i], U[1]); }
                float * const mine = us + (p & 1) * ST::PARTS + wave * 512 + lane * 4;
                *(cm_f32x4 *) mine = U[0];
                *(cm_f32x4 *) (mine + 256) = U[1];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2 * MT; i++) { O[0] = cm_mfma(Q[i >> 2][i & 3], S[i >> 2][i & 3], O[0]); O[1] = cm_mfma(Q[MT + (i >> 2)][i & 3], S[i >> 2][i & 3], O[1]); }
        }
        __syncthreads();                                               // the waves' parts of U are there, and the next piece; this one's buffer is free
        cm_f32x4 part[RULE == 0 ? 2 * NW : 1];
        if constexpr (RULE == 0)
#pragma unroll
            for (int i = 0; i < 2 * NW; i++) part[i] = *(const cm_f32x4 *) (us + (p & 1) * ST::PARTS + i * 256 + lane * 4);
        __builtin_amdgcn_sched_barrier(0);
        if (!odd) {                                                    // (the second half of Q' S: the parts arrive meanwhile)
#pragma unroll
            for (int i = 2 * MT; i < 4 * MT; i++) { O[0] = cm_mfma(Q[i >> 2][i & 3], S[i >> 2][i & 3], O[0]); O[1] = cm_mfma(Q[MT + (i >> 2)][i & 3], S[i >> 2][i & 3], O[1]); }
#pragma unroll
            for (int m = 0; m < MT; m++) S[m] *= G[m];
        }
        __builtin_amdgcn_sched_barrier(0);
        first(p + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (!odd) {
            if constexpr (RULE == 0) {
                U[0] = part[0]; U[1] = part[1];
#pragma unroll
                for (int w = 1; w < NW; w++) { U[0] += part[2 * w]; U[1] += part[2 * w + 1]; }
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int m = 0; m < MT; m++) S[m] = cm_mfma(K[2 * m][i], U[0][i], S[m]);
#pragma unroll
            for (int e = 0; e < 4 / NW; e++) {                        // P U: a part of the inner index per wave
                const int i = wave + NW * e;
                const float u0 = i == 0 ? U[0][0] : i == 1 ? U[0][1] : i == 2 ? U[0][2] : U[0][3], u1 = i == 0 ? U[1][0] : i == 1 ? U[1][1] : i == 2 ? U[1][2] : U[1][3];
                O[0] = cm_mfma(P[0][e], u0, O[0]);
                O[1] = cm_mfma(P[1][e], u0, O[1]);
                O[1] = cm_mfma(P[2][e], u1, O[1]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int m = 0; m < MT; m++) S[m] = cm_mfma(K[2 * m + 1][i], U[1][i], S[m]);
            __builtin_amdgcn_sched_barrier(0);
            float * o = op + (p & 1) * ST::OUT + wave * 512 + lane * 4;
            *(cm_f32x4 *) o = O[0];
            *(cm_f32x4 *) (o + 256) = O[1];
        }
        second(p + 1);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) S_hbm[(int64_t) (16 * (m0 + m) + 4 * g + r) * vdim] = S[m][r];
}

#define CR_LDS_MAX (150 * 1024)
template <int DPT, int RULE> static int cr_reserve_one() { PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_channel_recurrence<DPT, RULE>, hipFuncAttributeMaxDynamicSharedMemorySize, CR_LDS_MAX)); return 0; }
template <int DI, int RULE> static int cp_reserve_one() { PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_channel_walk<DI, RULE>, hipFuncAttributeMaxDynamicSharedMemorySize, cp_stage<DI, RULE>::LDS)); return 0; }
extern "C" int pi_op_channel_recurrence_reserve(void) {
    static bool done = false;
    if (done) return 0;
    if (cr_reserve_one<8, 0>() || cr_reserve_one<16, 0>() || cr_reserve_one<32, 0>() || cr_reserve_one<8, 1>() || cr_reserve_one<16, 1>() || cr_reserve_one<32, 1>()) return -1;
    if (cp_reserve_one<2, 0>() || cp_reserve_one<4, 0>() || cp_reserve_one<8, 0>() || cp_reserve_one<2, 1>() || cp_reserve_one<4, 1>() || cp_reserve_one<8, 1>()) return -1;
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_channel_state_scan<8>, hipFuncAttributeMaxDynamicSharedMemorySize, CR_LDS_MAX));
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_channel_state_scan<16>, hipFuncAttributeMaxDynamicSharedMemorySize, CR_LDS_MAX));
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_channel_state_scan<32>, hipFuncAttributeMaxDynamicSharedMemorySize, CR_LDS_MAX));
    done = true;
    return 0;
}
static int cr_max_pieces(int n_tok, int max_segments, int piece = CR_TB) { return n_tok / piece + std::min(n_tok, std::max(1, max_segments)) + 1; }
// whether the matrix cores take a pass (of pieces), and the floats of scratch it needs for them
static bool cp_takes(int dim, int vdim) { return (dim == 32 || dim == 64 || dim == 128) && vdim % 16 == 0; }
static size_t cp_floats(int heads, int dim, int vdim, int n_tok, int max_segments) { return (size_t) cr_max_pieces(n_tok, max_segments) * heads * cp_of(dim, vdim).total; }
// floats of scratch that the walks need
static size_t cr_floats(int heads, int dim, int vdim, int n_tok, int max_segments) { return (n_tok <= CR_TB || dim > CR_SCAN_MAXDIM) ? 0 : (size_t) cr_max_pieces(n_tok, max_segments) * heads * dim * (vdim + dim); }
// passes of more than 32 tokens cut the runs into pieces that run side by side: floats of scratch they need (0: such a pass is walked in one piece per run)
extern "C" size_t pi_op_channel_recurrence_scratch_floats(int heads, int dim, int vdim, int n_tok, int max_segments) {      // (sized for the delta rule, which needs more)
    const size_t need = cr_floats(heads, dim, vdim, n_tok, max_segments);
    return need > 0 && cp_takes(dim, vdim) ? std::max(need, cp_floats(heads, dim, vdim, n_tok, max_segments)) : need;
}
extern "C" int pi_op_channel_recurrence(int rule, const float * q, int64_t q_stride, const float * k, int64_t k_stride, const float * v, int64_t v_stride, const float * decay_raw, int64_t decay_stride, int decay_mode,
                                        const float * decay_bias_dev, const float * a_log_dev, const float * beta_raw, int64_t beta_stride, const float * bonus_dev, int qk_unit, float q_mult,
                                        int heads, int qk_heads, int dim, int vdim, float * state_dev, const int32_t * rec_dev, int n_tok, int max_segments, float * scratch_dev, size_t scratch_floats,
                                        float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0) return 0;
    if (rule != PI_RULE_DELTA && rule != PI_RULE_BONUS) { pi_set_error("pi_op_channel_recurrence: rule %d is unknown", rule); return -1; }
    if (qk_heads < 1 || heads % qk_heads) { pi_set_error("pi_op_channel_recurrence: %d heads do not divide over %d query / key heads", heads, qk_heads); return -1; }
    if (dim <= 0 || vdim <= 0 || heads <= 0 || dim > 1024) { pi_set_error("pi_op_channel_recurrence: head sizes %d x %d outside the kernel's range (key width <= 1024)", dim, vdim); return -1; }
    if (decay_mode < 0 || decay_mode > 2 || (decay_mode == 2 && !a_log_dev) || !decay_raw) { pi_set_error("pi_op_channel_recurrence: decays (mode %d) are missing a part", decay_mode); return -1; }
    if (max_segments > CR_MAXRUNS) { pi_set_error("pi_op_channel_recurrence: at most %d sequences in a pass", CR_MAXRUNS); return -1; }
    const int dpt = dim <= 8 ? 8 : dim <= 16 ? 16 : 32;                // state values a thread keeps in registers
    int R = 1; while (R * dpt < dim) R *= 2;
    const size_t need = cr_floats(heads, dim, vdim, n_tok, max_segments);
    const bool pieces = need > 0 && scratch_dev && scratch_floats >= need;       // (without scratch a long pass is still right, only serial)
    const int runs = std::max(1, std::min(n_tok, max_segments));
    const double bytes = 4.0 * n_tok * heads * (3.0 * dim + 2.0 * vdim) + 8.0 * heads * dim * vdim;
    hipStream_t s = (hipStream_t) stream;
    const int nta = std::min(n_tok, PI_KT_MAXNT - 1);
    // delta rule: the scan's work grows with the number of pieces, so pieces of 64 tokens where that still leaves a workgroup per compute unit; bonus rule (a scan of no weight): 32
    const int cols0 = std::min(256, (vdim * R + 63) / 64 * 64) / R;
    const int piece = (rule == PI_RULE_DELTA && (int64_t) heads * ((vdim + cols0 - 1) / cols0) * (n_tok / CR_PIECE) >= 256) ? CR_PIECE : CR_TB;
    auto launch = [&](int mode) -> int {
        const int ncol = mode == 1 ? vdim + (rule == PI_RULE_DELTA ? dim : 1) : vdim;
        const int threads = std::min(256, (ncol * R + 63) / 64 * 64);
        const int cols = threads / R;
        const dim3 grid((unsigned) heads, (unsigned) ((ncol + cols - 1) / cols), (unsigned) (mode ? cr_max_pieces(n_tok, max_segments, piece) : runs));
        int tb = CR_TB;                                                 // tokens staged at a time: as many as the LDS takes
        auto lds_of = [&](int n) { return ((size_t) 3 * n * R * (dpt + 4) + (size_t) n * cols) * sizeof(float); };
        while (tb > 1 && lds_of(tb) > CR_LDS_MAX) tb >>= 1;
        const size_t lds = lds_of(tb);
        if (lds > CR_LDS_MAX) { pi_set_error("pi_op_channel_recurrence: a key width of %d needs %zu bytes of LDS (at most %d)", dim, lds, CR_LDS_MAX); return -1; }
        if (lds > 48 * 1024 && pi_op_channel_recurrence_reserve() != 0) return -1;
#define CR_GO(D, RL) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_channel_recurrence<D, RL>), grid, dim3(threads), lds, s, q, q_stride, k, k_stride, v, v_stride, decay_raw, decay_stride, decay_mode, decay_bias_dev, a_log_dev, \
                                  beta_raw, beta_stride, bonus_dev, qk_unit, q_mult, heads, heads / qk_heads, dim, vdim, R, state_dev, rec_dev, n_tok, mode, tb, piece, scratch_dev, out, out_stride, pi_abort_word())
        if (rule == PI_RULE_DELTA) { if (dpt == 8) CR_GO(8, 0); else if (dpt == 16) CR_GO(16, 0); else CR_GO(32, 0); }
        else                       { if (dpt == 8) CR_GO(8, 1); else if (dpt == 16) CR_GO(16, 1); else CR_GO(32, 1); }
#undef CR_GO
        PI_CHECK_LAUNCH(); return 0;
    };
    // every pass that is not cut into pieces, of key widths and columns that the step kernel's threads share out whole (its figures: both kernels at every number of tokens)
    if (n_tok <= CS_TOKENS && (dim == 32 || dim == 64 || dim == 128) && vdim % 32 == 0 && v_stride % 4 == 0 && out_stride % 4 == 0 && (((uintptr_t) v | (uintptr_t) out | (uintptr_t) state_dev) & 15) == 0) {
        const dim3 grid((unsigned) heads, (unsigned) (vdim / 32), (unsigned) runs);
#define CS_GO(NR, RL, NW) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, (k_channel_step<NR, RL, NW>), grid, dim3(64 * NW), 0, s, q, q_stride, k, k_stride, v, v_stride, decay_raw, decay_stride, decay_mode, decay_bias_dev, a_log_dev, \
                                   beta_raw, beta_stride, bonus_dev, qk_unit, q_mult, heads, heads / qk_heads, vdim, state_dev, rec_dev, n_tok, out, out_stride, pi_abort_word())
        if (rule == PI_RULE_DELTA) { if (dim == 32) CS_GO(4, 0, 1); else if (dim == 64) CS_GO(2, 0, 4); else CS_GO(4, 0, 4); }
        else                       { if (dim == 32) CS_GO(4, 1, 1); else if (dim == 64) CS_GO(2, 1, 4); else CS_GO(4, 1, 4); }
#undef CS_GO
        PI_CHECK_LAUNCH(); return 0;
    }
    if (!pieces) return launch(0);
    if (cp_takes(dim, vdim) && (rule == PI_RULE_BONUS || qk_unit) && scratch_floats >= cp_floats(heads, dim, vdim, n_tok, max_segments) && ((uintptr_t) scratch_dev & 15) == 0) {
        const dim3 pg((unsigned) heads, (unsigned) cr_max_pieces(n_tok, max_segments, CP_TB)), wg((unsigned) heads, (unsigned) (vdim / 16), (unsigned) runs);
        if (pi_op_channel_recurrence_reserve() != 0) return -1;
        const double blocks = 4.0 * pg.y * heads * cp_of(dim, vdim).total;
#define CP_GO(DI, RL) do { PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes + blocks, (k_channel_pieces<DI, RL>), pg, dim3(CP_PIECE_THREADS), 0, s, q, q_stride, k, k_stride, v, v_stride, decay_raw, decay_stride, decay_mode, decay_bias_dev, a_log_dev, \
                                        beta_raw, beta_stride, bonus_dev, qk_unit, q_mult, heads, heads / qk_heads, vdim, rec_dev, n_tok, scratch_dev, pi_abort_word()); \
                           PI_CHECK_LAUNCH(); \
                           PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes + blocks, (k_channel_walk<DI, RL>), wg, dim3(64 * (CP_WAVES(DI) + CP_HELP(RL))), (cp_stage<DI, RL>::LDS), s, v, v_stride, heads, vdim, state_dev, rec_dev, n_tok, scratch_dev, out, out_stride, pi_abort_word()); } while (0)
#define CP_RULE(RL) do { if (dim == 32) CP_GO(2, RL); else if (dim == 64) CP_GO(4, RL); else CP_GO(8, RL); } while (0)
        if (rule == PI_RULE_DELTA) CP_RULE(0); else CP_RULE(1);
#undef CP_RULE
#undef CP_GO
        PI_CHECK_LAUNCH(); return 0;
    }
    if (launch(1) != 0) return -1;
    const int n_pieces = cr_max_pieces(n_tok, max_segments, piece);
    if (rule == PI_RULE_BONUS) {
        PI_KT_LAUNCH(PI_KT_ATT, 0, nta, 12.0 * n_pieces * heads * dim * vdim, k_channel_state_scan_diag, dim3((unsigned) heads, (unsigned) (((int64_t) dim * vdim + 255) / 256), (unsigned) runs), dim3(256), 0, s,
                     heads, dim, vdim, piece, state_dev, rec_dev, n_tok, scratch_dev, pi_abort_word());
    } else {
        // columns per workgroup: as few as it takes to put a workgroup on every compute unit (each one re-reads the transition matrices, which the others' reads keep in L2)
        int sc = 32;
        while (sc > 8 && (int64_t) heads * ((vdim + sc - 1) / sc) < 256) sc >>= 1;           // (a pass usually carries one run, whatever the slots allow)
        const size_t scan_lds = ((size_t) dim * ((dim + 3) / 4 * 4 + 4) + (size_t) 2 * dim * sc + 8) * sizeof(float);
        if (scan_lds > 48 * 1024 && pi_op_channel_recurrence_reserve() != 0) return -1;
        const dim3 sgrid((unsigned) heads, (unsigned) ((vdim + sc - 1) / sc), (unsigned) runs);
        const double sbytes = 4.0 * n_pieces * heads * dim * (2.0 * vdim + dim);
#define CR_SCAN(C) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, sbytes, k_channel_state_scan<C>, sgrid, dim3(256), scan_lds, s, heads, dim, vdim, piece, state_dev, rec_dev, n_tok, scratch_dev, pi_abort_word())
        if (sc == 8) CR_SCAN(8); else if (sc == 16) CR_SCAN(16); else CR_SCAN(32);
#undef CR_SCAN
    }
    PI_CHECK_LAUNCH();
    return launch(2);
}

// ---- per-head RMS norm, weight, gate ------------------------------------------------------------------------------------------------------------------------------
// out[t][h][i] = y[t][h][i] / sqrt(mean_i(y[t][h]^2) + eps) * w[(w_per_head ? h * n : 0) + i] * act(gate[t][h][i]);  a wave per (token, head); out may be y
__global__ void __launch_bounds__(256) k_head_norm_gate(const float * __restrict__ y, int64_t ys, int heads, int n, const float * __restrict__ w, int w_per_head, const float * __restrict__ gate, int64_t gs, int gate_act,
                                                        float eps, float * __restrict__ out, int64_t os, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int t = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= heads) return;
    const float * yr = y + (int64_t) t * ys + (int64_t) h * n;
    if (n <= 128) {                                                   // (two values a lane: what the row needs is on its way before its sum)
        float yv[2], wv[2], gv[2], ss = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int i = min(lane + 64 * j, n - 1);
            yv[j] = yr[i]; wv[j] = w[(w_per_head ? h * n : 0) + i]; gv[j] = gate ? gate[(int64_t) t * gs + (int64_t) h * n + i] : 1.0f;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) if (lane + 64 * j < n) ss = fmaf(yv[j], yv[j], ss);
        const float inv = 1.0f / sqrtf(pi_lanes_sum<64>(ss) / (float) n + eps);
        if (pi_abort_late(gone, abort_w)) return;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int i = lane + 64 * j;
            if (i >= n) break;
            float g = gv[j];
            if (gate && gate_act == PI_ACT_SIGMOID) g = cm_sigmoid(g);
            else if (gate && gate_act == PI_ACT_SILU) g = g / (1.0f + expf(-g));
            const float o = yv[j] * inv * wv[j] * g;
            if (!rd.only) out[(int64_t) t * os + (int64_t) h * n + i] = o;
            if (rd.h) rd.h[t * rd.stride + (int64_t) h * n + i] = pi_round_one(o);
        }
        return;
    }
    if (pi_abort_late(gone, abort_w)) return;
    float ss = 0.0f;
    for (int i = lane; i < n; i += 64) ss = fmaf(yr[i], yr[i], ss);
    const float inv = 1.0f / sqrtf(pi_lanes_sum<64>(ss) / (float) n + eps);
    for (int i = lane; i < n; i += 64) {
        float g = gate ? gate[(int64_t) t * gs + (int64_t) h * n + i] : 1.0f;
        if (gate && gate_act == PI_ACT_SIGMOID) g = cm_sigmoid(g);
        else if (gate && gate_act == PI_ACT_SILU) g = g / (1.0f + expf(-g));
        const float o = yr[i] * inv * w[(w_per_head ? h * n : 0) + i] * g;
        if (!rd.only) out[(int64_t) t * os + (int64_t) h * n + i] = o;
        if (rd.h) rd.h[t * rd.stride + (int64_t) h * n + i] = pi_round_one(o);
    }
}
extern "C" int pi_op_head_norm_gate(const float * y, int64_t y_stride, int heads, int n, const float * w_dev, int w_per_head, const float * gate, int64_t gate_stride, int gate_act, float eps, int n_tok,
                                    float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || heads <= 0 || n <= 0) return 0;
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 12.0 * n_tok * heads * n, k_head_norm_gate, dim3((unsigned) n_tok, (unsigned) ((heads + 3) / 4)), dim3(256), 0, (hipStream_t) stream, y, y_stride, heads, n, w_dev, w_per_head,
                 gate, gate_stride, gate_act, eps, out, out_stride, pi_round_asked(0, (int64_t) heads * n), pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
