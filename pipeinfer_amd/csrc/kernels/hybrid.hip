// Operators of hybrid decoder blocks (recurrent and low-rank-attention mixers, routed feed-forwards).  Everything here is fp32: norms, scores, soft-max, recurrent
// state, router.  Matrices are bfloat16 pi_weights (widened exactly); `exact` = 0 rounds the activations that enter an expert's matrices to bfloat16 as pi_op_dense does.
//
//   k_rms_scale          y = x / sqrt(mean(x^2) + eps) * (w + w_offset) [* gate];  out = [residual +] mult * y;  rows may be written into the cache cells of the pass
//   k_linear_attention   per head S <- lambda * S + k v^T, o = S^T q over a run of tokens of one sequence; S lives in HBM per (slot, head) between calls; optionally with a value column of
//                        ones behind the others (the running sum of keys a normalised memory divides by)
//   k_latent_attention   attention over a shared low-rank latent c: the key up-projection is folded into the query (q~ = W_uk^T q), the value up-projection applied to the
//                        probability-weighted sum of latents — the cache is read once for all heads of a tile and K / V are never materialised; soft-max with a sink term
//   k_norm_chain(_reg)   y = ((ca * a + cb * b) - mean) / sqrt(variance + eps) * w + bias;  out = [residual +] y   (layer norm of one input or of the weighted sum of two), and
//                        the three row operations at the end of a block in one launch: post-norm + residual, the depth average, the next sublayer's pre-norm
//   k_depth_mix          out = sum_j coef[j] * X_j over the stream's earlier states (a learned average over depth)
//   k_moe_route          router logits, soft-max over all router outputs, bias-corrected top-k choice, weights = uncorrected scores
//   k_moe_up / _down     the chosen experts of every token (gathered mat-vecs), identity experts pass their input through
#include "ops_common.h"
#include "kernel_timing.h"
#include "prompt_attention.h"
#include "dense_tile.h"
#include "dense_async.h"

#include <algorithm>
#include <cmath>
#include <initializer_list>
#include <type_traits>
#include <utility>

static __device__ __forceinline__ float hy_widen(uint16_t b) { return __uint_as_float((uint32_t) b << 16); }
static __device__ __forceinline__ float hy_round(float f) { const uint32_t u = __float_as_uint(f); return __uint_as_float(((u + 0x7fffu + ((u >> 16) & 1u)) >> 16) << 16); }

typedef uint16_t hy_u16x8v __attribute__((ext_vector_type(8)));
// this lane's share of w . x over n values (bfloat16 row w, fp32 row x); vec: n % 8 == 0 and both rows 16-byte aligned — 16-byte weight loads, several in flight
static __device__ __forceinline__ float hy_dot_lane(const uint16_t * __restrict__ w, const float * __restrict__ x, int64_t n, int lane, bool exact, bool vec) {
    float a = 0.0f;
    if (vec) {
#pragma unroll 4
        for (int64_t i = (int64_t) lane * 8; i < n; i += 512) {
            const hy_u16x8v wv = *(const hy_u16x8v *) (w + i);
            const float4 x0 = *(const float4 *) (x + i), x1 = *(const float4 *) (x + i + 4);
            const float xf[8] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
#pragma unroll
            for (int k = 0; k < 8; k++) a = fmaf(hy_widen(wv[k]), exact ? xf[k] : hy_round(xf[k]), a);
        }
    } else {
        for (int64_t i = lane; i < n; i += 64) a = fmaf(hy_widen(w[i]), exact ? x[i] : hy_round(x[i]), a);
    }
    return a;
}

// sum over the 256 threads of a block (every thread gets the total); red: 4 floats of LDS, reusable after the call
static __device__ __forceinline__ float hy_block_sum(float v, float * red) {
    v = pi_lanes_sum<64>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.0f;
    for (int i = 0; i < (int) (blockDim.x >> 6); i++) s += red[i];
    return s;
}
static __device__ __forceinline__ float hy_block_max(float v, float * red) {
    v = pi_wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = red[0];
    for (int i = 1; i < (int) (blockDim.x >> 6); i++) s = fmaxf(s, red[i]);
    return s;
}

// ---- RMS norm with its usual companions ---------------------------------------------------------------------------------------------------------
// A row of up to 1024 NV values in the registers of 256 threads (thread i: values 4 i .. of every 1024): its norm, gate, multiplier and residual, in place.  Further threads of the workgroup only take part in the sum
// (as zeros: a row's bits do not depend on their number).  red: a float for each wave.  gv, rv: looked at where gated and added say so (arrays and not pointers that may be null: behind a choice between a pointer and null
// the arrays went to scratch memory, 48 / 80 / 144 bytes a lane)
template <int NV>
static __device__ __forceinline__ void hy_rms_row(float4 (&xv)[NV], const float4 (&wv)[NV], float w_off, float eps, int n, bool gated, const float4 (&gv)[NV], bool added, const float4 (&rv)[NV], float mult, float * red) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++) if (threadIdx.x < 256 && (int) threadIdx.x * 4 + 1024 * j < n) { ss = fmaf(xv[j].x, xv[j].x, ss); ss = fmaf(xv[j].y, xv[j].y, ss); ss = fmaf(xv[j].z, xv[j].z, ss); ss = fmaf(xv[j].w, xv[j].w, ss); }
    ss = hy_block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) n + eps);
#pragma unroll
    for (int j = 0; j < NV; j++) {
        float y[4] = { xv[j].x * inv * (wv[j].x + w_off), xv[j].y * inv * (wv[j].y + w_off), xv[j].z * inv * (wv[j].z + w_off), xv[j].w * inv * (wv[j].w + w_off) };
        if (gated) { y[0] *= gv[j].x; y[1] *= gv[j].y; y[2] *= gv[j].z; y[3] *= gv[j].w; }
#pragma unroll
        for (int k = 0; k < 4; k++) y[k] *= mult;
        if (added) { y[0] = rv[j].x + y[0]; y[1] = rv[j].y + y[1]; y[2] = rv[j].z + y[2]; y[3] = rv[j].w + y[3]; }
        xv[j] = make_float4(y[0], y[1], y[2], y[3]);
    }
}
// the row's results: a second norm's where w2 is given (the one ahead of the output head: its input is this row), beside the row itself
struct hy_second { const float * w; float w_off; float * out; int64_t os; };
struct hy_norm { const float * w; float w_off, eps; const float * res; int64_t rs; float mult; float * out; int64_t os; hy_second two; };
template <int NV>
static __device__ __forceinline__ void hy_rms_store(float4 (&xv)[NV], int t, int64_t orow, int n, float eps, float * out, int64_t os, const hy_second & two, const pi_round_dst & rd, float * red) {
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = (int) threadIdx.x * 4 + 1024 * j;
        if (i >= n || threadIdx.x >= 256) break;
        if (two.w || !rd.only) *(float4 *) (out + orow * os + i) = xv[j];
        if (!two.w && rd.h) pi_round_store4(rd, t, i, xv[j].x, xv[j].y, xv[j].z, xv[j].w);
    }
    if (!two.w) return;
    float4 wv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) wv[j] = *(const float4 *) (two.w + min((int) threadIdx.x * 4 + 1024 * j, n - 4));
    hy_rms_row<NV>(xv, wv, two.w_off, eps, n, false, wv, false, wv, 1.0f, red);
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = (int) threadIdx.x * 4 + 1024 * j;
        if (i >= n || threadIdx.x >= 256) break;
        if (!rd.only) *(float4 *) (two.out + (int64_t) t * two.os + i) = xv[j];
        if (rd.h) pi_round_store4(rd, t, i, xv[j].x, xv[j].y, xv[j].z, xv[j].w);
    }
}
// rows of up to 1024 NV aligned values: everything the row needs is on its way before its sum (a row that was read again behind the sum: one more trip to memory, 3.4 us a launch instead of 3.1)
template <int NV>
__global__ void __launch_bounds__(256) k_rms_scale_once(const float * __restrict__ x, int64_t xs, const float * __restrict__ w, float w_off, float eps, int n, const float * __restrict__ gate, int64_t gs,
                                                        const float * __restrict__ res, int64_t rs, float mult, float * __restrict__ out, int64_t os, const int32_t * __restrict__ dyn, int to_cells, const hy_second two,
                                                        const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ float red[4];
    const int t = blockIdx.x;
    const int64_t orow = to_cells ? pi_cell_of(dyn, 0, t) : t;
    float4 xv[NV], wv[NV], gv[NV], rv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = min((int) threadIdx.x * 4 + 1024 * j, n - 4);
        xv[j] = *(const float4 *) (x + (int64_t) t * xs + i); wv[j] = *(const float4 *) (w + i);
        if (gate) gv[j] = *(const float4 *) (gate + (int64_t) t * gs + i);
        if (res) rv[j] = *(const float4 *) (res + (int64_t) t * rs + i);
    }
    hy_rms_row<NV>(xv, wv, w_off, eps, n, gate != nullptr, gv, res != nullptr, rv, mult, red);
    if (pi_abort_late(gone, abort_w)) return;
    hy_rms_store<NV>(xv, t, orow, n, eps, out, os, two, rd, red);
}
__global__ void __launch_bounds__(256) k_rms_scale(const float * __restrict__ x, int64_t xs, const float * __restrict__ w, float w_off, float eps, int n,
                                                   const float * __restrict__ gate, int64_t gs, const float * __restrict__ res, int64_t rs, float mult,
                                                   float * __restrict__ out, int64_t os, const int32_t * __restrict__ dyn, int to_cells, int vec, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    __shared__ float red[4];
    const int t = blockIdx.x;
    const float * xr = x + (int64_t) t * xs;
    float ss = 0.0f;
    if (vec) { for (int i = threadIdx.x * 4; i < n; i += 1024) { const float4 v = *(const float4 *) (xr + i); ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss); } }
    else for (int i = threadIdx.x; i < n; i += 256) ss = fmaf(xr[i], xr[i], ss);
    ss = hy_block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) n + eps);
    const int64_t orow = to_cells ? pi_cell_of(dyn, 0, t) : t;
    if (vec) {
        for (int i = threadIdx.x * 4; i < n; i += 1024) {
            const float4 xv = *(const float4 *) (xr + i), wv = *(const float4 *) (w + i);
            float y[4] = { xv.x * inv * (wv.x + w_off), xv.y * inv * (wv.y + w_off), xv.z * inv * (wv.z + w_off), xv.w * inv * (wv.w + w_off) };
            if (gate) { const float4 g = *(const float4 *) (gate + (int64_t) t * gs + i); y[0] *= g.x; y[1] *= g.y; y[2] *= g.z; y[3] *= g.w; }
#pragma unroll
            for (int k = 0; k < 4; k++) y[k] *= mult;
            if (res) { const float4 r = *(const float4 *) (res + (int64_t) t * rs + i); y[0] = r.x + y[0]; y[1] = r.y + y[1]; y[2] = r.z + y[2]; y[3] = r.w + y[3]; }
            *(float4 *) (out + orow * os + i) = make_float4(y[0], y[1], y[2], y[3]);
        }
        return;
    }
    for (int i = threadIdx.x; i < n; i += 256) {
        float y = xr[i] * inv * (w[i] + w_off);
        if (gate) y *= gate[(int64_t) t * gs + i];
        y *= mult;
        if (res) y = res[(int64_t) t * rs + i] + y;
        out[orow * os + i] = y;
    }
}

static bool rms_vec(int n, std::initializer_list<std::pair<const void *, int64_t>> rows) {
    bool ok = n % 4 == 0;
    for (const auto & r : rows) ok = ok && (!r.first || (((uintptr_t) r.first % 16) == 0 && r.second % 4 == 0));
    return ok;
}
extern "C" int pi_op_rms_scale(const float * x, int64_t x_stride, const float * w, float w_offset, float eps, int n, int n_tok, const float * gate, int64_t gate_stride,
                               const float * residual, int64_t residual_stride, float mult, float * out, int64_t out_stride, const int32_t * dyn_dev, int to_cells, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (to_cells && !dyn_dev) { pi_set_error("pi_op_rms_scale: rows go to cache cells but no cell table was given"); return -1; }
    const int vec = rms_vec(n, { { x, x_stride }, { w, 0 }, { gate, gate_stride }, { residual, residual_stride }, { out, out_stride } });
#define RS_GO(NV, TWO) do { PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 12.0 * n * n_tok, k_rms_scale_once<NV>, dim3((unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, x, x_stride, w, w_offset, eps, n, gate, gate_stride, residual, \
                                    residual_stride, mult, out, out_stride, dyn_dev, to_cells, TWO, to_cells ? pi_round_dst{} : pi_round_asked(0, n), pi_abort_word()); PI_CHECK_LAUNCH(); return 0; } while (0)
    if (vec && n <= 1024) RS_GO(1, hy_second{});
    if (vec && n <= 2048) RS_GO(2, hy_second{});
    if (vec && n <= 4096) RS_GO(4, hy_second{});
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 12.0 * n * n_tok, k_rms_scale, dim3((unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, x, x_stride, w, w_offset, eps, n, gate, gate_stride,
                 residual, residual_stride, mult, out, out_stride, dyn_dev, to_cells, vec, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
// pi_op_rms_scale of a row and, of the result, a second one (plain) -> out2, in one launch where the row's values stay in registers; an asked rounding is the second's.  us of the two launches / of this: one token of
// 2048 8.6 / 4.6; 512 of 2048 9.4 / 6.3; 2048 of 4096 36 / 30
extern "C" int pi_op_rms_scale_twice(const float * x, int64_t x_stride, const float * w, float w_offset, float eps, int n, int n_tok, const float * residual, int64_t residual_stride, float mult, float * out, int64_t out_stride,
                                     const float * w2, float w2_offset, float * out2, int64_t out2_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    const bool vec = rms_vec(n, { { x, x_stride }, { w, 0 }, { residual, residual_stride }, { out, out_stride }, { w2, 0 }, { out2, out2_stride } });
    const float * gate = nullptr; const int64_t gate_stride = 0; const int32_t * dyn_dev = nullptr; const int to_cells = 0;
    const hy_second two = { w2, w2_offset, out2, out2_stride };
    if (vec && n <= 1024) RS_GO(1, two);
    if (vec && n <= 2048) RS_GO(2, two);
    if (vec && n <= 4096) RS_GO(4, two);
#undef RS_GO
    const pi_round_dst asked = pi_round_take();
    if (pi_op_rms_scale(x, x_stride, w, w_offset, eps, n, n_tok, gate, gate_stride, residual, residual_stride, mult, out, out_stride, nullptr, 0, stream) != 0) return -1;
    pi_set_rounded_output(asked.h, asked.stride, asked.from, asked.n, asked.only);
    return pi_op_rms_scale(out, out_stride, w2, w2_offset, eps, n, n_tok, nullptr, 0, nullptr, 0, 1.0f, out2, out2_stride, nullptr, 0, stream);
}

// ---- layer norm (weight and bias) over one or the weighted sum of two inputs, optional residual; the row operations at the end of a block -----------------------------
// The end of a block as one launch, per token row:  v = [residual +] LN_A(ca * a + cb * b)  -> out_a;   (n_hist > 0)  v = sum_(j < n_hist - 1) coef[j] * hist[j] + coef[n_hist - 1] * v
// -> out_mix  (out_a is hist[n_hist - 1]: the block's result joins the history it is averaged with);   (w_c)  LN_C(v) -> out_c  (the next sublayer's input).
// A thread re-reads only what it wrote itself, so no barrier is needed between the stages beyond those of the sums.
__global__ void __launch_bounds__(256) k_norm_chain(const float * __restrict__ a, int64_t as, float ca, const float * __restrict__ b, int64_t bs, float cb, const float * __restrict__ w,
                                                    const float * __restrict__ bias, float eps, int n, const float * __restrict__ res, int64_t rs, float * __restrict__ out_a, int64_t oas,
                                                    const float * __restrict__ hist, int64_t hist_stride, int n_hist, const float * __restrict__ coef, float * __restrict__ out_mix, int64_t oms,
                                                    const float * __restrict__ w_c, const float * __restrict__ bias_c, float * __restrict__ out_c, int64_t ocs, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    __shared__ float red[4];
    const int t = blockIdx.x;
    const float * ar = a + (int64_t) t * as, * br = b ? b + (int64_t) t * bs : nullptr;
    auto val = [&](int i) { const float v = ca * ar[i]; return br ? fmaf(cb, br[i], v) : v; };
    float sum = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) sum += val(i);
    const float mean = hy_block_sum(sum, red) / (float) n;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) { const float d = val(i) - mean; ss = fmaf(d, d, ss); }
    const float inv = 1.0f / sqrtf(hy_block_sum(ss, red) / (float) n + eps);
    float * oa = out_a + (int64_t) t * oas;
    float * last = oa;                                                 // the row the next stage reads (this thread's own elements)
    float sum_c = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) {
        float y = (val(i) - mean) * inv * w[i] + (bias ? bias[i] : 0.0f);
        if (res) y = res[(int64_t) t * rs + i] + y;
        oa[i] = y;
        if (n_hist > 0) {
            float m = 0.0f;
            for (int j = 0; j < n_hist - 1; j++) m = fmaf(coef[j], hist[(int64_t) j * hist_stride + (int64_t) t * n + i], m);
            y = fmaf(coef[n_hist - 1], y, m);
            out_mix[(int64_t) t * oms + i] = y;
        }
        sum_c += y;
    }
    if (!w_c) return;
    if (n_hist > 0) last = out_mix + (int64_t) t * oms;
    const float mean_c = hy_block_sum(sum_c, red) / (float) n;
    float ss_c = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) { const float d = last[i] - mean_c; ss_c = fmaf(d, d, ss_c); }
    const float inv_c = 1.0f / sqrtf(hy_block_sum(ss_c, red) / (float) n + eps);
    for (int i = threadIdx.x; i < n; i += 256) out_c[(int64_t) t * ocs + i] = (last[i] - mean_c) * inv_c * w_c[i] + (bias_c ? bias_c[i] : 0.0f);
}
// The same with the row in registers (n <= 256 * NPT): every input is loaded once, all loads are issued before the first sum, and the stages only exchange their sums
template <int NPT>
__global__ void __launch_bounds__(256) k_norm_chain_reg(const float * __restrict__ a, int64_t as, float ca, const float * __restrict__ b, int64_t bs, float cb, const float * __restrict__ w,
                                                        const float * __restrict__ bias, float eps, int n, const float * __restrict__ res, int64_t rs, float * __restrict__ out_a, int64_t oas,
                                                        const float * __restrict__ hist, int64_t hist_stride, int n_hist, const float * __restrict__ coef, float * __restrict__ out_mix, int64_t oms,
                                                        const float * __restrict__ w_c, const float * __restrict__ bias_c, float * __restrict__ out_c, int64_t ocs, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    __shared__ float red[4];
    const int t = blockIdx.x;
    const float * ar = a + (int64_t) t * as, * br = b ? b + (int64_t) t * bs : nullptr;
    float v[NPT], wv[NPT], bv[NPT], rv[NPT], mv[NPT];
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int i = threadIdx.x + k * 256;
        const bool ok = i < n;
        float x = ok ? ca * ar[i] : 0.0f;
        if (ok && br) x = fmaf(cb, br[i], x);
        v[k] = x; sum += x;
        wv[k] = ok ? w[i] : 0.0f; bv[k] = ok && bias ? bias[i] : 0.0f; rv[k] = ok && res ? res[(int64_t) t * rs + i] : 0.0f;
        float m = 0.0f;
        if (ok) for (int j = 0; j < n_hist - 1; j++) m = fmaf(coef[j], hist[(int64_t) j * hist_stride + (int64_t) t * n + i], m);
        mv[k] = m;
    }
    const float mean = hy_block_sum(sum, red) / (float) n;
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NPT; k++) if (threadIdx.x + k * 256 < n) { const float d = v[k] - mean; ss = fmaf(d, d, ss); }
    const float inv = 1.0f / sqrtf(hy_block_sum(ss, red) / (float) n + eps);
    const float c_last = n_hist > 0 ? coef[n_hist - 1] : 0.0f;
    float sum_c = 0.0f;
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int i = threadIdx.x + k * 256;
        if (i < n) {
            float y = (v[k] - mean) * inv * wv[k] + bv[k];
            if (res) y = rv[k] + y;
            out_a[(int64_t) t * oas + i] = y;
            if (n_hist > 0) { y = fmaf(c_last, y, mv[k]); out_mix[(int64_t) t * oms + i] = y; }
            v[k] = y; sum_c += y;
        }
    }
    if (!w_c) return;
#pragma unroll
    for (int k = 0; k < NPT; k++) { const int i = threadIdx.x + k * 256; wv[k] = i < n ? w_c[i] : 0.0f; bv[k] = i < n && bias_c ? bias_c[i] : 0.0f; }
    const float mean_c = hy_block_sum(sum_c, red) / (float) n;
    float ss_c = 0.0f;
#pragma unroll
    for (int k = 0; k < NPT; k++) if (threadIdx.x + k * 256 < n) { const float d = v[k] - mean_c; ss_c = fmaf(d, d, ss_c); }
    const float inv_c = 1.0f / sqrtf(hy_block_sum(ss_c, red) / (float) n + eps);
#pragma unroll
    for (int k = 0; k < NPT; k++) { const int i = threadIdx.x + k * 256; if (i < n) out_c[(int64_t) t * ocs + i] = (v[k] - mean_c) * inv_c * wv[k] + bv[k]; }
}
// ... and with 16-byte accesses: a thread owns NG groups of four neighbouring values (n % 4 == 0, rows 16-byte aligned, n <= 1024 * NG); one barrier per sum (each has its own LDS words)
static __device__ __forceinline__ float hy_block_sum_once(float v, float * red) {
    v = pi_lanes_sum<64>(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}
template <int NG>
__global__ void __launch_bounds__(256) k_norm_chain_vec(const float * __restrict__ a, int64_t as, float ca, const float * __restrict__ b, int64_t bs, float cb, const float * __restrict__ w,
                                                        const float * __restrict__ bias, float eps, int n, const float * __restrict__ res, int64_t rs, float * __restrict__ out_a, int64_t oas,
                                                        const float * __restrict__ hist, int64_t hist_stride, int n_hist, const float * __restrict__ coef, float * __restrict__ out_mix, int64_t oms,
                                                        const float * __restrict__ w_c, const float * __restrict__ bias_c, float * __restrict__ out_c, int64_t ocs, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    __shared__ float red[4][4];
    const int t = blockIdx.x;
    const float * ar = a + (int64_t) t * as, * br = b ? b + (int64_t) t * bs : nullptr;
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 v[NG], wv[NG], bv[NG], rv[NG], mv[NG];
    float sum = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int i = (threadIdx.x + g * 256) * 4;
        const bool ok = i < n;
        float4 x = ok ? *(const float4 *) (ar + i) : zero;
        x.x *= ca; x.y *= ca; x.z *= ca; x.w *= ca;
        if (ok && br) { const float4 y = *(const float4 *) (br + i); x.x = fmaf(cb, y.x, x.x); x.y = fmaf(cb, y.y, x.y); x.z = fmaf(cb, y.z, x.z); x.w = fmaf(cb, y.w, x.w); }
        v[g] = x; sum += (x.x + x.y) + (x.z + x.w);
        wv[g] = ok ? *(const float4 *) (w + i) : zero;
        bv[g] = ok && bias ? *(const float4 *) (bias + i) : zero;
        rv[g] = ok && res ? *(const float4 *) (res + (int64_t) t * rs + i) : zero;
        float4 m = zero;
        if (ok) for (int j = 0; j < n_hist - 1; j++) {
            const float c = coef[j]; const float4 h = *(const float4 *) (hist + (int64_t) j * hist_stride + (int64_t) t * n + i);
            m.x = fmaf(c, h.x, m.x); m.y = fmaf(c, h.y, m.y); m.z = fmaf(c, h.z, m.z); m.w = fmaf(c, h.w, m.w);
        }
        mv[g] = m;
    }
    const float mean = hy_block_sum_once(sum, red[0]) / (float) n;
    float ss = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; g++) if ((threadIdx.x + g * 256) * 4 < n) {
        const float d0 = v[g].x - mean, d1 = v[g].y - mean, d2 = v[g].z - mean, d3 = v[g].w - mean;
        ss = fmaf(d0, d0, ss); ss = fmaf(d1, d1, ss); ss = fmaf(d2, d2, ss); ss = fmaf(d3, d3, ss);
    }
    const float inv = 1.0f / sqrtf(hy_block_sum_once(ss, red[1]) / (float) n + eps);
    const float c_last = n_hist > 0 ? coef[n_hist - 1] : 0.0f;
    float sum_c = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int i = (threadIdx.x + g * 256) * 4;
        if (i < n) {
            float4 y = make_float4((v[g].x - mean) * inv * wv[g].x + bv[g].x, (v[g].y - mean) * inv * wv[g].y + bv[g].y, (v[g].z - mean) * inv * wv[g].z + bv[g].z, (v[g].w - mean) * inv * wv[g].w + bv[g].w);
            if (res) { y.x = rv[g].x + y.x; y.y = rv[g].y + y.y; y.z = rv[g].z + y.z; y.w = rv[g].w + y.w; }
            *(float4 *) (out_a + (int64_t) t * oas + i) = y;
            if (n_hist > 0) {
                y.x = fmaf(c_last, y.x, mv[g].x); y.y = fmaf(c_last, y.y, mv[g].y); y.z = fmaf(c_last, y.z, mv[g].z); y.w = fmaf(c_last, y.w, mv[g].w);
                *(float4 *) (out_mix + (int64_t) t * oms + i) = y;
            }
            v[g] = y; sum_c += (y.x + y.y) + (y.z + y.w);
        }
    }
    if (!w_c) return;
#pragma unroll
    for (int g = 0; g < NG; g++) { const int i = (threadIdx.x + g * 256) * 4; wv[g] = i < n ? *(const float4 *) (w_c + i) : zero; bv[g] = i < n && bias_c ? *(const float4 *) (bias_c + i) : zero; }
    const float mean_c = hy_block_sum_once(sum_c, red[2]) / (float) n;
    float ss_c = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; g++) if ((threadIdx.x + g * 256) * 4 < n) {
        const float d0 = v[g].x - mean_c, d1 = v[g].y - mean_c, d2 = v[g].z - mean_c, d3 = v[g].w - mean_c;
        ss_c = fmaf(d0, d0, ss_c); ss_c = fmaf(d1, d1, ss_c); ss_c = fmaf(d2, d2, ss_c); ss_c = fmaf(d3, d3, ss_c);
    }
    const float inv_c = 1.0f / sqrtf(hy_block_sum_once(ss_c, red[3]) / (float) n + eps);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int i = (threadIdx.x + g * 256) * 4;
        if (i < n) *(float4 *) (out_c + (int64_t) t * ocs + i) = make_float4((v[g].x - mean_c) * inv_c * wv[g].x + bv[g].x, (v[g].y - mean_c) * inv_c * wv[g].y + bv[g].y,
                                                                              (v[g].z - mean_c) * inv_c * wv[g].z + bv[g].z, (v[g].w - mean_c) * inv_c * wv[g].w + bv[g].w);
    }
}
extern "C" int pi_op_layer_norm_mix(const float * a, int64_t a_stride, float ca, const float * b, int64_t b_stride, float cb, const float * w_dev, const float * bias_dev, float eps, int n, int n_tok,
                                    const float * residual, int64_t residual_stride, float * out, int64_t out_stride, void * stream) {
    return pi_op_norm_chain(a, a_stride, ca, b, b_stride, cb, w_dev, bias_dev, eps, n, n_tok, residual, residual_stride, out, out_stride, nullptr, 0, 0, nullptr, nullptr, 0, nullptr, nullptr, nullptr, 0, stream);
}
extern "C" int pi_op_norm_chain(const float * a, int64_t a_stride, float ca, const float * b, int64_t b_stride, float cb, const float * w_dev, const float * bias_dev, float eps, int n, int n_tok,
                                const float * residual, int64_t residual_stride, float * out_a, int64_t out_a_stride, const float * hist, int64_t hist_stride, int n_hist, const float * coef_dev,
                                float * out_mix, int64_t out_mix_stride, const float * w_next, const float * bias_next, float * out_next, int64_t out_next_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (n_hist > 0 && (!hist || !coef_dev || !out_mix || out_a != hist + (int64_t) (n_hist - 1) * hist_stride || out_a_stride != n)) {
        pi_set_error("pi_op_norm_chain: the block's result must be written into the last entry of the history it is averaged with"); return -1;
    }
    if (w_next && (!out_next || out_next == out_a || out_next == out_mix)) { pi_set_error("pi_op_norm_chain: the next norm needs an output of its own"); return -1; }
    const double bytes = 4.0 * n * n_tok * (3.0 + (b ? 1 : 0) + (residual ? 1 : 0) + n_hist + (w_next ? 2 : 0));
#define NC_GO(K) PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, bytes, K, dim3((unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, a, a_stride, ca, b, b_stride, cb, w_dev, bias_dev, eps, n, residual, residual_stride, \
                              out_a, out_a_stride, hist, hist_stride, n_hist, coef_dev, out_mix, out_mix_stride, w_next, bias_next, out_next, out_next_stride, pi_abort_word())
    auto al = [](const void * p, int64_t stride) { return !p || (((uintptr_t) p % 16) == 0 && stride % 4 == 0); };
    const bool vec = n % 4 == 0 && n <= 8192 && al(a, a_stride) && al(b, b_stride) && al(w_dev, 0) && al(bias_dev, 0) && al(residual, residual_stride) && al(out_a, out_a_stride) && al(hist, hist_stride) &&
                     al(out_mix, out_mix_stride) && al(w_next, 0) && al(bias_next, 0) && al(out_next, out_next_stride);
    if (vec) { if (n <= 1024) NC_GO(k_norm_chain_vec<1>); else if (n <= 2048) NC_GO(k_norm_chain_vec<2>); else if (n <= 4096) NC_GO(k_norm_chain_vec<4>); else NC_GO(k_norm_chain_vec<8>); }
    else if (n <= 1024) NC_GO(k_norm_chain_reg<4>); else if (n <= 2048) NC_GO(k_norm_chain_reg<8>); else if (n <= 4096) NC_GO(k_norm_chain_reg<16>); else if (n <= 8192) NC_GO(k_norm_chain_reg<32>); else NC_GO(k_norm_chain);
#undef NC_GO
    PI_CHECK_LAUNCH(); return 0;
}

// out[t][i] = sum_j coef[j] * hist[j][t][i], j ascending; hist: n_hist arrays [n_tok rows][n], `hist_stride` floats apart
__global__ void __launch_bounds__(256) k_depth_mix(const float * __restrict__ hist, int64_t hist_stride, int n_hist, const float * __restrict__ coef, int n, float * __restrict__ out, int64_t os,
                                                   const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float a = 0.0f;
    for (int j = 0; j < n_hist; j++) a = fmaf(coef[j], hist[(int64_t) j * hist_stride + (int64_t) t * n + i], a);
    out[(int64_t) t * os + i] = a;
}
extern "C" int pi_op_depth_mix(const float * hist, int64_t hist_stride, int n_hist, const float * coef_dev, int n, int n_tok, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || n <= 0 || n_hist <= 0) return 0;
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n * n_tok * (n_hist + 1.0), k_depth_mix, dim3((unsigned) ((n + 255) / 256), (unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, hist, hist_stride, n_hist, coef_dev, n,
                 out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// x <- cap * tanh(x / cap) in place
__global__ void k_softcap(float * __restrict__ x, int64_t n, float cap, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    for (int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t) gridDim.x * 256) x[i] = cap * tanhf(x[i] / cap);
}
extern "C" int pi_op_softcap(float * x, int64_t n, float cap, void * stream) {
    if (n <= 0) return 0;
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 8.0 * n, k_softcap, dim3((unsigned) std::max<int64_t>(1, std::min<int64_t>(4096, (n + 255) / 256))), dim3(256), 0, (hipStream_t) stream, x, n, cap, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// a gated hidden layer from its raw halves: PI_GLU_SILU silu(g) * u; PI_GLU_CLIPPED g' sigmoid(1.702 g') (u' + 1) with g' = min(g, limit), u' = clip(u, -limit, limit) (limit <= 0: no bounds)
static __device__ __forceinline__ float hy_glu(float g, float u, int glu, float limit) {
    if (glu == PI_GLU_CLIPPED) {
        if (limit > 0.0f) { g = fminf(g, limit); u = fminf(fmaxf(u, -limit), limit); }
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    return glu == PI_GLU_SILU ? g / (1.0f + expf(-g)) * u : g * u;
}
// the same for passes of many tokens, whose result the down-projection reads in bfloat16: eight values of a thread (1000 tokens of 1408: 6.3 us and 5.2 for the rounding behind it, now 5)
__global__ void __launch_bounds__(256) k_glu_rounded(const float * __restrict__ in, int64_t is, int ff, int glu, float limit, int64_t gate_col, float * __restrict__ out, int64_t os, const pi_round_dst rd,
                                                     const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w), t = blockIdx.y, f = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (f >= ff) return;
    const float * r = in + (int64_t) t * is + f;
    float4 g[2] = { *(const float4 *) r, *(const float4 *) (r + 4) }, u[2] = { *(const float4 *) (r + ff), *(const float4 *) (r + ff + 4) };
    const float m = gate_col >= 0 ? 1.0f / (1.0f + expf(-in[(int64_t) t * is + gate_col])) : 1.0f;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; i++) { y[i] = hy_glu(((const float *) g)[i], ((const float *) u)[i], glu, limit); if (gate_col >= 0) y[i] *= m; }
    if (pi_abort_late(gone, abort_w)) return;
    if (!rd.only) { float4 * o = (float4 *) (out + (int64_t) t * os + f); o[0] = make_float4(y[0], y[1], y[2], y[3]); o[1] = make_float4(y[4], y[5], y[6], y[7]); }
    pi_round_store4(rd, t, f, y[0], y[1], y[2], y[3]); pi_round_store4(rd, t, f + 4, y[4], y[5], y[6], y[7]);
}
static bool glu_rounded(const float * in, int64_t is, int ff, int glu, float limit, int64_t gate_col, int n_tok, float * out, int64_t os, hipStream_t s) {
    if (ff % 8 || is % 4 || os % 4 || (((uintptr_t) in | (uintptr_t) out) & 15)) return false;
    const pi_round_dst rd = pi_round_asked(0, ff);
    if (!rd.h) return false;
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 10.0 * ff * n_tok, k_glu_rounded, dim3((unsigned) ((ff + 2047) / 2048), (unsigned) n_tok), dim3(256), 0, s, in, is, ff, glu, limit, gate_col, out, os, rd, pi_abort_word());
    return true;
}

// out[t][f] = in[t][f] * in[t][ff + f]  (a gated feed-forward whose gate and up rows are one matrix; the gate's activation ran in the projection's epilogue)
__global__ void k_glu_mul(const float * __restrict__ in, int64_t is, int ff, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w), t = blockIdx.y, f = blockIdx.x * 256 + threadIdx.x;
    if (f >= ff) return;
    const float y = in[(int64_t) t * is + f] * in[(int64_t) t * is + ff + f];
    if (pi_abort_late(gone, abort_w)) return;
    out[(int64_t) t * os + f] = y;
}
extern "C" int pi_op_glu_mul(const float * in, int64_t in_stride, int ff, int n_tok, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || ff <= 0) return 0;
    if (glu_rounded(in, in_stride, ff, PI_GLU_OFF, 0.0f, -1, n_tok, out, out_stride, (hipStream_t) stream)) { PI_CHECK_LAUNCH(); return 0; }
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 12.0 * ff * n_tok, k_glu_mul, dim3((unsigned) ((ff + 255) / 256), (unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, in, in_stride, ff, out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

__global__ void k_glu_mul_ex(const float * __restrict__ in, int64_t is, int ff, int glu, float limit, int64_t gate_col, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w), t = blockIdx.y, f = blockIdx.x * 256 + threadIdx.x;
    if (f >= ff) return;
    const float * r = in + (int64_t) t * is;
    float y = hy_glu(r[f], r[ff + f], glu, limit);
    if (gate_col >= 0) y *= 1.0f / (1.0f + expf(-r[gate_col]));
    if (pi_abort_late(gone, abort_w)) return;
    out[(int64_t) t * os + f] = y;
}
extern "C" int pi_op_glu_mul_ex(const float * in, int64_t in_stride, int ff, int glu, float limit, int64_t gate_col, int n_tok, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0 || ff <= 0) return 0;
    if (glu < PI_GLU_OFF || glu > PI_GLU_CLIPPED || gate_col >= in_stride) { pi_set_error("pi_op_glu_mul_ex: hidden layer of kind %d, gate column %lld of rows %lld floats apart", glu, (long long) gate_col, (long long) in_stride); return -1; }
    if (glu_rounded(in, in_stride, ff, glu, limit, gate_col, n_tok, out, out_stride, (hipStream_t) stream)) { PI_CHECK_LAUNCH(); return 0; }
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 12.0 * ff * n_tok, k_glu_mul_ex, dim3((unsigned) ((ff + 255) / 256), (unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, in, in_stride, ff, glu, limit, gate_col, out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// ---- rows of the stream: copies, and a layer's end with the next tanh norm --------------------------------------------------------------------------------------
__global__ void k_copy_rows(const float * __restrict__ src, int64_t ss, float * __restrict__ dst, int64_t ds, int n, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[(int64_t) t * ds + i] = src[(int64_t) t * ss + i];
}
extern "C" int pi_op_copy_rows(const float * src, int64_t src_stride, float * dst, int64_t dst_stride, int n, int n_tok, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 8.0 * n * n_tok, k_copy_rows, dim3((unsigned) ((n + 255) / 256), (unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, src, src_stride, dst, dst_stride, n, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
// x_out = x + a + b + c (summed in this order); h = tanh(alpha * x_out) * w + bias: no statistics, so a thread needs nobody else's values
__global__ void k_sum_tanh_norm(const float * __restrict__ x, int64_t xs, const float * __restrict__ a, int64_t as, const float * __restrict__ b, int64_t bs, const float * __restrict__ c, int64_t cs, int n,
                                float * __restrict__ xo, int64_t xos, const float * __restrict__ alpha, const float * __restrict__ w, const float * __restrict__ bias, float * __restrict__ ho, int64_t hos,
                                const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float v = x[(int64_t) t * xs + i];
    if (a) v += a[(int64_t) t * as + i];
    if (b) v += b[(int64_t) t * bs + i];
    if (c) v += c[(int64_t) t * cs + i];
    if (xo) xo[(int64_t) t * xos + i] = v;
    if (w) ho[(int64_t) t * hos + i] = fmaf(tanhf(alpha[0] * v), w[i], bias ? bias[i] : 0.0f);
}
extern "C" int pi_op_sum_tanh_norm(const float * x, int64_t x_stride, const float * a, int64_t a_stride, const float * b, int64_t b_stride, const float * c, int64_t c_stride, int n, int n_tok,
                                   float * x_out, int64_t x_out_stride, const float * alpha_dev, const float * w_dev, const float * bias_dev, float * h_out, int64_t h_out_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (w_dev && (!alpha_dev || !h_out)) { pi_set_error("pi_op_sum_tanh_norm: the norm needs its scalar and an output"); return -1; }
    if (!w_dev && !x_out) return 0;
    const int rows = 1 + (a != nullptr) + (b != nullptr) + (c != nullptr) + (x_out != nullptr) + (w_dev != nullptr);
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n * n_tok * rows, k_sum_tanh_norm, dim3((unsigned) ((n + 255) / 256), (unsigned) n_tok), dim3(256), 0, (hipStream_t) stream, x, x_stride, a, a_stride, b, b_stride, c, c_stride, n,
                 x_out, x_out_stride, alpha_dev, w_dev, bias_dev, h_out, h_out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// the same with the token shift of the norm's output behind it, m = h + (h_prev - h) * mu (h_prev: the sequence's previous token; pi_op_token_shift's state and slot words), for passes of at most
// 32 tokens in ONE launch: the thread of a run's first token walks the run for its column with h_prev in a register and leaves the state, so nothing it writes is read by another thread
#define STN_FRESH (1 << 30)
#define STN_WALK_MAX_TOKENS 32
__global__ void __launch_bounds__(256) k_sum_tanh_norm_walk(const float * __restrict__ x, int64_t xs, const float * __restrict__ a, int64_t as, const float * __restrict__ b, int64_t bs, const float * __restrict__ c, int64_t cs,
                                                            int n, int n_tok, float * __restrict__ xo, int64_t xos, const float * __restrict__ alpha, const float * __restrict__ w, const float * __restrict__ bias,
                                                            float * __restrict__ ho, int64_t hos, const float * __restrict__ mu, float * __restrict__ state, const int32_t * __restrict__ rec, float * __restrict__ mo,
                                                            int64_t mos, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    const int word = rec[t], slot = word & ~STN_FRESH;
    if (i >= n || (t > 0 && (rec[t - 1] & ~STN_FRESH) == slot)) return;
    const float al = alpha[0], wi = w[i], bi = bias ? bias[i] : 0.0f, mi = mu[i];
    float prev = (word & STN_FRESH) ? 0.0f : state[(int64_t) slot * n + i];
    for (int tt = t; tt < n_tok && (rec[tt] & ~STN_FRESH) == slot; tt++) {
        float v = x[(int64_t) tt * xs + i];
        if (a) v += a[(int64_t) tt * as + i];
        if (b) v += b[(int64_t) tt * bs + i];
        if (c) v += c[(int64_t) tt * cs + i];
        if (xo) xo[(int64_t) tt * xos + i] = v;
        const float h = fmaf(tanhf(al * v), wi, bi);
        ho[(int64_t) tt * hos + i] = h;
        mo[(int64_t) tt * mos + i] = fmaf(prev - h, mi, h);
        prev = h;
    }
    state[(int64_t) slot * n + i] = prev;
}
extern "C" int pi_op_sum_tanh_norm_shift(const float * x, int64_t x_stride, const float * a, int64_t a_stride, const float * b, int64_t b_stride, const float * c, int64_t c_stride, int n, int n_tok,
                                         float * x_out, int64_t x_out_stride, const float * alpha_dev, const float * w_dev, const float * bias_dev, float * h_out, int64_t h_out_stride,
                                         const float * mu_dev, float * state_dev, const int32_t * rec_dev, float * m_out, int64_t m_out_stride, void * stream) {
    if (n_tok <= 0 || n <= 0) return 0;
    if (!w_dev || !alpha_dev || !h_out || !mu_dev || !state_dev || !rec_dev || !m_out || m_out == h_out) { pi_set_error("pi_op_sum_tanh_norm_shift: the norm, the shift factors, the sequences' state and slot words and two outputs are required"); return -1; }
    if (n_tok > STN_WALK_MAX_TOKENS) {
        if (pi_op_sum_tanh_norm(x, x_stride, a, a_stride, b, b_stride, c, c_stride, n, n_tok, x_out, x_out_stride, alpha_dev, w_dev, bias_dev, h_out, h_out_stride, stream) != 0) return -1;
        return pi_op_token_shift(h_out, h_out_stride, n, mu_dev, 1, state_dev, rec_dev, n_tok, m_out, m_out_stride, stream);
    }
    const int rows = 3 + (a != nullptr) + (b != nullptr) + (c != nullptr) + (x_out != nullptr);
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n * n_tok * rows + 8.0 * n, k_sum_tanh_norm_walk, dim3((unsigned) n_tok, (unsigned) ((n + 255) / 256)), dim3(256), 0, (hipStream_t) stream, x, x_stride, a, a_stride, b, b_stride,
                 c, c_stride, n, n_tok, x_out, x_out_stride, alpha_dev, w_dev, bias_dev, h_out, h_out_stride, mu_dev, state_dev, rec_dev, m_out, m_out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// ---- linear attention with a per-head decay -------------------------------------------------------------------------------------------------------
// rec[t] = state slot of token t (| 1 << 30 on the first token of a sequence whose state starts from zero), tokens of one slot are consecutive.  Workgroup (head, column block,
// piece): thread (column j, part sp of R) keeps S[i][j] for its DPT rows i in registers and walks the piece's tokens in order.
// A pass of up to LA_TB tokens is one launch: a piece is a sequence's whole run, S comes from and goes back to HBM.  Longer passes cut every sequence's run into pieces of LA_TB
// tokens and take three launches, so that the serial depth is two pieces instead of the whole prompt (the recurrence is linear in S):
//   mode 1  every piece but a run's last: the state it would build from ZERO, L_p = sum_j lambda^(len-1-j) k_j v_j^T, into scratch
//   k_linear_state_scan  per run, piece by piece: S_in(p + 1) = lambda^len_p * S_in(p) + L_p, S_in(0) = the slot's state (or zero); scratch[p] <- S_in(p)
//   mode 2  every piece from its true S_in(p): outputs; a run's last piece leaves the slot's new state
// Key widths of 32, 64, 96 and 128 take the fp32 matrix cores instead: up to LM_TB tokens one launch (k_linear_pieces), more of them two over pieces of LW_TB (k_linear_scores, k_linear_walk).
#define LA_TB 32                                  // tokens of a piece; q, k and v of a piece are staged in LDS
#define LA_FRESH (1 << 30)
#define LA_MAXRUNS 256                            // sequences a pass may carry (the host checks)
// the first tokens of the pass's runs, in order (every thread of the block, 64 at least, calls; bnd / nb in LDS): a thread looks at its own tokens only, then every run finds its place by counting the ones ahead of
// it.  (One thread that sorted them: with 64 runs 200 us and more of every launch, 16 heads of 64 x 64, 96 tokens: 719 us for the three, now 75)
static __device__ __forceinline__ int la_runs(const int * recs, int n_tok, int * bnd, int * nb) {
    if (threadIdx.x == 0) *nb = 0;
    __syncthreads();
    for (int t = threadIdx.x; t < n_tok; t += blockDim.x)
        if (t == 0 || (recs[t] & ~LA_FRESH) != (recs[t - 1] & ~LA_FRESH)) { const int k = atomicAdd(nb, 1); if (k < LA_MAXRUNS) bnd[k] = t; }
    __syncthreads();
    const int n = min(*nb, LA_MAXRUNS);
    if (n > 1) {
        int at[LA_MAXRUNS / 64], v[LA_MAXRUNS / 64];
#pragma unroll
        for (int k = 0; k < LA_MAXRUNS / 64; k++) {
            const int i = threadIdx.x + k * blockDim.x;
            at[k] = 0;
            if (i < n) { v[k] = bnd[i]; for (int o = 0; o < n; o++) at[k] += bnd[o] < v[k]; }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < LA_MAXRUNS / 64; k++) if ((int) (threadIdx.x + k * blockDim.x) < n) bnd[at[k]] = v[k];
    }
    __syncthreads();
    return n;
}
// The pieces of lseg tokens (0: pieces are whole runs) that lie ahead of a lane's four runs (the first wave calls; run 4 lane + k has own[k])
static __device__ __forceinline__ int la_pieces_before(const int * bnd, int n_runs, int n_tok, int lseg, int (&own)[4]) {
    const int lane = threadIdx.x;
    int sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int r = 4 * lane + k;
        own[k] = r >= n_runs ? 0 : lseg > 0 ? ((r + 1 < n_runs ? bnd[r + 1] : n_tok) - bnd[r] + lseg - 1) / lseg : 1;
        sum += own[k];
    }
    int upto = sum;
    if (n_runs > 4)
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int x = __shfl_up(upto, o, 64); if (lane >= o) upto += x; }
    return upto - sum;
}
static_assert(LA_MAXRUNS <= 4 * 64, "four runs to a lane");
// piece number `want` of the pass into seg (LDS; the first wave calls): first token, length (0: there is none), slot word, whether it is its run's last piece
static __device__ __forceinline__ void la_find_piece(const int * recs, int n_tok, const int * bnd, int n_runs, int lseg, int want, int * seg) {
    int own[4], ord = la_pieces_before(bnd, n_runs, n_tok, lseg, own);
    if (threadIdx.x == 0) { seg[0] = 0; seg[1] = 0; seg[2] = -1; seg[3] = 1; }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (want >= ord && want < ord + own[k]) {
            const int r = 4 * (int) threadIdx.x + k, t = bnd[r], e = r + 1 < n_runs ? bnd[r + 1] : n_tok, p = want - ord, first = lseg > 0 ? t + p * lseg : t;
            seg[0] = first; seg[1] = lseg > 0 ? min(lseg, e - first) : e - t; seg[2] = recs[t]; seg[3] = p == own[k] - 1;
        }
        ord += own[k];
    }
}
// whether all tokens of the pass are one sequence's (every thread of the block calls): most prompts, for which nothing has to be searched
static __device__ __forceinline__ bool la_one_run(const int32_t * __restrict__ rec, int n_tok) {
    const int own = rec[0];
    int other = 0;
    for (int t = threadIdx.x; t < n_tok; t += blockDim.x) other |= (rec[t] ^ own) & ~LA_FRESH;
    return !__syncthreads_or(other);
}
template <int DPT>
__global__ void __launch_bounds__(256) k_linear_attention(const float * __restrict__ q, const float * __restrict__ k, const float * __restrict__ v, int64_t stride, int heads, int hpg, int dim, int vdim, int vstored, int R,
                                                          const float * __restrict__ decay, const float * __restrict__ tdecay, const float * __restrict__ tscale, int64_t tds, const float * __restrict__ skip,
                                                          float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, int mode, float * __restrict__ scratch,
                                                          float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    extern __shared__ float lds[];                // q tile [LA_TB][dim] | k tile [LA_TB][dim] | v tile [LA_TB][cols] | the slot words of the pass [n_tok]
    __shared__ int seg[4], bnd[LA_MAXRUNS], nbnd; // seg: first token, length, slot word, last piece of its run
    __shared__ float lam_t[LA_TB], sc_t[LA_TB];   // per token of the tile: decay and the factor on k v^T
    const int h = blockIdx.x, tid = threadIdx.x;
    int * recs = (int *) (lds + 2 * LA_TB * dim + LA_TB * (blockDim.x / R));
    if (n_tok == 1) { if (tid == 0) { seg[0] = 0; seg[1] = blockIdx.z == 0; seg[2] = rec[0]; seg[3] = 1; } }      // (a single token is its own run: no search)
    else {
    for (int t = tid; t < n_tok; t += blockDim.x) recs[t] = rec[t];
    __syncthreads();
    const int n_runs = la_runs(recs, n_tok, bnd, &nbnd);
    if (tid < 64) la_find_piece(recs, n_tok, bnd, n_runs, mode ? LA_TB : 0, blockIdx.z, seg);
    }
    __syncthreads();
    const int first = seg[0], len = seg[1], word = seg[2], last = seg[3];
    if (pi_abort_late(gone, abort_w)) return;
    if (len == 0 || word < 0 || (mode == 1 && last)) return;
    const int slot = word & ~LA_FRESH;
    const int cols = blockDim.x / R;
    const int j = blockIdx.y * cols + tid / R, sp = tid % R;
    const bool col_ok = j < vdim;
    const float lam = decay ? decay[h] : 1.0f, skp = skip ? skip[h] : 0.0f;
    const int hq = h / hpg;                                            // the q / k head this head reads (hpg heads share one)
    float * S_hbm = state + ((int64_t) slot * heads + h) * dim * vdim;
    float * S_scr = scratch ? scratch + ((int64_t) blockIdx.z * heads + h) * dim * vdim : nullptr;
    const float * S_from = mode == 2 ? S_scr : mode == 1 || (word & LA_FRESH) ? nullptr : S_hbm;
    float S[DPT];
#pragma unroll
    for (int ii = 0; ii < DPT; ii++) {
        const int i = sp * DPT + ii;
        S[ii] = (col_ok && i < dim && S_from) ? S_from[(int64_t) i * vdim + j] : 0.0f;
    }
    float * qt = lds, * kt = lds + LA_TB * dim, * vt = kt + LA_TB * dim;
    const bool dim4 = (dim & 3) == 0;
    for (int t0 = 0; t0 < len; t0 += LA_TB) {
        const int nt = min(LA_TB, len - t0);
        __syncthreads();
        for (int idx = tid; idx < nt * dim; idx += blockDim.x) {
            const int tt = idx / dim, i = idx % dim;
            const int64_t off = (int64_t) (first + t0 + tt) * stride + (int64_t) hq * dim + i;
            if (mode != 1) qt[idx] = q[off];
            kt[idx] = k[off];
        }
        if (tid < nt) {
            lam_t[tid] = tdecay ? tdecay[(int64_t) (first + t0 + tid) * tds + h] : lam;
            sc_t[tid] = tscale ? tscale[(int64_t) (first + t0 + tid) * tds + h] : 1.0f;
        }
        for (int idx = tid; idx < nt * cols; idx += blockDim.x) {
            const int tt = idx / cols, jj = blockIdx.y * cols + idx % cols;
            vt[idx] = jj < vstored ? v[(int64_t) (first + t0 + tt) * stride + (int64_t) h * vstored + jj] : jj < vdim ? 1.0f : 0.0f;      // (a column the values do not have: ones)
        }
        __syncthreads();
        if (mode == 1) {                                              // the state only
            for (int tt = 0; tt < nt; tt++) {
                const float vj = vt[tt * cols + tid / R] * sc_t[tt], lam = lam_t[tt];
                const float * kr = kt + tt * dim + sp * DPT;
#pragma unroll
                for (int ii = 0; ii < DPT; ii++) if (sp * DPT + ii < dim) S[ii] = fmaf(kr[ii], vj, lam * S[ii]);
            }
            continue;
        }
        for (int tt = 0; tt < nt; tt++) {
            const float vraw = vt[tt * cols + tid / R], vj = vraw * sc_t[tt], lam = lam_t[tt];
            const float * kr = kt + tt * dim + sp * DPT, * qr = qt + tt * dim + sp * DPT;
            float o = 0.0f;
            if (dim4) {
#pragma unroll
                for (int ii = 0; ii < DPT; ii += 4) {
                    if (sp * DPT + ii < dim) {
                        const float4 kv = *(const float4 *) (kr + ii), qv = *(const float4 *) (qr + ii);
                        S[ii] = fmaf(kv.x, vj, lam * S[ii]);         o = fmaf(S[ii], qv.x, o);
                        S[ii + 1] = fmaf(kv.y, vj, lam * S[ii + 1]); o = fmaf(S[ii + 1], qv.y, o);
                        S[ii + 2] = fmaf(kv.z, vj, lam * S[ii + 2]); o = fmaf(S[ii + 2], qv.z, o);
                        S[ii + 3] = fmaf(kv.w, vj, lam * S[ii + 3]); o = fmaf(S[ii + 3], qv.w, o);
                    }
                }
            } else {
#pragma unroll
                for (int ii = 0; ii < DPT; ii++)
                    if (sp * DPT + ii < dim) { S[ii] = fmaf(kr[ii], vj, lam * S[ii]); o = fmaf(S[ii], qr[ii], o); }
            }
            if (R == 2) o += pi_partner<1>(o);
            else if (R == 4) { o += pi_partner<2>(o); o += pi_partner<1>(o); }
            else for (int d = R >> 1; d > 0; d >>= 1) o += __shfl_xor(o, d, PI_WAVE);
            if (col_ok && sp == 0) out[(int64_t) (first + t0 + tt) * os + (int64_t) h * vdim + j] = fmaf(skp, vraw, o);
        }
    }
    float * S_to = mode == 1 ? S_scr : last ? S_hbm : nullptr;
    if (col_ok && S_to)
#pragma unroll
        for (int ii = 0; ii < DPT; ii++) { const int i = sp * DPT + ii; if (i < dim) S_to[(int64_t) i * vdim + j] = S[ii]; }
}

// The same for a step: a few tokens, most of them a run of their own, whole key widths and columns.  What bounds it: the trips to memory in front of a state's one.  Nothing goes through LDS but the sums over the rows: a wave finds its
// run by a ballot, its first token's operands leave beside the state, the next one's ahead of the sums.  Workgroup (head, 32 columns of values, run); thread (four columns, rows rg + 32 m), states in runs of 128 bytes.
// Measured, us (k_linear_attention or k_linear_pieces, whichever it was / this): 16 heads of 128 x 128, one token 7.7 / 3.1, eight of a sequence each 10.5 / 4.4, eight of one 22.2 / 7.2, 16 of one 23.0 / 12.2; 16 heads of 64 x 64 7.4 / 2.9,
// 9.6 / 3.1, 16.9 / 6.4, 11.4 / 10.4.  (There a token's operands were staged for 32, behind a search through LDS, and a state came in runs of 64 bytes.)
template <int NR>
__global__ void __launch_bounds__(256) k_linear_step(const float * __restrict__ q, const float * __restrict__ k, const float * __restrict__ v, int64_t stride, int heads, int hpg, int vdim,
                                                     const float * __restrict__ decay, const float * __restrict__ tdecay, const float * __restrict__ tscale, int64_t tds, const float * __restrict__ skip,
                                                     float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int DIM = 32 * NR;
    __shared__ __attribute__((aligned(16))) float meet[2][4][32];       // [token % 2][wave][column]
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), quad = tid & 7, rg = tid >> 3, col = blockIdx.y * 32 + quad * 4, hq = h / hpg;
    const int own = rec[min(lane, n_tok - 1)], before = rec[max(min(lane, n_tok - 1) - 1, 0)];
    const float lam0 = decay ? decay[h] : 1.0f, skp = skip ? skip[h] : 0.0f;
    uint64_t starts = __ballot(lane < n_tok && (lane == 0 || (own & ~LA_FRESH) != (before & ~LA_FRESH)));
    for (int r = 0; r < (int) blockIdx.z; r++) starts &= starts - 1;
    if (!starts) return;
    const int first = __ffsll((unsigned long long) starts) - 1, rest = __ffsll((unsigned long long) (starts & (starts - 1))), end = rest ? rest - 1 : n_tok, word = __builtin_amdgcn_readlane(own, first);
    if (word < 0) return;
    float * const S_hbm = state + ((int64_t) (word & ~LA_FRESH) * heads + h) * DIM * vdim + (int64_t) rg * vdim + col;
    float4 S[NR];
    if (word & LA_FRESH) {
#pragma unroll
        for (int m = 0; m < NR; m++) S[m] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
#pragma unroll
        for (int m = 0; m < NR; m++) S[m] = *(const float4 *) (S_hbm + (int64_t) 32 * m * vdim);
    }
    struct token { float q[NR], k[NR], lam, sc; float4 v; };
    auto ask = [&](token & T, int t) __attribute__((always_inline)) {
        const float * qr = q + (int64_t) t * stride + (int64_t) hq * DIM, * kr = k + (int64_t) t * stride + (int64_t) hq * DIM;
#pragma unroll
        for (int m = 0; m < NR; m++) { T.q[m] = qr[rg + 32 * m]; T.k[m] = kr[rg + 32 * m]; }
        T.lam = tdecay ? tdecay[(int64_t) t * tds + h] : lam0;
        T.sc = tscale ? tscale[(int64_t) t * tds + h] : 1.0f;
        T.v = *(const float4 *) (v + (int64_t) t * stride + (int64_t) h * vdim + col);
    };
    token T;
    ask(T, first);
    if (pi_abort_late(gone, abort_w)) return;
    for (int t = first; t < end; t++) {
        const float4 vv = T.v;
        const float vx = vv.x * T.sc, vy = vv.y * T.sc, vz = vv.z * T.sc, vw = vv.w * T.sc, lam = T.lam;
        float o[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int m = 0; m < NR; m++) {
            const float kk = T.k[m], qq = T.q[m];
            S[m].x = fmaf(kk, vx, lam * S[m].x); S[m].y = fmaf(kk, vy, lam * S[m].y); S[m].z = fmaf(kk, vz, lam * S[m].z); S[m].w = fmaf(kk, vw, lam * S[m].w);
            o[0] = fmaf(S[m].x, qq, o[0]); o[1] = fmaf(S[m].y, qq, o[1]); o[2] = fmaf(S[m].z, qq, o[2]); o[3] = fmaf(S[m].w, qq, o[3]);
        }
        if (t + 1 < end) ask(T, t + 1);
        // over the wave's eight rows: lanes 8 apart
#pragma unroll
        for (int x = 0; x < 4; x++) { o[x] += pi_partner<8>(o[x]); o[x] += pi_partner<16>(o[x]); o[x] += pi_partner<32>(o[x]); }
        float (* const M)[32] = meet[t & 1];
        if (lane < 8) *(float4 *) &M[wave][quad * 4] = make_float4(o[0], o[1], o[2], o[3]);
        __syncthreads();
        if (tid < 8) {
            const float4 w0 = *(const float4 *) &M[0][quad * 4], w1 = *(const float4 *) &M[1][quad * 4], w2 = *(const float4 *) &M[2][quad * 4], w3 = *(const float4 *) &M[3][quad * 4];
            *(float4 *) (out + (int64_t) t * os + (int64_t) h * vdim + col) = make_float4(fmaf(skp, vv.x, (w0.x + w1.x) + (w2.x + w3.x)), fmaf(skp, vv.y, (w0.y + w1.y) + (w2.y + w3.y)),
                                                                                       fmaf(skp, vv.z, (w0.z + w1.z) + (w2.z + w3.z)), fmaf(skp, vv.w, (w0.w + w1.w) + (w2.w + w3.w)));
        }
    }
#pragma unroll
    for (int m = 0; m < NR; m++) *(float4 *) (S_hbm + (int64_t) 32 * m * vdim) = S[m];
}

// Long passes on the fp32 matrix cores (v_mfma_f32_16x16x4_f32), pieces of 64 or 32 tokens, for key widths of 32 DI <= 128.  What bounds the token loop of k_linear_attention is its chain: a token's state
// value waits for the one before, two products per state value on the vector units.  Per head and piece, with a_t = lambda_1 .. lambda_t and D[t][j] = lambda_{j+1} .. lambda_t (products only, no quotients):
//   O = a_t (Q S_in) + (Q K^T o D s) V,   S_out = a_64 S_in + sum_j (lambda_{j+1} .. lambda_64 s_j k_j) v_j^T
// k_linear_pieces: a pass of up to 64 tokens, every run one piece of up to 16, 32 or 64 tokens (a run of 16 tokens alone: 42 us with all four tiles, 23).  More tokens: k_linear_scores and k_linear_walk.
#define LM_TB 64
#define LM_MAX_TOKENS 16384                       // (the pass's slot words in LDS beside the 54 KB of a piece)
typedef float hy_f32x4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ hy_f32x4 hy_mfma(float a, float b, hy_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// base[i] with a 32-bit offset from a uniform base (an address per load in flight would not stay in registers)
typedef float hy_f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
static __device__ __forceinline__ float lm_at(const float * __restrict__ base, uint32_t i) { return *(const float *) ((const char *) base + i * 4u); }
static __device__ __forceinline__ hy_f32x4 lm_at4(const float * __restrict__ base, uint32_t i) { return *(const hy_f32x4_u *) ((const char *) base + i * 4u); }
// the value of token j of the piece in column c: the values end at vstored, a further column is ones
static __device__ __forceinline__ float lm_value(const float * __restrict__ vp, uint32_t j, uint32_t stride, int c, int vstored) { const float x = lm_at(vp, j * stride + (uint32_t) min(c, vstored - 1)); return c < vstored ? x : 1.0f; }
// the decays of a piece's tokens (a wave, a lane per token): decay, factor on k v^T (0 behind the piece's end), products of a tile of 16 up to this token and from the next one on, products 1 .. t, t + 1 .. 64 times the factor, a tile's
static __device__ __forceinline__ void lm_factors(int lane, int len, int64_t at, const float * __restrict__ decay, const float * __restrict__ tdecay, const float * __restrict__ tscale, int h, float * lam, float * sc, float * pre,
                                                  float * suf, float * upto, float * from, float * whole) {
    const int n = lane & 15, g = lane >> 4;
    const float l = lane >= len ? 1.0f : tdecay ? tdecay[at] : decay[h], s = lane < len ? (tscale ? tscale[at] : 1.0f) : 0.0f;
    float a = l, b = l;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) { const float x = __shfl_up(a, o, 16), y = __shfl_down(b, o, 16); if (n >= o) a *= x; if (n + o < 16) b *= y; }
    const float after = __shfl_down(b, 1, 16);
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = __shfl(a, 16 * i + 15, 64);
    float before = 1.0f, behind = 1.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) { if (i < g) before *= w[i]; if (i > g) behind *= w[i]; }
    const float s1 = n == 15 ? 1.0f : after;
    lam[lane] = l; sc[lane] = s;
    pre[lane] = a; suf[lane] = s1; upto[lane] = before * a; from[lane] = s1 * behind * s;
    if (n == 15) whole[g] = a;
}
// lambda_{j+1} .. lambda_t inside a tile of 16, in that order (a loop over them made a trip to LDS for each)
static __device__ __forceinline__ float lm_inside(const float * lam, int j, int t) {
    float d = 1.0f;
#pragma unroll
    for (int m = 1; m < 16; m++) { const float l = lam[m]; d *= m > j && m <= t ? l : 1.0f; }
    return d;
}
template <int DI>
__global__ void __launch_bounds__(256, 2) k_linear_pieces(const float * __restrict__ q, const float * __restrict__ k, const float * __restrict__ v, int64_t stride, int heads, int hpg, int vdim, int vstored,
                                                       const float * __restrict__ decay, const float * __restrict__ tdecay, const float * __restrict__ tscale, int64_t tds, const float * __restrict__ skip,
                                                       float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int DIM = 32 * DI, PITCH = DIM + 4, PP = LM_TB + 4;
    __shared__ __attribute__((aligned(16))) float qk[LM_TB * PITCH];  // the queries, then the keys
    __shared__ __attribute__((aligned(16))) float pt[LM_TB * PP];
    __shared__ int seg[4], bnd[LA_MAXRUNS], nbnd;
    __shared__ __attribute__((aligned(16))) float lam[LM_TB]; __shared__ float sc[LM_TB], upto[LM_TB], from[LM_TB], pre[LM_TB], suf[LM_TB], whole[4];     // decay, factor on k v^T; products: 1 .. t, t + 1 .. 64, and the same inside a tile of 16; a tile's
    extern __shared__ int lm_recs[];              // the slot words of the pass
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    for (int t = tid; t < n_tok; t += 256) lm_recs[t] = rec[t];
    if (pi_aborted_together(gone, abort_w)) return;
    const int n_runs = la_runs(lm_recs, n_tok, bnd, &nbnd);
    if (tid < 64) la_find_piece(lm_recs, n_tok, bnd, n_runs, 0, blockIdx.y, seg);
    __syncthreads();
    const int first = seg[0], len = seg[1], word = seg[2];
    if (len == 0 || word < 0) return;
    const int hq = h / hpg;
    const float * qp = q + (int64_t) first * stride + (int64_t) hq * DIM, * kp = k + (int64_t) first * stride + (int64_t) hq * DIM, * vp = v + (int64_t) first * stride + (int64_t) h * vstored;
    const int tiles = len <= 16 ? 1 : len <= 32 ? 2 : 4;              // of 16 tokens
    auto stage = [&](const float * src) {                             // rows behind the last repeat it: nothing of theirs is used
        for (int i = tid; i < 16 * tiles * DIM; i += 256) { const int t = i / DIM, d = i % DIM; qk[t * PITCH + d] = src[(int64_t) min(t, len - 1) * stride + d]; }
    };
    stage(qp);
    if (wave == 0) lm_factors(lane, len, (int64_t) (first + min(lane, len - 1)) * tds + h, decay, tdecay, tscale, h, lam, sc, pre, suf, upto, from, whole);
    __syncthreads();
    const int64_t per = (int64_t) DIM * vdim;
    float * S_hbm = state + ((int64_t) (word & ~LA_FRESH) * heads + h) * per;
    const bool zero = (word & LA_FRESH) != 0;
    const int n_tiles = (vdim + 15) / 16;
    {
        // (Q K^T o D s) transposed: tiles (rows j, columns t) on and below the diagonal, shared out among the waves; a lane's four rows are consecutive values of row t of pt
        for (int i = wave; i < tiles * (tiles + 1) / 2; i += 4) {
            const int tt = i < 1 ? 0 : i < 3 ? 1 : i < 6 ? 2 : 3, jt = i - tt * (tt + 1) / 2, j = 16 * jt + n;
            const float * kr = kp + (int64_t) min(j, len - 1) * stride;
            hy_f32x4 a = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int s = 0; s < 2 * DI; s++) {
                const hy_f32x4 qv = *(const hy_f32x4 *) &qk[(16 * tt + n) * PITCH + 16 * s + 4 * g];
#pragma unroll
                for (int c = 0; c < 4; c++) a = hy_mfma(kr[16 * s + 4 * g + c], qv[c], a);
            }
            const int t = 16 * tt + n;
            float between = 1.0f;
            for (int m = jt + 1; m < tt; m++) between *= whole[m];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int jr = 16 * jt + 4 * g + r;
                const float d = jt < tt ? suf[jr] * between * pre[t] : lm_inside(lam + 16 * tt, 4 * g + r, n);
                a[r] = jr <= t && jr < len ? a[r] * d * sc[jr] : 0.0f;
            }
            *(hy_f32x4 *) &pt[t * PP + 16 * jt + 4 * g] = a;
        }
        __syncthreads();
        auto outputs = [&](auto n_mt) {
            constexpr int MT = decltype(n_mt)::value;
            for (int nt = wave; nt < n_tiles; nt += 4) {
                const int c = 16 * nt + n, cc = min(c, vdim - 1);
                float sv[8 * DI];                                          // S_in: rows 16 s + 4 g + i of column c
#pragma unroll
                for (int s = 0; s < 2 * DI; s++)
#pragma unroll
                    for (int i = 0; i < 4; i++) { const float x = lm_at(S_hbm, (uint32_t) (16 * s + 4 * g + i) * (uint32_t) vdim + (uint32_t) cc); sv[4 * s + i] = zero ? 0.0f : x; }
                float vv[4 * MT];                                          // values: rows 16 jt + 4 g + r
#pragma unroll
                for (int i = 0; i < 4 * MT; i++) { const int j = 16 * (i >> 2) + 4 * g + (i & 3); vv[i] = lm_value(vp, min(j, len - 1), (uint32_t) stride, cc, vstored); }
                hy_f32x4 acc[MT];
#pragma unroll
                for (int m = 0; m < MT; m++) acc[m] = hy_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
                for (int s = 0; s < 2 * DI; s++) {
                    __builtin_amdgcn_sched_barrier(0);
                    hy_f32x4 qv[MT];
#pragma unroll
                    for (int m = 0; m < MT; m++) qv[m] = *(const hy_f32x4 *) &qk[(16 * m + n) * PITCH + 16 * s + 4 * g];
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int m = 0; m < MT; m++) acc[m] = hy_mfma(qv[m][i], sv[4 * s + i], acc[m]);
                }
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[m][r] *= upto[16 * m + 4 * g + r];
#pragma unroll
                for (int jt = 0; jt < MT; jt++) {
                    __builtin_amdgcn_sched_barrier(0);
                    uint32_t big = 0;                                      // (an infinity or a NaN among the values must not meet the zero weights of the tokens before it)
#pragma unroll
                    for (int r = 0; r < 4; r++) big = max(big, __float_as_uint(vv[4 * jt + r]) & 0x7fffffffu);
                    const bool odd = __any(big >= 0x7f800000u);
#pragma unroll
                    for (int m = jt; m < MT; m++) {
                        if (m == jt && odd) {
                            for (int j = 16 * jt; j < min(16 * jt + 16, len); j++) {
                                const float x = lm_value(vp, j, (uint32_t) stride, cc, vstored);
#pragma unroll
                                for (int r = 0; r < 4; r++) if (j <= 16 * m + 4 * g + r) acc[m][r] = fmaf(pt[(16 * m + 4 * g + r) * PP + j], x, acc[m][r]);
                            }
                            continue;
                        }
                        const hy_f32x4 pv = *(const hy_f32x4 *) &pt[(16 * m + n) * PP + 16 * jt + 4 * g];
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[m] = hy_mfma(pv[r], vv[4 * jt + r], acc[m]);
                    }
                }
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int t = 16 * m + 4 * g + r;
                        if (t >= len || c >= vdim) continue;
                        __builtin_amdgcn_sched_barrier(0);
                        float o = acc[m][r];
                        if (skip) o = fmaf(skip[h], lm_value(vp, t, (uint32_t) stride, c, vstored), o);
                        out[(int64_t) (first + t) * os + (int64_t) h * vdim + c] = o;
                    }
            }
        };
        if (tiles == 1) outputs(std::integral_constant<int, 1>{});
        else if (tiles == 2) outputs(std::integral_constant<int, 2>{});
        else outputs(std::integral_constant<int, 4>{});
        __syncthreads();
        stage(kp);
        __syncthreads();
    }
    // the slot's new state
    const float all = upto[LM_TB - 1];
    auto states = [&](auto n_mt) {
        constexpr int MT = decltype(n_mt)::value;
        for (int nt = wave; nt < n_tiles; nt += 4) {
            const int c = 16 * nt + n, cc = min(c, vdim - 1);
            float vv[4 * MT];
#pragma unroll
            for (int i = 0; i < 4 * MT; i++) { const int j = 16 * (i >> 2) + 4 * g + (i & 3); vv[i] = j < len ? lm_value(vp, min(j, len - 1), (uint32_t) stride, cc, vstored) * from[j] : 0.0f; }
            hy_f32x4 acc[2 * DI];
#pragma unroll
            for (int m = 0; m < 2 * DI; m++) acc[m] = hy_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int i = 0; i < 4 * MT; i++) {
                __builtin_amdgcn_sched_barrier(0);
                const float * kr = &qk[(16 * (i >> 2) + 4 * g + (i & 3)) * PITCH + n];
#pragma unroll
                for (int m = 0; m < 2 * DI; m++) acc[m] = hy_mfma(kr[16 * m], vv[i], acc[m]);
            }
            if (c < vdim)
#pragma unroll
                for (int m = 0; m < 2 * DI; m++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const uint32_t at = ((uint32_t) (16 * m + 4 * g + r) * (uint32_t) vdim + (uint32_t) c) * 4u;
                        if (r == 0) __builtin_amdgcn_sched_barrier(0);
                        *(float *) ((char *) S_hbm + at) = zero ? acc[m][r] : fmaf(all, *(const float *) ((const char *) S_hbm + at), acc[m][r]);
                    }
        }
    };
    if (tiles == 1) states(std::integral_constant<int, 1>{});
    else if (tiles == 2) states(std::integral_constant<int, 2>{});
    else states(std::integral_constant<int, 4>{});
}

// A pass of more than 64 tokens, in pieces of 32: the scores of every piece side by side, then every run walked piece by piece with its state in registers.  (States of all pieces from zero, a scan that chains them and the outputs
// from every piece's true state moved 64 KB per piece and head four times: 2048 tokens, 32 heads of 128 x 128: 93 + 31 + 140 us, now 30 + 87; 512 tokens, 16 heads: 27 + 8 + 60, now 9 + 24.)
// scratch per (piece, head): (Q K^T o D s) [32 t][32 j], nothing in the tile above the diagonal | lambda_1 .. lambda_t [32] | lambda_{j+1} .. lambda_32 s_j [32] (0 behind the piece's end)
#define LW_TB 32
#define LW_SCR (LW_TB * LW_TB + 2 * LW_TB)
#define LW_LDS(DI) (4 * LW_TB * (32 * (DI) + 4) * 4)        /* k_linear_walk: two buffers of queries and of keys */
// grid (head, piece): queries and keys through LDS (a matrix operand straight from memory is sixteen rows at a time, 59 clocks of the address unit a load), a wave to each of the three tiles
template <int DI>
__global__ void __launch_bounds__(256) k_linear_scores(const float * __restrict__ q, const float * __restrict__ k, int64_t stride, int heads, int hpg, const float * __restrict__ decay, const float * __restrict__ tdecay,
                                                       const float * __restrict__ tscale, int64_t tds, const int32_t * __restrict__ rec, int n_tok, float * __restrict__ scratch, const int32_t * __restrict__ abort_w) {
    if (pi_aborted_together(pi_abort_peek(abort_w), abort_w)) return;
    constexpr int DIM = 32 * DI, PITCH = DIM + 4;
    __shared__ __attribute__((aligned(16))) float qs[LW_TB * PITCH], ks[LW_TB * PITCH];
    __shared__ int seg[4], bnd[LA_MAXRUNS], nbnd;
    __shared__ __attribute__((aligned(16))) float lam[64];
    __shared__ float sc[64], pre[64], suf[64], upto[64], from[64], whole[4];
    extern __shared__ int lm_recs[];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    if (la_one_run(rec, n_tok)) {
        if (tid == 0) { seg[0] = (int) blockIdx.y * LW_TB; seg[1] = max(0, min(LW_TB, n_tok - (int) blockIdx.y * LW_TB)); seg[2] = rec[0]; }
    } else {
        for (int t = tid; t < n_tok; t += 256) lm_recs[t] = rec[t];
        __syncthreads();
        const int n_runs = la_runs(lm_recs, n_tok, bnd, &nbnd);
        if (tid < 64) la_find_piece(lm_recs, n_tok, bnd, n_runs, LW_TB, blockIdx.y, seg);
    }
    __syncthreads();
    const int first = seg[0], len = seg[1], word = seg[2];
    if (len == 0 || word < 0) return;
    const float * qp = q + (int64_t) first * stride + (int64_t) (h / hpg) * DIM, * kp = k + (int64_t) first * stride + (int64_t) (h / hpg) * DIM;
    hy_f32x4 x[2 * DI];
#pragma unroll
    for (int i = 0; i < DI; i++) {
        const int at = tid + 256 * i, t = at / (DIM / 4), d = at % (DIM / 4) * 4;
        const uint32_t o = (uint32_t) min(t, len - 1) * (uint32_t) stride + d;
        x[2 * i] = lm_at4(qp, o); x[2 * i + 1] = lm_at4(kp, o);
    }
    if (wave == 3) lm_factors(lane, len, (int64_t) (first + min(lane, len - 1)) * tds + h, decay, tdecay, tscale, h, lam, sc, pre, suf, upto, from, whole);
#pragma unroll
    for (int i = 0; i < DI; i++) {
        const int at = tid + 256 * i, t = at / (DIM / 4), d = at % (DIM / 4) * 4;
        *(hy_f32x4 *) &qs[t * PITCH + d] = x[2 * i]; *(hy_f32x4 *) &ks[t * PITCH + d] = x[2 * i + 1];
    }
    __syncthreads();
    float * own = scratch + ((int64_t) blockIdx.y * heads + h) * LW_SCR;
    if (wave == 3) { own[LW_TB * LW_TB + lane] = lane < LW_TB ? upto[lane] : from[lane - LW_TB]; return; }
    const int tt = wave == 0 ? 0 : 1, jt = wave == 2 ? 1 : 0, t = 16 * tt + n;
    if (16 * tt >= len) return;
    hy_f32x4 a = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
    for (int s = 0; s < 2 * DI; s++) {
        const hy_f32x4 kv = *(const hy_f32x4 *) &ks[(16 * jt + n) * PITCH + 16 * s + 4 * g], qv = *(const hy_f32x4 *) &qs[t * PITCH + 16 * s + 4 * g];
#pragma unroll
        for (int e = 0; e < 4; e++) a = hy_mfma(kv[e], qv[e], a);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {                                     // transposed: a lane's four rows j are consecutive values of row t
        const int jr = 16 * jt + 4 * g + r;
        const float d = jt < tt ? suf[jr] * pre[t] : lm_inside(lam + 16 * tt, 4 * g + r, n);
        a[r] = jr <= t && jr < len ? a[r] * d * sc[jr] : 0.0f;
    }
    *(hy_f32x4 *) (own + t * LW_TB + 16 * jt + 4 * g) = a;
}
// grid (head, sixteen columns of values, run): the run's pieces in order.  Wave w keeps 16 MW rows of the state in registers as the matrix cores leave them, which is how they take them for Q S: row 16 MW w + MW (4 g + r) + i in
// register r of tile i, so that a lane's keys are MW neighbours.  Of a piece it computes Q S over those rows for all tokens, a quarter of P V (value r = w of every four), and its rows' new state; the four waves' shares of an output
// meet in LDS.  Four more waves bring the pieces' queries, keys, values and scores through LDS in two buffers, two pieces ahead in registers, and add up and write the outputs: one barrier a piece.  Bound by the chain of a piece, whatever the number of heads: 35 products of 32 clocks
// and two trips through LDS.
template <int DI>
__global__ void __launch_bounds__(512, 2) k_linear_walk(const float * __restrict__ q, const float * __restrict__ k, const float * __restrict__ v, int64_t stride, int heads, int hpg, int vdim, int vstored,
                                                        const float * __restrict__ skip, float * __restrict__ state, const int32_t * __restrict__ rec, int n_tok, const float * __restrict__ scratch, float * __restrict__ out,
                                                        int64_t os, const int32_t * __restrict__ abort_w) {
    if (pi_aborted_together(pi_abort_peek(abort_w), abort_w)) return;
    constexpr int DIM = 32 * DI, MW = (2 * DI + 3) / 4, PITCH = DIM + 4, PP = LW_TB + 4;
    __shared__ int seg[4], bnd[LA_MAXRUNS], nbnd;
    __shared__ __attribute__((aligned(16))) float vs[2][LW_TB * 16], ps[2][LW_TB * PP], fs[2][2 * LW_TB];
    __shared__ hy_f32x4 part[2][4][2][64];                             // [piece % 2][wave][tile of tokens][lane]
    extern __shared__ __attribute__((aligned(16))) float lw_lds[];     // queries and keys, two buffers each; ahead of them the slot words of the pass
    int * const lm_recs = (int *) lw_lds; float * const qs = lw_lds, * const ks = lw_lds + 2 * LW_TB * PITCH;
    constexpr int BUF = LW_TB * PITCH;
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, g = lane >> 4;
    if (la_one_run(rec, n_tok)) {
        if (tid == 0) { seg[0] = 0; seg[1] = 0; seg[2] = blockIdx.z == 0 ? n_tok : 0; seg[3] = rec[0]; }
    } else {
        for (int t = tid; t < n_tok; t += 512) lm_recs[t] = rec[t];
        __syncthreads();
        const int n_runs = la_runs(lm_recs, n_tok, bnd, &nbnd);
        if (tid < 64) {
            int own[4], ord = la_pieces_before(bnd, n_runs, n_tok, LW_TB, own);
            if (tid == 0) seg[2] = 0;
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const int r = 4 * tid + x;
                if (r == (int) blockIdx.z && r < n_runs) { seg[0] = bnd[r]; seg[1] = ord; seg[2] = (r + 1 < n_runs ? bnd[r + 1] : n_tok) - bnd[r]; seg[3] = lm_recs[bnd[r]]; }
                ord += own[x];
            }
        }
    }
    __syncthreads();
    const int run0 = seg[0], run_len = seg[2], word = seg[3], c0 = (int) blockIdx.y * 16, c = c0 + n, cc = min(c, vdim - 1);
    const int64_t ord0 = seg[1];
    if (run_len == 0 || word < 0) return;
    const int pieces = (run_len + LW_TB - 1) / LW_TB;
    float * S_hbm = state + ((int64_t) (word & ~LA_FRESH) * heads + h) * (int64_t) DIM * vdim;
    const float skp = skip ? skip[h] : 0.0f;
    const bool walks = wave < 4;
    const int st = tid & 255;                                          // of the four waves that bring the pieces
    auto row_of = [&](int i, int r) { return 16 * MW * wave + MW * (4 * g + r) + i; };
    hy_f32x4 S[MW];
    if (walks)
#pragma unroll
    for (int i = 0; i < MW; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) { const int row = row_of(i, r); const float x = lm_at(S_hbm, (uint32_t) min(row, DIM - 1) * (uint32_t) vdim + (uint32_t) cc); S[i][r] = (word & LA_FRESH) || row >= DIM ? 0.0f : x; }
    // what this thread brings of a piece: DI runs of four values of the queries and of the keys, two values, four scores, one factor
    struct piece_regs { hy_f32x4 q[DI], k[DI], p; float v[2], f; } R[2];
    const int vt = st >> 4, vc = min(c0 + (st & 15), vstored - 1);
    auto fetch = [&](piece_regs & F, int p) __attribute__((always_inline)) {
        const int len = min(LW_TB, run_len - p * LW_TB);
        const int64_t first = run0 + (int64_t) p * LW_TB;
        const float * qp = q + first * stride + (int64_t) (h / hpg) * DIM, * kp = k + first * stride + (int64_t) (h / hpg) * DIM, * vp = v + first * stride + (int64_t) h * vstored;
        const float * own = scratch + ((ord0 + p) * heads + h) * LW_SCR;
#pragma unroll
        for (int i = 0; i < DI; i++) {
            const int at = st + 256 * i, t = at / (DIM / 4), d = at % (DIM / 4) * 4;      // (rows behind the last repeat it)
            const uint32_t o = (uint32_t) min(t, len - 1) * (uint32_t) stride + d;
            F.q[i] = lm_at4(qp, o); F.k[i] = lm_at4(kp, o);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) F.v[i] = lm_at(vp, (uint32_t) min(vt + 16 * i, len - 1) * (uint32_t) stride + (uint32_t) vc);
        F.p = *(const hy_f32x4 *) (own + 4 * st);
        F.f = own[LW_TB * LW_TB + (st & 63)];
    };
    auto stage = [&](piece_regs & F, int p) __attribute__((always_inline)) {
        const int b = p & 1, len = min(LW_TB, run_len - p * LW_TB);
#pragma unroll
        for (int i = 0; i < DI; i++) {
            const int at = st + 256 * i, t = at / (DIM / 4), d = at % (DIM / 4) * 4;
            *(hy_f32x4 *) &qs[b * BUF + t * PITCH + d] = F.q[i]; *(hy_f32x4 *) &ks[b * BUF + t * PITCH + d] = F.k[i];
        }
#pragma unroll
        for (int i = 0; i < 2; i++) vs[b][st + 256 * i] = vt + 16 * i >= len ? 0.0f : c0 + (st & 15) < vstored ? F.v[i] : 1.0f;      // (a column the values do not have: ones)
        *(hy_f32x4 *) &ps[b][(st >> 3) * PP + (st & 7) * 4] = F.p;
        if (st < 64) fs[b][st] = F.f;
    };
    const int own_rows = 16 * MW * min(wave, 2 * DI / MW - 1);        // (a wave without rows repeats the last ones: its state is zero and stays so)
    typedef float keys __attribute__((ext_vector_type(MW)));
    auto compute = [&](int p) __attribute__((always_inline)) {
        const int b = p & 1, len = min(LW_TB, run_len - p * LW_TB);
        hy_f32x4 qv[2][MW], o[2], up[2], w[2]; keys kv[8]; float vv[8], pv[2], pw[3];
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int i = 0; i < MW; i++) qv[tt][i] = *(const hy_f32x4 *) &qs[b * BUF + (16 * tt + n) * PITCH + own_rows + 4 * MW * g + 4 * i];
#pragma unroll
        for (int tt = 0; tt < 2; tt++) { w[tt] = *(const hy_f32x4 *) &fs[b][LW_TB + 16 * tt + 4 * g]; up[tt] = *(const hy_f32x4 *) &fs[b][16 * tt + 4 * g]; }
        const float all = fs[b][LW_TB - 1];
#pragma unroll
        for (int x = 0; x < 8; x++) { const int t = 16 * (x >> 2) + 4 * g + (x & 3); vv[x] = vs[b][t * 16 + n]; kv[x] = *(const keys *) &ks[b * BUF + t * PITCH + own_rows + MW * n]; }
#pragma unroll
        for (int jt = 0; jt < 2; jt++) pv[jt] = vs[b][(16 * jt + 4 * g + wave) * 16 + n];
        pw[0] = ps[b][n * PP + 4 * g + wave]; pw[1] = ps[b][(16 + n) * PP + 4 * g + wave]; pw[2] = ps[b][(16 + n) * PP + 16 + 4 * g + wave];
        o[0] = o[1] = hy_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < MW; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int tt = 0; tt < 2; tt++) o[tt] = hy_mfma(qv[tt][(MW * e + i) >> 2][(MW * e + i) & 3], S[i][e], o[tt]);
        // the piece's new state: what is left of its keys' products at its end
#pragma unroll
        for (int i = 0; i < MW; i++) S[i] *= all;
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const float vw = wave * MW < 2 * DI && 16 * (x >> 2) + 4 * g + (x & 3) < len ? vv[x] * w[x >> 2][x & 3] : 0.0f;
#pragma unroll
            for (int i = 0; i < MW; i++) S[i] = hy_mfma(kv[x][i], vw, S[i]);
        }
        o[0] *= up[0]; o[1] *= up[1];
        // an infinity or a NaN among the values must not meet the zero weights of the tokens before it: the diagonal's tiles then go value by value, in the first wave
        const uint32_t big = max(__float_as_uint(pv[0]) & 0x7fffffffu, __float_as_uint(pv[1]) & 0x7fffffffu);
        const bool odd = __any(big >= 0x7f800000u);
        hy_f32x4 (* meet)[2][64] = part[b];
        if (!odd) { o[0] = hy_mfma(pw[0], pv[0], o[0]); o[1] = hy_mfma(pw[2], pv[1], o[1]); }
        else
#pragma unroll
            for (int tt = 0; tt < 2; tt++)
                for (int gg = 0; gg < 4; gg++) {                       // (the keys 4 gg + w: this wave's share of them)
                    const int j = 16 * tt + 4 * gg + wave;
                    const float x = vs[b][j * 16 + n];
#pragma unroll
                    for (int r = 0; r < 4; r++) if (j <= 16 * tt + 4 * g + r && j < len) o[tt][r] = fmaf(ps[b][(16 * tt + 4 * g + r) * PP + j], x, o[tt][r]);
                }
        o[1] = hy_mfma(pw[1], pv[0], o[1]);
        meet[wave][0][lane] = o[0]; meet[wave][1][lane] = o[1];
    };
    auto finish = [&](int p) __attribute__((always_inline)) {
        const int b = p & 1, len = min(LW_TB, run_len - p * LW_TB), tt = (wave & 3) >> 1, half = wave & 1;
        const int64_t first = run0 + (int64_t) p * LW_TB;
        typedef float two __attribute__((ext_vector_type(2)));
        two y[4];
#pragma unroll
        for (int x = 0; x < 4; x++) y[x] = *(const two *) ((const float *) &part[b][x][tt][lane] + 2 * half);
        const two sum = (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int t = 16 * tt + 4 * g + 2 * half + r;
            if (t >= len || c >= vdim) continue;
            out[(first + t) * os + (int64_t) h * vdim + c] = skip ? fmaf(skp, lm_value(v + first * stride + (int64_t) h * vstored, t, (uint32_t) stride, c, vstored), sum[r]) : sum[r];
        }
    };
    auto meet_all = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };      // (loads stay on their way)
    // Between two barriers the walking waves compute piece p while the others sum up piece p - 1, put piece p + 1 into the other buffer and ask for piece p + 3.  (The walkers doing all of it, one thing after another: 120 us, now 87)
    if (!walks) {
        // (always two next ones, behind the last piece that again, and no way out between two pieces: where paths with different loads on their way meet, the compiler waits for the younger ones too)
        fetch(R[0], 0);
        fetch(R[1], min(1, pieces - 1));
        stage(R[0], 0);
        fetch(R[0], min(2, pieces - 1));
        meet_all();
        auto step = [&](int p, piece_regs & F) __attribute__((always_inline)) {
            if (p > 0) finish(p - 1);
            stage(F, p + 1);                                           // (behind the last piece: of no use)
            fetch(F, min(p + 3, pieces - 1));
            meet_all();
        };
        int p = 0;
        for (; p + 2 <= pieces; p += 2) { step(p, R[1]); step(p + 1, R[0]); }
        if (p < pieces) step(p, R[1]);
        finish(pieces - 1);
        return;
    }
    meet_all();
    for (int p = 0; p < pieces; p++) { compute(p); meet_all(); }
    if (c < vdim)
#pragma unroll
        for (int i = 0; i < MW; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) { const int row = row_of(i, r); if (row < DIM) S_hbm[(int64_t) row * vdim + c] = S[i][r]; }
}

// grid (head, blocks over dim * vdim, run): scratch[piece] holds L_p coming in and S_in(p) going out
template <int TB>
__global__ void __launch_bounds__(256) k_linear_state_scan(int heads, int dim, int vdim, const float * __restrict__ decay, const float * __restrict__ tdecay, int64_t tds, const float * __restrict__ state,
                                                           const int32_t * __restrict__ rec, int n_tok, float * __restrict__ scratch, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ int seg[4], bnd[LA_MAXRUNS], nbnd; // seg: slot word, first piece ordinal, pieces of the run (0: no such run), the run's first token
    extern __shared__ int recs[];                 // the slot words of the pass
    for (int t = threadIdx.x; t < n_tok; t += 256) recs[t] = rec[t];
    if (pi_aborted_together(gone, abort_w)) return;
    const int n_runs = la_runs(recs, n_tok, bnd, &nbnd);
    if (threadIdx.x < 64) {
        int own[4], ord = la_pieces_before(bnd, n_runs, n_tok, TB, own);
        if (threadIdx.x == 0) seg[2] = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int r = 4 * (int) threadIdx.x + k;
            if (r == (int) blockIdx.z && r < n_runs) { seg[0] = recs[bnd[r]]; seg[1] = ord; seg[2] = own[k]; seg[3] = bnd[r]; }
            ord += own[k];
        }
    }
    __syncthreads();
    const int word = seg[0], sub0 = seg[1], nsub = seg[2], tfirst = seg[3];
    if (nsub == 0 || word < 0) return;
    const int h = blockIdx.x, slot = word & ~LA_FRESH;
    const int64_t per = (int64_t) dim * vdim, idx = (int64_t) blockIdx.y * 256 + threadIdx.x;
    const bool in = idx < per;
    constexpr int ND = 256 / TB;                                       // pieces whose per-token decays are multiplied out in a round, a thread per token (the TB <= 64 lanes of a piece meet)
    __shared__ float lps[8];
    float lp = 1.0f;                                                   // lambda^TB: every piece but a run's last has TB tokens
    if (!tdecay) for (int i = 0; i < TB; i++) lp *= decay[h];
    float run = !in || (word & LA_FRESH) ? 0.0f : state[((int64_t) slot * heads + h) * per + idx];
    for (int p0 = 0; p0 < nsub; p0 += 8) {                             // eight pieces at a time: their loads are in flight together, then the chain runs on registers
        float lpart[8];
#pragma unroll
        for (int i = 0; i < 8; i++) lpart[i] = in && p0 + i < nsub - 1 ? scratch[((int64_t) (sub0 + p0 + i) * heads + h) * per + idx] : 0.0f;
        if (tdecay) {
            __syncthreads();                                           // (the previous eight are no longer read)
            for (int pb = 0; pb < 8; pb += ND) {
                const int pi = pb + threadIdx.x / TB;
                float d = p0 + pi < nsub - 1 ? tdecay[(int64_t) (tfirst + (p0 + pi) * TB + threadIdx.x % TB) * tds + h] : 1.0f;        // (only whole pieces are multiplied out)
                for (int o = TB >> 1; o > 0; o >>= 1) d *= __shfl_xor(d, o, PI_WAVE);
                if (threadIdx.x % TB == 0) lps[pi] = d;
            }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (in && p0 + i < nsub) {
                scratch[((int64_t) (sub0 + p0 + i) * heads + h) * per + idx] = run;
                run = fmaf(tdecay ? lps[i] : lp, run, lpart[i]);
            }
    }
}

// once per process, outside graph capture: the tiles of wide keys (q, k of 32 tokens) need more dynamic LDS than a kernel gets by default
#define LA_LDS_MAX (150 * 1024)
extern "C" int pi_op_linear_attention_reserve(void) {
    static bool done = false;
    if (done) return 0;
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_attention<8>, hipFuncAttributeMaxDynamicSharedMemorySize, LA_LDS_MAX));
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_attention<16>, hipFuncAttributeMaxDynamicSharedMemorySize, LA_LDS_MAX));
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_attention<32>, hipFuncAttributeMaxDynamicSharedMemorySize, LA_LDS_MAX));
#define LM_RES(DI) PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_scores<DI>, hipFuncAttributeMaxDynamicSharedMemorySize, 4 * LM_MAX_TOKENS)); \
                   PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_walk<DI>, hipFuncAttributeMaxDynamicSharedMemorySize, std::max(4 * LM_MAX_TOKENS, LW_LDS(DI))));
    LM_RES(1) LM_RES(2) LM_RES(3) LM_RES(4)
#undef LM_RES
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_linear_state_scan<LA_TB>, hipFuncAttributeMaxDynamicSharedMemorySize, LA_LDS_MAX));
    done = true;
    return 0;
}
static int la_max_pieces(int n_tok, int max_segments) { return n_tok / LA_TB + std::min(n_tok, std::max(1, max_segments)) + 1; }
extern "C" size_t pi_op_linear_attention_scratch_floats(int heads, int dim, int vdim, int n_tok, int max_segments) {
    return n_tok <= LA_TB ? 0 : (size_t) heads * std::max((size_t) la_max_pieces(n_tok, max_segments) * dim * vdim, dim % 32 == 0 && dim <= 128 ? (size_t) la_max_pieces(n_tok, max_segments) * LW_SCR : (size_t) 0);
}
extern "C" int pi_op_linear_attention(const float * q, const float * k, const float * v, int64_t stride, int heads, int dim, int vdim, const float * decay_dev, float * state_dev,
                                      const int32_t * rec_dev, int n_tok, int max_segments, float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride, void * stream) {
    return pi_op_linear_attention_ex(q, k, v, stride, heads, heads, dim, vdim, decay_dev, nullptr, nullptr, 0, nullptr, state_dev, rec_dev, n_tok, max_segments, scratch_dev, scratch_floats, out, out_stride, stream);
}
extern "C" int pi_op_linear_attention_ex(const float * q, const float * k, const float * v, int64_t stride, int heads, int qk_heads, int dim, int vdim, const float * decay_dev, const float * tdecay_dev,
                                         const float * tscale_dev, int64_t t_stride, const float * skip_dev, float * state_dev, const int32_t * rec_dev, int n_tok, int max_segments, float * scratch_dev,
                                         size_t scratch_floats, float * out, int64_t out_stride, void * stream) {
    return pi_op_linear_attention_keysum(q, k, v, stride, heads, qk_heads, dim, vdim, 0, decay_dev, tdecay_dev, tscale_dev, t_stride, skip_dev, state_dev, rec_dev, n_tok, max_segments, scratch_dev, scratch_floats, out, out_stride, stream);
}
extern "C" int pi_op_linear_attention_keysum(const float * q, const float * k, const float * v, int64_t stride, int heads, int qk_heads, int dim, int value_cols, int key_sum, const float * decay_dev, const float * tdecay_dev,
                                             const float * tscale_dev, int64_t t_stride, const float * skip_dev, float * state_dev, const int32_t * rec_dev, int n_tok, int max_segments, float * scratch_dev,
                                             size_t scratch_floats, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0) return 0;
    const int vdim = value_cols + (key_sum ? 1 : 0);                   // columns of the state and of an output row per head
    if (qk_heads < 1 || heads % qk_heads) { pi_set_error("pi_op_linear_attention: %d heads do not divide over %d query / key heads", heads, qk_heads); return -1; }
    if (!decay_dev && !tdecay_dev) { pi_set_error("pi_op_linear_attention: neither per-head nor per-token decays were given"); return -1; }
    const int hpg = heads / qk_heads;
    if (dim <= 0 || value_cols <= 0 || heads <= 0 || dim > 1024) { pi_set_error("pi_op_linear_attention: head sizes %d x %d outside the kernel's range (key width <= 1024)", dim, vdim); return -1; }
    if (max_segments > LA_MAXRUNS) { pi_set_error("pi_op_linear_attention: at most %d sequences in a pass", LA_MAXRUNS); return -1; }
    const int dpt = dim <= 8 ? 8 : dim <= 16 ? 16 : 32;                // state values a thread keeps in registers (more would spill in the token loop)
    int R = 1; while (R * dpt < dim) R *= 2;
    int threads = std::min(256, (vdim * R + 63) / 64 * 64);
    if (key_sum && R <= 64) {                                          // one column more than a round number: blocks of the size that leaves the fewest lanes without a column
        int best = 1 << 30;
        const int b0 = (vdim * R + 255) / 256;
        for (int b = b0; b < b0 + 8; b++) {
            const int waves = ((vdim + b - 1) / b * R + 63) / 64;
            if (b * waves < best) { best = b * waves; threads = waves * 64; }
        }
    }
    const int cols = threads / R;
    const bool pieces = n_tok > LA_TB;
    if (pieces && (!scratch_dev || scratch_floats < pi_op_linear_attention_scratch_floats(heads, dim, vdim, n_tok, max_segments))) { pi_set_error("pi_op_linear_attention: a pass of %d tokens needs %zu floats of scratch", n_tok, pi_op_linear_attention_scratch_floats(heads, dim, vdim, n_tok, max_segments)); return -1; }
    const unsigned gz = pieces ? (unsigned) la_max_pieces(n_tok, max_segments) : (unsigned) std::max(1, std::min(n_tok, max_segments));
    const dim3 grid((unsigned) heads, (unsigned) ((vdim + cols - 1) / cols), gz);
    const size_t lds = ((size_t) 2 * LA_TB * dim + (size_t) LA_TB * cols + (size_t) n_tok) * sizeof(float);
    if (lds > LA_LDS_MAX) { pi_set_error("pi_op_linear_attention: a key width of %d with %d tokens in the pass needs %zu bytes of LDS (at most %d)", dim, n_tok, lds, LA_LDS_MAX); return -1; }
    if (lds > 48 * 1024 && pi_op_linear_attention_reserve() != 0) return -1;
    const double bytes = 4.0 * n_tok * heads * (2.0 * dim + 2.0 * vdim) + 8.0 * heads * dim * vdim;
    hipStream_t s = (hipStream_t) stream;
    const int nta = std::min(n_tok, PI_KT_MAXNT - 1);
#define LA_GO(D, MODE) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, k_linear_attention<D>, grid, dim3(threads), lds, s, q, k, v, stride, heads, hpg, dim, vdim, value_cols, R, decay_dev, tdecay_dev, tscale_dev, t_stride, skip_dev, state_dev, rec_dev, n_tok, MODE, scratch_dev, out, out_stride, pi_abort_word())
#define LA_ANY(MODE) do { if (dpt == 8) LA_GO(8, MODE); else if (dpt == 16) LA_GO(16, MODE); else LA_GO(32, MODE); } while (0)
    const bool matrix = dim % 32 == 0 && dim <= 128 && n_tok <= LM_MAX_TOKENS && stride < (1 << 24) && vdim <= (1 << 22);       // (32-bit offsets within a piece)
    const unsigned gr = (unsigned) std::max(1, std::min(n_tok, max_segments)), gb = (unsigned) (((int64_t) dim * vdim + 255) / 256);
#define LM_ANY(GO) do { if (dim == 32) GO(1); else if (dim == 64) GO(2); else if (dim == 96) GO(3); else GO(4); } while (0)
#define LM_PIECES(DI) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, k_linear_pieces<DI>, dim3((unsigned) heads, gr), dim3(256), (size_t) 4 * n_tok, s, q, k, v, stride, heads, hpg, vdim, value_cols, decay_dev, tdecay_dev, tscale_dev, t_stride, \
                                   skip_dev, state_dev, rec_dev, n_tok, out, out_stride, pi_abort_word())
#define LM_SCORES(DI) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, 4.0 * n_tok * heads * (2 * dim + LW_TB), k_linear_scores<DI>, dim3((unsigned) heads, (unsigned) la_max_pieces(n_tok, max_segments)), dim3(256), (size_t) 4 * n_tok, s, q, k, stride, heads, hpg, \
                                   decay_dev, tdecay_dev, tscale_dev, t_stride, rec_dev, n_tok, scratch_dev, pi_abort_word())
#define LM_WALK(DI) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, k_linear_walk<DI>, dim3((unsigned) heads, (unsigned) ((vdim + 15) / 16), gr), dim3(512), std::max((size_t) 4 * n_tok, (size_t) LW_LDS(DI)), s, q, k, v, stride, heads, hpg, vdim, value_cols, skip_dev, state_dev, \
                                 rec_dev, n_tok, scratch_dev, out, out_stride, pi_abort_word())
    // Up to 64 tokens every run is one piece: one launch from the slots' states to the slots' states.  Beyond LA_TB always (32 heads of 128 x 128, three launches against it: a run of 64 tokens 55 -> 48 us, 64 runs of a
    // token 450 -> 123, for the pieces are walked twice and the scan starts for every run); up to there where the walk, whose time is its longest run's (7 us and 1.9 a token), has more than eight tokens in one whatever the runs are
    // (24 tokens 53 -> 29, 9 about even; eight runs of a token or two 14 .. 18, here 25 .. 29)
    // The step's kernel walks a run at 0.6 us a token, the pieces below take 9 .. 29 us for up to 32: us of one run, step / pieces, 16 heads: key width 32 12 tokens 8.0 / 9.5, 16 10.1 / 9.4; 64 20 tokens 13.0 / 13.9, 24 14.3 / 14.0; 96 32
    // tokens 19.5 / 25.8; 128 32 tokens 20.9 / 29.1; of values of 64 and less, whose states are the fewer loads, 96 28 tokens 17.6 / 18.8, 32 19.9 / 19.0, 128 32
    // tokens 21.0 / 20.1.  The host knows how many runs there may be, not how many there are: one may have all tokens, so the line is a single run's; and no fewer tokens than those that k_linear_attention's walk would take otherwise
    // (24 tokens of width 32 as one run: where there may be two 13.4 by the step and 10.5 by the pieces, where there may be three 13.3 by the step and 38 by that walk; 32 of width 64, two 18.7 and 14.3)
    const int alone = dim == 32 ? 12 : dim == 64 ? 20 : vdim <= 64 ? 28 : LA_TB;
    if (n_tok <= LA_TB && matrix && n_tok <= std::max(alone, 8 * (int) gr) && !key_sum && vdim % 32 == 0 && stride % 4 == 0 && out_stride % 4 == 0 && (((uintptr_t) v | (uintptr_t) out | (uintptr_t) state_dev) & 15) == 0) {
#define LS_GO(NR) PI_KT_LAUNCH(PI_KT_ATT, 0, nta, bytes, k_linear_step<NR>, dim3((unsigned) heads, (unsigned) (vdim / 32), gr), dim3(256), 0, s, q, k, v, stride, heads, hpg, vdim, decay_dev, tdecay_dev, tscale_dev, t_stride, skip_dev, state_dev, \
                               rec_dev, n_tok, out, out_stride, pi_abort_word())
        LM_ANY(LS_GO);
#undef LS_GO
        PI_CHECK_LAUNCH(); return 0;
    }
    if (matrix && n_tok <= LM_TB && (pieces || n_tok > 8 * gr)) {
        LM_ANY(LM_PIECES);
        PI_CHECK_LAUNCH(); return 0;
    }
    if (!pieces) { LA_ANY(0); PI_CHECK_LAUNCH(); return 0; }
    if (matrix) {
        if (pi_op_linear_attention_reserve() != 0) return -1;
        LM_ANY(LM_SCORES);
        PI_CHECK_LAUNCH();
        LM_ANY(LM_WALK);
        PI_CHECK_LAUNCH(); return 0;
    }
#undef LM_ANY
#undef LM_PIECES
#undef LM_SCORES
#undef LM_WALK
    LA_ANY(1);
    PI_CHECK_LAUNCH();
    PI_KT_LAUNCH(PI_KT_ATT, 0, nta, 12.0 * gz * heads * dim * vdim, k_linear_state_scan<LA_TB>, dim3((unsigned) heads, gb, gr), dim3(256), (size_t) 4 * n_tok, s,
                 heads, dim, vdim, decay_dev, tdecay_dev, t_stride, state_dev, rec_dev, n_tok, scratch_dev, pi_abort_word());
    PI_CHECK_LAUNCH();
    LA_ANY(2);
#undef LA_ANY
#undef LA_GO
    PI_CHECK_LAUNCH(); return 0;
}

// copies the state of one slot to another, all heads of one layer (sequence copy)
__global__ void k_copy_f32(const float * __restrict__ src, float * __restrict__ dst, int64_t n) {
    for (int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t) gridDim.x * 256) dst[i] = src[i];
}
extern "C" int pi_op_copy_f32(const float * src, float * dst, int64_t n, void * stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_copy_f32, dim3((unsigned) std::max<int64_t>(1, std::min<int64_t>(1024, (n + 255) / 256))), dim3(256), 0, (hipStream_t) stream, src, dst, n);
    PI_CHECK_LAUNCH(); return 0;
}

// ---- attention over a shared latent -----------------------------------------------------------------------------------------------------------------
// Three launches.  (1) k_latent_absorb folds the key up-projection and the score scale into the query: qa[t][h][:] = scale * W_uk[h]^T q[t][h] (rank values per head).
// (2) k_latent_scores, grid (token, head tile of M heads, split of the cell range): a thread owns a cell in the score phase — its latent row streams through registers once and
// feeds M accumulators, the M queries come through wave-uniform (scalar) loads — and a slice of the latent's rank in the value phase, where the probabilities of a cell are
// broadcast from LDS to M x RPT accumulators; every split leaves an un-normalised partial (max, sum, sum of p * c) in scratch.  (3) k_latent_combine merges the splits with
// the sink term, normalises and applies the value up-projection.  K / V are never materialised; passes of up to eight tokens are spread over the chip by the splits (64 cells each),
// longer ones take splits only when a score row would not fit LDS.  k_latent_rows takes (2) for few tokens of ranks 256 and 512 (lat_rows_takes), prompt_attention.hip passes of nine tokens and more that are not
// k_latent_rows's; where sizes, alignment or scratch memory keep a pass off both it comes here.
// A cached row is [latent (rank) | rotated key part (rot values, shared by the heads; none by default)]: the folded query carries its own rotated part behind the rank values, so a score is one
// dot product over the row's width; only the latent is summed with the probabilities.  Which cells a token sees is the mask's alone (a window of positions: pi_op_window_mask).
// scratch (floats): qa [n_tok][heads][rank + rot] | pol [n_tok][heads][S][rank] | pml [n_tok][heads][S][2]
#define LAT_LDS_BUDGET (128 * 1024)
struct lat_plan { int M, RPT, cap, S; size_t lds, scratch; };
static lat_plan latent_plan(int heads, int rank, int rot, int n_tok, int n_ctx) {
    lat_plan p;
    const bool single = n_tok <= 8;
    int best = 1;                                                     // heads per workgroup: the largest tile that leaves at most a quarter of its accumulator rows idle
    for (int m : { 2, 4, 8, 16 }) { if (single && m > 4) break; if (3 * ((heads + m - 1) / m * m) <= 4 * heads) best = m; }
    p.M = best;
    p.RPT = rank > 512 ? 4 : rank > 256 ? 2 : 1;
    const int rthreads = (rank + p.RPT - 1) / p.RPT, G = std::max(1, 256 / rthreads);
    const int cap_max = std::max(64, (int) (((LAT_LDS_BUDGET / 4 - (size_t) G * p.M * rank - 256 * p.M) / p.M) / 64 * 64));
    p.cap = single ? 64 : std::min(cap_max, 2048);
    p.cap = std::min(p.cap, (n_ctx + 63) / 64 * 64);
    p.S = (n_ctx + p.cap - 1) / p.cap;
    p.lds = ((size_t) p.cap * p.M + (size_t) G * p.M * rank + 8 * p.M + 8 + 256 * p.M) * 4;
    p.scratch = (size_t) n_tok * heads * (rank + rot) + (size_t) n_tok * heads * rank * p.S + (size_t) n_tok * heads * p.S * 2;
    return p;
}

// Passes that take k_latent_rows: ranks of whole tiles, up to eight tokens, and as many more as leave rows (token, head) x rank small: there the tiles of a prompt, a workgroup per head that walks all cells, leave most of
// the chip idle (16 heads, rank 512, us of the per-token kernels / the tiles / here: 9 tokens alone 71 / 25 / 22, of 512 cells 178 / 54 / 28, of 4096 439 / 274 / 89, of 16384 510 / 1060 / 292; 32 tokens alone
// 82 / 32 / 29, of 4096 cells 431 / 280 / 174).  Beyond 512 rows of rank 512 the shares of the splits cost more than the tiles of a short context (32 heads, 24 tokens alone 31, here 36).  The shares are kept to
// 560 MB of scratch memory from nine tokens on.
static size_t lat_rows_floats(int heads, int rank, int rot, int n_tok, int n_ctx) { return (size_t) n_tok * heads * ((size_t) (rank + rot) + (size_t) (n_ctx + 31) / 32 * (rank + 2)); }
static bool lat_rows_takes(int heads, int rank, int rot, int n_tok, int n_ctx) {
    return (rank == 256 || rank == 512) && rot <= 64 && (rot & 3) == 0 && (n_tok <= 8 || (n_tok <= 32 && (int64_t) n_tok * heads * rank <= 512 * 512 && lat_rows_floats(heads, rank, rot, n_tok, n_ctx) <= (size_t) 140 << 20 &&
                                                                                                 (n_ctx >= 64 || (int64_t) n_tok * heads * rank <= 384 * 512)));
}

// the tokens' own latents on their way to their cells: a norm of rows of `rank` values (256 or 512), of no rows where w is null
struct lat_kv { const float * x; int64_t xs; const float * w; float eps; float * cache; };
// grid (token tile of 4, head, 64 values of the rank, then 64 values of the rotated part, then the tokens' latents): lane = one rank value, the four waves take a quarter of the head's dim each and meet in LDS.  A query head is
// [dim values | rot values]; the last are turned in pairs by the token's position (cs: the rotation table) and go behind the rank values
__global__ void __launch_bounds__(256) k_latent_absorb(const float * __restrict__ q, int64_t qs, const uint16_t * __restrict__ wuk, float scale, int heads, int dim, int rank, int rot, const float2 * __restrict__ cs, int n_pos,
                                                       int pairing, const int32_t * __restrict__ pos, int n_tok, float * __restrict__ qa, const int32_t * __restrict__ dyn, int live_min, const lat_kv kv, const int32_t * __restrict__ abort_w) {
    if (live_min > 0 && dyn[1] <= live_min) return;                    // (a pass that prompt_attention.hip takes: latent_tiles_to)
    const int gone = pi_abort_peek(abort_w);
    if (kv.w && blockIdx.z == gridDim.z - 1) {                         // wave = token; the bits of k_rms_scale_once, whose waves sum 256 values each
        const int t = blockIdx.x * 4 + (threadIdx.x >> 6), i = (threadIdx.x & 63) * 4;
        if (blockIdx.y != 0 || t >= n_tok) return;
        const float * x = kv.x + (int64_t) t * kv.xs;
        const int64_t cell = pi_cell_of(dyn, 0, t);
        float4 v[2], w[2];
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; j++) { const int at = min(i + 256 * j, rank - 4); v[j] = *(const float4 *) (x + at); w[j] = *(const float4 *) (kv.w + at); }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (256 * j >= rank) break;
            float a = fmaf(v[j].x, v[j].x, 0.0f);
            a = fmaf(v[j].y, v[j].y, a); a = fmaf(v[j].z, v[j].z, a); a = fmaf(v[j].w, v[j].w, a);
            ss += pi_lanes_sum<64>(a);
        }
        const float inv = 1.0f / sqrtf(ss / (float) rank + kv.eps);
        if (pi_abort_late(gone, abort_w, 5)) return;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (256 * j >= rank) break;
            *(float4 *) (kv.cache + cell * rank + i + 256 * j) = make_float4(v[j].x * inv * (w[j].x + 0.0f), v[j].y * inv * (w[j].y + 0.0f), v[j].z * inv * (w[j].z + 0.0f), v[j].w * inv * (w[j].w + 0.0f));
        }
        return;
    }
    __shared__ float part[4][4][64];
    extern __shared__ float4 qsh[];                                    // [dim]: the head's query values of the four tokens, side by side
    const int t0 = blockIdx.x * 4, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = blockIdx.z * 64 + lane;
    const int n_rank_blocks = (rank + 63) / 64, hw = dim + rot;
    if ((int) blockIdx.z >= n_rank_blocks) {                           // the rotated part: wave = token
        const int d = (blockIdx.z - n_rank_blocks) * 64 + lane, t = t0 + wave;
        if (d >= rot || t >= n_tok) return;
        const float * qr = q + (int64_t) t * qs + (int64_t) h * hw + dim;
        const pi_turn u = pi_turn_of(d, rot / 2, pairing);
        const float2 c = cs[(int64_t) min(pos[t], n_pos - 1) * (rot / 2) + u.angle];
        const float own = qr[d], other = qr[u.mate];
        if (pi_abort_late(gone, abort_w, 5)) return;
        qa[((int64_t) t * heads + h) * (rank + rot) + rank + d] = (u.lead ? own * c.x - other * c.y : own * c.x + other * c.y) * scale;
        return;
    }
    for (int idx = threadIdx.x; idx < 4 * dim; idx += 256) {
        const int tt = idx / dim, d = idx % dim;
        ((float *) qsh)[d * 4 + tt] = q[(int64_t) min(t0 + tt, n_tok - 1) * qs + (int64_t) h * hw + d];
    }
    __syncthreads();
    const int dq = (dim + 3) / 4, d0 = wave * dq, d1 = min(dim, d0 + dq);
    float acc[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
    const uint16_t * w = wuk + (int64_t) h * dim * rank + min(r, rank - 1);
#pragma unroll 8
    for (int d = d0; d < d1; d++) {
        const float wv = hy_widen(w[(int64_t) d * rank]);
        const float4 qv = qsh[d];
        acc[0] = fmaf(qv.x, wv, acc[0]); acc[1] = fmaf(qv.y, wv, acc[1]); acc[2] = fmaf(qv.z, wv, acc[2]); acc[3] = fmaf(qv.w, wv, acc[3]);
    }
#pragma unroll
    for (int tt = 0; tt < 4; tt++) part[wave][tt][lane] = acc[tt];
    __syncthreads();
    const int tt = wave;                                              // wave tt writes token t0 + tt
    if (pi_abort_late(gone, abort_w, 5)) return;                       // (32 rows of 128 bytes per wave: an earlier look keeps them behind the queries, 4.7 us a launch instead of 3.8)
    if (t0 + tt < n_tok && r < rank) qa[((int64_t) (t0 + tt) * heads + h) * (rank + rot) + r] = (part[0][tt][lane] + part[1][tt][lane] + part[2][tt][lane] + part[3][tt][lane]) * scale;
}

template <int M, int RPT>
__global__ void __launch_bounds__(256) k_latent_scores(const float * __restrict__ qa, const float * __restrict__ cache, const uint32_t * __restrict__ mask, int heads, int rank, int rot, int n_kv_arg,
                                                       int cap, int S, float * __restrict__ pol, float * __restrict__ pml, const int32_t * __restrict__ dyn, int live_min, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 5) || (live_min > 0 && dyn[1] <= live_min)) return;
    extern __shared__ float lds[];
    const int t = blockIdx.x, h0 = blockIdx.y * M, split = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rthreads = (rank + RPT - 1) / RPT, G = max(1, 256 / rthreads);
    float * sc = lds, * part = sc + (size_t) cap * M, * red = part + (size_t) G * M * rank, * wsc = red + 8 * M + 8;     // red: [4 waves][M] twice; wsc: [4 waves][64 cells][M]
    __shared__ int hi_s, lo_s;
    const int n_kv = min(dyn ? dyn[1] : n_kv_arg, n_kv_arg);
    const int words = (n_kv_arg + 31) / 32;
    const uint32_t * mrow = mask + (int64_t) t * words;
    int c0 = split * cap;
    int c1 = min(n_kv, c0 + cap);
    if (tid == 0) { hi_s = 0; lo_s = 0x7fffffff; }
    __syncthreads();
    {   // cells past the last visible one of this token are not walked (a prompt's early tokens see little of the pass's cells), nor those ahead of the first (a window's)
        int hi = 0, lo = 0x7fffffff;
        for (int w = (c0 >> 5) + tid; w < (c1 + 31) >> 5; w += 256) { const uint32_t bits = mrow[w]; if (bits) { hi = max(hi, w * 32 + 32 - __clz(bits)); lo = min(lo, w * 32 + __ffs(bits) - 1); } }
        if (hi) { atomicMax(&hi_s, hi); atomicMin(&lo_s, lo); }
    }
    __syncthreads();
    c1 = min(c1, hi_s); c0 = max(c0, lo_s);
    const int W = rank + rot;                                          // a cached row
    const int nh = min(M, heads - h0);
    const float * qat = qa + ((int64_t) t * heads + h0) * W;
    float * pol_t = pol + (((int64_t) t * heads + h0) * S + split) * rank, * pml_t = pml + (((int64_t) t * heads + h0) * S + split) * 2;
    if (c1 <= c0) {                                                   // nothing of this token lives in this split: its maximum says so, and nobody reads its sums
        if (tid < nh) { pml_t[(int64_t) tid * S * 2] = -INFINITY; pml_t[(int64_t) tid * S * 2 + 1] = 0.0f; }
        return;
    }
    // scores: a thread per cell; a split of 64 cells (single tokens) gives every wave a quarter of the rank instead, so that all four waves stream the 64 latents
    float lmax[M];
#pragma unroll
    for (int m = 0; m < M; m++) lmax[m] = -INFINITY;
    if (cap == 64 && (W & 15) == 0) {
        const int j = c0 + lane, rq = W >> 2, rb = wave * rq;
        const bool vis = j < c1 && ((mrow[j >> 5] >> (j & 31)) & 1u);
        float a[M];
#pragma unroll
        for (int m = 0; m < M; m++) a[m] = 0.0f;
        if (vis) {
            const float * c = cache + (int64_t) j * W + rb;
#pragma unroll 8
            for (int r = 0; r < rq; r += 4) {
                const float4 cv = *(const float4 *) (c + r);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const float * qq = qat + (m < nh ? m : 0) * W + rb + r;                    // (wave-uniform address)
                    a[m] = fmaf(qq[0], cv.x, a[m]); a[m] = fmaf(qq[1], cv.y, a[m]); a[m] = fmaf(qq[2], cv.z, a[m]); a[m] = fmaf(qq[3], cv.w, a[m]);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++) wsc[((size_t) wave * 64 + lane) * M + m] = a[m];
        __syncthreads();
        if (wave == 0 && j < c1) {
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float sv = vis ? wsc[(size_t) lane * M + m] + wsc[((size_t) 64 + lane) * M + m] + wsc[((size_t) 128 + lane) * M + m] + wsc[((size_t) 192 + lane) * M + m] : -INFINITY;
                sc[(size_t) lane * M + m] = sv; lmax[m] = sv;
            }
        }
        __syncthreads();
    } else
    for (int j = c0 + tid; j < c1; j += 256) {
        const bool vis = (mrow[j >> 5] >> (j & 31)) & 1u;
        float a[M];
#pragma unroll
        for (int m = 0; m < M; m++) a[m] = 0.0f;
        if (vis) {
            const float * c = cache + (int64_t) j * W;
            if ((W & 3) == 0) {
#pragma unroll 2
                for (int r = 0; r < W; r += 4) {
                    const float4 cv = *(const float4 *) (c + r);
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        const float * qq = qat + (m < nh ? m : 0) * W + r;                     // (wave-uniform address)
                        a[m] = fmaf(qq[0], cv.x, a[m]); a[m] = fmaf(qq[1], cv.y, a[m]); a[m] = fmaf(qq[2], cv.z, a[m]); a[m] = fmaf(qq[3], cv.w, a[m]);
                    }
                }
            } else {
                for (int r = 0; r < W; r++) {
                    const float cv = c[r];
#pragma unroll
                    for (int m = 0; m < M; m++) a[m] = fmaf(qat[(m < nh ? m : 0) * W + r], cv, a[m]);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++) { const float sv = vis ? a[m] : -INFINITY; sc[(size_t) (j - c0) * M + m] = sv; lmax[m] = fmaxf(lmax[m], sv); }
    }
    // per head: max over the split, then p = exp(s - max) and its sum (every thread revisits its own cells)
#pragma unroll
    for (int m = 0; m < M; m++) { const float v = pi_wave_max(lmax[m]); if (lane == 0) red[wave * M + m] = v; }
    __syncthreads();
    float mx[M], lsum[M];
#pragma unroll
    for (int m = 0; m < M; m++) { mx[m] = fmaxf(fmaxf(red[m], red[M + m]), fmaxf(red[2 * M + m], red[3 * M + m])); lsum[m] = 0.0f; }
    for (int j = c0 + tid; j < c1; j += 256)
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float sv = sc[(size_t) (j - c0) * M + m];
            const float pv = sv == -INFINITY ? 0.0f : expf(sv - mx[m]);
            sc[(size_t) (j - c0) * M + m] = pv; lsum[m] += pv;
        }
    float * red2 = red + 4 * M;
#pragma unroll
    for (int m = 0; m < M; m++) { const float v = pi_lanes_sum<64>(lsum[m]); if (lane == 0) red2[wave * M + m] = v; }
    __syncthreads();
    if (tid < nh) {
        pml_t[(int64_t) tid * S * 2] = fmaxf(fmaxf(red[tid], red[M + tid]), fmaxf(red[2 * M + tid], red[3 * M + tid]));
        pml_t[(int64_t) tid * S * 2 + 1] = red2[tid] + red2[M + tid] + red2[2 * M + tid] + red2[3 * M + tid];
    }
    // sum of p * c: thread (cell group g, rank slice rt)
    const int g = tid / rthreads, rt = tid % rthreads, r0 = rt * RPT;
    float o[M][RPT];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int i = 0; i < RPT; i++) o[m][i] = 0.0f;
    if (g < G) {
#pragma unroll 8
        for (int j = c0 + g; j < c1; j += G) {                          // (a masked cell has p = 0: its latent — zeros or an earlier owner's finite values — adds nothing)
            float cv[RPT];
#pragma unroll
            for (int i = 0; i < RPT; i++) cv[i] = r0 + i < rank ? cache[(int64_t) j * W + r0 + i] : 0.0f;
            const float * pj = sc + (size_t) (j - c0) * M;
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float pv = pj[m];
#pragma unroll
                for (int i = 0; i < RPT; i++) o[m][i] = fmaf(pv, cv[i], o[m][i]);
            }
        }
        if (G > 1)
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int i = 0; i < RPT; i++) if (r0 + i < rank) part[((size_t) g * M + m) * rank + r0 + i] = o[m][i];
    }
    if (G > 1) {
        __syncthreads();
        for (int idx = tid; idx < nh * rank; idx += 256) {
            const int m = idx / rank, r = idx % rank;
            float v = 0.0f;
            for (int gg = 0; gg < G; gg++) v += part[((size_t) gg * M + m) * rank + r];
            pol_t[(int64_t) m * S * rank + r] = v;
        }
    } else if (g == 0) {
#pragma unroll
        for (int m = 0; m < M; m++)
            if (m < nh)
#pragma unroll
                for (int i = 0; i < RPT; i++) if (r0 + i < rank) pol_t[(int64_t) m * S * rank + r0 + i] = o[m][i];
    }
}

// The same for a few tokens on the fp32 matrix cores, sixteen rows (token, head) and a split of 32 cells per workgroup.  What bounds it: one trip to memory and back - every load of the workgroup goes out before the first
// product.  With a lane per cell and a chain of loads each, 4 tokens x 16 heads over 700 cells of 512 + 64 took 20 us (now 11.5); 1 token x 16 heads of 256, 32 cells: 9.7 (6.4).
// NJ: a wave sums 16 NJ of the rank's values (rank = 64 NJ); EX: steps of 16 values behind the rank.  Lane l holds, with n = l % 16 and g = l / 16, of the scores row n and the wave's cells 4 g + r, of the sums
// row n and the values NJ (4 g + r) + j.  (Splits of 64 cells, every wave its sixteen over the whole width: 17 us.)
// LOOP: fewer workgroups than splits, each takes several (a loop of one round costs 77 -> 85 us: 4 tokens x 16 heads, 16384 cells)
template <int NJ, int EX, bool LOOP>
__global__ void __launch_bounds__(256, NJ == 4 ? 3 : EX == 0 ? 2 : 1) k_latent_rows(const float * __restrict__ qa, const float * __restrict__ cache, const uint32_t * __restrict__ mask, int heads, int W, int n_rows, int n_kv_arg, int S,
                                                        float * __restrict__ pol, float * __restrict__ pml, const int32_t * __restrict__ dyn, int live_max, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    constexpr int RANK = 64 * NJ, NS = RANK / 16 + EX, NH = NS / 2;
    __shared__ __attribute__((aligned(16))) float ps[16][36], half[2][16][20];
    __shared__ float top[2][16], sum[2][16];
    const int words = (n_kv_arg + 31) / 32, n_kv = min(dyn ? dyn[1] : n_kv_arg, n_kv_arg);
    const uint32_t first = mask[(int64_t) (min((int) (blockIdx.x * 16 + (threadIdx.x & 15)), n_rows - 1) / heads) * words + blockIdx.y];      // (on its way beside the number of live cells)
    int split = blockIdx.y;
    if (split * 32 >= n_kv || (live_max > 0 && n_kv > live_max)) return;       // (cells of the context that hold nothing yet; a pass that the kernels per token take)
    do {                                                               // (a barrier lies between a round's last look at the LDS and the next one's writes to the same place)
        int tid = threadIdx.x;
        if constexpr (LOOP) asm volatile("" : "+v"(tid));              // (queries and addresses are made again in every round: kept from one to the next they take the registers of a second workgroup)
        const int lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4, ct = wave & 1, wh = wave >> 1, row = min((int) blockIdx.x * 16 + n, n_rows - 1);
        const int c0 = split * 32;
        uint32_t vis = split == (int) blockIdx.y ? first : mask[(int64_t) (row / heads) * words + split];
        if (n_kv - c0 < 32) vis &= (1u << (n_kv - c0)) - 1u;
        uint32_t some = vis;                                              // the cells that any row sees; what the others hold is not read
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) some |= __shfl_xor(some, o, 64);
        float * pml_r = pml + ((int64_t) ((int) blockIdx.x * 16 + n) * S + split) * 2;
        const bool real = (int) blockIdx.x * 16 + n < n_rows;
        if (pi_abort_late(gone, abort_w, 5)) return;                       // (behind the mask, requested after it)
        if (!some) {                                                      // (the same in every lane: the rows of a tile are the same sixteen in all four)
            if (tid < 16 && real) { pml_r[0] = -INFINITY; pml_r[1] = 0.0f; }
            continue;
        }
        const int spare = __ffs(some) - 1;
        auto cell = [&](int c) { return (uint32_t) (c0 + ((some >> c) & 1u ? c : spare)); };
        hy_f32x4 kf[NH], qf[NH], vf[2][4][NJ / 4];
        {   // a wave scores sixteen cells over half of the row's width
            const uint32_t ko = cell(16 * ct + n) * (uint32_t) W, qo = (uint32_t) row * (uint32_t) W;
#pragma unroll
            for (int i = 0; i < NH; i++) {
                const uint32_t d = 16u * (wh * NH + i) + 4u * g, at = EX == 0 ? d : min(d, (uint32_t) W - 4u);
                kf[i] = *(const hy_f32x4 *) (cache + ko + at); qf[i] = *(const hy_f32x4 *) (qa + qo + at);
                if (EX && d >= (uint32_t) W) qf[i] = hy_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
            }
        }
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t o = cell(16 * jt + 4 * g + c) * (uint32_t) W + (uint32_t) (wave * (RANK / 4) + NJ * n);
#pragma unroll
                for (int j = 0; j < NJ / 4; j++) vf[jt][c][j] = *(const hy_f32x4 *) (cache + o + 4 * j);
            }
        __builtin_amdgcn_sched_barrier(0);
        hy_f32x4 s0 = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < NH; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) s0 = hy_mfma(kf[i][c], qf[i][c], s0);
        if (wh) *(hy_f32x4 *) &half[ct][n][4 * g] = s0;
        __syncthreads();
        const uint32_t mine = vis >> (16 * ct + 4 * g);
        float m = -INFINITY;
        if (!wh) {
            s0 += *(const hy_f32x4 *) &half[ct][n][4 * g];
#pragma unroll
            for (int r = 0; r < 4; r++) if (mine >> r & 1u) m = fmaxf(m, s0[r]);
            m = fmaxf(m, __shfl_xor(m, 16, 64)); m = fmaxf(m, __shfl_xor(m, 32, 64));
            if (g == 0) top[ct][n] = m;
        }
        __syncthreads();
        m = fmaxf(top[0][n], top[1][n]);
        if (!wh) {
            float l = 0.0f;
            hy_f32x4 p;
#pragma unroll
            for (int r = 0; r < 4; r++) { p[r] = mine >> r & 1u ? expf(s0[r] - m) : 0.0f; l += p[r]; }
            l += __shfl_xor(l, 16, 64); l += __shfl_xor(l, 32, 64);
            if (g == 0) sum[ct][n] = l;
            *(hy_f32x4 *) &ps[n][16 * ct + 4 * g] = p;
        }
        __syncthreads();
        if (tid < 16 && real) { pml_r[0] = m; pml_r[1] = sum[0][n] + sum[1][n]; }
        hy_f32x4 acc[NJ];
        auto sums = [&]() {
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[j] = hy_f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                const hy_f32x4 w = *(const hy_f32x4 *) &ps[n][16 * jt + 4 * g];
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[j] = hy_mfma(vf[jt][c][j >> 2][j & 3], w[c], acc[j]);
            }
        };
        sums();
        // an infinity or a NaN must not meet the zero weight of a row that does not see its cell (rows of several tokens share a tile, a cell that nobody sees repeats another): where a sum is no number it is left out of all
        // of them and joins at the end
        bool odd = false;
        if (__any(vis != 0xffffffffu)) {
            hy_f32x4 z = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) z[r] = fmaf(acc[j][r], 0.0f, z[r]);
            odd = __any((z[0] + z[1]) + (z[2] + z[3]) != 0.0f);
            if (odd) {
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) if ((__float_as_uint(vf[i >> 2][i & 3][j >> 2][j & 3]) & 0x7fffffffu) >= 0x7f800000u) vf[i >> 2][i & 3][j >> 2][j & 3] = 0.0f;
                sums();
            }
        }
        if (!real || vis == 0) continue;
        if (odd)
            for (int c = 0; c < 32; c++) {
                if (!(vis >> c & 1u)) continue;
                const float * row = cache + cell(c) * (uint32_t) W + wave * (RANK / 4) + NJ * 4 * g;
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) if ((__float_as_uint(row[NJ * r + j]) & 0x7fffffffu) >= 0x7f800000u) acc[j][r] += row[NJ * r + j];
            }
        float * o = pol + ((int64_t) row * S + split) * RANK + wave * (RANK / 4);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < NJ; j += 4) *(hy_f32x4 *) (o + NJ * (4 * g + r) + j) = hy_f32x4{ acc[j][r], acc[j + 1][r], acc[j + 2][r], acc[j + 3][r] };
    } while (LOOP && (split += gridDim.y) * 32 < n_kv);
}

// grid (token tile of 4, head, 16 output values): merges the splits (with the sink if there is one), normalises, applies its rows of W_uv[h], then the gate if there is one: one value per head, or (gate_width = vdim)
// one per output value
// MANY: more than eight splits (the code for them costs the launches of fewer 0.3 us of 9.5)
template <bool MANY, int NT>
__global__ void __launch_bounds__(NT) k_latent_combine(const float * __restrict__ pol, const float * __restrict__ pml, const uint16_t * __restrict__ wuv, const float * __restrict__ sink,
                                                        const float * __restrict__ gate, int64_t gs, int gate_act, int gate_width, int heads, int vdim, int rank, int S, int n_tok, int n_kv, int cap, const int32_t * __restrict__ dyn, int live_min, int live_max, int vec, float * __restrict__ out, int64_t os,
                                                        const int32_t * __restrict__ abort_w) {
    if ((live_min > 0 && dyn[1] <= live_min) || (live_max > 0 && dyn[1] > live_max)) return;
    const int gone = pi_abort_peek(abort_w);
    extern __shared__ __attribute__((aligned(16))) float ol[];                                     // [4][rank]
    __shared__ float wgt[4][64];                                      // per token: weight of the splits that hold something, 64 splits at a time,
    __shared__ int num[4][64], cnt[4];                                // their numbers, how many they are
    __shared__ float gsh[4];                                          // per token: the head's gate (one value per head)
    const int t0 = blockIdx.x * 4, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nt = min(4, n_tok - t0), n_s = min(S, (min(dyn ? dyn[1] : n_kv, n_kv) + cap - 1) / cap);      // (splits of cap cells: the ones behind the live cells hold nothing)
    constexpr int NW = NT / 64, RW = 16 / NW;                         // waves, rows of W_uv of a wave
    hy_u16x8v wrow[RW]; float gv[RW];      // (wide: eight weights of the rank per lane; the wave's rows and their gates are on their way while the splits are merged)
    const bool wide = vec && rank > 64;                             // (of fewer values a lane per value is quicker: rank 64, 6.0 us against 6.9; calls of rank 96 with one split, 4 tokens, 17.1 that way, 16.3 so)
    if (wide) {
#pragma unroll
        for (int k = 0; k < RW; k++) wrow[k] = *(const hy_u16x8v *) (wuv + ((int64_t) h * vdim + min((int) blockIdx.z * 16 + wave + NW * k, vdim - 1)) * rank + min(lane * 8, rank - 8));
        if (gate && gate_width > 1)
#pragma unroll
            for (int k = 0; k < RW; k++) gv[k] = gate[(int64_t) (t0 + min(lane, nt - 1)) * gs + (int64_t) h * vdim + min((int) blockIdx.z * 16 + wave + NW * k, vdim - 1)];
    }
    // many splits: a thread per four values of the rank, for all tokens at a time or, where that leaves some threads idle but no second group of them and the splits are many, for one token after the other; the groups take eight splits
    // in turn (1 token of 8 heads, rank 256, over 16384 cells: 83 us with one group, now 43)
    __shared__ __attribute__((aligned(16))) float4 shares[MANY && NT == 256 ? 4 : 1][MANY ? NT : 1];
    int groups = 1, per = 1, at_once = 1, grp = 0, mine = 0, col = 0;
    float4 share[NT == 256 ? 4 : 1];
    if (MANY && vec) {
        const int cols = rank >> 2;
        at_once = nt * cols <= NT / 2 ? nt : 1; per = at_once * cols;
        if (n_s > (NT == 256 ? 16 : 8) && (at_once == nt || (NT == 256 && n_s > 64 && (nt * cols & 255))) && per <= NT / 2) { groups = NT / per; grp = tid / per; mine = tid % per / cols; col = tid % cols; }
#pragma unroll
        for (int i = 0; i < (NT == 256 ? 4 : 1); i++) share[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    for (int idx = tid; idx < 4 * rank; idx += NT) ol[idx] = 0.0f;
    if (tid < 4) {
        float g = 1.0f;
        if (gate && gate_width == 1 && tid < nt) { g = gate[(int64_t) (t0 + tid) * gs + h]; if (gate_act == PI_ACT_SIGMOID) g = 1.0f / (1.0f + expf(-g)); }
        gsh[tid] = g;
    }
    // (the wave `tt` owns token t0 + tt's bookkeeping)
    float mstar = -INFINITY, den = 0.0f;
    const float sk = sink ? sink[h] : -INFINITY;
    const float * pml_t = pml + ((int64_t) (t0 + min(wave, nt - 1)) * heads + h) * S * 2;
    const float m_own = lane < S ? pml_t[lane * 2] : -INFINITY, l_own = lane < S ? pml_t[lane * 2 + 1] : 0.0f;      // (on their way beside the number of live cells)
    {
        float m = lane < n_s ? fmaxf(sk, m_own) : sk;
        for (int s = lane + 64; s < n_s; s += 64) m = fmaxf(m, pml_t[s * 2]);
        mstar = pi_wave_max(m);
        float d = lane < n_s && m_own != -INFINITY ? l_own * expf(m_own - mstar) : 0.0f;
        for (int s = lane + 64; s < n_s; s += 64) { const float ms = pml_t[s * 2]; if (ms != -INFINITY) d += pml_t[s * 2 + 1] * expf(ms - mstar); }
        den = pi_lanes_sum<64>(d) + (sink ? expf(sk - mstar) : 0.0f);
    }
    if (pi_aborted_together(gone, abort_w, 5)) return;                 // (behind the splits' maxima, requested after it)
    for (int sb = 0; sb < n_s; sb += 64) {
        if (sb) __syncthreads();
        if (wave < nt) {
            const int s = sb + lane;
            const float ms = s >= n_s ? -INFINITY : sb == 0 ? m_own : pml_t[s * 2];
            const unsigned long long some = __ballot(ms != -INFINITY);
            if (ms != -INFINITY) { const int at = __popcll(some & ((1ull << lane) - 1ull)); wgt[wave][at] = expf(ms - mstar) / den; num[wave][at] = s; }
            if (lane == 0) cnt[wave] = __popcll(some);
        }
        __syncthreads();
        if (MANY && groups > 1) {
#pragma unroll
            for (int i = 0; i < (NT == 256 ? 4 : 1); i++) {
                const int tt = min(i * at_once + mine, nt - 1), n = i * at_once < nt && grp < groups ? cnt[tt] : 0;
                const float * p = pol + (((int64_t) (t0 + tt) * heads + h) * S) * rank + col * 4;
                for (int s0 = 8 * grp; s0 < n; s0 += 8 * groups) {
                    float4 x[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) x[u] = *(const float4 *) (p + (int64_t) num[tt][min(s0 + u, n - 1)] * rank);
#pragma unroll
                    for (int u = 0; u < 8; u++)
                        if (s0 + u < n) { const float w = wgt[tt][s0 + u]; share[i].x = fmaf(w, x[u].x, share[i].x); share[i].y = fmaf(w, x[u].y, share[i].y); share[i].z = fmaf(w, x[u].z, share[i].z); share[i].w = fmaf(w, x[u].w, share[i].w); }
                }
            }
            continue;
        }
        if (vec) {                                                     // four values of the rank per thread, eight splits on their way at a time (one by one, every split was a trip to memory: 23 us for 11 of 4 tokens)
            for (int idx = tid; idx < nt * (rank >> 2); idx += NT) {
                const int tt = idx / (rank >> 2), r = idx % (rank >> 2) * 4, n = cnt[tt];
                if (n == 0) continue;
                const float * p = pol + (((int64_t) (t0 + tt) * heads + h) * S) * rank + r;
                float4 v = *(const float4 *) (ol + tt * rank + r);
                for (int s0 = 0; s0 < n; s0 += 8) {
                    float4 x[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) x[u] = *(const float4 *) (p + (int64_t) num[tt][min(s0 + u, n - 1)] * rank);
#pragma unroll
                    for (int u = 0; u < 8; u++)
                        if (s0 + u < n) { const float w = wgt[tt][s0 + u]; v.x = fmaf(w, x[u].x, v.x); v.y = fmaf(w, x[u].y, v.y); v.z = fmaf(w, x[u].z, v.z); v.w = fmaf(w, x[u].w, v.w); }
                }
                *(float4 *) (ol + tt * rank + r) = v;
            }
            continue;
        }
        for (int idx = tid; idx < nt * rank; idx += NT) {
            const int tt = idx / rank, r = idx % rank;
            const float * p = pol + (((int64_t) (t0 + tt) * heads + h) * S) * rank + r;
            float v = ol[idx];
            const int n = cnt[tt];
#pragma unroll 8
            for (int s = 0; s < n; s++) v = fmaf(wgt[tt][s], p[(int64_t) num[tt][s] * rank], v);
            ol[idx] = v;
        }
    }
    if (MANY && groups > 1) {
#pragma unroll
        for (int i = 0; i < (NT == 256 ? 4 : 1); i++) if (i * at_once < nt) shares[i][tid] = share[i];
        __syncthreads();
        const int cols = rank >> 2;
        for (int idx = tid; idx < nt * cols; idx += NT) {
            const float4 * from = shares[idx / per];
            float4 v = from[idx % per];
            for (int g = 1; g < groups; g++) { const float4 x = from[g * per + idx % per]; v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w; }
            *(float4 *) (ol + idx / cols * rank + idx % cols * 4) = v;
        }
    }
    __syncthreads();
    if (wide) {
        const int v0 = blockIdx.z * 16 + wave;
        float a[RW][4];
#pragma unroll
        for (int k = 0; k < RW; k++)
#pragma unroll
            for (int tt = 0; tt < 4; tt++) a[k][tt] = 0.0f;
        for (int rb = 0; rb < rank; rb += 512) {
            const int r = rb + lane * 8;
            if (r >= rank) break;
#pragma unroll
            for (int k = 0; k < RW; k++) {
                const hy_u16x8v w = rb == 0 ? wrow[k] : *(const hy_u16x8v *) (wuv + ((int64_t) h * vdim + min(v0 + NW * k, vdim - 1)) * rank + r);
#pragma unroll
                for (int tt = 0; tt < 4; tt++)
#pragma unroll
                    for (int i = 0; i < 8; i++) a[k][tt] = fmaf(hy_widen(w[i]), ol[tt * rank + r + i], a[k][tt]);
            }
        }
#pragma unroll
        for (int k = 0; k < RW; k++) {
            const int vv = v0 + NW * k;
            if (vv >= vdim) break;
            float v = 0.0f;
#pragma unroll
            for (int tt = 0; tt < 4; tt++) { const float s = pi_lanes_sum<64>(a[k][tt]); if (lane == tt) v = s; }
            if (lane >= nt) continue;
            float g = gsh[lane];
            if (gate && gate_width > 1) { g = gv[k]; if (gate_act == PI_ACT_SIGMOID) g = 1.0f / (1.0f + expf(-g)); }
            out[(int64_t) (t0 + lane) * os + (int64_t) h * vdim + vv] = v * g;
        }
        return;
    }
    for (int vv = blockIdx.z * 16 + wave; vv < min(vdim, (int) blockIdx.z * 16 + 16); vv += NW) {
        const uint16_t * wv = wuv + ((int64_t) h * vdim + vv) * rank;
        float a[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
        const bool mine = lane < nt;                                   // lane tt writes token t0 + tt; its gate is on the way while the row is summed
        float g = mine ? gsh[lane] : 1.0f;
        if (gate && gate_width > 1 && mine) g = gate[(int64_t) (t0 + lane) * gs + (int64_t) h * vdim + vv];
#pragma unroll 4
        for (int r = lane; r < rank; r += 64) {
            const float w = hy_widen(wv[r]);
#pragma unroll
            for (int tt = 0; tt < 4; tt++) a[tt] = fmaf(w, ol[tt * rank + r], a[tt]);
        }
        if (gate && gate_width > 1 && gate_act == PI_ACT_SIGMOID) g = 1.0f / (1.0f + expf(-g));
        float v = 0.0f;
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
            const float s = pi_lanes_sum<64>(a[tt]);
            if (lane == tt) v = s;
        }
        if (mine) out[(int64_t) (t0 + lane) * os + (int64_t) h * vdim + vv] = v * g;
    }
}

extern "C" int pi_op_latent_attention_max_cells(int rank) { (void) rank; return 1 << 22; }       // (long contexts are cut into splits: no score row has to fit LDS whole)
extern "C" size_t pi_op_latent_attention_scratch_floats(int heads, int rank, int n_tok, int n_ctx) { return pi_op_latent_attention_rot_scratch_floats(heads, rank, 0, n_tok, n_ctx); }
extern "C" size_t pi_op_latent_attention_rot_scratch_floats(int heads, int rank, int rot_dim, int n_tok, int n_ctx) {
    size_t need = std::max(latent_plan(heads, rank, rot_dim, n_tok, n_ctx).scratch, latent_plan(heads, rank, rot_dim, std::min(n_tok, 8), n_ctx).scratch);
    for (int few = 1; few <= std::min(n_tok, 32); few++) if (lat_rows_takes(heads, rank, rot_dim, few, n_ctx)) need = std::max(need, lat_rows_floats(heads, rank, rot_dim, few, n_ctx));
    return need;
}
extern "C" size_t pi_op_latent_attention_prompt_scratch_floats(int heads, int dim, int rot_dim, int vdim, int rank, int n_tok, int n_ctx) {
    return n_tok >= PA_LATENT_TOKENS && sa_sizes(dim, rot_dim, vdim, rank) ? ((size_t) n_ctx + 63) / 64 * 64 * sa_cell_floats(heads, dim, rot_dim, vdim) : 0;
}
template <int M, int RPT> static int latent_reserve_one() {
    PI_CHECK_HIP(hipFuncSetAttribute((const void *) k_latent_scores<M, RPT>, hipFuncAttributeMaxDynamicSharedMemorySize, LAT_LDS_BUDGET + 4096));
    return 0;
}
extern "C" int pi_op_latent_attention_reserve(void) {
    static bool done = false;
    if (done) return 0;
#define LAT_RES(M) if (latent_reserve_one<M, 1>() || latent_reserve_one<M, 2>() || latent_reserve_one<M, 4>()) return -1;
    LAT_RES(1) LAT_RES(2) LAT_RES(4) LAT_RES(8) LAT_RES(16)
#undef LAT_RES
    done = true;
    return 0;
}
template <int M, int RPT>
static void latent_scores_launch(const lat_plan & p, dim3 grid, hipStream_t s, double bytes, int nta, const float * qa, const float * cache, const uint32_t * mask, int heads, int rank, int rot, int n_kv,
                                 float * pol, float * pml, const int32_t * dyn, int live_min) {
    PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, nta, bytes, (k_latent_scores<M, RPT>), grid, dim3(256), p.lds, s, qa, cache, mask, heads, rank, rot, n_kv, p.cap, p.S, pol, pml, dyn, live_min, pi_abort_word());
}
extern "C" int pi_op_latent_attention(const float * q, int64_t q_stride, const float * cache, const uint32_t * mask, const pi_weight * wuk, const pi_weight * wuv, const float * sink_dev,
                                      float scale, int heads, int dim, int vdim, int rank, int n_tok, int n_kv, float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride,
                                      const int32_t * dyn_dev, void * stream) {
    if (!sink_dev) { pi_set_error("pi_op_latent_attention: the sink is required"); return -1; }
    return pi_op_latent_attention_rot(q, q_stride, cache, mask, wuk, wuv, sink_dev, nullptr, 0, PI_ACT_NONE, scale, heads, dim, 0, vdim, rank, nullptr, nullptr, n_tok, n_kv, scratch_dev, scratch_floats, out, out_stride, dyn_dev, stream);
}
extern "C" int pi_op_latent_attention_rot(const float * q, int64_t q_stride, const float * cache, const uint32_t * mask, const pi_weight * wuk, const pi_weight * wuv, const float * sink_dev, const float * gate_dev,
                                          int64_t gate_stride, int gate_act, float scale, int heads, int dim, int rot, int vdim, int rank, const void * rotary_table, const int32_t * pos_dev, int n_tok, int n_kv,
                                          float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride, const int32_t * dyn_dev, void * stream) {
    return pi_op_latent_attention_gated(q, q_stride, cache, mask, wuk, wuv, sink_dev, gate_dev, gate_stride, gate_act, 1, scale, heads, dim, rot, vdim, rank, rotary_table, PI_PAIR_NEIGHBOURS, pos_dev, n_tok, n_kv, scratch_dev,
                                        scratch_floats, out, out_stride, dyn_dev, stream);
}
// How many live cells the tiles of a prompt are the better for.  They walk all cells with a workgroup per head and 32 tokens: few heads and tokens over a long context leave most of the chip idle, where k_latent_scores has
// a workgroup per token, tile of heads and 1280 .. 2048 cells.  Both by what was measured (8 .. 128 heads, ranks 128 .. 768, 9 .. 256 tokens, 40 .. 16000 cells), us: a tile's round of 128 cells 2 + 0.385 per step, the keys
// and values written out at 1000 TFLOP/s, 8 for every pair of launches; a round of 256 workgroups per token 0.19 + 0.029 per head of the tile for 1000 cells x values.  The tiles give way where they are clearly slower:
// tiles / workgroups per token 33 tokens of 16000 cells, 8 heads of rank 256 610 / 455, 16 of 512 + 64 1205 / 1060, 16 of 128 + 32 (in several launches) 1576 / 360, 9 tokens of them 1587 / 199; 128 heads, 9 tokens of
// 4000 cells 751 / 480, of 300 100 / 184; 33 tokens of 512 of 65536, rank 512 114 / 202.
// 0: none; n_kv: all.  The line between is looked at on the device, where the number of live cells is known: both sets of launches go out and one returns at once
// split: keys and values in three parts (split_attention.hip): a round of 256 workgroups and 128 cells 1.2 + 0.085 per step, the parts written out at 800 TFLOP/s, 20 for every pair of launches (tiles / workgroups per token there: 33 tokens
// of 1033 cells, 16 heads of 128, rank 512 60 / 362, of 12033 465 / 899, 32 heads of 4033 238 / 468; 8 heads of 128 + 64, 33 tokens of 12033 338 / 554)
static int latent_tiles_to(const lat_plan & p, const pa_args & a, int rank, int launches, bool split) {
    const double steps = (a.dim1 + 15) / 16 + (a.dim2 + 15) / 16 + 4 * ((a.vdim + 63) / 64);
    const int64_t slots = split ? 256 : 512, rounds = ((int64_t) a.heads * ((a.n_tok + 31) / 32) + slots - 1) / slots, heads = (a.heads + p.M - 1) / p.M;
    auto tiles = [&](int64_t live) {
        return (double) ((live + 127) / 128 * rounds) * (split ? 1.2 + 0.085 * steps : 2.0 + 0.385 * steps) + (split ? 7.8e-9 : 6e-9) * (double) live * a.heads * (a.dim1 + a.vdim) * rank + (split ? 20.0 : 8.0) * launches;
    };
    auto tokens = [&](int64_t live) { return std::ceil((double) (a.n_tok * heads) * live / p.cap / 256) * (double) std::min<int64_t>(live, p.cap) * (rank + a.dim2) * (1.9e-4 + 2.9e-5 * p.M) + 25.0; };
    int64_t to = a.n_kv, live = a.n_kv;                                // down from all cells as long as the tiles lose
    while (live >= 64 && 0.72 * tiles(live) > tokens(live)) { to = live = live * 5 / 7; }
    return to == a.n_kv ? a.n_kv : live < 64 ? 0 : (int) to;          // (33 tokens alone in a context of 33 cells: 20 us, a workgroup per token 80)
}
// A prompt with its keys and values written out (prompt_attention.hip), in as few launches over the cells as the scratch memory allows.  How many live cells it took the pass for: 0 none, a.n_kv any
static int latent_prompt(pa_args a, const lat_plan & p, const float * cache, int rank, const pi_weight * wuk, const pi_weight * wuv, float * scratch, size_t scratch_floats, double bytes, hipStream_t s) {
    if ((rank & 7) || (a.k2_row & 3) || ((uintptr_t) cache & 15) || ((uintptr_t) scratch & 15)) return 0;
    const size_t state = (size_t) a.n_tok * a.heads * (a.vdim + 2) + 3, whole = ((size_t) a.n_kv + 63) / 64 * 64;
    auto fits = [&](size_t per_cell) -> size_t {                       // the cells of a launch, 0: too few
        if (whole * per_cell <= scratch_floats) return whole;
        const size_t cells = scratch_floats > state ? (scratch_floats - state) / per_cell / 64 * 64 : 0;
        return cells >= 1024 ? cells : 0;
    };
    // In three parts where they are the quicker (sa_pays: of one launch each) and take no more launches than keys and values as they are: behind a launch that holds all live cells another one still costs two idle launches and
    // the sums' way to memory and back.  us as they are in one / in parts in one / in parts in two, cells 3072: 32 heads of 128, rank 512, 512 tokens alone 66 / 53 / 70, 64 alone 27 / 24 / 33; 64 heads of 64 + 32, rank 256, 512 alone
    // 87 / 74 / 98 (all 3072 cells 311 / 237 / 262 and 355 / 273 / 312: how many are live is not known here)
    const size_t plain_cell = (size_t) a.heads * (a.dim1 + a.vdim), part_cell = sa_cell_floats(a.heads, a.dim1, a.dim2, a.vdim), plain = fits(plain_cell), parts = sa_takes(a, rank) ? fits(part_cell) : 0;
    if (plain == 0) return 0;
    auto launches = [](int to, size_t cells) { return (int) ((to + cells - 1) / cells); };
    const int to_plain = latent_tiles_to(p, a, rank, launches(a.n_kv, plain), false), to_parts = parts > 0 ? latent_tiles_to(p, a, rank, launches(a.n_kv, parts), true) : 0;
    const bool split = to_parts > 0 && launches(to_parts, parts) <= std::max(1, launches(to_plain, plain)) && sa_pays(a, rank, to_parts);
    const size_t cells = split ? parts : plain;
    const int to = split ? to_parts : to_plain;
    a.state = cells < whole ? scratch + cells * (split ? part_cell : plain_cell) : nullptr;
    a.k1 = scratch; a.k1_row = (int64_t) a.heads * a.dim1; a.k1_head = a.dim1;
    a.v = scratch + cells * (size_t) a.k1_row; a.v_row = (int64_t) a.heads * a.vdim; a.v_head = a.vdim;
    a.k2 = cache + rank;
    if (!pa_takes(a, 1, PA_LATENT_TOKENS)) return 0;
    if (to == 0 || (to < a.n_kv && !a.dyn)) return 0;
    a.live_max = to < a.n_kv ? to : 0;
    if (to == a.n_kv) a.rd = pi_round_asked(0, (int64_t) a.heads * a.vdim);      // (else other launches may be the ones that write)
    for (size_t c = 0; c < (size_t) to; c += cells) {
        a.cell0 = (int) c; a.cell1 = (int) std::min((size_t) to, c + cells); a.first = c == 0; a.last = c + cells >= (size_t) to;
        if (split) { sa_launch(a, cache, rank, wuk, wuv, scratch, bytes, s); continue; }
        pa_expand(cache, a.k2_row, rank, wuk, wuv, a.cell0, a.cell1, a.n_kv, a.live_max, a.dyn, scratch, scratch + cells * (size_t) a.k1_row, s);
        pa_launch(a, 1, bytes, s);
    }
    return to;
}
static int latent_attention(const float * q, int64_t q_stride, const float * cache, const uint32_t * mask, const pi_weight * wuk, const pi_weight * wuv, const float * sink_dev, const float * gate_dev,
                                            int64_t gate_stride, int gate_act, int gate_width, float scale, int heads, int dim, int rot, int vdim, int rank, const void * rotary_table, int pairing, const int32_t * pos_dev,
                                            int n_tok, int n_kv, float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride, const int32_t * dyn_dev, const lat_kv & tokens, void * stream) {
    if (n_tok <= 0) return 0;
    const float2 * cs = nullptr; int n_pos = 0, half = 0;
    if (rot < 0 || (rot & 1)) { pi_set_error("pi_op_latent_attention: %d rotated dimensions (an even number)", rot); return -1; }
    if (rot > 0) {
        pi_rotary_table_view(rotary_table, &cs, &n_pos, &half);
        if (!cs || half != rot / 2 || !pos_dev) { pi_set_error("pi_op_latent_attention: a rotation table over the %d rotated dimensions and the tokens' positions are required", rot); return -1; }
    }
    if (pairing != PI_PAIR_HALVES && pairing != PI_PAIR_NEIGHBOURS) { pi_set_error("pi_op_latent_attention: pairing %d is unknown", pairing); return -1; }
    if (gate_dev && gate_act != PI_ACT_NONE && gate_act != PI_ACT_SIGMOID) { pi_set_error("pi_op_latent_attention: gate activation %d is unknown", gate_act); return -1; }
    if (gate_dev && gate_width != 1 && gate_width != vdim) { pi_set_error("pi_op_latent_attention: a gate has one value per head or one per output value (%d), not %d", vdim, gate_width); return -1; }
    if (q_stride < (int64_t) heads * (dim + rot)) { pi_set_error("pi_op_latent_attention: query rows of %lld floats hold no %d heads of %d + %d values", (long long) q_stride, heads, dim, rot); return -1; }
    if (!wuk || !wuv || wuk->type != PI_BF16 || wuv->type != PI_BF16 || wuk->ne0 != rank || wuv->ne0 != rank || wuk->ne1 != (int64_t) heads * dim || wuv->ne1 != (int64_t) heads * vdim) {
        pi_set_error("pi_op_latent_attention: the up-projections must be bfloat16 [heads * dim][rank] and [heads * vdim][rank]"); return -1;
    }
    if (rank > 1024) { pi_set_error("pi_op_latent_attention: latent width %d above 1024", rank); return -1; }
    lat_plan p = latent_plan(heads, rank, rot, n_tok, n_kv);
    if (p.scratch > scratch_floats) { pi_set_error("pi_op_latent_attention: %zu floats of scratch needed, %zu given", p.scratch, scratch_floats); return -1; }
    if (p.lds > LAT_LDS_BUDGET + 4096 || (size_t) 4 * rank * 4 > 64 * 1024) { pi_set_error("pi_op_latent_attention: LDS plan does not fit"); return -1; }
    if (pi_op_latent_attention_reserve() != 0) return -1;
    hipStream_t s = (hipStream_t) stream;
    float * qa = scratch_dev, * pol = qa + (size_t) n_tok * heads * (rank + rot), * pml = pol + (size_t) n_tok * heads * p.S * rank;
    const int nta = std::min(n_tok, PI_KT_MAXNT - 1);
    const int acct = pi_account_n_kv() > 0 ? pi_account_n_kv() : n_kv;
    pa_args a = {};
    a.q = q; a.qs = q_stride; a.dim1 = dim; a.k2_row = rank + rot; a.dim2 = rot; a.vdim = vdim; a.heads = heads; a.per_kv = 1; a.n_tok = n_tok; a.n_kv = n_kv; a.dyn = dyn_dev; a.mask = mask; a.pos = rot > 0 ? pos_dev : nullptr;
    a.cs = cs; a.n_pos = n_pos; a.pairing = pairing; a.scale = scale; a.weights = PI_WEIGHTS_SOFTMAX; a.sink = sink_dev; a.gate = gate_dev; a.gs = gate_stride; a.gate_act = gate_act; a.gate_width = gate_width; a.out_mult = 1.0f;
    a.out = out; a.os = out_stride;
    // few tokens, sizes of whole steps (more scratch memory than the per-token kernels': its size is pi_op_latent_attention_rot_scratch_floats'); fewer than eight rows over a long context: those (1 head, 1 token of 16384
    // cells 34 us, 40 here)
    const int S32 = (n_kv + 31) / 32;
    const bool whole = lat_rows_takes(heads, rank, rot, n_tok, n_kv) && (n_tok * heads >= 8 || n_kv < 4096) && lat_rows_floats(heads, rank, rot, n_tok, n_kv) <= scratch_floats &&
                       (((uintptr_t) cache | (uintptr_t) scratch_dev) & 15) == 0 && (int64_t) n_kv * (rank + rot) < (1ll << 30);
    int live_min = 0;                                                  // the launches below are for passes of more live cells
    // the tokens' latents, normed on their way: beside the queries where those kernels follow, which read nothing of the cells' (us a step's layer less: 5), else ahead of everything
    lat_kv kv = tokens;
    if (kv.w && (!whole || rot > 0 || ((uintptr_t) kv.x & 15) || kv.xs % 4 || ((uintptr_t) kv.w & 15))) {
        if (pi_op_rms_scale(kv.x, kv.xs, kv.w, 0.0f, kv.eps, rank, n_tok, nullptr, 0, nullptr, 0, 1.0f, kv.cache, rank + rot, dyn_dev, 1, stream) != 0) return -1;
        kv.w = nullptr;
    }
    if (!whole && (live_min = latent_prompt(a, p, cache, rank, wuk, wuv, scratch_dev, scratch_floats, 4.0 * acct * heads * (double) (dim + vdim) + 4.0 * n_tok * heads * (double) (dim + rot + vdim), s)) > 0) {
        PI_CHECK_LAUNCH();
        if (live_min >= n_kv) return 0;
    }
    PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, nta, 2.0 * rank * heads * dim + 4.0 * n_tok * heads * (dim + rank + 2.0 * rot), k_latent_absorb, dim3((unsigned) ((n_tok + 3) / 4), (unsigned) heads, (unsigned) ((rank + 63) / 64 + (rot + 63) / 64 + (kv.w ? 1 : 0))), dim3(256), (size_t) 16 * dim, s,
                 q, q_stride, (const uint16_t *) wuk->p0, scale, heads, dim, rank, rot, cs, n_pos, pairing, pos_dev, n_tok, qa, dyn_dev, live_min, kv, pi_abort_word());
    PI_CHECK_LAUNCH();
    const double bytes = 4.0 * acct * (rank + rot) + 4.0 * n_tok * heads * (rank + rot + (double) rank * p.S);
    // most rows and more shares of the splits than the 256 MB of the last cache: the kernels per token (32 tokens of 16 heads, rank 512 + 64, us here / per token: 6000 cells 327 / 482, 9000 611 / 510, 16000 1029 / 968; of
    // 24 tokens, 384 rows, 16000 cells still 695 / 973)
    const int64_t rows_to = n_tok > 8 && dyn_dev && (int64_t) n_tok * heads * rank > 448 * 512 ? ((int64_t) 1 << 31) / ((int64_t) n_tok * heads * rank) : n_kv;
    const int live_max = whole && rows_to < n_kv ? (int) rows_to : 0;
#define LAT_COMBINE(MANY, NT) PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, nta, 2.0 * rank * heads * vdim + 4.0 * n_tok * heads * (rank * S + vdim), (k_latent_combine<MANY, NT>), dim3((unsigned) ((n_tok + 3) / 4), (unsigned) heads, (unsigned) ((vdim + 15) / 16)), \
                 dim3(NT), (size_t) 16 * rank, s, pol, pml, (const uint16_t *) wuv->p0, sink_dev, gate_dev, gate_stride, gate_act, gate_width, heads, vdim, rank, S, n_tok, n_kv, rows ? 32 : p.cap, dyn_dev, rows ? 0 : live_min, rows ? live_max : 0, \
                 vec, out, out_stride, pi_abort_word())
    auto combine = [&](int S, bool rows) -> int {
        const int vec = (rank & 7) == 0 && (rank > 64 || S > 32) && (((uintptr_t) wuv->p0 | (uintptr_t) pol) & 15) == 0;      // (rank 64: one split 16.3 us, 17.1 so; 64 splits 18.9 and 18.3)
        // Many splits of whole rows: eight waves, as a thread's trips to memory one behind the other are what is waited for; up to two workgroups a compute unit.  us of 256 / 512 threads, rank 512: 4 tokens x 16 heads, 23 splits
        // 12.7 / 10.6, 10 splits 10.9 / 8.3, 1 token 23 splits 9.1 / 7.4, 250 splits 27.6 / 19.6, 8 tokens x 32 heads (512 workgroups), 32 splits 17.7 / 14.8, x 64 heads 22.5 / 26.8.  (How many splits are live is not known here: 2 tokens x 64 heads
        // with the launches ahead, over 204 of 4096 cells 22.3 / 23.5, over 4096 65 / 59)
        const int64_t wgs = (int64_t) ((n_tok + 3) / 4) * heads * ((vdim + 15) / 16);
        if (S > 8 && vec && rank > 64 && wgs <= 2 * pi_cu_count()) LAT_COMBINE(true, 512); else if (S > 8) LAT_COMBINE(true, 256); else LAT_COMBINE(false, 256);
        PI_CHECK_LAUNCH(); return 0;
    };
    if (whole) {
        pml = pol + (size_t) n_tok * heads * S32 * rank;
        const unsigned row_tiles = (unsigned) ((n_tok * heads + 15) / 16);
        const dim3 rgrid(row_tiles, std::min((unsigned) S32, std::max(1u, 4096u / row_tiles)));      // (a context that holds less than it could: 8 tokens x 32 heads, 512 cells of 65536, a workgroup for each of the 2048 splits: 129 us, so 35)
#define LAT_ROWS2(NJ, EX, LOOP) PI_KT_LAUNCH(PI_KT_ATT, PI_BF16, nta, bytes, (k_latent_rows<NJ, EX, LOOP>), rgrid, dim3(256), 0, s, qa, cache, mask, heads, rank + rot, n_tok * heads, n_kv, S32, pol, pml, dyn_dev, live_max, pi_abort_word())
#define LAT_ROWS(NJ, EX) do { if (rgrid.y < (unsigned) S32) LAT_ROWS2(NJ, EX, true); else LAT_ROWS2(NJ, EX, false); } while (0)
        if (rank == 256) { if (rot) LAT_ROWS(4, 4); else LAT_ROWS(4, 0); } else { if (rot) LAT_ROWS(8, 4); else LAT_ROWS(8, 0); }
#undef LAT_ROWS2
#undef LAT_ROWS
        PI_CHECK_LAUNCH();
        if (combine(S32, true) != 0) return -1;
        if (live_max == 0) return 0;
        live_min = live_max;
        pml = pol + (size_t) n_tok * heads * p.S * rank;
    }
    const dim3 grid((unsigned) n_tok, (unsigned) ((heads + p.M - 1) / p.M), (unsigned) p.S);
#define LAT_GO(M) do { if (p.RPT == 1) latent_scores_launch<M, 1>(p, grid, s, bytes, nta, qa, cache, mask, heads, rank, rot, n_kv, pol, pml, dyn_dev, live_min); \
                       else if (p.RPT == 2) latent_scores_launch<M, 2>(p, grid, s, bytes, nta, qa, cache, mask, heads, rank, rot, n_kv, pol, pml, dyn_dev, live_min); \
                       else latent_scores_launch<M, 4>(p, grid, s, bytes, nta, qa, cache, mask, heads, rank, rot, n_kv, pol, pml, dyn_dev, live_min); } while (0)
    switch (p.M) { case 16: LAT_GO(16); break; case 8: LAT_GO(8); break; case 4: LAT_GO(4); break; case 2: LAT_GO(2); break; default: LAT_GO(1); }
#undef LAT_GO
    PI_CHECK_LAUNCH();
    return combine(p.S, false);
#undef LAT_COMBINE
    PI_CHECK_LAUNCH(); return 0;
}
extern "C" int pi_op_latent_attention_gated(const float * q, int64_t q_stride, const float * cache, const uint32_t * mask, const pi_weight * wuk, const pi_weight * wuv, const float * sink_dev, const float * gate_dev,
                                            int64_t gate_stride, int gate_act, int gate_width, float scale, int heads, int dim, int rot, int vdim, int rank, const void * rotary_table, int pairing, const int32_t * pos_dev,
                                            int n_tok, int n_kv, float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride, const int32_t * dyn_dev, void * stream) {
    return latent_attention(q, q_stride, cache, mask, wuk, wuv, sink_dev, gate_dev, gate_stride, gate_act, gate_width, scale, heads, dim, rot, vdim, rank, rotary_table, pairing, pos_dev, n_tok, n_kv, scratch_dev, scratch_floats, out,
                            out_stride, dyn_dev, {}, stream);
}
// pi_op_rms_scale of the tokens' latents into their cells, and pi_op_latent_attention
extern "C" int pi_op_latent_attention_tokens(const float * kv, int64_t kv_stride, const float * kv_norm, float eps, const float * q, int64_t q_stride, float * cache, const uint32_t * mask, const pi_weight * wuk, const pi_weight * wuv,
                                             const float * sink_dev, float scale, int heads, int dim, int vdim, int rank, int n_tok, int n_kv, float * scratch_dev, size_t scratch_floats, float * out, int64_t out_stride,
                                             const int32_t * dyn_dev, void * stream) {
    if (!sink_dev || !kv || !kv_norm || !dyn_dev) { pi_set_error("pi_op_latent_attention_tokens: the latents, their norm, the sink and the cell table are required"); return -1; }
    return latent_attention(q, q_stride, cache, mask, wuk, wuv, sink_dev, nullptr, 0, PI_ACT_NONE, 1, scale, heads, dim, 0, vdim, rank, nullptr, PI_PAIR_HALVES, nullptr, n_tok, n_kv, scratch_dev, scratch_floats, out, out_stride, dyn_dev,
                            { kv, kv_stride, kv_norm, eps, cache }, stream);
}

// ---- routed feed-forward ------------------------------------------------------------------------------------------------------------------------------
// one workgroup per token: logits of all router outputs (a wave per output; few tokens: up to sixteen waves, so that ten outputs are one trip to memory: 7.2 us on four, 5.4 so), soft-max, choice = score + correction, `top` rounds of arg-max (lowest index wins a tie)
// n_groups > 0: the scores are sigmoid(logit), consecutive outputs are bundled into n_groups groups of equal size, a group is ranked by top1 + top2 of its members' scores, and the
// choice is restricted to members of the `keep` highest-ranked groups (then by their own score; lowest index wins a tie, among groups as among outputs)
// (moe_choose: one wave, from the logits in z.  Up to 64 outputs, whose corrections (c0: the lane's) have come with the launch's first loads: an output to a lane, a round is the largest across the lanes and the first that has it.  With
// rounds through LDS, corrections asked for at the end and the chosen logits read back from memory: k_rms_route of ten outputs in a model's step 5.2 us, 3.8 so; of 512 tokens of 2048 8.5 and 7.2, of 2048 of 4096 34 and 32)
static __device__ __forceinline__ void moe_choose(float * z, int n_out, const float * __restrict__ corr, float c0, int top, int n_groups, int keep, int t, int lane, int32_t * __restrict__ sel, float * __restrict__ selw) {
    if (n_groups <= 0 && n_out <= 64 && (n_groups == 0 || top <= 16)) {
        const bool there = lane < n_out;
        float score = there ? z[lane] : -INFINITY, choice;
        if (n_groups < 0) choice = score = score + c0;
        else {
            const float m = pi_wave_max(score), p = there ? expf(score - m) : 0.0f;
            score = p / pi_lanes_sum<64>(p);
            choice = score + c0;
        }
        float chosen[16], own = 0.0f; int which = 0;                    // the chosen scores (by logit); lane kk: the kk-th's score and number
#pragma unroll
        for (int i = 0; i < 16; i++) chosen[i] = -INFINITY;
        for (int k0 = 0; k0 < top; k0 += 64) {
            const int k1 = min(top - k0, 64);
            for (int kk = 0; kk < k1; kk++) {
                const float best = pi_wave_max(there && choice == choice ? choice : -INFINITY);
                const uint64_t who = __ballot(there && choice == best);
                const int bi = who ? __ffsll((unsigned long long) who) - 1 : 0;       // (fewer finite choices than `top`: cannot happen with finite logits)
                const float sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(score), bi));
                if (lane == kk) { own = sc; which = bi; }
                if (lane == bi) choice = -INFINITY;
#pragma unroll
                for (int i = 0; i < 16; i++) if (i == kk) chosen[i] = sc;
            }
            if (n_groups < 0) {                                         // soft-max over the chosen logits alone (the first chosen is the largest)
                float l = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; i++) if (i < top) l += expf(chosen[i] - chosen[0]);
                own = expf(own - chosen[0]) / l;
            }
            if (lane < k1) { sel[(int64_t) t * top + k0 + lane] = which; selw[(int64_t) t * top + k0 + lane] = own; }
        }
        return;
    }
    float * ch = z + n_out, * gsc = ch + n_out;   // [n_out] logits -> scores | [n_out] choice | [n_groups] group scores
    if (n_groups < 0) {                           // by logit (+ bias); the weights are worked out over the chosen ones below
        for (int e = lane; e < n_out; e += 64) { z[e] += corr ? corr[e] : 0.0f; ch[e] = z[e]; }
    } else if (n_groups > 0) {
        const int per = n_out / n_groups;
        for (int e = lane; e < n_out; e += 64) { z[e] = 1.0f / (1.0f + expf(-z[e])); ch[e] = -INFINITY; }
        for (int g = lane; g < n_groups; g += 64) {
            float b0 = -INFINITY, b1 = -INFINITY;
            for (int e = g * per; e < (g + 1) * per; e++) { const float v = z[e]; if (v > b0) { b1 = b0; b0 = v; } else if (v > b1) b1 = v; }
            gsc[g] = b1 == -INFINITY ? b0 : b0 + b1;
        }
        for (int kk = 0; kk < keep; kk++) {
            float bv = -INFINITY; int bi = 0x7fffffff;
            for (int g = lane; g < n_groups; g += 64) { const float c = gsc[g]; if (c > bv || (c == bv && g < bi)) { bv = c; bi = g; } }
            for (int d = 32; d > 0; d >>= 1) {
                const float ov = __shfl_xor(bv, d, PI_WAVE); const int oi = __shfl_xor(bi, d, PI_WAVE);
                if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
            }
            if (bi == 0x7fffffff) break;
            for (int e = bi * per + lane; e < (bi + 1) * per; e += 64) ch[e] = z[e];
            if (lane == 0) gsc[bi] = -INFINITY;
        }
    } else {
    float m = -INFINITY;
    for (int e = lane; e < n_out; e += 64) m = fmaxf(m, z[e]);
    m = pi_wave_max(m);
    float l = 0.0f;
    for (int e = lane; e < n_out; e += 64) { const float p = expf(z[e] - m); z[e] = p; l += p; }
    l = pi_lanes_sum<64>(l);
    for (int e = lane; e < n_out; e += 64) { z[e] = z[e] / l; ch[e] = z[e] + corr[e]; }
    }
    for (int kk = 0; kk < top; kk++) {
        float bv = -INFINITY; int bi = 0x7fffffff;
        for (int e = lane; e < n_out; e += 64) { const float c = ch[e]; if (c > bv || (c == bv && e < bi)) { bv = c; bi = e; } }
        for (int d = 32; d > 0; d >>= 1) {
            const float ov = __shfl_xor(bv, d, PI_WAVE); const int oi = __shfl_xor(bi, d, PI_WAVE);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (bi == 0x7fffffff) bi = 0;             // (fewer finite choices than `top`: cannot happen with finite logits)
        if (lane == 0) { sel[(int64_t) t * top + kk] = bi; selw[(int64_t) t * top + kk] = z[bi]; ch[bi] = -INFINITY; }
    }
    if (n_groups < 0 && lane == 0) {              // soft-max over the chosen logits alone (the first chosen is the largest)
        float * wt = selw + (int64_t) t * top;
        const float m = wt[0];
        float l = 0.0f;
        for (int kk = 0; kk < top; kk++) { wt[kk] = expf(wt[kk] - m); l += wt[kk]; }
        for (int kk = 0; kk < top; kk++) wt[kk] = wt[kk] / l;
    }
}
__global__ void __launch_bounds__(1024) k_moe_route(const uint16_t * __restrict__ router, int64_t width, int n_out, const float * __restrict__ corr, const float * __restrict__ x, int64_t xs,
                                                   int top, int exact, int vec, int n_groups, int keep, int32_t * __restrict__ sel, float * __restrict__ selw, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    extern __shared__ float z[];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float c0 = corr && lane < n_out ? corr[lane] : 0.0f;
    const float * xr = x + (int64_t) t * xs;
    for (int e = wave; e < n_out; e += (int) (blockDim.x >> 6)) {
        const float a = pi_lanes_sum<64>(hy_dot_lane(router + (int64_t) e * width, xr, width, lane, exact != 0, vec != 0));
        if (gone & 1) break;                                           // (no further outputs for a cancelled run)
        if (lane == 0) z[e] = a;
    }
    __syncthreads();
    if (wave != 0 || pi_abort_late(gone, abort_w)) return;
    moe_choose(z, n_out, corr, c0, top, n_groups, keep, t, lane, sel, selw);
}
// The norm ahead of the router and the router, a workgroup per token: the row goes from the norm's registers to LDS as the products read it (exact: as it is; else rounded once, not once per output), and a wave's first
// output's weights leave ahead of the norm.  us of the two launches / of this, 10 outputs: 1 token of
// 2048 7.9 / 5.5, of 4096 10.0 / 6.7; 512 tokens of 2048 12.4 / 7.5, 2048 of 4096 50 / 23; 64 outputs, 2048 tokens of 4096 143 / 57
template <int NV>
__global__ void __launch_bounds__(1024) k_rms_route(const float * __restrict__ y, int64_t ys, const hy_norm p, const uint16_t * __restrict__ router, int width, int n_out, const float * __restrict__ corr, int top, int exact,
                                                    int32_t * __restrict__ sel, float * __restrict__ selw, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    extern __shared__ __attribute__((aligned(16))) float row[];        // [width] | z
    __shared__ float red[16];
    float * const z = row + width;
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (int) (blockDim.x >> 6);
    const float c0 = corr && lane < n_out ? corr[lane] : 0.0f;
    hy_u16x8v rw[2 * NV];
#pragma unroll
    for (int j = 0; j < 2 * NV; j++) rw[j] = *(const hy_u16x8v *) (router + (int64_t) min(wave, n_out - 1) * width + min(lane * 8 + 512 * j, width - 8));
    float4 xv[NV], wv[NV], rv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = min(((int) threadIdx.x & 255) * 4 + 1024 * j, width - 4);
        xv[j] = *(const float4 *) (y + (int64_t) t * ys + i); wv[j] = *(const float4 *) (p.w + i); rv[j] = *(const float4 *) (p.res + (int64_t) t * p.rs + i);
    }
    hy_rms_row<NV>(xv, wv, p.w_off, p.eps, width, false, wv, true, rv, p.mult, red);
    if (pi_abort_late(gone, abort_w)) return;
    if (threadIdx.x < 256) {
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int i = (int) threadIdx.x * 4 + 1024 * j;
            if (i < width) *(float4 *) (row + i) = exact ? xv[j] : make_float4(hy_round(xv[j].x), hy_round(xv[j].y), hy_round(xv[j].z), hy_round(xv[j].w));
        }
    }
    hy_rms_store<NV>(xv, t, t, width, p.eps, p.out, p.os, hy_second{}, rd, red);
    __syncthreads();
    for (int e = wave; e < n_out; e += nw) {
        float a = 0.0f;
#pragma unroll
        for (int j = 0; j < 2 * NV; j++) {
            const int i = lane * 8 + 512 * j;
            if (i >= width) break;
            const float4 x0 = *(const float4 *) (row + i), x1 = *(const float4 *) (row + i + 4);
            const float xf[8] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
#pragma unroll
            for (int k = 0; k < 8; k++) a = fmaf(hy_widen(rw[j][k]), xf[k], a);
        }
        if (e + nw < n_out) {
#pragma unroll
            for (int j = 0; j < 2 * NV; j++) rw[j] = *(const hy_u16x8v *) (router + (int64_t) (e + nw) * width + min(lane * 8 + 512 * j, width - 8));
        }
        a = pi_lanes_sum<64>(a);
        if (lane == 0) z[e] = a;
    }
    __syncthreads();
    if (wave == 0) moe_choose(z, n_out, corr, c0, top, 0, 0, t, lane, sel, selw);
}

// up[t][kk][f] = relu(W_up[e] x_t)^2 for the kk-th chosen expert e of token t (nothing for identity experts); a wave per row f.
// glu: an expert's first matrix holds 2 * ff rows [gate | up] and up[t][kk][f] = silu(gate_f . x) * (up_f . x)
// (this kernel and the next: the abort word and the choice leave together, and the word is looked at before the choice is used.  In a cancelled run the router has written none: what stands there may be anything, and
// an expert's matrix is not read for nothing.  A choice below zero is nobody's)
__global__ void __launch_bounds__(256) k_moe_up(const uint16_t * __restrict__ wup, int64_t width, int ff, int n_exp, const float * __restrict__ x, int64_t xs, const int32_t * __restrict__ sel,
                                                int top, int exact, int vec, int glu, float limit, float * __restrict__ up, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int lane = threadIdx.x & 63, f = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int slot = blockIdx.y, e = sel[slot];
    if (pi_abort_late(gone, abort_w, 0) || f >= ff || (uint32_t) e >= (uint32_t) n_exp) return;
    const int t = slot / top;
    const float * xr = x + (int64_t) t * xs;
    if (glu) {
        const float g = pi_lanes_sum<64>(hy_dot_lane(wup + ((int64_t) e * 2 * ff + f) * width, xr, width, lane, exact != 0, vec != 0));
        const float u = pi_lanes_sum<64>(hy_dot_lane(wup + ((int64_t) e * 2 * ff + ff + f) * width, xr, width, lane, exact != 0, vec != 0));
        if (lane == 0) up[(int64_t) slot * ff + f] = hy_glu(g, u, glu, limit);
        return;
    }
    const float a = pi_lanes_sum<64>(hy_dot_lane(wup + ((int64_t) e * ff + f) * width, xr, width, lane, exact != 0, vec != 0));
    if (lane == 0) { const float r = fmaxf(a, 0.0f); up[(int64_t) slot * ff + f] = r * r; }
}
// out[t][n] = sum_kk w_kk * (identity ? x[t][n] : W_down[e_kk][n] . up[t][kk]); a wave per output n
__global__ void __launch_bounds__(256) k_moe_down(const uint16_t * __restrict__ wdown, int64_t width, int ff, int n_exp, int top, const float * __restrict__ x, int64_t xs,
                                                  const int32_t * __restrict__ sel, const float * __restrict__ selw, const float * __restrict__ up, int exact, int vec, float * __restrict__ out, int64_t os,
                                                  const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    const int lane = threadIdx.x & 63;
    const int64_t n = (int64_t) blockIdx.x * 4 + (threadIdx.x >> 6);
    const int t = blockIdx.y;
    const int32_t * own = sel + (int64_t) t * top;
    int e = own[0];
    if (pi_abort_late(gone, abort_w, 0) || n >= width) return;
    float acc = 0.0f;
    for (int kk = 0; kk < top; kk++) {
        if (kk > 0) e = own[kk];
        const float wgt = selw[(int64_t) t * top + kk];
        if (e < 0) continue;
        if (e >= n_exp) { acc = fmaf(wgt, x[(int64_t) t * xs + n], acc); continue; }
        const float a = pi_lanes_sum<64>(hy_dot_lane(wdown + ((int64_t) e * width + n) * ff, up + ((int64_t) t * top + kk) * ff, ff, lane, exact != 0, vec != 0));
        acc = fmaf(wgt, a, acc);
    }
    if (lane == 0) out[(int64_t) t * os + n] = acc;
}

static int moe_route_launch(const pi_weight * router, const float * correction_dev, const float * x, int64_t x_stride, int n_tok, int top, int exact, int n_groups, int keep, int32_t * sel_dev, float * selw_dev, void * stream) {
    if (n_tok <= 0) return 0;
    if (!router || router->type != PI_BF16 || top < 1 || top > router->ne1 || router->ne1 > 8192) { pi_set_error("pi_op_moe_route: a bfloat16 router of at most 8192 outputs and 1 <= top <= outputs are required"); return -1; }
    PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 2.0 * router->ne0 * router->ne1 + 4.0 * n_tok * router->ne0, k_moe_route, dim3((unsigned) n_tok), dim3((unsigned) (64 * (n_tok <= 64 ? std::min<int64_t>(16, router->ne1) : 4))), (size_t) 8 * router->ne1 + (size_t) 4 * std::max(n_groups, 1), (hipStream_t) stream,
                 (const uint16_t *) router->p0, router->ne0, (int) router->ne1, correction_dev, x, x_stride, top, exact,
                 (int) (router->ne0 % 8 == 0 && ((uintptr_t) router->p0 % 16) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0), n_groups, keep, sel_dev, selw_dev, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
// pi_op_rms_scale with a residual, and pi_op_moe_route of the result
extern "C" int pi_op_rms_scale_route(const float * y, int64_t y_stride, const float * w, float w_offset, float eps, const float * residual, int64_t residual_stride, float mult, float * out, int64_t out_stride,
                                     const pi_weight * router, const float * correction_dev, int n_tok, int top, int exact, int32_t * sel_dev, float * selw_dev, void * stream) {
    if (n_tok <= 0) return 0;
    if (!router || router->type != PI_BF16 || top < 1 || top > router->ne1 || router->ne1 > 8192) { pi_set_error("pi_op_rms_scale_route: a bfloat16 router of at most 8192 outputs and 1 <= top <= outputs are required"); return -1; }
    const int n = (int) router->ne0, n_out = (int) router->ne1;
    const size_t lds = 4 * ((size_t) n + 2 * n_out + 1);
    const bool one = residual && n <= 4096 && n % 8 == 0 && n_out <= 4096 && rms_vec(n, { { y, y_stride }, { w, 0 }, { residual, residual_stride }, { out, out_stride }, { router->p0, 0 } });
    if (!one) {
        if (pi_op_rms_scale(y, y_stride, w, w_offset, eps, n, n_tok, nullptr, 0, residual, residual_stride, mult, out, out_stride, nullptr, 0, stream) != 0) return -1;
        return moe_route_launch(router, correction_dev, out, out_stride, n_tok, top, exact, 0, 0, sel_dev, selw_dev, stream);
    }
    const hy_norm p = { w, w_offset, eps, residual, residual_stride, mult, out, out_stride, {} };
    const int waves = n_tok <= 64 ? std::max(4, std::min(16, n_out)) : 4;
    const pi_round_dst rd = pi_round_asked(0, n);
#define RR_GO(NV) PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 2.0 * n * n_out + 16.0 * n_tok * n, k_rms_route<NV>, dim3((unsigned) n_tok), dim3(64 * waves), lds, (hipStream_t) stream, y, y_stride, p, (const uint16_t *) router->p0, \
                               n, n_out, correction_dev, top, exact, sel_dev, selw_dev, rd, pi_abort_word())
    if (n <= 1024) RR_GO(1); else if (n <= 2048) RR_GO(2); else RR_GO(4);
#undef RR_GO
    PI_CHECK_LAUNCH(); return 0;
}
extern "C" int pi_op_moe_route(const pi_weight * router, const float * correction_dev, const float * x, int64_t x_stride, int n_tok, int top, int exact, int32_t * sel_dev, float * selw_dev, void * stream) {
    return moe_route_launch(router, correction_dev, x, x_stride, n_tok, top, exact, 0, 0, sel_dev, selw_dev, stream);
}
extern "C" int pi_op_moe_route_top_logits(const pi_weight * router, const float * bias_dev, const float * x, int64_t x_stride, int n_tok, int top, int exact, int32_t * sel_dev, float * selw_dev, void * stream) {
    return moe_route_launch(router, bias_dev, x, x_stride, n_tok, top, exact, -1, 0, sel_dev, selw_dev, stream);
}
extern "C" int pi_op_moe_route_groups(const pi_weight * router, const float * x, int64_t x_stride, int n_tok, int top, int n_groups, int keep, int exact, int32_t * sel_dev, float * selw_dev, void * stream) {
    if (!router || n_groups < 1 || router->ne1 % n_groups || keep < 1 || keep > n_groups || (int64_t) keep * (router->ne1 / n_groups) < top) {
        pi_set_error("pi_op_moe_route_groups: the router's outputs must divide into the groups, and the kept groups must hold at least `top` outputs"); return -1;
    }
    return moe_route_launch(router, nullptr, x, x_stride, n_tok, top, exact, n_groups, keep, sel_dev, selw_dev, stream);
}
// wup: [n_exp * ff][width], wdown: [n_exp * width][ff] (the experts' matrices one after the other); up_dev: scratch [n_tok][top][ff]
extern "C" int pi_op_moe_experts(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev, int n_tok, int top,
                                 int exact, float * up_dev, float * out, int64_t out_stride, void * stream) {
    return pi_op_moe_experts_act(wup, wdown, n_exp, ff, 0, x, x_stride, sel_dev, selw_dev, n_tok, top, exact, up_dev, out, out_stride, stream);
}
extern "C" int pi_op_moe_experts_act(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int glu, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev, int n_tok, int top,
                                     int exact, float * up_dev, float * out, int64_t out_stride, void * stream) {
    return pi_op_moe_experts_glu(wup, wdown, n_exp, ff, glu, 0.0f, x, x_stride, sel_dev, selw_dev, n_tok, top, exact, up_dev, out, out_stride, stream);
}
extern "C" int pi_op_moe_experts_glu(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int glu, float limit, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev, int n_tok,
                                     int top, int exact, float * up_dev, float * out, int64_t out_stride, void * stream) {
    if (n_tok <= 0) return 0;
    if (glu < PI_GLU_OFF || glu > PI_GLU_CLIPPED) { pi_set_error("pi_op_moe_experts: hidden layer of kind %d is unknown", glu); return -1; }
    const int upr = glu ? 2 : 1;                                       // rows of an expert's first matrix, in units of ff
    hipStream_t s = (hipStream_t) stream;
    int64_t width = 0;
    if (n_exp > 0) {
        if (!wup || !wdown || wup->type != PI_BF16 || wdown->type != PI_BF16 || wup->ne1 != (int64_t) n_exp * ff * upr || wdown->ne0 != ff || wdown->ne1 != (int64_t) n_exp * wup->ne0) {
            pi_set_error("pi_op_moe_experts: expert matrices must be bfloat16 [experts * ff (twice with a gate)][width] and [experts * width][ff]"); return -1;
        }
        width = wup->ne0;
        const double b_up = std::min<double>(n_tok * top, n_exp) * 2.0 * upr * ff * width + 4.0 * n_tok * (width + (double) top * ff);
        PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, std::min(n_tok, PI_KT_MAXNT - 1), b_up, k_moe_up, dim3((unsigned) ((ff + 3) / 4), (unsigned) (n_tok * top)), dim3(256), 0, s,
                     (const uint16_t *) wup->p0, width, ff, n_exp, x, x_stride, sel_dev, top, exact,
                     (int) (width % 8 == 0 && ((uintptr_t) wup->p0 % 16) == 0 && ((uintptr_t) x % 16) == 0 && x_stride % 4 == 0), glu, limit, up_dev, pi_abort_word());
        PI_CHECK_LAUNCH();
    } else width = out_stride;
    const double b_dn = std::min<double>(n_tok * top, std::max(n_exp, 1)) * 2.0 * ff * width + 4.0 * n_tok * (width + (double) top * ff);
    PI_KT_LAUNCH(PI_KT_MATVEC, PI_BF16, std::min(n_tok, PI_KT_MAXNT - 1), b_dn, k_moe_down, dim3((unsigned) ((width + 3) / 4), (unsigned) n_tok), dim3(256), 0, s,
                 n_exp > 0 ? (const uint16_t *) wdown->p0 : nullptr, width, ff, n_exp, top, x, x_stride, sel_dev, selw_dev, up_dev, exact,
                 (int) (n_exp > 0 && ff % 8 == 0 && ((uintptr_t) wdown->p0 % 16) == 0 && ((uintptr_t) up_dev % 16) == 0), out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}

// ---- the same for a prompt's worth of tokens: grouped by expert, on the matrix cores ---------------------------------------------------------------------
// k_moe_group sorts the (token, choice) slots of a pass by expert (a counting sort in one workgroup) and cuts every expert's run into tiles of 64 or 128 slots; k_moe_tile computes the products of a tile with
// its expert's rows on the matrix cores — an expert's matrices are read once per tile of its tokens instead of once per token; k_moe_combine sums a token's weighted choices (identity experts: the input itself).
// idx layout (int32): [0] number of tiles | tile expert [max_tiles] | tile start [max_tiles] | tile length [max_tiles] | order [n_slots]
#define MOE_GROUP_MAX_EXPERTS 1024
static inline int moe_max_tiles(int n_slots, int n_exp) { return (n_slots + 63) / 64 + std::min(n_exp, n_slots); }

// (one workgroup: the slots of a thread are asked for together and stay in registers for the second look.  With 256 threads that read them one after the other, twice: 1024 slots 5.0 us, 4096 12.0; now 4.6 and 6.2)
#define MOE_GROUP_KEEP 8
__global__ void __launch_bounds__(1024) k_moe_group(const int32_t * __restrict__ sel, int n_slots, int n_exp, int max_tiles, int tile_len, int32_t * __restrict__ idx, const int32_t * __restrict__ abort_w) {
    const int gone = pi_abort_peek(abort_w);
    __shared__ int cnt[MOE_GROUP_MAX_EXPERTS], cur[MOE_GROUP_MAX_EXPERTS];
    int32_t * tile_e = idx + 1, * tile_s = tile_e + max_tiles, * tile_n = tile_s + max_tiles, * order = tile_n + max_tiles;
    int own[MOE_GROUP_KEEP];
#pragma unroll
    for (int u = 0; u < MOE_GROUP_KEEP; u++) { const int i = (int) threadIdx.x + 1024 * u; own[u] = i < n_slots ? sel[i] : -1; }
    for (int e = threadIdx.x; e < n_exp; e += 1024) cnt[e] = 0;
    if (pi_aborted_together(gone, abort_w)) return;
#pragma unroll
    for (int u = 0; u < MOE_GROUP_KEEP; u++) if (own[u] >= 0 && own[u] < n_exp) atomicAdd(&cnt[own[u]], 1);
    for (int i = threadIdx.x + 1024 * MOE_GROUP_KEEP; i < n_slots; i += 1024) { const int e = sel[i]; if (e >= 0 && e < n_exp) atomicAdd(&cnt[e], 1); }
    __syncthreads();
    if (threadIdx.x == 0) {
        int at = 0, nt = 0;
        for (int e = 0; e < n_exp; e++) {
            const int n = cnt[e];
            cur[e] = at;
            for (int k = 0; k < n; k += tile_len) { tile_e[nt] = e; tile_s[nt] = at + k; tile_n[nt] = min(tile_len, n - k); nt++; }
            at += n;
        }
        idx[0] = nt;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MOE_GROUP_KEEP; u++) if (own[u] >= 0 && own[u] < n_exp) order[atomicAdd(&cur[own[u]], 1)] = (int) threadIdx.x + 1024 * u;
    for (int i = threadIdx.x + 1024 * MOE_GROUP_KEEP; i < n_slots; i += 1024) { const int e = sel[i]; if (e >= 0 && e < n_exp) order[atomicAdd(&cur[e], 1)] = i; }
}

// A tile of slots x BN rows of its expert's matrix (dense_tile.h).  UP: X rows are the tokens' inputs x[slot / top], W rows W_up[e], out up[slot][f] = relu(.)^2; !UP: X rows up[slot] (K = ff), W rows W_down[e],
// out dn[slot][n].  glu: UP leaves the 2 * ff rows [gate | up] of an expert raw, !UP (PAIR) joins them while it stages them (bs = 2 * ff, K = ff).  What bounds it: as k_dense_tile, whose tiles these are.  Operands
// straight from memory, 64 x 64 without prefetch, took 623 and 702 us for 2048 tokens' two choices of 8 experts 4096 x 2048 (now 91 and 98: 605 and 562 TFLOP/s), 44 and 23 us for 24 tokens' of 1024 x 512
// (10 and 7).
template <int BN, int BT, int WN, int WT, int KG, bool UP, bool PAIR>
__global__ void __launch_bounds__(64 * WN * WT * KG, 2) k_moe_tile(const uint16_t * __restrict__ W, int64_t K, int rows, const float * __restrict__ B, int64_t bs, int top, const int32_t * __restrict__ idx,
                                                          int max_tiles, int glu, float limit, float * __restrict__ out, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 1)) return;
    __shared__ __attribute__((aligned(16))) uint8_t lds[DT_LDS_BYTES(BN, BT, KG)];
    // workgroup n runs on XCD n % 8: an XCD takes a contiguous run of the work, eight tiles of slots (mostly one expert's) by all of its rows
    const int row_blocks = (rows + BN - 1) / BN, total = idx[0] * row_blocks, per = (total + 7) / 8, at = (int) (blockIdx.x >> 3), work = (int) (blockIdx.x & 7) * per + at;
    if (at >= per || work >= total) return;
    const int grp = work / (8 * row_blocks), in_grp = work % (8 * row_blocks), gsz = min(8, idx[0] - 8 * grp), tile = 8 * grp + in_grp % gsz, n0 = in_grp / gsz * BN;
    const int32_t * tile_e = idx + 1, * tile_s = tile_e + max_tiles, * tile_n = tile_s + max_tiles, * order = tile_n + max_tiles;
    const int e = tile_e[tile], start = tile_s[tile], len = tile_n[tile];
    constexpr int SR = 8 * WN * WT;
    const int tid = threadIdx.x % (64 * WN * WT), lane = tid & 63, wave = tid >> 6;
    dt_offs wo; dt_offs64 xo;                                          // the rows this thread stages
#pragma unroll
    for (int i = 0; i < BN / SR; i++) wo[i] = (uint32_t) ((min(n0 + (tid >> 3) + SR * i, rows - 1) - n0) * K);
#pragma unroll
    for (int i = 0; i < BT / SR; i++) { const int slot = order[start + min((tid >> 3) + SR * i, len - 1)]; xo[i] = (uint64_t) (UP ? slot / top : slot) * (uint64_t) bs; }
    dt_f32x4 acc[BN / WN / 16][BT / WT / 16];
    dt_tile<BN, BT, WN, WT, 2, KG, PAIR>(W + ((int64_t) e * rows + n0) * K, wo, B, xo, K, [=](float a, float b) { return hy_glu(a, b, glu, limit); }, K, lds, acc);
    if (KG > 1 && threadIdx.x >= 64 * WN * WT) return;
#pragma unroll
    for (int b = 0; b < BT / WT / 16; b++) {
        const int si = (wave % WT) * (BT / WT) + b * 16 + (lane & 15);
        if (si >= len) continue;
        float * o = out + (int64_t) order[start + si] * rows;
#pragma unroll
        for (int a = 0; a < BN / WN / 16; a++) {
            const int row = n0 + (wave / WT) * (BN / WN) + a * 16 + (lane >> 4) * 4;
            dt_f32x4 v = acc[a][b];
            if (UP && !glu) {
#pragma unroll
                for (int r = 0; r < 4; r++) { v[r] = fmaxf(v[r], 0.0f); v[r] *= v[r]; }
            }
            if (row < rows) *(dt_f32x4 *) (o + row) = v;               // (rows % 8 == 0)
        }
    }
}

// The same tiles from inputs that are bfloat16 already (dense_async.h), the hidden layer left in bfloat16 for the second product: what the engine's prompts take where the experts have no gate.  us for both products of top-2 of 8
// experts, k_moe_tile / these: 4096 x 2048 at 2048 tokens 88 + 98 / 71 + 81, 2048 x 1024 at 512 23.7 + 22 / 19.9 + 18.2
template <int BN, int BT, int WN, int WT, int S, bool UP>
__global__ void __launch_bounds__(64 * WN * WT, 1) k_moe_async(const uint16_t * __restrict__ W, int64_t K, int rows, const uint16_t * __restrict__ B, int64_t bs, int top, const int32_t * __restrict__ idx, int max_tiles,
                                                               float * __restrict__ out, uint16_t * __restrict__ out_h, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w, 1)) return;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[DA_LDS_BYTES(BN, BT, S)];
    const int row_blocks = (rows + BN - 1) / BN, total = idx[0] * row_blocks, per = (total + 7) / 8, at = (int) (blockIdx.x >> 3), work = (int) (blockIdx.x & 7) * per + at;
    if (at >= per || work >= total) return;
    const int grp = work / (8 * row_blocks), in_grp = work % (8 * row_blocks), gsz = min(8, idx[0] - 8 * grp), tile = 8 * grp + in_grp % gsz, n0 = in_grp / gsz * BN;
    const int32_t * tile_e = idx + 1, * tile_s = tile_e + max_tiles, * tile_n = tile_s + max_tiles, * order = tile_n + max_tiles;
    const int e = tile_e[tile], start = tile_s[tile], len = tile_n[tile], wave = threadIdx.x >> 6;
    dt_f32x4 acc[BN / WN / 16][BT / WT / 16];
    da_tile<BN, BT, WN, WT, S>(W + ((int64_t) e * rows + n0) * K, [&](int r) { return (uint32_t) (min(r, rows - 1 - n0) * K * 2); },
                               B, [&](int r) { const int slot = order[start + min(r, len - 1)]; return (uint32_t) ((UP ? slot / top : slot) * bs * 2); }, (int) (K / 64), lds, acc);
    __syncthreads();                                                   // (the operands of every wave are read)
    constexpr int SHARE = DA_LDS_BYTES(BN, BT, S) / (WN * WT) & ~15;
    const int row0 = n0 + (wave / WT) * (BN / WN), si0 = (wave % WT) * (BT / WT);
    da_rows<BN / WN / 16, BT / WT / 16, SHARE>(acc, lds + wave * SHARE, [&](int t, int r, dt_f32x4 v) __attribute__((always_inline)) {
        if (si0 + t >= len || row0 + r >= rows) return;               // (rows % 64 == 0)
        const int64_t at = (int64_t) order[start + si0 + t] * rows + row0 + r;
        if (UP) {
#pragma unroll
            for (int i = 0; i < 4; i++) { v[i] = fmaxf(v[i], 0.0f); v[i] *= v[i]; }
            *(uint2 *) (out_h + at) = make_uint2(pi_round_pair(v[0], v[1]), pi_round_pair(v[2], v[3]));
        } else *(dt_f32x4 *) (out + at) = v;
    });
}

__global__ void __launch_bounds__(256) k_moe_combine(const float * __restrict__ dn, int64_t width, int n_exp, int top, const float * __restrict__ x, int64_t xs, const int32_t * __restrict__ sel,
                                                     const float * __restrict__ selw, float * __restrict__ out, int64_t os, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    const int t = blockIdx.y;
    const int64_t n = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (n >= width) return;
    float acc = 0.0f;
    for (int kk = 0; kk < top; kk++) {
        const int e = sel[(int64_t) t * top + kk];
        acc = fmaf(selw[(int64_t) t * top + kk], e >= n_exp ? x[(int64_t) t * xs + n] : dn[((int64_t) t * top + kk) * width + n], acc);
    }
    out[(int64_t) t * os + n] = acc;
}

// The same and the norm behind it, a workgroup per token (the sum stays in registers: 2048 tokens' top-2 rows of 4096 35 us and the norm 17, 27 so; 512 tokens of 2048 6 and 5, 6 so).  What a combination does not
// need to know - the norm's weights, the residual - leaves ahead of it
template <int NV>
__global__ void __launch_bounds__(256) k_moe_combine_norm(const float * __restrict__ dn, int64_t width, int n_exp, int top, const float * x, int64_t xs, const int32_t * __restrict__ sel,
                                                          const float * __restrict__ selw, const hy_norm p, const pi_round_dst rd, const int32_t * __restrict__ abort_w) {
    if (pi_aborted(abort_w)) return;
    __shared__ float red[4];
    const int t = blockIdx.x, n = (int) width;
    float4 acc[NV], wv[NV], rv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = min((int) threadIdx.x * 4 + 1024 * j, n - 4);
        wv[j] = *(const float4 *) (p.w + i); rv[j] = *(const float4 *) (p.res + (int64_t) t * p.rs + i);
        acc[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    for (int kk = 0; kk < top; kk++) {
        const float g = selw[(int64_t) t * top + kk];
        const float * from = sel[(int64_t) t * top + kk] >= n_exp ? x + (int64_t) t * xs : dn + ((int64_t) t * top + kk) * width;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const float4 v = *(const float4 *) (from + min((int) threadIdx.x * 4 + 1024 * j, n - 4));
            acc[j].x = fmaf(g, v.x, acc[j].x); acc[j].y = fmaf(g, v.y, acc[j].y); acc[j].z = fmaf(g, v.z, acc[j].z); acc[j].w = fmaf(g, v.w, acc[j].w);
        }
    }
    hy_rms_row<NV>(acc, wv, p.w_off, p.eps, n, false, wv, true, rv, p.mult, red);
    hy_rms_store<NV>(acc, t, t, n, p.eps, p.out, p.os, p.two, rd, red);
}

// slots of a tile
static int moe_tile_len(int n_slots, int n_exp) { return n_slots / n_exp >= 256 ? 128 : 64; }
// rows of a tile: as for k_dense_tile, the largest that gives every compute unit a workgroup; where none does, two groups of waves share K.  Of 128 slots 256 rows as soon as tiles of 128 rows would be more than a round
// of workgroups (some more: the number of tiles is an estimate).  us for both products of top-2 of 8 experts, 128 / 256 rows: 4096 x 2048 at 1024 tokens 210 / 190, 2048 356 / 328, 4000 549 / 434; 2048 x 2048 at 1400
// 113 / 96, 3000 227 / 200; and at less than a round 2048 x 1024 at 1400 the one of 208 workgroups + 8.7, the one of 416 - 5.7.  (128 rows by 4 x 2 waves instead of 2 x 4: 1 - 3 % more)
template <bool UP>
static void moe_tile_launch(const uint16_t * w, int64_t K, int rows, const float * b, int64_t bs, int top, const int32_t * idx, int mt, int tl, int est, int glu, float limit, float * out, int nta, double bytes, hipStream_t s) {
#define MOE_GO2(BN, BT, WN, WT, KG, PAIR) PI_KT_LAUNCH(PI_KT_MMQ, PI_BF16, nta, bytes, (k_moe_tile<BN, BT, WN, WT, KG, UP, PAIR>), dim3((unsigned) ((mt * ((rows + BN - 1) / BN) + 7) / 8 * 8)), dim3(64 * WN * WT * KG), 0, s, \
                                               w, K, rows, b, bs, top, idx, mt, glu, limit, out, pi_abort_word())
#define MOE_GO(BN, BT, KG) do { if constexpr (UP) MOE_GO2(BN, BT, 2, 2, KG, false); else if (glu) MOE_GO2(BN, BT, 2, 2, KG, true); else MOE_GO2(BN, BT, 2, 2, KG, false); } while (0)
    const int wg128 = est * ((rows + 127) / 128);
    if constexpr (!UP) if (tl == 128 && glu) { MOE_GO2(64, 128, 2, 4, 1, true); return; }            // (two values for each of X: the registers do not hold the larger tile)
    if (tl == 128 && wg128 > 280 && K < (1 << 23)) MOE_GO2(256, 128, 4, 2, 1, false);                 // (256 rows of weights in 32 bits, in bytes)
    else if (tl == 128) MOE_GO2(128, 128, 2, 4, 1, false);
    else if (wg128 >= 256) MOE_GO(128, 64, 1);
    else if (wg128 >= 128) MOE_GO(128, 64, 2);
    else MOE_GO(64, 64, 2);
#undef MOE_GO
#undef MOE_GO2
}
// the tile that needs the least time by rounds of 256 workgroups, as async_tile_of (dense.hip)
template <bool UP>
static void moe_async_launch(const uint16_t * w, int64_t K, int rows, const uint16_t * b, int64_t bs, int top, const int32_t * idx, int mt, int tl, int est, float * out, uint16_t * out_h, int nta, double bytes, hipStream_t s) {
    auto cost = [&](int bn, double us) { return std::max(1.0, (double) est * ((rows + bn - 1) / bn) / 256) * us; };      // (the number of tiles is an estimate: no whole rounds)
#define MOE_GO(BN, BT, WN, WT, S) PI_KT_LAUNCH(PI_KT_MMQ, PI_BF16, nta, bytes, (k_moe_async<BN, BT, WN, WT, S, UP>), dim3((unsigned) (((int64_t) mt * ((rows + BN - 1) / BN) + 7) / 8 * 8)), dim3(64 * WN * WT), 0, s, \
                                               w, K, rows, b, bs, top, idx, mt, out, out_h, pi_abort_word())
    if (tl == 128) { if (cost(256, 31.0) < cost(128, 19.5)) MOE_GO(256, 128, 4, 2, 3); else MOE_GO(128, 128, 4, 2, 4); }
    else if (cost(64, 6.3) < cost(32, 4.6)) MOE_GO(64, 64, 4, 2, 4);
    else MOE_GO(32, 64, 2, 2, 4);
#undef MOE_GO
}
// ints of index scratch the grouped path needs for a pass of n_tok tokens
extern "C" size_t pi_op_moe_grouped_index_ints(int n_tok, int top, int n_exp) { const int ns = n_tok * top; return (size_t) 1 + 3 * (size_t) moe_max_tiles(ns, n_exp) + (size_t) ns; }
// whether a pass of this shape takes the grouped matrix-core path (otherwise pi_op_moe_experts: gathered mat-vecs)
extern "C" int pi_op_moe_grouped_ok(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int glu, int n_tok, int top, int exact) {
    (void) glu;
    static const int min_slots = getenv("PI_MOE_GROUPED_MIN") ? atoi(getenv("PI_MOE_GROUPED_MIN")) : 32;
    return !exact && n_exp > 0 && n_exp <= MOE_GROUP_MAX_EXPERTS && wup && wdown && n_tok * top >= min_slots && wup->ne0 % 8 == 0 && ff % 8 == 0 &&
           wup->ne0 < (1 << 24) && ff < (1 << 24) &&                   // (a tile's 128 rows of weights in 32 bits, in bytes)
           ((uintptr_t) wup->p0 % 16) == 0 && ((uintptr_t) wdown->p0 % 16) == 0;
}
// up_dev: [n_tok * top][ff], dn_dev: [n_tok * top][width], idx_dev: pi_op_moe_grouped_index_ints ints
extern "C" int pi_op_moe_experts_grouped(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev, int n_tok, int top,
                                         float * up_dev, float * dn_dev, int32_t * idx_dev, float * out, int64_t out_stride, void * stream) {
    return pi_op_moe_experts_grouped_act(wup, wdown, n_exp, ff, 0, x, x_stride, sel_dev, selw_dev, n_tok, top, up_dev, dn_dev, idx_dev, out, out_stride, stream);
}
// glu: w_up holds [gate | up] per expert (2 * ff rows) and up_dev is [n_tok * top][2 * ff]
extern "C" int pi_op_moe_experts_grouped_act(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int glu, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev, int n_tok, int top,
                                             float * up_dev, float * dn_dev, int32_t * idx_dev, float * out, int64_t out_stride, void * stream) {
    return pi_op_moe_experts_grouped_glu(wup, wdown, n_exp, ff, glu, 0.0f, x, x_stride, sel_dev, selw_dev, n_tok, top, up_dev, dn_dev, idx_dev, out, out_stride, stream);
}
extern "C" int pi_op_moe_experts_grouped_glu(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int glu, float limit, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev,
                                             int n_tok, int top, float * up_dev, float * dn_dev, int32_t * idx_dev, float * out, int64_t out_stride, void * stream) {
    if (glu < PI_GLU_OFF || glu > PI_GLU_CLIPPED) { pi_set_error("pi_op_moe_experts_grouped: hidden layer of kind %d is unknown", glu); return -1; }
    if (!pi_op_moe_grouped_ok(wup, wdown, n_exp, ff, glu, n_tok, top, 0)) { pi_set_error("pi_op_moe_experts_grouped: this shape takes pi_op_moe_experts"); return -1; }
    const int upr = glu ? 2 : 1;
    if (wup->type != PI_BF16 || wdown->type != PI_BF16 || wup->ne1 != (int64_t) n_exp * ff * upr || wdown->ne0 != ff || wdown->ne1 != (int64_t) n_exp * wup->ne0 || x_stride % 4 || ((uintptr_t) x % 16)) {
        pi_set_error("pi_op_moe_experts_grouped: expert matrices must be bfloat16 [experts * ff][width] and [experts * width][ff], inputs 16-byte aligned rows"); return -1;
    }
    hipStream_t s = (hipStream_t) stream;
    const int64_t width = wup->ne0;
    const int ns = n_tok * top, mt = moe_max_tiles(ns, n_exp), nta = std::min(n_tok, PI_KT_MAXNT - 1);
    const double wbytes = std::min<double>(ns, n_exp) * 2.0 * ff * width * (glu ? 1.5 : 1.0);
    const int tl = moe_tile_len(ns, n_exp), est = (ns + tl - 1) / tl + std::min(n_exp, ns) / 2;      // (tiles, if the experts' runs end in the middle of one)
    PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 8.0 * ns, k_moe_group, dim3(1), dim3(1024), 0, s, sel_dev, ns, n_exp, mt, tl, idx_dev, pi_abort_word());
    PI_CHECK_LAUNCH();
    const double bytes = wbytes + 4.0 * ns * (width + ff);
    moe_tile_launch<true>((const uint16_t *) wup->p0, width, ff * upr, x, x_stride, top, idx_dev, mt, tl, est, glu, limit, up_dev, nta, bytes, s);
    PI_CHECK_LAUNCH();
    moe_tile_launch<false>((const uint16_t *) wdown->p0, ff, (int) width, up_dev, (int64_t) ff * upr, top, idx_dev, mt, tl, est, glu, limit, dn_dev, nta, bytes, s);
    PI_CHECK_LAUNCH();
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n_tok * width * (top + 2), k_moe_combine, dim3((unsigned) ((width + 255) / 256), (unsigned) n_tok), dim3(256), 0, s,
                 dn_dev, width, n_exp, top, x, x_stride, sel_dev, selw_dev, out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
// whether pi_op_moe_experts_rounded takes the pass: whole steps of both products' K, offsets of a tile's rows in 32 bits
extern "C" int pi_op_moe_rounded_ok(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, int64_t x_stride, int n_tok, int top) {
    return pi_op_moe_grouped_ok(wup, wdown, n_exp, ff, PI_GLU_OFF, n_tok, top, 0) && wup->ne0 % 64 == 0 && ff % 64 == 0 && wup->ne0 < (1 << 22) && ff < (1 << 22) && (int64_t) n_tok * x_stride < (1ll << 31) && (int64_t) n_tok * top * ff < (1ll << 31);
}
// pi_op_moe_experts_grouped from inputs in bfloat16 (xh); x: the same in fp32, what identity experts hand on.  up_dev holds the hidden layer, bfloat16 [n_tok * top][ff]
static int moe_experts_rounded(const char * name, const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, const uint16_t * xh, int64_t xh_stride, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev,
                                         int n_tok, int top, uint16_t * up_dev, float * dn_dev, int32_t * idx_dev, float * out, int64_t out_stride, const hy_norm * norm, void * stream) {
    if (n_tok <= 0) return 0;
    if (!pi_op_moe_rounded_ok(wup, wdown, n_exp, ff, xh_stride, n_tok, top)) { pi_set_error("%s: this shape takes pi_op_moe_experts or pi_op_moe_experts_grouped", name); return -1; }
    if (wup->type != PI_BF16 || wdown->type != PI_BF16 || wup->ne1 != (int64_t) n_exp * ff || wdown->ne0 != ff || wdown->ne1 != (int64_t) n_exp * wup->ne0 || xh_stride % 8 || xh_stride < wup->ne0 || (((uintptr_t) xh | (uintptr_t) up_dev | (uintptr_t) dn_dev) & 15)) {
        pi_set_error("%s: expert matrices must be bfloat16 [experts * ff][width] and [experts * width][ff], inputs 16-byte aligned rows", name); return -1;
    }
    hipStream_t s = (hipStream_t) stream;
    const int64_t width = wup->ne0;
    const int ns = n_tok * top, mt = moe_max_tiles(ns, n_exp), nta = std::min(n_tok, PI_KT_MAXNT - 1), tl = moe_tile_len(ns, n_exp), est = (ns + tl - 1) / tl + std::min(n_exp, ns) / 2;
    const double bytes = std::min<double>(ns, n_exp) * 2.0 * ff * width + 2.0 * ns * (width + ff);
    PI_KT_LAUNCH(PI_KT_OTHER, PI_BF16, 1, 8.0 * ns, k_moe_group, dim3(1), dim3(1024), 0, s, sel_dev, ns, n_exp, mt, tl, idx_dev, pi_abort_word());
    PI_CHECK_LAUNCH();
    moe_async_launch<true>((const uint16_t *) wup->p0, width, ff, xh, xh_stride, top, idx_dev, mt, tl, est, nullptr, up_dev, nta, bytes, s);
    PI_CHECK_LAUNCH();
    moe_async_launch<false>((const uint16_t *) wdown->p0, ff, (int) width, up_dev, ff, top, idx_dev, mt, tl, est, dn_dev, nullptr, nta, bytes, s);
    PI_CHECK_LAUNCH();
    if (norm) {
#define CN_GO(NV) PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n_tok * width * (top + 3), k_moe_combine_norm<NV>, dim3((unsigned) n_tok), dim3(256), 0, s, dn_dev, width, n_exp, top, x, x_stride, sel_dev, selw_dev, *norm, pi_round_asked(0, (int) width), pi_abort_word())
        if (width <= 1024) CN_GO(1); else if (width <= 2048) CN_GO(2); else CN_GO(4);
#undef CN_GO
        PI_CHECK_LAUNCH(); return 0;
    }
    PI_KT_LAUNCH(PI_KT_OTHER, 0, 1, 4.0 * n_tok * width * (top + 2), k_moe_combine, dim3((unsigned) ((width + 255) / 256), (unsigned) n_tok), dim3(256), 0, s,
                 dn_dev, width, n_exp, top, x, x_stride, sel_dev, selw_dev, out, out_stride, pi_abort_word());
    PI_CHECK_LAUNCH(); return 0;
}
extern "C" int pi_op_moe_experts_rounded(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, const uint16_t * xh, int64_t xh_stride, const float * x, int64_t x_stride, const int32_t * sel_dev, const float * selw_dev,
                                         int n_tok, int top, uint16_t * up_dev, float * dn_dev, int32_t * idx_dev, float * out, int64_t out_stride, void * stream) {
    return moe_experts_rounded("pi_op_moe_experts_rounded", wup, wdown, n_exp, ff, xh, xh_stride, x, x_stride, sel_dev, selw_dev, n_tok, top, up_dev, dn_dev, idx_dev, out, out_stride, nullptr, stream);
}
// the same and pi_op_rms_scale of the result with a residual (w2: pi_op_rms_scale_twice); sum: where the result stands in between, if it has to
extern "C" int pi_op_moe_experts_rounded_norm(const pi_weight * wup, const pi_weight * wdown, int n_exp, int ff, const uint16_t * xh, int64_t xh_stride, const float * x, int64_t x_stride, const int32_t * sel_dev,
                                              const float * selw_dev, int n_tok, int top, uint16_t * up_dev, float * dn_dev, int32_t * idx_dev, float * sum, int64_t sum_stride, const float * w, float w_offset, float eps,
                                              const float * residual, int64_t residual_stride, float mult, float * out, int64_t out_stride, const float * w2, float w2_offset, float * out2, int64_t out2_stride, void * stream) {
    if (n_tok <= 0 || !wup) return 0;
    const int n = (int) wup->ne0;
    const hy_norm norm = { w, w_offset, eps, residual, residual_stride, mult, out, out_stride, { w2, w2_offset, out2, out2_stride } };
    const bool one = residual && n <= 4096 && rms_vec(n, { { x, x_stride }, { w, 0 }, { residual, residual_stride }, { out, out_stride }, { w2, 0 }, { w2 ? out2 : nullptr, out2_stride } });
    if (one) return moe_experts_rounded("pi_op_moe_experts_rounded_norm", wup, wdown, n_exp, ff, xh, xh_stride, x, x_stride, sel_dev, selw_dev, n_tok, top, up_dev, dn_dev, idx_dev, nullptr, 0, &norm, stream);
    if (moe_experts_rounded("pi_op_moe_experts_rounded_norm", wup, wdown, n_exp, ff, xh, xh_stride, x, x_stride, sel_dev, selw_dev, n_tok, top, up_dev, dn_dev, idx_dev, sum, sum_stride, nullptr, stream) != 0) return -1;
    if (w2) return pi_op_rms_scale_twice(sum, sum_stride, w, w_offset, eps, n, n_tok, residual, residual_stride, mult, out, out_stride, w2, w2_offset, out2, out2_stride, stream);
    return pi_op_rms_scale(sum, sum_stride, w, w_offset, eps, n, n_tok, nullptr, 0, residual, residual_stride, mult, out, out_stride, nullptr, 0, stream);
}
