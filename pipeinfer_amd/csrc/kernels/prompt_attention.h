// Attention of a prompt's many tokens on the matrix cores (prompt_attention.hip): what the operators of hybrid.hip and parallel_mixer.hip hand over.  Internal to the kernels.
#pragma once
#include "ops_common.h"

struct pa_args {
    const float * q; int64_t qs;                                       // [token][qs]: heads of MAPS x (dim1 + dim2) values
    const float * k1; int64_t k1_row, k1_head; int dim1;               // a cell's key: dim1 values of its head at k1 + cell * k1_row + (head / per_kv) * k1_head, ...
    const float * k2; int64_t k2_row; int dim2;                        // ... then dim2 values that the heads share
    const float * v; int64_t v_row, v_head; int vdim;
    int cell0, cell1;                                                  // the cells of this launch; k1 and v begin at cell0, everything else at cell 0
    int live_max;                                                      // > 0: a launch for passes of no more live cells than that (others return)
    int heads, per_kv, n_tok, n_kv; const int32_t * dyn;
    const uint32_t * mask; const int32_t * cell_pos, * pos;            // cell_pos null: what a token sees is the mask's alone
    int mask_kind, chunk, keep_first;
    const float2 * cs; int n_pos, pairing;                             // dim2 > 0: the query's last dim2 values are turned by the token's position
    float scale; const float * hbias; float softcap; int weights; const float * sink;
    const float * gate; int64_t gs; int gate_act, gate_width;
    float out_mult, lam, eps;
    float * out; int64_t os;
    pi_round_dst rd;                                                   // of the output (the launch that writes it)
    float * state; int first, last;                                    // the cells in several launches: [token][head][vdim sums | maximum | denominator] between them
};
typedef float pa_f32x4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ pa_f32x4 pa_mfma(float a, float b, pa_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// a launch over the cells [cell0, cell1); maps = 2: see ca_join_maps.  false: sizes or alignment that the kernel does not take (pa_takes)
bool pa_takes(const pa_args & a, int maps, int min_tokens);
void pa_launch(const pa_args & a, int maps, double bytes, hipStream_t s);
// Which passes take tiles of 32 tokens rather than a workgroup per token (measured against each other over 9 .. 128 tokens, 16 and 32 heads, contexts of the pass's own tokens, 512 .. 1000 and 4096 cells, us):
//   keys in a cache     from 32 tokens on: 16 heads of 128 over 4: 32 tokens in a window of 256 of 1000 cells 76 -> 36, all of 4000 cells 1060 -> 251, alone in the
//                       cache 15.7 -> 14.8; 128 tokens alone 38 -> 17.  Fewer tokens: k_few_attention (31 of them over all of 1000 cells 31)
//   keys of a latent    from 9 tokens on, but for the long contexts of latent_tiles_to (hybrid.hip) and for the passes that k_latent_rows (hybrid.hip: splits of 32 cells) takes: 16 heads of 128, rank 512, without those: 9 tokens alone 74 -> 27, of 512 cells 179 -> 65, of 4096
//                       440 -> 379; 128 tokens 123 -> 38, 213 -> 69, 836 -> 374
#define PA_CACHE_TOKENS 32
#define PA_LATENT_TOKENS 9
// keys [cell][heads * dim] and values [cell][heads * vdim] of the cells [cell0, cell1) from their latents (row stride `width` floats)
void pa_expand(const float * cache, int64_t width, int rank, const pi_weight * wuk, const pi_weight * wuv, int cell0, int cell1, int n_kv, int live_max, const int32_t * dyn, float * k, float * v, hipStream_t s);
// a few tokens over keys and values in a cache: splits of 32 cells (or of several times 32), sixteen query heads of a key head at a time, every split's [vdim sums | maximum | denominator] per (token, head, map)
// into a.state for the caller's merge.  pa_few_split: cells of a split and their number, 0: not for this kernel
int pa_few_split(const pa_args & a, int maps, size_t scratch_floats, int * split_cells);
void pa_few_launch(const pa_args & a, int maps, int n_cs, int split_cells, double bytes, hipStream_t s);
#define PA_FEW_SPLITS 32
// Keys and values of a latent in three bfloat16 parts and the attention over them (split_attention.hip).  sa_sizes: heads and ranks that the kernels take, sa_takes: passes, sa_pays: which of them are the quicker that way; sa_cell_floats: scratch memory for a cell
bool sa_sizes(int dim, int rot, int vdim, int rank);
bool sa_takes(const pa_args & a, int rank);
bool sa_pays(const pa_args & a, int rank, int live_max);
size_t sa_cell_floats(int heads, int dim, int rot, int vdim);
void sa_launch(const pa_args & a, const float * cache, int rank, const pi_weight * wuk, const pi_weight * wuv, float * scratch, double bytes, hipStream_t s);
