/*
 * mi355_ops.h -- kernel-level entry points of libmi355_decode.so.
 *
 * These expose the individual HIP kernels behind mi355_decode.h on caller-owned DEVICE
 * buffers (e.g. torch tensors) so that each fused stage can be checked against the oracle at
 * its own scale and timed on its own (bench.py roofline leg).  They are not needed to use the
 * engine.  Every call runs on the HIP null stream of the current device and synchronises
 * before returning.  Error convention as in mi355_decode.h.
 *
 * Reference op each one replaces (MLX call sites in the reference):
 *   mi_op_gemv        nn.Linear / nn.QuantizedLinear (+ fused RMSNorm / residual / SwiGLU):
 *                     llama.py:64-67,93,143,160-165,175-177,188-190,250-252; qwen3.py:37-40,63,115
 *   mi_op_embed       nn.Embedding / QuantizedEmbedding: llama.py:212; qwen3.py:166
 *   mi_op_rope_append q_norm/k_norm + nn.RoPE + cache.update_and_fetch:
 *                     qwen3.py:65-70; llama.py:107-125; base.py:66-85,119-140
 *   mi_op_attention   mx.fast.scaled_dot_product_attention + causal mask: llama.py:139-141; base.py:17-40
 *   mi_op_sample      sample closure + top_p_sampling: utils.py:345-364; sample_utils.py:3-38
 */
#ifndef MI355_OPS_H
#define MI355_OPS_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* weight kinds */
#define MI_WK_F32 0
#define MI_WK_BF16 1
#define MI_WK_F16 2
#define MI_WK_Q4_F32 3
#define MI_WK_Q4_BF16 4
#define MI_WK_Q4_F16 5
#define MI_WK_Q8_F32 6
#define MI_WK_Q8_BF16 7
#define MI_WK_Q8_F16 8

/* run-time logical rounding on top of the storage dtype */
#define MI_RND_NONE 0
#define MI_RND_BF16 1
#define MI_RND_F16 2

#define MI_PRO_NONE 0
#define MI_PRO_NORM 1

#define MI_EPI_STORE 0
#define MI_EPI_STORE_F32 1
#define MI_EPI_RESID 2
#define MI_EPI_SWIGLU 3

typedef struct mi_op_linear {
  int32_t wk;            /* MI_WK_* */
  int32_t N, K, group;
  const void* w;         /* [N][K] dense, or MLX-packed [N][K*bits/32] */
  const void* scales;    /* [N][K/group] */
  const void* biases;
  int32_t layout;        /* 0 = row-major (checkpoint order), 1 = tile-major (mi_op_repack_tiled; then w is
                            the tiled buffer and scales/biases are unused) */
} mi_op_linear;

typedef struct mi_op_gemv_args {
  const void* x;         /* [M][ldx] */
  int32_t ldx, M;
  int32_t act, rnd;      /* MI_F32/BF16/F16 storage, MI_RND_* */
  int32_t pro;           /* MI_PRO_* */
  int32_t epi;           /* MI_EPI_* */
  const void* norm_w;    /* [K] */
  float eps;
  int32_t ldo;
  void* out;
  void* resid;
  int32_t pair_offset;
  int32_t force_generic; /* 1 = never take the MFMA path */
} mi_op_gemv_args;

typedef struct mi_op_attn_shape {
  int32_t B, L, Hq, Hkv, D;
  int32_t act, kv, rnd, cap;
} mi_op_attn_shape;

int mi_op_gemv(const mi_op_linear* w, const mi_op_gemv_args* a);
int mi_op_gemv_uses_mfma(const mi_op_linear* w, const mi_op_gemv_args* a);
/* launches the same call `iters` times back to back and returns the mean launch time (HIP events) */
int mi_op_gemv_bench(const mi_op_linear* w, const mi_op_gemv_args* a, int iters, float* avg_ms);
/* the split-K weight-streaming GEMM the engine uses for decode steps of 9..128 rows (int4 / int8 weights: 1..128), on its own:
 * a->M in that range, a->pro = MI_PRO_NONE, tile-major 16-bit, int4 or int8 (group 64) weights.  ksplit 0 = the library's
 * cost model (returned in *ksplit_used); iters >= 1 also times that many back-to-back launches into *avg_ms.
 * wide int4 matrices above 16 rows, and narrow ones where its rule says so, with ksplit <= 0 run gemm_q4.hip (x prepared once per launch, K split over the
 * waves of a workgroup; in front of a wide matrix a->pro may then be MI_PRO_NORM); ksplit < 0 forces it, and its plan, for tests and A/B runs:
 * -(row_tiles | ksplit << 11 | 1 << 15 for the narrow matrices' kernel), 0 = the cost model's choice; what the fields between carried (tile units, K lanes, staging waves) is fixed by the kernel and is ignored. */
int mi_op_gemm_skinny(const mi_op_linear* w, const mi_op_gemv_args* a, int ksplit, int* ksplit_used, int iters,
                      float* avg_ms);
/* gemm_prefill.hip on its own: the tile GEMM of the prefill call (generate_step's first model call, utils.py:243-262: every
 * nn.Linear over B x L rows at once).  a->M rows of 16-bit activations, tile-major dense 16-bit weights, a->pro =
 * MI_PRO_NONE; plain / residual / SwiGLU epilogues.  iters >= 1 also times that many back-to-back launches into *avg_ms. */
int mi_op_gemm_prefill(const mi_op_linear* w, const mi_op_gemv_args* a, int iters, float* avg_ms);
/* the same for tile-major int4 / int8 weights (group 64): the tile GEMM on their codes where it takes the call, else on their [hi | lo] copy.
 * a->act: 16-bit, or float32 on a bf16 model (split into three terms here; a->rnd = MI_RND_BF16, plain stores only: one).
 * iters < 0: on the codes whatever the size, or an error. */
int mi_op_gemm_codes(const mi_op_linear* w, const mi_op_gemv_args* a, int iters, float* avg_ms);
/* what a prefill call of a->M rows on tile-major int4 / int8 weights runs on: 2 the tile GEMM on their codes, 1 the tile GEMM on their [hi | lo] copy, 0
 * another kernel (float32 activations: 32 rows per launch of the streaming one); a negative error code.  No device needed; no pointer is read.
 * For calls that make their copy of the codes, as mi_op_gemm_codes does; an engine's float32 rows are priced without that copy and take the codes from fewer rows on. */
int mi_op_gemm_quant_route(const mi_op_linear* w, const mi_op_gemv_args* a);
/* gemv_reg.hip on its own: the decode linears of at most 8 rows on tile-major weights -- int4 / int8 (group 64) with scales of the
 * activations' type (plain / float32 / residual / SwiGLU epilogues, the last with the norm), dense 16-bit ones with activations of
 * their type or float32 on bf16 (plain / float32 / residual; float32 also MI_EPI 4, SwiGLU on a row-interleaved gate|up matrix:
 * 8 gate rows, their 8 up rows, ...).  a->pro MI_PRO_NONE or MI_PRO_NORM. */
int mi_op_gemv_reg(const mi_op_linear* w, const mi_op_gemv_args* a);
/* tile-major weight layout of the streaming kernels (what mi_engine_finalize applies to eligible
 * matrices): returns the size of the tiled buffer (0 if the matrix is not eligible) / fills `dst`. */
uint64_t mi_op_tiled_bytes(const mi_op_linear* row_major);
int mi_op_repack_tiled(const mi_op_linear* row_major, void* dst);
int mi_op_embed(const mi_op_linear* w, const int32_t* tokens, int rows, int act, int rnd, void* out);
int mi_op_rope_tables(float* cos_tab, float* sin_tab, int max_pos, int head_dim, float base, float scale);
int mi_op_rope_append(const mi_op_attn_shape* s, const void* qkv, void* q_out, void* kcache, void* vcache,
                      const int32_t* offsets, const void* q_norm_w, const void* k_norm_w, float eps,
                      const float* cos_tab, const float* sin_tab, int max_pos);
int mi_op_attention(const mi_op_attn_shape* s, const void* q, const void* kcache, const void* vcache,
                    const int32_t* offsets, void* out, float scale, int nsplit, float* partial);
/* causal prefill attention on the matrix cores alone (L > 1), its keys split over up to 16 workgroups, `nsplit` for the longest row and
 * fewer for rows of few keys.  partial: ceil(L / 16) x B x Hkv x nsplit x Hq / Hkv x 64 x (D / 16 + 1) x 4 floats, counters:
 * ceil(L / 16) x B x Hkv ints, zero before and after (both may be NULL for nsplit 1).  btab: block table of a paged cache
 * ([row][bt_stride], blocks of 2^bs_shift tokens), NULL: contiguous. */
int mi_op_attention_prefill(const mi_op_attn_shape* s, const int32_t* btab, int bt_stride, int bs_shift, const void* q,
                            const void* kcache, const void* vcache, const int32_t* offsets, void* out, float scale,
                            int nsplit, float* partial, int32_t* counters);
/* slices over which the engine splits the keys of a prefill call whose longest row reaches max_keys keys, on ncu compute units (no device
 * needed) */
int mi_op_attention_prefill_slices(const mi_op_attn_shape* s, int max_keys, int ncu);
/* fused decode attention (L == 1): q/k norm + RoPE + append + split-KV attention + combine.
 * counters: [B*Hkv] zero-initialised ints.  variant 0: MFMA kernel where it applies (16-bit caches,
 * head_dim % 32 == 0; float32 caches, head_dim 64 / 128), 1: VALU kernel (2: the MFMA kernel in its twelve-wave form,
 * only in a library built with -DMI_ATTN_WIDE; otherwise the same as 0).  iters > 1 repeats the launch (timing; avg_ms may be NULL). */
int mi_op_attention_decode(const mi_op_attn_shape* s, const void* qkv, void* kcache, void* vcache,
                           const int32_t* offsets, const void* q_norm_w, const void* k_norm_w, float eps,
                           const float* cos_tab, const float* sin_tab, void* out, float scale, int rnd_out,
                           int nsplit, float* partial, int32_t* counters, int variant, int iters, float* avg_ms);
/* splits that a decode step's attention is launched with: `groups` (rows x kv heads) whose rows have `keys` cached keys of kv_dtype, on
 * ncu compute units (no device needed) */
int mi_op_attention_decode_splits(int ncu, int groups, int keys, int kv_dtype);
/* row tiles a slab in which an int4 linear of a->M rows (17..128) takes its x as the launch in front of it left it, in the order that it multiplies; 0: it prepares x itself, or is
 * another kernel's (no device needed) */
int mi_op_gemm_q4_prepared(const mi_op_linear* w, const mi_op_gemv_args* a);
/* 1: decoding rows (L == 1) and a chunk of another row's prompt (B == 1), its keys in `slices` workgroups, share one attention launch on paged caches and ncu compute units (no device
 * needed) */
int mi_op_attention_mixed(const mi_op_attn_shape* rows, const mi_op_attn_shape* chunk, int slices, int ncu);
/* 1: logits (rounded = 0) or layer 0's rounded q|k|v (1) of `rows` rows of float32 activations go to the tile GEMM, 0: 32 rows at a time to the
 * streaming kernel.  codes: int4 weights too small for the tile GEMM on codes (the others: mi_op_gemm_quant_route), hilo: an
 * f16 matrix through its [hi | lo] copy (no device needed) */
int mi_op_gemm_prefill_pays(int codes, int hilo, int rounded, int rows);
int mi_op_sample(float* logits, int B, int V, float temperature, float top_p, const float* uniforms,
                 int top_logprobs, int32_t* tokens_out, float* logprob_out, float* prob_row0_out,
                 int32_t* topk_ids, float* topk_logprobs, float* row_stats);

#ifdef __cplusplus
}
#endif
#endif /* MI355_OPS_H */
