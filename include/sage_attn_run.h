/*
 * sage_attn_run.h — whole-call entry points of libsage_attn.so.
 *
 * sage_attn.h offers the stages (pre-pass, V tiles, attention) one by one;
 * the calls here take a user's Q, K, V and O and choose the stages, kernels
 * and launch shapes themselves.  They share its conventions: strides are the
 * element strides of batch, head and sequence, rows are 16-byte aligned, the
 * caller owns every buffer, calls are asynchronous on `stream`, a non-zero
 * status leaves a message in sage_last_error().
 *
 *   sage_run()       <- run_sage_attn  (kernels/sage_attn/triton_impl.py:162-200)
 *   sage_flash_run() <- run_flash_attn (kernels/flash_attn/triton_impl.py:103-121)
 */
#ifndef SAGE_ATTN_RUN_H
#define SAGE_ATTN_RUN_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* One call.  Every field is 8 bytes, so a binding can pack it as an array. */
typedef struct sage_call {
  int64_t size; /* sizeof(sage_call): a caller built for another layout is refused */
  const void* q;
  const void* k;
  const void* v;
  void* o;         /* [B,Hq,Nq,D] in dtype */
  void* workspace; /* device memory, 256-byte aligned; holds nothing between calls */
  int64_t workspace_bytes;
  int64_t q_strides[3], k_strides[3], v_strides[3], o_strides[3];
  int64_t B, Hq, Hkv, Nq, Nkv, D;
  double mul;     /* fp32(sm_scale * 1.44269504): scores in log2 units */
  int64_t dtype;  /* of q, k, v and o: SAGE_DTYPE_* */
  int64_t causal; /* 1: key j is visible to query i iff j <= i */
  /* sage_run only */
  int64_t pv_mode;  /* SAGE_PV_* */
  int64_t q_sub;    /* rows per Q scale: 128, 32 or 1 */
  int64_t smooth_k; /* 1: subtract the per-channel K mean */
  int64_t fuse_q;   /* where Q is quantized: 1 the attention kernel's prologue (the pre-pass where the keys
                       are split or heads share a work-group), 0 the pre-pass, -1 the faster of the two
                       (the pre-pass with q8): the same Q8 and scales, and the same output, bit for bit.
                       1, and -1 at D = 128, need mul > 0 and finite, a head's Q rows within 2^31 bytes */
  /* optional outputs (NULL: kept in the workspace), as sage_prepass writes them with blkq 128, blkk 64 */
  void* q8; /* with q's strides when fuse_q is 1 (multiples of 16 then), else q8_strides */
  void* q_scale;
  void* k8; /* k8_strides */
  void* k_scale;
  void* km;
  void* v_scale;
  int64_t q8_strides[3], k8_strides[3];
} sage_call;

/* Bytes of workspace the call needs (reads the shape, the options and which optional outputs are NULL). */
size_t sage_run_workspace_bytes(const sage_call* call);
size_t sage_flash_run_workspace_bytes(const sage_call* call);

/* Which parts of the pre-pass sage_run() makes for this call: Q quantized there (or in the attention's
   prologue), V tiles (or V read in place).  For whoever times or repeats the stages one by one. */
int sage_run_stages(const sage_call* call, int* quant_q, int* v_tiles);

/* SageAttention forward: sage_prepass_vt and the fused attention. */
int sage_run(const sage_call* call, void* stream);

/*
 * Unquantized attention on fp16 / bf16 inputs: sage_flash_fwd with V read
 * where it is (no V tiles).  Row strides of V must be below 2^25 elements.
 */
int sage_flash_run(const sage_call* call, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* SAGE_ATTN_RUN_H */
