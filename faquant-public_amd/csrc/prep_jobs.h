/*
 * The call between this package's Python modules and the library that runs the operand prologues
 * of one attention call together.  Not part of the public C ABI (include/faquant_amd.h), whose
 * single entries give the same outputs.
 */
#pragma once
#include "../../include/faquant_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * One operand of an attention call for faq_operand_prep_jobs: the arguments of
 * faq_operand_prep (y: bf16 rows), of faq_operand_prep_hif4_kv (codes and meta non-NULL: packed
 * rows instead of y) or, with vt non-NULL, of faq_operand_prep_vt (no key offset, Smooth-QK,
 * Hadamard or packed rows), which then also writes the same values as natural rows to y where y
 * is non-NULL.
 */
typedef struct faq_prep_job {
  const void* x;
  int in_dtype;
  int64_t sb, sh, sl;
  int B, H, L;
  const float* key_offset;
  int64_t off_sh;
  const float* smooth;
  int64_t smooth_sh;
  int smooth_divide, hadamard, round_dtype;
  void* y;
  int64_t yb, yh, yl;
  int levels;
  uint32_t* codes;
  uint32_t* meta;
  int64_t p_sb, p_sh;
  uint16_t* vt;
  int Lpad;
} faq_prep_job;

/*
 * The prologues of one attention call (Q, K and V; simulated_flash_attention.py:592-619,
 * qwen3.py:97-136), the same outputs as the single entries, bit for bit.  At most three row jobs
 * and one vt job (the last) that are bf16 in and round to bf16 run as one launch; any other
 * list runs job by job.  Outputs must not overlap any job's input.
 */
int faq_operand_prep_jobs(const faq_prep_job* jobs, int n, faq_stream_t stream);

#ifdef __cplusplus
}
#endif
