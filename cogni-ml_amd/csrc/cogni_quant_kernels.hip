// The gfx950 code object: every kernel is an unmangled extern "C" __global__ symbol so a host can
// fetch it by name with hipModuleGetFunction after hipModuleLoadData, the way the reference loads
// its PTX modules (src/ml/cuda/driver.cr:115-127).
#include "kernels/dequant.hpp"
#include "kernels/gemv.hpp"
#include "kernels/gemv_plain.hpp"
#include "kernels/gemv_mfma.hpp"
#include "kernels/gemv_mfma_q6k.hpp"
#include "kernels/gemv_mt.hpp"
#include "kernels/gemm_q4k.hpp"
#include "kernels/gemm_q4k_wide.hpp"
#include "kernels/gemm_q6k.hpp"
#include "kernels/gemm_q6k_wide.hpp"
#include "kernels/norm.hpp"

GEMV_MFMA_ENTRY(q4_k_gemv_mfma_f32_tbatch2, 2)
GEMV_MFMA_ENTRY(q4_k_gemv_mfma_f32_tbatch3, 3)
GEMV_MFMA_ENTRY(q4_k_gemv_mfma_f32_tbatch4, 4)
GEMV_MFMA_ADD_ENTRY(q4_k_gemv_mfma_add_f32_tbatch2, 2)
GEMV_MFMA_ADD_ENTRY(q4_k_gemv_mfma_add_f32_tbatch3, 3)
GEMV_MFMA_ADD_ENTRY(q4_k_gemv_mfma_add_f32_tbatch4, 4)
GEMV_MFMA_Q6K_ENTRY(q6_k_gemv_mfma_f32_tbatch3, 3)
GEMV_MFMA_Q6K_ENTRY(q6_k_gemv_mfma_f32_tbatch4, 4)
GEMV_MFMA_Q6K_ADD_ENTRY(q6_k_gemv_mfma_add_f32_tbatch3, 3)
GEMV_MFMA_Q6K_ADD_ENTRY(q6_k_gemv_mfma_add_f32_tbatch4, 4)
GEMV_MFMA_TOP1_ENTRY(q4_k_gemv_mfma_top1_partial_f32_tbatch3, 3)
GEMV_MFMA_TOP1_ENTRY(q4_k_gemv_mfma_top1_partial_f32_tbatch4, 4)
GEMV_MFMA_Q6K_TOP1_ENTRY(q6_k_gemv_mfma_top1_partial_f32_tbatch3, 3)
GEMV_MFMA_Q6K_TOP1_ENTRY(q6_k_gemv_mfma_top1_partial_f32_tbatch4, 4)
GEMV_MFMA_DUAL_ENTRY(q4_k_dual_gemv_mfma_f32_tbatch2, 2)
GEMV_MFMA_DUAL_ENTRY(q4_k_dual_gemv_mfma_f32_tbatch3, 3)
GEMV_MFMA_DUAL_ENTRY(q4_k_dual_gemv_mfma_f32_tbatch4, 4)
GEMV_MFMA_MANY_ENTRY(q4_k_many_gemv_mfma_f32_tbatch2, 2)
GEMV_MFMA_MANY_ENTRY(q4_k_many_gemv_mfma_f32_tbatch3, 3)
GEMV_MFMA_MANY_ENTRY(q4_k_many_gemv_mfma_f32_tbatch4, 4)
GEMV_MFMA_SWIGLU_ENTRY(q4_k_dual_gemv_swiglu_mfma_f32_tbatch2, 2)
GEMV_MFMA_SWIGLU_ENTRY(q4_k_dual_gemv_swiglu_mfma_f32_tbatch3, 3)
GEMV_MFMA_SWIGLU_ENTRY(q4_k_dual_gemv_swiglu_mfma_f32_tbatch4, 4)
GEMV_MFMA_Q5K_ENTRY(q5_k_gemv_mfma_f32_tbatch3, 3)
GEMV_MFMA_Q5K_ENTRY(q5_k_gemv_mfma_f32_tbatch4, 4)
GEMV_MFMA_Q5K_ADD_ENTRY(q5_k_gemv_mfma_add_f32_tbatch3, 3)
GEMV_MFMA_Q5K_ADD_ENTRY(q5_k_gemv_mfma_add_f32_tbatch4, 4)
// Behind the decode kernels, whose distances in the code object stay what they were: with these in front of and among them the
// projections of eight tokens took 58.7 us, with them here 58.4 (58.0 without), in one session each and with the same instructions
// in every kernel that runs. Why is not known, and the difference is hardly more than that of two sessions.
GEMV_TOP1_LOGITS_ENTRY(q4_k_gemv_top1_logits_partial_f32, FmtQ4K, 1)
GEMV_TOP1_LOGITS_ENTRY(q4_k_gemv_top1_logits_partial_f32_tbatch2, FmtQ4K, 2)
GEMV_TOP1_LOGITS_ENTRY(q5_k_gemv_top1_logits_partial_f32, FmtQ5K, 1)
GEMV_TOP1_LOGITS_ENTRY(q6_k_gemv_top1_logits_partial_f32, FmtQ6K, 1)
GEMV_TOP1_LOGITS_ENTRY(q6_k_gemv_top1_logits_partial_f32_tbatch2, FmtQ6K, 2)
GEMV_TOP1_LOGITS_ENTRY(q8_0_gemv_top1_logits_partial_f32, FmtQ80, 1)
GEMV_MT_TOP1_LOGITS_ENTRY(q4_k_gemv_mt_top1_logits_partial_f32, MtQ4K)
GEMV_MT_TOP1_LOGITS_ENTRY(q6_k_gemv_mt_top1_logits_partial_f32, MtQ6K)
#include "kernels/gemm_terms.hpp"
#include "kernels/gemm_stream.hpp"
#include "kernels/gemm_q4k_tall.hpp"
