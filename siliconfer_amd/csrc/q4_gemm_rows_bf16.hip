// q4_gemm_rows_bf16.hip — the k_q4_gemm_rows variants for bf16 activations.
#include "q4_gemm_rows.h"

bool sf_gemm_rows_bf16(const sf_gemm::RowsArgs &a, const sf_gemm::RowsGroupArgs *group, bool asym, int rb,
                      int kw, hipStream_t s) {
  return sf_gemm::rows_dispatch<SF_BF16>(a, group, asym, rb, kw, s);
}
