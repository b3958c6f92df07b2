// q4_gemm_rows_f16.hip — the k_q4_gemm_rows variants for f16 activations.
#include "q4_gemm_rows.h"

bool sf_gemm_rows_f16(const sf_gemm::RowsArgs &a, const sf_gemm::RowsGroupArgs *group, bool asym, int rb,
                      int kw, hipStream_t s) {
  return sf_gemm::rows_dispatch<SF_F16>(a, group, asym, rb, kw, s);
}
