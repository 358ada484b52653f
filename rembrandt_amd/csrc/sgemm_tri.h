// Column-major products with exactly split operands (sgemm_tri.hip).
#pragma once
#include "gemm_core.h"

namespace rh {

struct SgemmTriPlan {
  int groups;   // of eight k, whole K steps
  int bm, splits;
  size_t rows_bytes, cols_bytes, part_bytes;
  bool ok;
  size_t part_at() const { return rows_bytes + cols_bytes; }
  size_t total() const { return part_at() + part_bytes; }
};
SgemmTriPlan plan_sgemm_tri(bool a_trans, bool b_trans, int m, int n, int k);
// rows: op(B)'s columns (b_trans: contiguous, else k contiguous); cols: op(A)'s rows, 16-byte aligned, ld a multiple of 4.
// ep: where the result goes, or with p.splits > 1 the partial sums, *used slices of them.
int launch_sgemm_tri(const SgemmTriPlan& p, bool a_trans, bool b_trans, const DenseParams& rows, const DenseParams& cols, EpiParams ep,
                     void* ws, hipStream_t stream, int* used);

}  // namespace rh
