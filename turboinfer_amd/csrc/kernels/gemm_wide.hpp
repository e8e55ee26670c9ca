// gemm_wide.hpp -- the many-rows GEMM (gemm_wide.hip): row-major fp16 x against packed weights of every format.
#pragma once
#include "gemm_common.hpp"

namespace ti {

struct WidePlan {
  int shape;             // workgroup shape (gemm_wide.hip), -1: none
  int n_cb, n_rb, n_ks;  // column blocks x row blocks x k-slices
  int rows, tiles;       // of a block
};
// fmt: the bits of ti_gemm_wq_a16.  fold: a call with a folded input or output.  False: not a call of this kernel (shape
// or format).
bool wide_plan(int fmt, int M, int N, int K, int cus, int64_t ws_bytes, bool fold, WidePlan* p);
long wide_workgroups(const WidePlan& p);
int wide_launch(int fmt, const WidePlan& p, const GemvArgs& a, hipStream_t s);
int gemm_cus();       // CUs of the current device (gemv.hip)
int wide_prepare();   // dynamic-LDS limits on the current device

}  // namespace ti
