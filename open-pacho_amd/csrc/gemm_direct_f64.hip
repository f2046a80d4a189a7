// Direct products in f64 (see gemm_direct.h).
#include "gemm_direct_kernels.h"

void hpgemm::direct_f64(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const void* a, const void* b, void* c,
                        int64_t m, int64_t n, int64_t k, const BatchDesc& bd, int64_t batch) {
  run_direct<double>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
}
