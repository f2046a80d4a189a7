// Direct products in f32 (see gemm_direct.h).
#include "gemm_direct_kernels.h"

void hpgemm::direct_f32(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const void* a, const void* b, void* c,
                        int64_t m, int64_t n, int64_t k, const BatchDesc& bd, int64_t batch) {
  run_direct<float>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
}
