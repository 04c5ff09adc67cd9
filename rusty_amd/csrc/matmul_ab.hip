// C = A.B on the matrix cores (kernels.wgsl:7-54).
#include "matmul_mfma.hpp"

namespace rq {

int launch_mfma_ab(const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus,
                   hipStream_t s) {
    return launch_mfma<MM_AB>(a, b, out, m, k, n, num_cus, s);
}

}  // namespace rq
