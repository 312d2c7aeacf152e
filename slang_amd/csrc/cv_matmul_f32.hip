// cv_matmul_f32.hip -- fp32 instantiations of the batched matMul kernel
// (bfloat16 pieces on v_mfma_f32_16x16x32_bf16, F32Mma; fp32 vectors, matrix, bias and results).
#include "cv_matmul_impl.h"

namespace cv {

hipError_t launchMatMulF32(hipStream_t stream, const MatMulArgs& a, int numCUs)
{
    return dispatchShape<VecAsMatrix<F32Mma>, float>(stream, a, numCUs);
}

} // namespace cv
