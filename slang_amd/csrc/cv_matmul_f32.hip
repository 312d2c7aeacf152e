// cv_matmul_f32.hip -- fp32 instantiations of the batched matMul kernel (fp32 vectors, matrix, bias and results): the operators on
// bfloat16 pieces (v_mfma_f32_16x16x32_bf16, F32Mma), the products of the training step over memory on v_mfma_f32_16x16x4_f32
// (F32WholeMma).
#include "cv_matmul_impl.h"

namespace cv {

hipError_t launchMatMulF32(hipStream_t stream, const MatMulArgs& a, int numCUs)
{
    return dispatchShape<VecAsMatrix<F32Mma>, float>(stream, a, numCUs);
}

hipError_t launchMatMulF32Whole(hipStream_t stream, const MatMulArgs& a, int numCUs)
{
    return dispatchShape<VecAsMatrix<F32WholeMma>, float>(stream, a, numCUs);
}

} // namespace cv
