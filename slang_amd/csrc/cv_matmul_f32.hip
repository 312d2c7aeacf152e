// cv_matmul_f32.hip -- fp32 instantiations of the batched matMul kernel (fp32 vectors, matrix, bias and results): the operators on
// bfloat16 pieces (v_mfma_f32_16x16x32_bf16, F32Mma) where these are the faster ones, else, and the products of the training step over memory, on
// v_mfma_f32_16x16x4_f32 (F32WholeMma).
#include "cv_matmul_impl.h"

namespace cv {

hipError_t launchMatMulF32(hipStream_t stream, const MatMulArgs& a, int numCUs)
{
    // Pieces take half as much again of LDS and have to be made: with many terms a block of the matrix holds half the rows that it
    // does whole, and with few rows nothing else shares the work.  Pieces against whole, over 2^11 / 2^15 (32 and 16 rows: 2^14) / 2^17 samples:
    // 64 x 384 17.9, 21.1, 54.5 against 19.1, 33.3, 89.9 us; 64 x 400 26.5, 40.6, 128 against 23.1, 39.9, 111; 64 x 480 35.7, 47.8, 154
    // against 25.0, 41.7, 123; 64 x 640 39.1, 50.6, 190 against 31.7, 52.8, 168; 32 x 320 11.6, 12.0, 38.6 against 12.3, 12.6, 55.6; 32 x 384
    // 13.2, 13.8, 42.0 against 11.5, 12.1, 41.6; 16 x 192 7.7, 8.0, 23.1 against 7.2, 7.5, 38.5; 16 x 256 9.1, 9.6, 27.7 against 6.7, 7.1, 27.4.
    // (By the matrix alone: what a sample's result is does not depend on how many come with it.)
    const int most = a.m <= 16 ? 192 : a.m <= 32 ? 320 : 384;
    return a.k <= most ? dispatchShape<VecAsMatrix<F32Mma>, float>(stream, a, numCUs) : dispatchShape<VecAsMatrix<F32WholeMma>, float>(stream, a, numCUs);
}

hipError_t launchMatMulF32Whole(hipStream_t stream, const MatMulArgs& a, int numCUs)
{
    return dispatchShape<VecAsMatrix<F32WholeMma>, float>(stream, a, numCUs);
}

} // namespace cv
