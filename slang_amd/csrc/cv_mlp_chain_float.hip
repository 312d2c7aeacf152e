// cv_mlp_chain_float.hip -- mlpChainKernel for networks of float and of bfloat16.
#include "cv_mlp_chain.h"
#include "cv_mlp_equal_f32.h"

namespace cv {

hipError_t launchMlpChainFloat(hipStream_t stream, MmaKind kind, const MlpArgs& a, int numCUs)
{
    if (kind == MmaKind::F32) {
        const hipError_t e = launchEqualF32(stream, a, numCUs);
        if (e != hipErrorInvalidValue) return e;
    }
    return kind == MmaKind::F32 ? launchChain<F32Mma>(stream, a, numCUs) : launchChain<Bf16Mma>(stream, a, numCUs);
}

} // namespace cv
