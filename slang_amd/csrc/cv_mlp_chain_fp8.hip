// cv_mlp_chain_fp8.hip -- mlpChainKernel for e4m3 networks, on the fp16 matrix pipeline or on the fp8 one.
#include "cv_mlp_chain.h"

namespace cv {

hipError_t launchMlpChainFp8(hipStream_t stream, MmaKind kind, const MlpArgs& a, int numCUs)
{
    return kind == MmaKind::Fp8Native ? launchChain<Fp8NativeMma>(stream, a, numCUs) : launchChain<Fp8AsF16Mma>(stream, a, numCUs);
}

} // namespace cv
