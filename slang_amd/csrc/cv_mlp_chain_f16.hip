// cv_mlp_chain_f16.hip -- mlpChainKernel for fp16 networks.
#include "cv_mlp_chain.h"

namespace cv {

hipError_t launchMlpChainF16(hipStream_t stream, const MlpArgs& a, int numCUs) { return launchChain<F16Mma>(stream, a, numCUs); }

} // namespace cv
