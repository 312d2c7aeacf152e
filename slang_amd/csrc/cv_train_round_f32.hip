// cv_train_round_f32.hip -- trainRoundKernel for networks of float, and the choice between the kernels of cv_train_round.h.
#include "cv_train_round.h"
#include "cv_error.h"
#include "cv_launch.h"

namespace cv {

hipError_t launchTrainRoundF16(hipStream_t stream, const TrainLaunch& t, int numCUs);
hipError_t launchTrainWave(hipStream_t stream, const TrainLaunch& t, int numCUs);

size_t trainRoundWorkspaceBytes(const MlpArgs& shapes, int numCUs, int carrierCt)
{
    RoundArgs a = {};
    int maxTiles = 0;
    if (!planRound(shapes, carrierCt, a, maxTiles)) return 0;
    // a partial per workgroup: one per round of the batch, as long as they are all resident (trainWaveKernel: per two rounds and
    // per compute unit, never more)
    return (size_t)roundBlocks(shapes.batch, a.samples, roundWorkgroups(a, shapes.numLayers, roundTiles(maxTiles), numCUs)) * a.partialFloats * sizeof(float);
}

hipError_t launchTrainRound(hipStream_t stream, const TrainLaunch& t, int numCUs)
{
    if (t.mlp.batch == 0) return hipSuccess;
    if (t.carrierCt != kF32) return launchTrainRoundF16(stream, t, numCUs);
    const hipError_t e = launchTrainWave(stream, t, numCUs);
    return e != hipErrorInvalidValue ? e : launchRoundTyped<float>(stream, t, numCUs);
}

} // namespace cv
