// cv_train_wave.hip -- instantiations and launcher of trainWaveKernel.
#include "cv_train_wave.h"
#include "cv_error.h"
#include "cv_launch.h"

namespace cv {

// hipErrorInvalidValue where no instantiation takes the network (hidden layers beyond 64 units, more than 64 inputs, more
// gradients than a wave can hold)
hipError_t launchTrainWave(hipStream_t stream, const TrainLaunch& t, int numCUs)
{
    RoundArgs a = {};
    int maxTiles = 0;
    if (!fillRoundArgs<float>(t, a, maxTiles)) return hipErrorInvalidValue;
    const int L = t.mlp.numLayers;
    auto round = [](int v) { return v <= 2 ? v : v <= 4 ? 4 : v; };
    int hidden = 1;
    for (int l = 0; l + 1 < L; ++l) hidden = a.layers[l].rowTiles > hidden ? a.layers[l].rowTiles : hidden;
    switch ((round(hidden) * 8 + L) * 8 + round(a.layers[0].colTiles)) {
#define CV_N(HT, NL, IT) \
    case (HT * 8 + NL) * 8 + IT: \
        if constexpr (WaveNet<HT, NL, IT>::fits) return launchWave<WaveNet<HT, NL, IT>>(stream, t, a, numCUs); \
        break;
#define CV_I(HT, NL) CV_N(HT, NL, 1) CV_N(HT, NL, 2) CV_N(HT, NL, 4)
#define CV_L(HT) CV_I(HT, 2) CV_I(HT, 3) CV_I(HT, 4) CV_I(HT, 5)
    CV_L(1) CV_L(2) CV_L(4)
#undef CV_L
#undef CV_I
#undef CV_N
    }
    return hipErrorInvalidValue;
}

} // namespace cv
