// cv_train_round_f16.hip -- trainRoundKernel for networks of half.
#include "cv_train_round.h"
#include "cv_error.h"
#include "cv_launch.h"

namespace cv {

hipError_t launchTrainRoundF16(hipStream_t stream, const TrainLaunch& t, int numCUs) { return launchRoundTyped<half_t>(stream, t, numCUs); }

} // namespace cv
