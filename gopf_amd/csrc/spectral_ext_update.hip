// spectral_ext_update.hip -- FP32 update pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_pencil_update_set<float, 1>(const PencilUpdateArgs<float>&, int, hipStream_t);

}  // namespace gpf
