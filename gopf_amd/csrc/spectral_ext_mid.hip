// spectral_ext_mid.hip -- FP32 instantiations of the middle pass k_mid (the extended lengths).
#include "spectral_mid_kernels.h"

namespace gpf {

template hipError_t launch_mid_set<float, 1>(const MidArgs<float>&, int, hipStream_t);

}  // namespace gpf
