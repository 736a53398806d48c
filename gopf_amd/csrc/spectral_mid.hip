// spectral_mid.hip -- FP32 instantiations of the middle pass k_mid (the core lengths).
#include "spectral_mid_kernels.h"

namespace gpf {

template hipError_t launch_mid<float>(const MidArgs<float>&, int, hipStream_t);

}  // namespace gpf
