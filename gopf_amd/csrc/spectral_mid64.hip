// spectral_mid64.hip -- FP64 instantiations of the middle pass k_mid (the core lengths).
#include "spectral_mid_kernels.h"

namespace gpf {

template hipError_t launch_mid<double>(const MidArgs<double>&, int, hipStream_t);

}  // namespace gpf
