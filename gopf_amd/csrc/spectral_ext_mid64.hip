// spectral_ext_mid64.hip -- FP64 instantiations of the middle pass k_mid (the extended lengths).
#include "spectral_mid_kernels.h"

namespace gpf {

template hipError_t launch_mid_set<double, 1>(const MidArgs<double>&, int, hipStream_t);

}  // namespace gpf
