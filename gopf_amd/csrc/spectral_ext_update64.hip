// spectral_ext_update64.hip -- FP64 update pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_pencil_update_set<double, 1>(const PencilUpdateArgs<double>&, int, hipStream_t);

}  // namespace gpf
