// spectral_ext_r2c.hip -- FP32 forward and inverse row passes of the general path of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_r2c_set<float, 1>(const RowR2CArgs<float>&, hipStream_t);
template hipError_t launch_rows_c2r_set<float, 1>(const RowC2RArgs<float>&, hipStream_t);

}  // namespace gpf
