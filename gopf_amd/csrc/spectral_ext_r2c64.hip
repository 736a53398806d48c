// spectral_ext_r2c64.hip -- FP64 forward and inverse row passes of the general path of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_r2c_set<double, 1>(const RowR2CArgs<double>&, hipStream_t);
template hipError_t launch_rows_c2r_set<double, 1>(const RowC2RArgs<double>&, hipStream_t);

}  // namespace gpf
