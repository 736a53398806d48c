// spectral_ext_rows64.hip -- FP64 fused row pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_fused_set<double, 1>(const RowFusedArgs<double>&, hipStream_t);

}  // namespace gpf
