// spectral_ext_rows.hip -- FP32 fused row pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_fused_set<float, 1>(const RowFusedArgs<float>&, hipStream_t);

}  // namespace gpf
