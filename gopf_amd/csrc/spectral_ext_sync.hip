// spectral_ext_sync.hip -- FP32 between-stage row pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_sync_set<float, 1>(const RowSyncArgs<float>&, hipStream_t);

}  // namespace gpf
