// spectral_ext_sync64.hip -- FP64 between-stage row pass of the extended lengths.
#include "spectral_kernels.h"

namespace gpf {

template hipError_t launch_rows_sync_set<double, 1>(const RowSyncArgs<double>&, hipStream_t);

}  // namespace gpf
