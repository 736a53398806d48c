// spectral_adjoint64.hip -- FP64 instantiations of the adjoint's reverse pass k_adj_mid (every compiled
// length and the direct DFT).
#include "spectral_adjoint_kernels.h"

namespace gpf {

template long adj_mid_blocks<double>(const AdjMidArgs<double>&);
template hipError_t launch_adj_mid<double>(const AdjMidArgs<double>&, int, hipStream_t);

}  // namespace gpf
