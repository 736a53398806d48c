// spectral_adjoint.hip -- FP32 instantiations of the adjoint's reverse pass k_adj_mid (every compiled
// length and the direct DFT).
#include "spectral_adjoint_kernels.h"

namespace gpf {

template long adj_mid_blocks<float>(const AdjMidArgs<float>&);
template hipError_t launch_adj_mid<float>(const AdjMidArgs<float>&, int, hipStream_t);

}  // namespace gpf
