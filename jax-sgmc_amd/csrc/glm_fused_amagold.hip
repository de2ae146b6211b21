// The fused GLM step in mode SGMC_MODE_AMAGOLD, every D class.
#include "glm_fused.h"

namespace sgmc {
template void launch_fused<SGMC_MODE_AMAGOLD>(int, int, hipStream_t, const FusedArgs&);
}  // namespace sgmc
