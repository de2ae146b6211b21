// The fused GLM step in mode SGMC_MODE_SGGMC, every D class.
#include "glm_fused.h"

namespace sgmc {
template void launch_fused<SGMC_MODE_SGGMC>(int, int, hipStream_t, const FusedArgs&);
}  // namespace sgmc
