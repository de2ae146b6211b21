// The loop launch of the GLM step in mode SGMC_MODE_OBABO, every D class.
#include "glm_fused.h"

namespace sgmc {
template void launch_loop<SGMC_MODE_OBABO>(int, int, int, hipStream_t, const FusedArgs&);
}  // namespace sgmc
