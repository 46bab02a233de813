// hip_part.hip — the template kernels of one part of hip_instances.inl (SP_PART), compiled apart from the launching code so
// that the parts build side by side.
#include "hip_kernels.h"

#define SP_KERNEL(...) template __global__ void __VA_ARGS__;
namespace sphip_kernels {
#include "hip_instances.inl"
}  // namespace sphip_kernels
