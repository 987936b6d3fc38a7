// The kernels of env_device.hpp for any task (the common ones run those of env.hip).

#define MYA_GENERAL_TASKS 1
#include "env_device.hpp"

namespace mya
{
EnvKernels env_kernels_general() { return env_kernels(); }
}  // namespace mya
