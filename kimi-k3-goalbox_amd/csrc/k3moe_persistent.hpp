// The persistent kernels' instantiations (k3moe_persistent.hip).
#pragma once

#include "k3moe_decode.hpp"
#include "k3moe_plan.hpp"

namespace k3moe {

typedef void (*PersistentKernel)(Plan, DecodeArgs);
constexpr int kPersistentKernels = 20;

// The instantiation of a persistent plan, and its number.
PersistentKernel persistent_kernel(const Plan &p, int &slot);

}  // namespace k3moe
