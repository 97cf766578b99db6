// How a contraction runs.  No HIP: decided and tested on the CPU.
#pragma once

#include "direct_args.hpp"
#include "plan.hpp"

namespace tal {

// A plain product by the direct kernels straight from the tensors, or on copies
// of the operands the planner transposes (with D written in place or through
// D'), or a product by the fast-math GEMMs on such copies.
enum Route { kRouteDirect, kRouteCopies, kRouteSplit };

// direct_choose on the GPU at hand.
using DirectChooser = DirectChoice (*)(int dk, int64_t M, int64_t N, int64_t K, int64_t batch);

// Of a plan without fast math.
Route contract_route(const ContractPlan &plan, int dk, DirectChooser choose);

}  // namespace tal
