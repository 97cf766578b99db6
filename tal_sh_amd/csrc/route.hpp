// How a contraction runs.  No HIP: decided and tested on the CPU.
#pragma once

#include "direct_args.hpp"
#include "plan.hpp"

namespace tal {

// A plain product by the direct kernels straight from the tensors, or on copies
// of the operands the planner transposes (with D written in place or through
// D'), or a product by the fast-math GEMMs on such copies.
enum Route { kRouteDirect, kRouteCopies, kRouteSplit };

// Of a plan without fast math; c: the direct kernels' choice for its product.
Route contract_route(const ContractPlan &plan, int dk, const DirectChoice &c);

}  // namespace tal
