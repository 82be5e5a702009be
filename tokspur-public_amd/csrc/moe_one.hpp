// Internal interface of the one-token routed MoE products (moe_one.hip), used by the T <= 8 entry points.
#pragma once
#include "skinny.hpp"

namespace tsp {

bool one_gate_up_takes(const SkinnyMoe& m);
bool one_down_takes(const SkinnyMoe& m);
int launch_one_gate_up(const SkinnyMoe& m, hipStream_t stream);
int launch_one_down(const SkinnyMoe& m, hipStream_t stream);

}  // namespace tsp
