// Internal interface of the streaming products of the T <= 8 routed MoE (record_stream.hip): gate/up + SwiGLU on Q4_K planes
// and the down product on Q8_0, Q5_1 or Q6_K planes, for rows of any whole number of blocks up to 2560 columns.
#pragma once
#include "skinny.hpp"

namespace tsp {

bool record_stream_gate_up_takes(const SkinnyMoe& m);
int launch_record_stream_gate_up(const SkinnyMoe& m, hipStream_t stream);  // builds the union records itself when m.meta is there
bool record_stream_down_takes(const SkinnyMoe& m);
int launch_record_stream_down(const SkinnyMoe& m, hipStream_t stream);

}  // namespace tsp
