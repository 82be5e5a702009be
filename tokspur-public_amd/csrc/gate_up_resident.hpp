// Launch interface of the two grouped gate/up kernels: activations resident in registers (gate_up_resident.hip, 2048 channels), weights
// and activations both streaming through LDS (gate_up_stream.hip, any multiple of 256).
#pragma once
#include "grouping_device.hpp"

namespace tsp {

struct ResidentGateUpArgs {
    const _Float16* xh;       // [tokens][channels] activations as halves, columns 1 <-> 2 and 5 <-> 6 of every eight swapped
    const _Float16* sx;       // [tokens][channels / 256][16] sub-block sums of those rows: eight high halves, eight residuals
    const uint8_t* pair_lo;   // co-located [gate_e, up_e] Pack v3 Q4_K experts 0 .. experts/2-1
    const uint8_t* pair_hi;   // the same for experts/2 .. experts-1
    const uint8_t* shared_gate;  // an always-on expert whose tasks carry expert id == experts (null: none)
    const uint8_t* shared_up;
    tsp_planar_spec spec;     // one expert: `channels` columns, `hidden` rows
    uint32_t experts, tokens, selected, channels, hidden;
    const uint32_t* tasks;    // [2 + 2 * task_slots]: live tasks, routes, then (expert, first row) per 64-row task
    const uint32_t* classes;  // [2 + 2 * task_slots]: tasks of <= 32 rows, tasks of 33..64 rows, then the two kinds' task indices
    const uint32_t* counts;
    const uint32_t* token_map;
    const uint32_t* ids;
    uint32_t task_slots;
    const OrderedTask* order;  // the streaming kernel's: the same tasks as it takes them (task_order_block)
    _Float16* hbuf;           // [task_slots * 64][hidden]: SwiGLU output rows by task slot, as halves of h / 256
    uint32_t* error_word;
};

bool resident_gate_up_takes(uint32_t channels, uint32_t hidden);
int launch_resident_gate_up(const ResidentGateUpArgs& args, hipStream_t stream);
uint32_t stream_gate_up_tail(uint32_t hidden);  // task_order_block's tail for it
int launch_stream_gate_up(const ResidentGateUpArgs& args, hipStream_t stream);  // hidden units in 32s

}  // namespace tsp
