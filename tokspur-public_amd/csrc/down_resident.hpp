// Launch interface of the grouped down kernels that keep a task's h rows: in registers (down_resident.hip) or in LDS (down_wide.hip).
#pragma once
#include "tsp_common.hpp"

namespace tsp {

struct ResidentDownArgs {
    const _Float16* hbuf;        // [task_slots * 64][hidden units]: SwiGLU output rows by task slot, as halves of h / 256
    const uint8_t* down;         // Q6_K planes (ql / qh / sub-scales / d), Q8_0 planes (quants / d) or Q5_1 planes (nibbles / fifth bits / d, m) per expert, `channels` rows of hidden units
    const uint8_t* shared_down;  // an always-on expert whose tasks carry expert id == experts (null: none)
    tsp_planar_spec spec;        // one expert
    uint32_t experts, tokens, selected, channels;
    const uint32_t* tasks;       // [2 + 2 * task_slots]: live tasks, routes, then (expert, first row) per 64-row task
    const uint32_t* classes;     // [2 + 2 * task_slots]: tasks of <= 32 rows, tasks of 33..64 rows, then the two kinds' task indices
    const uint32_t* counts;
    const uint32_t* token_map;
    const uint32_t* ids;
    uint32_t task_slots;
    float* y;                    // [tokens * selected] rows by route, y_stride bytes apart; the whole output spans less than 0xffffff00 bytes, and so does shared_y
    uint64_t y_stride;
    uint32_t out_bytes;          // y from its first row's first byte to its last row's last
    float* shared_y;             // the always-on expert's rows by token
    uint64_t shared_y_stride;
    float out_scale;             // 256: undoes the 2^-8 that h carries (a power of two)
    uint32_t* error_word;
};

bool resident_down_takes(uint32_t source_type, uint32_t channels, uint32_t hidden);  // source_type: 14 (Q6_K planes), 8 (Q8_0 planes) or 7 (Q5_1 planes)
int launch_resident_down(const ResidentDownArgs& args, hipStream_t stream);

// down_wide.hip: Q8_0 and Q5_1 planes, `hidden` columns, no always-on expert; the output spans at most 0xffff0000 bytes
bool wide_down_takes(uint32_t source_type, uint32_t channels, uint32_t hidden);
int launch_wide_down(const ResidentDownArgs& args, uint32_t hidden, hipStream_t stream);

}  // namespace tsp
