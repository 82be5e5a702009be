// Internal interface of the kernels for up to eight tokens (moe_few.hip), used by the T <= 8 routed MoE entry points.
#pragma once
#include "tsp_common.hpp"

namespace tsp {

struct FewMoe {
    const uint8_t* pair_lo;  // experts 0..E/2-1 as [gate_e, up_e]
    const uint8_t* pair_hi;  // experts E/2..E-1
    const uint8_t* down;     // [experts] planar
    const uint32_t* ids;     // [tokens * selected]
    uint32_t* meta;          // the caller's union block (the gate/up launch writes it), or nullptr for one token
    const float* x;          // token rows
    float* h;                // route rows
    float* y;                // route rows
    uint64_t x_stride, h_stride, y_stride;  // bytes
    uint32_t channels, hidden, experts, selected, tokens;
    tsp_planar_spec gu, dn;
    uint32_t* error_word;
    // optional always-on expert riding in the same launches (one Pack v3 expert each; rows = the tokens)
    const uint8_t* shared_gate = nullptr;
    const uint8_t* shared_up = nullptr;
    const uint8_t* shared_down = nullptr;
    float* shared_h = nullptr;  // [tokens, hidden]
    float* shared_y = nullptr;  // [tokens, channels]
    uint64_t shared_h_stride = 0, shared_y_stride = 0;
};

bool few_gate_up_takes(const FewMoe& m);
bool few_down_takes(const FewMoe& m);
int launch_few_gate_up(const FewMoe& m, hipStream_t stream);
int launch_few_down(const FewMoe& m, hipStream_t stream);

}  // namespace tsp
