// Loads from memory straight into LDS, for the products whose operands take that way.
#pragma once
#include "common.h"

// A number that picks a ring's slot at compile time.
template <int N> struct Index { static constexpr int value = N; };

// sixteen bytes a lane: lane l's land at `to` + 16 l, `to` the same in all lanes
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t from, char* to, int lane_at, int at) {
    typedef __attribute__((address_space(3))) char lds_char;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)(lds_char*)to, 16, lane_at, at, 0, 0);
}
