// va_int8.hpp — the int8 scan's launch arguments, shared by its kernels.
#pragma once

#include "va_internal.hpp"

namespace va {

struct I8Args {
    const int8_t* q = nullptr;
    const uint32_t* qrow = nullptr;
    int64_t ldq = 0;
    const int8_t* x = nullptr;
    int64_t ldx = 0;
    uint32_t Q = 0, N = 0, D = 0;
    uint32_t* out_k = nullptr;
    int64_t ldo = 0;
    const uint32_t* thr = nullptr;
    uint32_t* cnt = nullptr;
    uint32_t* cand_key = nullptr;
    uint32_t* cand_id = nullptr;
    uint32_t cap = 0;
};

// The scan for batches of at most 128 queries (va_int8_small.hip): whether it takes a launch (of any
// batch: past 128 queries each 128 read the rows again), and the launch.
constexpr uint32_t kI8SmallQueries = 128;
bool i8_small_ok(const I8Args& a);
va_status launch_i8_small(va_context* ctx, const I8Args& a, bool filter);

}  // namespace va
