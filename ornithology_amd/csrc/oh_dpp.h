// oh_dpp.h - ordered sums whose common factor sits in one lane of a 16-lane row.
#pragma once
#include "oh_common.h"
#include <utility>

template <class F, int... I>
OH_DEV void static_for_(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
// f(integral_constant<0>) ... f(integral_constant<N - 1>)
template <int N, class F>
OH_DEV void static_for(F &&f) { static_for_(f, std::make_integer_sequence<int, N>{}); }
// lane L of each 16-lane row, in every lane of the row (folds into the
// consuming instruction's DPP operand, so it costs nothing)
template <int L>
OH_DEV float row_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + L, 0xf, 0xf, true));
}
// base (uniform) + a 32-bit byte offset: one address register per load
template <typename T>
OH_DEV T ldo(const void *base, unsigned bytes) { return ldg((const T *)((const char *)base + bytes)); }
// an index that the compiler takes as new at this point: addresses are formed
// from it where they are used instead of being kept, one register pair each,
// across a loop
OH_DEV int again(int i) { asm volatile("" : "+v"(i)); return i; }
// nothing is scheduled across this point. A DPP instruction waits two issue
// slots for any register that a vector instruction has just written, also for
// one that it only overwrites, so products and sums are kept in groups: left
// to itself the compiler pairs each product with its sum and a wait.
OH_DEV void order() { __builtin_amdgcn_sched_barrier(0); }
// lane l + I of the 16-lane row, in lane l; opaque, so that a chain of adds over
// several of them is plain adds: folded into its add's DPP operand each would
// wait two slots for the running sum that the add before it wrote
template <int I>
OH_DEV float row_ahead(float v) {
    float u = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x100 + I, 0xf, 0xf, true));
    asm volatile("" : "+v"(u));
    return u;
}
