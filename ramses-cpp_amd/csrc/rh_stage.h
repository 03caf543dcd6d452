// rh_stage.h -- pinned host memory for results on their way to the caller.
#pragma once
#include <cstddef>

struct rh_ctx;

namespace rhi {

// Pinned memory of a context for small results (PIN_BYTES), null when none
// can be had.
constexpr size_t PIN_BYTES = 65536;
void* pinned_small(rh_ctx* c);

// Gives it back; the context's stream is idle.
void stage_release(rh_ctx* c);

}  // namespace rhi
