// rh_stage.cpp -- pinned host memory for results on their way to the caller.
#include "rh_stage.h"

#include "rh_context.h"

namespace rhi {

void* pinned_small(rh_ctx* c) {
    if (!c->h_pin && hipHostMalloc(&c->h_pin, PIN_BYTES, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        c->h_pin = nullptr;
    }
    return c->h_pin;
}

void stage_release(rh_ctx* c) {
    if (c->h_pin) (void)hipHostFree(c->h_pin);
    c->h_pin = nullptr;
}

}  // namespace rhi
