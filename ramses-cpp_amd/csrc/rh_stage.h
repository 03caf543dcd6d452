// rh_stage.h -- copies between the caller's (pageable) arrays and the device
// through pinned staging slots.
//
// A plain copy of pageable memory runs at 17-18 GB/s to the host here and 27-30
// to the device, staged by one thread of the runtime.  Long copies instead move
// pieces of STAGE_PIECE bytes through pinned slots, several host threads each
// owning one: a thread queues its piece on the context's stream, waits for it
// and copies it out while the others' pieces are on the bus (to the host 767 MB
// 43 -> 19 ms, 96 MB 5.5 -> 2.5 ms, 32 MB 1.9 -> 0.9 ms, 12 MB 0.72 -> 0.40 ms;
// to the device 25 -> 19, 3.3 -> 2.5, 1.07 -> 0.92 and 0.45 -> 0.43 ms).  A
// context that binds 12 MB, takes a Courant step, reads the state back and goes
// takes 1.61 ms, slots and threads included, 1.81 with plain copies; one that
// makes no launch at all pays up to 3 ms for its slots.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

struct rh_ctx;

namespace rhi {

// A run of host memory; the runs of a copy, in order, correspond to one
// contiguous device range.
struct HostRun {
    void* ptr;
    size_t bytes;
};

// Copies between host runs and device memory on the context's stream.  They
// are complete, and the host memory free for other use, once the caller has
// synchronised the stream; later work on the stream sees an upload.
int stage_to_host(rh_ctx* c, const std::vector<HostRun>& host, const void* dev);
int stage_to_device(rh_ctx* c, const std::vector<HostRun>& host, void* dev);

// Pinned memory of a context for small results (PIN_BYTES), null when none
// can be had.
constexpr size_t PIN_BYTES = 65536;
void* pinned_small(rh_ctx* c);

// Gives back what the context holds of the shared slots and threads; its
// stream is idle.
void stage_release(rh_ctx* c);

}  // namespace rhi
