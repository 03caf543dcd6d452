// rh_stage.cpp -- see rh_stage.h.  The slots are shared by the contexts of a
// process, one set per device: STAGE_SLOTS pieces of pinned memory and a thread
// for all but one of them, allocated by the first copy that needs them and
// given back with the last context that used them.  Copies of different
// contexts on one device take turns; those on different devices, and the
// worker threads of adaptive runs, do not wait for one another.
#include "rh_stage.h"

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>

#include "rh_context.h"
#include "rh_pool.h"

namespace rhi {

namespace {

// Four lanes reach what eight do (96 MB 2.46 ms each way with either), in half
// the pinned memory and threads that a context alone on its device allocates
// and gives back; pieces of 1 MB take 3.1 ms.
constexpr int STAGE_SLOTS = 4;
constexpr size_t STAGE_PIECE = (size_t)2 << 20;
constexpr size_t STAGE_LANES = (size_t)10 << 20;
constexpr size_t STAGE_FEW_RUNS = 4;
constexpr int STAGE_MAX_DEVICES = 64;

struct Slot {
    char* mem = nullptr;
    hipEvent_t done = nullptr;  // recorded after the slot's last copy
};

struct Stage {
    std::mutex mu;  // one copy at a time
    char* mem = nullptr;
    Slot slots[STAGE_SLOTS];
    std::unique_ptr<HostPool> lanes;  // joined before the slots go
    int users = 0;
};

std::mutex g_users_mu;  // guards users of every stage
Stage g_stages[STAGE_MAX_DEVICES];

// The stage of the context's device, with the context counted as its user.
Stage* stage_of(rh_ctx* c) {
    if (c->p.device < 0 || c->p.device >= STAGE_MAX_DEVICES) return nullptr;
    Stage* s = &g_stages[c->p.device];
    if (!c->stage_user) {
        std::lock_guard<std::mutex> lk(g_users_mu);
        ++s->users;
        c->stage_user = true;
    }
    return s;
}

// Whether a host pointer is memory that the runtime knows (pinned or managed):
// a copy moves such memory at the bus's rate by itself (767 MB 13.4 ms each way,
// through slots 18.8).
bool known_memory(const void* p) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

// Every slot, in one allocation: freeing them one by one takes longer (eight,
// 2 ms).
bool ensure_slots(Stage& s) {
    if (!s.mem && hipHostMalloc((void**)&s.mem, STAGE_SLOTS * STAGE_PIECE, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        s.mem = nullptr;
        return false;
    }
    for (int i = 0; i < STAGE_SLOTS; ++i) {
        Slot& sl = s.slots[i];
        sl.mem = s.mem + i * STAGE_PIECE;
        if (!sl.done && hipEventCreateWithFlags(&sl.done, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            sl.done = nullptr;
            return false;
        }
    }
    return true;
}

// Copies bytes [off, off + n) of the host runs to or from a slot.
void host_bytes(const std::vector<HostRun>& host, const std::vector<size_t>& start, size_t off, size_t n, char* mem,
                bool to_host) {
    size_t r = std::upper_bound(start.begin(), start.end(), off) - start.begin() - 1;
    while (n > 0) {
        const size_t in = off - start[r], k = std::min(n, host[r].bytes - in);
        char* h = (char*)host[r].ptr + in;
        if (to_host) std::memcpy(h, mem, k);
        else std::memcpy(mem, h, k);
        mem += k;
        off += k;
        n -= k;
        ++r;
    }
}

int plain(rh_ctx* c, const std::vector<HostRun>& host, char* dev, bool to_host) {
    for (const HostRun& h : host) {
        if (h.bytes) {
            if (to_host) RH_HIP(c, hipMemcpyAsync(h.ptr, dev, h.bytes, hipMemcpyDeviceToHost, c->stream));
            else RH_HIP(c, hipMemcpyAsync(dev, h.ptr, h.bytes, hipMemcpyHostToDevice, c->stream));
        }
        dev += h.bytes;
    }
    return RH_OK;
}

int staged(rh_ctx* c, const std::vector<HostRun>& host, char* dev, bool to_host) {
    std::vector<size_t> start;
    size_t total = 0;
    for (const HostRun& h : host) {
        start.push_back(total);
        total += h.bytes;
    }
    if (total == 0) return RH_OK;
    // A first use allocates the slots (some ms) and waking the lanes costs about
    // 150 us, so one run of middle size is left to the runtime (1.5 MB: 70 us
    // each way against 190).  Many runs always go through slots: the runtime
    // takes 10-20 us for each.
    if (host.size() <= STAGE_FEW_RUNS) {
        if (total < STAGE_LANES) return plain(c, host, dev, to_host);
        for (const HostRun& h : host)
            if (h.bytes && known_memory(h.ptr)) return plain(c, host, dev, to_host);
    }
    Stage* s = stage_of(c);
    if (!s) return plain(c, host, dev, to_host);
    const size_t npiece = (total + STAGE_PIECE - 1) / STAGE_PIECE;
    const int most = std::min(STAGE_SLOTS, host_threads());
    const int lanes = (int)std::min<size_t>(npiece, most);
    std::lock_guard<std::mutex> lk(s->mu);
    if (!ensure_slots(*s)) return plain(c, host, dev, to_host);
    if (lanes > 1 && !s->lanes) s->lanes.reset(new HostPool(most - 1));
    hipError_t err[STAGE_SLOTS] = {};
    auto lane = [&](int i) {
        Slot& sl = s->slots[i];
        hipError_t e = hipSetDevice(c->p.device);
        for (size_t k = i; k < npiece && e == hipSuccess; k += lanes) {
            const size_t off = k * STAGE_PIECE, n = std::min(STAGE_PIECE, total - off);
            // The slot's previous copy, which may be another context's.
            e = hipEventSynchronize(sl.done);
            if (e != hipSuccess) break;
            if (to_host) {
                e = hipMemcpyAsync(sl.mem, dev + off, n, hipMemcpyDeviceToHost, c->stream);
                if (e == hipSuccess) e = hipEventRecord(sl.done, c->stream);
                if (e == hipSuccess) e = hipEventSynchronize(sl.done);
                if (e == hipSuccess) host_bytes(host, start, off, n, sl.mem, true);
            } else {
                host_bytes(host, start, off, n, sl.mem, false);
                e = hipMemcpyAsync(dev + off, sl.mem, n, hipMemcpyHostToDevice, c->stream);
                if (e == hipSuccess) e = hipEventRecord(sl.done, c->stream);
            }
        }
        err[i] = e;
    };
    if (lanes == 1) lane(0);
    else s->lanes->run(lanes, lane);
    for (int i = 0; i < lanes; ++i)
        if (err[i] != hipSuccess) return hip_fail(c, err[i], "staged copy");
    return RH_OK;
}

}  // namespace

int stage_to_host(rh_ctx* c, const std::vector<HostRun>& host, const void* dev) {
    return staged(c, host, const_cast<char*>((const char*)dev), true);
}
int stage_to_device(rh_ctx* c, const std::vector<HostRun>& host, void* dev) { return staged(c, host, (char*)dev, false); }

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
    if (c->stage_user) {
        std::lock_guard<std::mutex> lk(g_users_mu);
        Stage& s = g_stages[c->p.device];
        if (--s.users == 0) {
            s.lanes.reset();
            for (Slot& sl : s.slots) {
                if (sl.done) (void)hipEventDestroy(sl.done);
                sl = Slot{};
            }
            if (s.mem) (void)hipHostFree(s.mem);
            s.mem = nullptr;
        }
        c->stage_user = false;
    }
}

}  // namespace rhi
