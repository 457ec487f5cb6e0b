// hostio.hpp -- pinned staging of the host-array entry points (abi.cpp).
#pragma once
#include <memory>

#include "common.hpp"

namespace tbfg {

// A few pinned slots that fields pass through in chunks of whole planes, so that the
// host's gather of one chunk overlaps the copy of the one before (and likewise the
// scatter on the way back).  Copies run on the null stream.
struct HostRing {
    static constexpr int kSlots = 3;                       // or as many as the field has chunks
    static constexpr size_t kSlotBytes = (size_t)4 << 20;  // or one plane, if that is larger; the field, if smaller
    // Small fields (one chunk) go through ordinary memory, whose copies the runtime stages:
    // up to kPageable always, up to kPageableFirst in the first call since there are handles.
    // Pinning takes 25 us (0.1 to 0.4 ms the first time in a process) and giving back 40 to 80.
    // Create, one call, destroy at 32^3: 190 us this way, 300 pinned, of which the call 83 and 77;
    // 48^3: the call 165 (the first) and 100, two calls pay for the ring.
    static constexpr size_t kPageable = (size_t)512 << 10, kPageableFirst = (size_t)1 << 20;
    int dev = 0;
    double* pin = nullptr;
    std::vector<double> page;  // in its place: one slot of ordinary memory, blocking copies
    size_t capacity = 0;       // doubles
    size_t slot = 0;           // doubles per slot, as the present call divides it
    hipEvent_t ev[kSlots] = {};
    bool busy[kSlots] = {};  // a copy from or to the slot is on the stream, ev after it

    HostRing() = default;
    HostRing(const HostRing&) = delete;
    HostRing& operator=(const HostRing&) = delete;
    ~HostRing();
    double* at(int sl) { return pin ? pin + (size_t)sl * slot : page.data(); }
    int wait(int sl)
    {
        if (busy[sl]) TBFG_HIP(hipEventSynchronize(ev[sl]));
        busy[sl] = false;
        return TBFG_OK;
    }
    int record(int sl)
    {
        TBFG_HIP(hipEventRecord(ev[sl], nullptr));
        busy[sl] = true;
        return TBFG_OK;
    }
};

// The rings of the process: a call takes one for its duration and gives it back, so a
// new handle's first call does not pin memory again.  A ring is no larger than the field
// needs.  Each thread in a call holds its own; at most kHostRingsKept idle ones are kept, the
// largest, and none once the last solver handle is gone (HostRingUser).
constexpr int kHostRingsKept = 4;
int host_ring_take(const int32_t* n, std::unique_ptr<HostRing>& out);
void host_ring_give(std::unique_ptr<HostRing> r);

// a member of every solver handle
struct HostRingUser {
    HostRingUser();
    ~HostRingUser();
    HostRingUser(const HostRingUser&) = delete;
    HostRingUser& operator=(const HostRingUser&) = delete;
};

}  // namespace tbfg
