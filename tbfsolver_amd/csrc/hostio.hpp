// hostio.hpp -- pinned staging of the host-array entry points (abi.cpp).
#pragma once
#include <memory>

#include "common.hpp"

namespace tbfg {

// A few pinned slots that fields pass through in chunks of whole planes, so that the
// host's gather of one chunk overlaps the copy of the one before (and likewise the
// scatter on the way back).  Copies run on the null stream.
struct HostRing {
    static constexpr int kSlots = 3;
    static constexpr size_t kSlotBytes = (size_t)4 << 20;  // or one plane, if that is larger
    int dev = 0;
    double* pin = nullptr;
    size_t slot = 0;  // doubles per slot
    hipEvent_t ev[kSlots] = {};
    bool busy[kSlots] = {};  // a copy from or to the slot is on the stream, ev after it

    HostRing() = default;
    HostRing(const HostRing&) = delete;
    HostRing& operator=(const HostRing&) = delete;
    ~HostRing();
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
// new handle's first call does not pin memory again (milliseconds, more than the call
// itself).  Each thread in a call holds its own; at most kHostRingsKept idle ones
// are kept, and none once the last solver handle is gone (HostRingUser).
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
