// oxr_copy.h -- copies between pageable host memory and the device through pinned staging.
//
// A copy runs in slots of a pinned ring: while one slot crosses PCIe the host side of
// another is copied by a few threads. One thread moves 10-20 GB/s into fresh pageable memory
// (page faults included) where the link moves 50, and chunk after chunk in turn adds the two
// times up: 108 MB of hits took 5.9 ms, now 2.9. Up to 1 MB a copy is one piece with no
// helper and no event, the stream is waited for instead; up to 2 MB it is two, without the
// helpers, whose waking costs more than they bring (512 KB: 121 us with them, 76 without).
#pragma once
#include <hip/hip_runtime.h>
#include "oxr_pool.h"

namespace oxh {

// The pinned ring of one engine; all its copies run on the engine's stream.
struct Stager {
    static constexpr int SLOTS = 4;
    static constexpr size_t SLOT = size_t(2) << 20, SHORT = SLOT / 2;
    char* ring = nullptr;
    size_t slot_bytes = 0;             // allocated per slot: grows from small copies to SLOT
    hipEvent_t done[SLOTS] = {};
    bool pending[SLOTS] = {};          // the slot's last upload may still be under way
    hipStream_t on[SLOTS] = {};        // where it is when it left no event
    bool marked[SLOTS] = {};           // it left one
    CopyPool pool;
    hipError_t ready(size_t bytes);    // ring and events for a copy of this size
    static size_t piece(size_t bytes); // how much of it goes through one slot
    hipError_t wait(int slot);         // the slot's last copy has finished
    void idle() { for (bool& p : pending) p = false; }   // the stream has been waited for
    hipError_t d2h(hipStream_t s, void* dst, const void* src, size_t bytes);
    hipError_t h2d(hipStream_t s, void* dst, const void* src, size_t bytes);
    void release();
};

} // namespace oxh
