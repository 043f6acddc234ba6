// Helpers shared by the library's translation units (not part of the C ABI).
#pragma once

#include <stddef.h>

#include <atomic>

namespace z1detail {

// Gives each workspace one of N slots for good, on its first use.  What a launch keeps in its workspace's slot is then as
// safe as the workspace itself: launches that could meet in a slot write the same workspace, which the caller orders,
// whether they are enqueued, captured or replayed, and on whichever streams.  Any thread may call.
template <int N>
class WorkspaceSlots {
    std::atomic<const void*> owner_[N] = {};

public:
    // The slot of `workspace` (not NULL); -1 when N other workspaces have them all.
    int slot(const void* workspace) {
        for (int i = 0; i < N; ++i) {
            const void* w = owner_[i].load(std::memory_order_relaxed);
            if (!w && owner_[i].compare_exchange_strong(w, workspace, std::memory_order_relaxed)) return i;
            if (w == workspace) return i;             // w: the owner, also when another thread has just become it
        }
        return -1;
    }
};

// Dynamic LDS (bytes) that caps a launch at `per_cu` resident workgroups per CU on device `dev`; 0 when the
// device does not report its LDS size.  Returns Z1_OK or a hipError_t.
int occupancy_lds(int dev, int per_cu, size_t* bytes);

}  // namespace z1detail
