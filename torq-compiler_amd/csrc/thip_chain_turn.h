// Launches of dec_chain on a device, of all the executables that have one.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <vector>

namespace thip {

// An executable's part.
struct ChainMember {
    hipStream_t stream = nullptr;
    std::atomic<bool> abandoned{false};  // a wait for its work timed out
};

// The workgroups of a launch wait for one another and need a CU each at the same time.  Two such launches at once could each hold
// CUs that the other waits for, so the executables of a device take turns: a dispatch on another stream than the last one's starts behind it.
// Behind an abandoned executable's unfinished work (or what waits for that) nobody is put: dispatches then run record by record, which waits for nothing.
class ChainTurns {
public:
    static ChainTurns &of(int ordinal);  // one per device and process

    // When an executable is made (its device is current): what turns need is there from then on.
    hipError_t join(ChainMember *m);
    // Its stream is idle.  (An abandoned one whose work is unfinished stays.)
    void leave(ChainMember *m);

    // Of one dispatch, from before its launches until they are enqueued.
    class Turn {
    public:
        // *chained: as one launch; otherwise record by record.
        hipError_t take(ChainTurns *turns, ChainMember *m, bool *chained);

    private:
        std::unique_lock<std::mutex> lock;
    };

private:
    std::mutex mutex;
    std::vector<ChainMember *> members;
    ChainMember *last = nullptr;  // whose launch was the last one
    hipEvent_t event = nullptr;   // behind it, recorded when another one's follows
};

}  // namespace thip
