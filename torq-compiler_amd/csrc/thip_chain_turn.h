// Launches of dec_chain on a device, of all the executables that have one.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <vector>

namespace thip {

// An executable's part.
struct ChainMember {
    hipStream_t stream = nullptr;
    bool always = false;                 // as one launch also beside others (THIP_DEC_CHAIN=1)
    std::atomic<bool> abandoned{false};  // a wait for its work timed out
    uint32_t *gaveUp = nullptr;          // null, or in host memory: a launch whose workgroups gave up waiting for one another sets it

    // What a wait for the executable's stream tells: it has begun, everything enqueued is done.
    void waiting();
    void finished();

private:
    friend class ChainTurns;
    std::atomic<int64_t> busyUntil{0};   // a point of the steady clock, 0: all its work is known to be done
    bool missesCus();
    uint32_t apart = 0;                  // dispatches that still go record by record since one gave up
    uint32_t penalty = 0;                // how many of them the last one cost
    uint32_t since = 0;                  // launches since then
};

// A decoder's step is one launch (dec_chain) while no other executable that has such launches is at work on the device, and otherwise runs record by
// record.  One launch holds every CU for the whole step; as launches of their own the records of several decoders fill each other's gaps.
// us a step, dispatches of one row from a thread for each decoder, one launch in turn / record by record, one decoder, two, three and four:
//   26 layers, 1152, 6912, vocabulary 262144   620 / 865   623 / 516   625 / 393   625 / 506
//   4 layers of it, vocabulary 4096             99 / 128   101 / 71    108 / 56    109 / 47
//   4 layers, 512, 2048                         79 / 113    81 / 60     82 / 42     82 / 33
// (and by this rule 622, 510, 393 and 504; 99, 72, 56 and 48; 79, 59, 42 and 33).  Where one thread enqueues for all of them its launches bound the
// records; in turn / record by record / by this rule, two decoders and four: 622 / 527 / 562  621 / 525 / 554;  99 / 88 / 82  105 / 83 / 79;  79 / 85 / 74  78 / 81 / 77.
// The two ways differ in the order of fp32 sums.  Who wants the same bits in company as alone asks for one of them when the executable is made
// (THIP_DEC_CHAIN=0 or 1).
// At work is who has been dispatched and not waited for in the last kAtWork, and who is being waited for.  The runtime is not asked: a
// query of a stream fails while another thread or library of the program captures a graph, and so does its capture then.
//
// The workgroups of a launch wait for one another and need a CU each at the same time.  Two such launches at once could each hold
// CUs that the other waits for, so they take turns: a dispatch as one launch starts behind the last one, unless that is known to be done.
// While there is an abandoned executable nobody is put behind it (or behind what waits for it): record by record a dispatch waits for nothing.
//
// A launch that does not get all CUs (another process, a CU mask, somebody's long kernels) costs its patience of 200 ms and the whole step by one
// workgroup (26 layers 51 ms; four 7).  What kept the CUs is likely to be there still, so the next kGivenUpFirst dispatches run record by record: at 26 layers
// these lose the same 0.25 s by not being one launch.  Twice as many after each further launch that gives up, and as at first again when as many
// launches went well.
class ChainTurns {
public:
    static constexpr uint32_t kGivenUpFirst = 1024, kGivenUpMost = 65536;
    static constexpr int64_t kAtWork = 10000000;  // ns; a step is well below

    static ChainTurns &of(int ordinal);  // one per device and process

    // When an executable is made (its device is current): what turns need is there from then on.
    hipError_t join(ChainMember *m);
    // Its stream is idle.
    void leave(ChainMember *m);

    // Of one dispatch, from before its launches until they are enqueued.
    class Turn {
    public:
        ~Turn();
        // *chained: as one launch, if `wanted`; no other executable's turn is taken until this one ends.  Otherwise record by record.
        hipError_t take(ChainTurns *turns, ChainMember *m, bool wanted, bool *chained);

    private:
        ChainMember *member = nullptr;
        std::unique_lock<std::mutex> lock;
    };

private:
    std::mutex mutex;
    std::vector<ChainMember *> members;
    ChainMember *last = nullptr;  // whose launch was the last one
    hipEvent_t event = nullptr;   // behind it, recorded when another one's follows
};

}  // namespace thip
