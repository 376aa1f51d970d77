#include "thip_chain_turn.h"

#include <algorithm>
#include <new>

namespace thip {

ChainTurns &ChainTurns::of(int ordinal) {
    static ChainTurns turns[64];
    return turns[ordinal & 63];
}

hipError_t ChainTurns::join(ChainMember *m) {
    std::lock_guard<std::mutex> held(mutex);
    if (!event) {
        if (hipError_t err = hipEventCreateWithFlags(&event, hipEventDisableTiming)) return err;
    }
    try {
        members.push_back(m);
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
    return hipSuccess;
}

void ChainTurns::leave(ChainMember *m) {
    std::lock_guard<std::mutex> held(mutex);
    if (last == m) last = nullptr;
    members.erase(std::remove(members.begin(), members.end(), m), members.end());
}

static bool idle(const ChainMember *m) {
    if (hipStreamQuery(m->stream) == hipSuccess) return true;
    (void)hipGetLastError();  // not-ready is no error
    return false;
}

hipError_t ChainTurns::Turn::take(ChainTurns *turns, ChainMember *m, bool *chained) {
    *chained = false;
    lock = std::unique_lock<std::mutex>(turns->mutex);
    for (const ChainMember *x : turns->members) {
        if (x != m && x->abandoned && !idle(x)) return hipSuccess;
    }
    if (turns->last && turns->last != m) {
        hipError_t err = hipEventRecord(turns->event, turns->last->stream);
        if (err == hipSuccess) err = hipStreamWaitEvent(m->stream, turns->event, 0);
        if (err != hipSuccess) return err;
    }
    turns->last = m;
    *chained = true;
    return hipSuccess;
}

}  // namespace thip
