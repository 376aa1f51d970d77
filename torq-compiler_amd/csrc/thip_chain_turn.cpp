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

// Whether this dispatch is one of those behind a launch that gave up.
bool ChainMember::missesCus() {
    if (gaveUp && __atomic_exchange_n(gaveUp, 0u, __ATOMIC_RELAXED) != 0) {
        penalty = std::min(std::max(2 * penalty, ChainTurns::kGivenUpFirst), ChainTurns::kGivenUpMost);
        apart = penalty;
        since = 0;
    }
    if (apart == 0) {
        if (penalty > 0 && ++since > penalty) penalty = 0;
        return false;
    }
    apart--;
    return true;
}

hipError_t ChainTurns::Turn::take(ChainTurns *turns, ChainMember *m, bool wanted, bool *chained) {
    *chained = false;
    lock = std::unique_lock<std::mutex>(turns->mutex);
    member = m;
    m->enqueuing = m->busy = true;
    bool apart = !wanted;
    for (ChainMember *x : turns->members) {
        if (apart || x == m || !x->busy || (m->always && !x->abandoned)) continue;
        if (!x->enqueuing && hipStreamQuery(x->stream) == hipSuccess) {
            x->busy = false;
        } else {
            (void)hipGetLastError();  // not-ready is no error
            apart = true;
        }
    }
    if (!apart && !m->always) apart = m->missesCus();
    if (apart) {  // others may enqueue at the same time
        lock.unlock();
        return hipSuccess;
    }
    if (m->always && turns->last && turns->last != m) {  // otherwise nobody else is at work
        hipError_t err = hipEventRecord(turns->event, turns->last->stream);
        if (err == hipSuccess) err = hipStreamWaitEvent(m->stream, turns->event, 0);
        if (err != hipSuccess) return err;
    }
    turns->last = m;
    *chained = true;
    return hipSuccess;
}

ChainTurns::Turn::~Turn() {
    if (!member) return;
    if (!lock.owns_lock()) lock.lock();
    member->enqueuing = false;
}

}  // namespace thip
