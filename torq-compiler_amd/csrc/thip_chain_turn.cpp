#include "thip_chain_turn.h"

#include <algorithm>
#include <chrono>
#include <new>

namespace thip {

static int64_t nanoseconds() { return std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

void ChainMember::waiting() { busyUntil.store(INT64_MAX, std::memory_order_relaxed); }
void ChainMember::finished() { busyUntil.store(0, std::memory_order_relaxed); }

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

hipError_t ChainTurns::Turn::take(ChainTurns *turns, ChainMember *m, bool wanted, bool *chained) {
    *chained = false;
    lock = std::unique_lock<std::mutex>(turns->mutex);
    member = m;
    const int64_t now = nanoseconds();
    m->busyUntil.store(now + kAtWork, std::memory_order_relaxed);
    bool apart = !wanted;
    for (const ChainMember *x : turns->members) {
        apart = apart || (x != m && (x->abandoned || (!m->always && x->busyUntil.load(std::memory_order_relaxed) > now)));
    }
    if (!apart && !m->always) apart = m->missesCus();
    if (apart) {  // others may enqueue at the same time
        lock.unlock();
        return hipSuccess;
    }
    if (turns->last && turns->last != m && turns->last->busyUntil.load(std::memory_order_relaxed) != 0) {
        hipError_t err = hipEventRecord(turns->event, turns->last->stream);
        if (err == hipSuccess) err = hipStreamWaitEvent(m->stream, turns->event, 0);
        if (err != hipSuccess) return err;
    }
    turns->last = m;
    *chained = true;
    return hipSuccess;
}

ChainTurns::Turn::~Turn() {
    if (member) member->busyUntil.store(nanoseconds() + kAtWork, std::memory_order_relaxed);
}

}  // namespace thip
