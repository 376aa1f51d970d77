#include "thip_chain_turn.h"

namespace thip {

ChainTurns &ChainTurns::of(int ordinal) {
    static ChainTurns turns[64];
    return turns[ordinal & 63];
}

hipError_t ChainTurns::join(ChainMember *) {
    std::lock_guard<std::mutex> held(mutex);
    return event ? hipSuccess : hipEventCreateWithFlags(&event, hipEventDisableTiming);
}

void ChainTurns::leave(ChainMember *m) {
    std::lock_guard<std::mutex> held(mutex);
    if (last == m) last = nullptr;
}

hipError_t ChainTurns::Turn::take(ChainTurns *turns, ChainMember *m) {
    lock = std::unique_lock<std::mutex>(turns->mutex);
    if (turns->last && turns->last != m) {
        hipError_t err = hipEventRecord(turns->event, turns->last->stream);
        if (err == hipSuccess) err = hipStreamWaitEvent(m->stream, turns->event, 0);
        if (err != hipSuccess) return err;
    }
    turns->last = m;
    return hipSuccess;
}

}  // namespace thip
