// The turns of executables that have a dec_chain launch, on a HIP of this file's own: which dispatches wait for which, and what is asked of
// the runtime when.
#include <stdio.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "thip_chain_turn.h"

using namespace thip;

// A stream is busy while it is in `busy`.  An event remembers the stream that it was recorded on last.
static std::mutex held;
static std::set<hipStream_t> busy;
static std::map<hipEvent_t, hipStream_t> recorded;
static std::vector<std::pair<hipStream_t, hipStream_t>> waits;  // who waits, for whose work
static int created, failures;

extern "C" hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t)(intptr_t)++created;
    return hipSuccess;
}
extern "C" hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    recorded[e] = s;
    return e ? hipSuccess : hipErrorInvalidHandle;
}
extern "C" hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    waits.push_back({s, recorded[e]});
    return hipSuccess;
}
extern "C" hipError_t hipStreamQuery(hipStream_t s) {
    std::lock_guard<std::mutex> lock(held);
    return busy.count(s) ? hipErrorNotReady : hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

#define CHECK(what) do { if (!(what)) failures++, printf("line %d: %s\n", __LINE__, #what); } while (0)

static hipStream_t streamOf(int n) { return (hipStream_t)(intptr_t)(100 * n); }

// One dispatch; whether it is one launch.
static bool dispatch(ChainTurns *turns, ChainMember *m, bool wanted = true) {
    waits.clear();
    ChainTurns::Turn turn;
    bool chained = false;
    CHECK(turn.take(turns, m, wanted, &chained) == hipSuccess);
    busy.insert(m->stream);
    return chained;
}

static void inTurn() {
    ChainTurns turns;
    ChainMember a, b;
    a.stream = streamOf(1);
    b.stream = streamOf(2);
    a.always = b.always = true;
    const int before = created;
    CHECK(turns.join(&a) == hipSuccess && turns.join(&b) == hipSuccess);
    // a dispatch makes nothing (thip_executable_enqueue_noalloc)
    const int made = created;
    CHECK(made > before);
    CHECK(dispatch(&turns, &a));
    CHECK(waits.empty());
    CHECK(dispatch(&turns, &a));
    CHECK(waits.empty());
    CHECK(dispatch(&turns, &b));
    CHECK(waits.size() == 1 && waits[0] == std::make_pair(b.stream, a.stream));
    CHECK(dispatch(&turns, &a));
    CHECK(waits.size() == 1 && waits[0] == std::make_pair(a.stream, b.stream));
    CHECK(created == made);
    busy.clear();
    turns.leave(&a);
    CHECK(dispatch(&turns, &b));
    CHECK(waits.empty());
    busy.clear();
    turns.leave(&b);
}

// Nobody is put behind work that does not end: neither an abandoned executable's nor what waits for that.
static void abandoned() {
    ChainTurns turns;
    ChainMember a, b, c;
    a.stream = streamOf(1);
    b.stream = streamOf(2);
    c.stream = streamOf(3);
    a.always = b.always = c.always = true;
    for (ChainMember *m : {&a, &b, &c}) CHECK(turns.join(m) == hipSuccess);
    CHECK(dispatch(&turns, &a));
    CHECK(dispatch(&turns, &b));
    a.abandoned = true;
    CHECK(!dispatch(&turns, &c) && waits.empty());
    CHECK(!dispatch(&turns, &b) && waits.empty());
    busy.clear();  // its work has ended after all
    CHECK(dispatch(&turns, &c));
    CHECK(dispatch(&turns, &b));
    CHECK(waits.size() == 1 && waits[0] == std::make_pair(b.stream, c.stream));
    busy.clear();
    for (ChainMember *m : {&a, &b, &c}) turns.leave(m);
}

// One launch while nobody else is at work, records beside others; nobody waits.
static void beside() {
    ChainTurns turns;
    ChainMember a, b;
    a.stream = streamOf(1);
    b.stream = streamOf(2);
    CHECK(turns.join(&a) == hipSuccess && turns.join(&b) == hipSuccess);
    CHECK(dispatch(&turns, &a) && dispatch(&turns, &a));
    CHECK(!dispatch(&turns, &b) && !dispatch(&turns, &a) && !dispatch(&turns, &b));
    busy.erase(b.stream);
    CHECK(dispatch(&turns, &a) && !dispatch(&turns, &b));
    busy.clear();
    CHECK(dispatch(&turns, &b));
    CHECK(!dispatch(&turns, &b, false));
    {
        // its launches are on their way, though its stream has none yet
        ChainTurns::Turn turn;
        bool chained = true;
        CHECK(turn.take(&turns, &a, true, &chained) == hipSuccess && !chained);
        busy.clear();
        CHECK(!dispatch(&turns, &b));
        busy.clear();
    }
    CHECK(dispatch(&turns, &b) && waits.empty());
    busy.clear();
    turns.leave(&a);
    turns.leave(&b);
}

// Behind a launch that gave up, records for a while, longer each time; then launches again.
static void gaveUp() {
    ChainTurns turns;
    ChainMember a;
    uint32_t word = 0;
    a.stream = streamOf(1);
    a.gaveUp = &word;
    CHECK(turns.join(&a) == hipSuccess);
    auto records = [&] {
        uint32_t n = 0;
        while (n < 1000000 && !dispatch(&turns, &a)) n++;
        return n;
    };
    CHECK(records() == 0);
    uint32_t wanted = ChainTurns::kGivenUpFirst;
    for (int i = 0; i < 9; i++) {
        word = 1;
        CHECK(records() == wanted);
        wanted = std::min(2 * wanted, ChainTurns::kGivenUpMost);
    }
    CHECK(wanted == ChainTurns::kGivenUpMost);
    word = 1;
    CHECK(records() == wanted);
    for (uint32_t i = 0; i < wanted; i++) CHECK(dispatch(&turns, &a));
    word = 1;
    CHECK(records() == ChainTurns::kGivenUpFirst);
    // who asked for the launch always has it
    a.always = true;
    word = 1;
    CHECK(dispatch(&turns, &a) && dispatch(&turns, &a));
    busy.clear();
    turns.leave(&a);
}

// From several threads: nobody else's work is on its way when one launches.
static void threads() {
    ChainTurns turns;
    ChainMember members[4];
    std::atomic<int> bad{0}, launches{0};
    std::vector<std::thread> all;
    for (int t = 0; t < 4; t++) {
        members[t].stream = streamOf(t + 1);
        CHECK(turns.join(&members[t]) == hipSuccess);
    }
    for (int t = 0; t < 4; t++) {
        all.emplace_back([&, t] {
            for (int i = 0; i < 2000; i++) {
                {
                    ChainTurns::Turn turn;
                    bool chained = false;
                    bad += turn.take(&turns, &members[t], i % 7 != 0, &chained) != hipSuccess;
                    std::lock_guard<std::mutex> lock(held);
                    bad += chained && !busy.empty();
                    launches += chained;
                    busy.insert(members[t].stream);
                }
                if (i % 3 == 0) std::this_thread::yield();
                std::lock_guard<std::mutex> lock(held);
                busy.erase(members[t].stream);
            }
        });
    }
    for (std::thread &t : all) t.join();
    CHECK(bad == 0 && launches > 0);
    for (ChainMember &m : members) turns.leave(&m);
}

int main() {
    inTurn();
    beside();
    gaveUp();
    threads();
    abandoned();
    if (failures == 0) puts("in order");
    return failures != 0;
}
