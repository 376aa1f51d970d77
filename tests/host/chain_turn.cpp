// The turns of executables that have a dec_chain launch, on a HIP of this file's own: which dispatches are one launch, which of them wait for
// which, and what is asked of the runtime when.
#include <stdio.h>

#include <algorithm>
#include <chrono>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "thip_chain_turn.h"

using namespace thip;

// An event remembers the stream that it was recorded on last.
static std::mutex held;
static std::map<hipEvent_t, hipStream_t> recorded;
static thread_local std::vector<std::pair<hipStream_t, hipStream_t>> waits;  // who waits, for whose work
static std::atomic<int> created{0}, failures{0};

#define CHECK(what) do { if (!(what)) failures++, printf("line %d: %s\n", __LINE__, #what); } while (0)

extern "C" hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t)(intptr_t)++created;
    return hipSuccess;
}
extern "C" hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> lock(held);
    recorded[e] = s;
    return e ? hipSuccess : hipErrorInvalidHandle;
}
extern "C" hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::lock_guard<std::mutex> lock(held);
    waits.push_back({s, recorded[e]});
    return hipSuccess;
}
// Neither is allowed while somebody captures a graph.
extern "C" hipError_t hipStreamQuery(hipStream_t) {
    CHECK(!"a query of a stream");
    return hipSuccess;
}
extern "C" hipError_t hipEventQuery(hipEvent_t) {
    CHECK(!"a query of an event");
    return hipSuccess;
}

static hipStream_t streamOf(int n) { return (hipStream_t)(intptr_t)(100 * n); }
static bool waited(const ChainMember &m, const ChainMember &behind) { return waits.size() == 1 && waits[0] == std::make_pair(m.stream, behind.stream); }
static void later() { std::this_thread::sleep_for(std::chrono::nanoseconds(ChainTurns::kAtWork * 3 / 2)); }

// One dispatch; whether it is one launch.
static bool dispatch(ChainTurns *turns, ChainMember *m, bool wanted = true) {
    waits.clear();
    ChainTurns::Turn turn;
    bool chained = false;
    CHECK(turn.take(turns, m, wanted, &chained) == hipSuccess);
    return chained;
}

struct Three {
    ChainTurns turns;
    ChainMember a, b, c;
    explicit Three(bool always) {
        int n = 0;
        for (ChainMember *m : {&a, &b, &c}) {
            m->stream = streamOf(++n);
            m->always = always;
            CHECK(turns.join(m) == hipSuccess);
        }
    }
};

// Launches that are asked for beside others, one behind the other.
static void inTurn() {
    const int before = created;
    Three t(true);
    // a dispatch makes nothing (thip_executable_enqueue_noalloc)
    const int made = created;
    CHECK(made > before);
    CHECK(dispatch(&t.turns, &t.a) && waits.empty());
    CHECK(dispatch(&t.turns, &t.a) && waits.empty());
    CHECK(dispatch(&t.turns, &t.b) && waited(t.b, t.a));
    CHECK(dispatch(&t.turns, &t.a) && waited(t.a, t.b));
    CHECK(created == made);
    later();  // not known to be done
    CHECK(dispatch(&t.turns, &t.c) && waited(t.c, t.a));
    t.c.finished();
    CHECK(dispatch(&t.turns, &t.b) && waits.empty());
    t.turns.leave(&t.b);
    CHECK(dispatch(&t.turns, &t.a) && waits.empty());
}

// Nobody is put behind work that does not end: neither an abandoned executable's nor what waits for that.
static void abandoned(bool always) {
    Three t(always);
    CHECK(dispatch(&t.turns, &t.a));
    t.a.finished();
    CHECK(dispatch(&t.turns, &t.b));
    t.a.abandoned = true;
    t.b.finished();
    later();
    CHECK(!dispatch(&t.turns, &t.c) && waits.empty());
    t.c.finished();
    CHECK(!dispatch(&t.turns, &t.b) && waits.empty());
    t.b.finished();
    t.turns.leave(&t.a);  // its work has ended after all
    CHECK(dispatch(&t.turns, &t.c));
}

// One launch while nobody else is at work, records beside others.
static void beside() {
    Three t(false);
    CHECK(dispatch(&t.turns, &t.a) && dispatch(&t.turns, &t.a));
    CHECK(!dispatch(&t.turns, &t.b) && !dispatch(&t.turns, &t.a) && !dispatch(&t.turns, &t.b));
    t.b.finished();
    CHECK(dispatch(&t.turns, &t.a) && !dispatch(&t.turns, &t.b) && waits.empty());
    t.a.finished();
    CHECK(dispatch(&t.turns, &t.b) && waits.empty());
    CHECK(!dispatch(&t.turns, &t.b, false));
    // a caller that waits by other means is at work for a while; a launch of its is waited for all the same
    CHECK(!dispatch(&t.turns, &t.c));
    t.c.finished();
    later();
    CHECK(dispatch(&t.turns, &t.c) && waited(t.c, t.b));
    // as long as it is being waited for
    t.c.waiting();
    later();
    CHECK(!dispatch(&t.turns, &t.a));
    t.a.finished();
    t.c.finished();
    CHECK(dispatch(&t.turns, &t.a) && waits.empty());
    t.a.finished();
    {
        // while its launches are enqueued, also if they are many
        ChainTurns::Turn turn;
        bool chained = false;
        CHECK(turn.take(&t.turns, &t.a, false, &chained) == hipSuccess && !chained);
        CHECK(!dispatch(&t.turns, &t.b));
        t.b.finished();
    }
    CHECK(!dispatch(&t.turns, &t.b));
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
}

// From several threads: a launch waits for another one's, or that is done.
static void threads(bool always) {
    ChainTurns turns;
    ChainMember members[4];
    std::atomic<int> bad{0}, launches{0};
    hipStream_t launched = nullptr;  // whose launch is on its way
    std::vector<std::thread> all;
    for (int t = 0; t < 4; t++) {
        members[t].stream = streamOf(t + 1);
        members[t].always = always;
        CHECK(turns.join(&members[t]) == hipSuccess);
    }
    for (int t = 0; t < 4; t++) {
        all.emplace_back([&, t] {
            ChainMember &m = members[t];
            for (int i = 0; i < 2000; i++) {
                {
                    ChainTurns::Turn turn;
                    bool chained = false;
                    waits.clear();
                    bad += turn.take(&turns, &m, i % 7 != 0, &chained) != hipSuccess;
                    std::lock_guard<std::mutex> lock(held);
                    bad += chained && launched && launched != m.stream && !(waits.size() == 1 && waits[0] == std::make_pair(m.stream, launched));
                    launches += chained;
                    if (chained) launched = m.stream;
                }
                if (i % 3 == 0) continue;  // the next one behind it
                std::this_thread::yield();
                m.waiting();
                {
                    std::lock_guard<std::mutex> lock(held);
                    if (launched == m.stream) launched = nullptr;
                }
                m.finished();
            }
            m.finished();
        });
    }
    for (std::thread &t : all) t.join();
    CHECK(bad == 0 && launches > 0);
}

int main() {
    inTurn();
    abandoned(false);
    abandoned(true);
    beside();
    gaveUp();
    threads(false);
    threads(true);
    if (failures == 0) puts("in order");
    return failures != 0;
}
