// CopyCrew: every byte is copied, at sizes around its pieces, with helpers and without, from several threads, and when a copy is left half-way.
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

#define private public  // what a copy does between the steps of another one's end
#include "thip_host_copy.h"
#undef private

using thip::CopyCrew;

static bool once(CopyCrew *crew, size_t bytes, unsigned seed, int steps) {
    std::vector<uint8_t> src(bytes + 1), dst(bytes + 1, 0xa5);
    for (size_t i = 0; i < bytes; i++) src[i] = (uint8_t)((i * 2654435761u + seed) >> 11);
    size_t there = 0;
    {
        CopyCrew::Copy copy(crew, dst.data(), src.data(), bytes);
        while (there < bytes && steps-- != 0) {
            if (!copy.step()) std::this_thread::yield();
            there = copy.ready();
            if (there > bytes || memcmp(dst.data(), src.data(), there) != 0) return false;
        }
    }
    src.assign(src.size(), 0);  // nobody reads or writes behind the end of a copy
    return dst[bytes] == 0xa5;
}

// A copy ends while another one takes over the helpers: that one keeps them.
static bool takenOver() {
    CopyCrew crew;
    char bytes[8] = {0};
    CopyCrew::Copy next(nullptr, bytes, bytes + 4, 4);
    std::thread other;
    {
        CopyCrew::Copy last(nullptr, bytes, bytes + 4, 4);
        last.crew = &crew;
        crew.copy = &last;
        crew.inside = 1;  // a helper that is on its way out
        other = std::thread([&] {
            for (;; std::this_thread::yield()) {
                std::lock_guard<std::mutex> lock(crew.mutex);
                if (crew.copy) continue;  // `last` has not begun to end
                crew.inside = 0;
                crew.copy = &next;
                return;
            }
        });
    }
    other.join();
    std::lock_guard<std::mutex> lock(crew.mutex);
    return crew.copy == &next;
}

int main() {
    for (int i = 0; i < 20; i++) {
        if (!takenOver()) return puts("the helpers were taken away"), 1;
    }
    const size_t piece = CopyCrew::kPiece, most = piece * CopyCrew::kMaxPieces;
    const size_t sizes[] = {0, 1, piece - 1, piece, piece + 1, CopyCrew::kAlone, CopyCrew::kAlone + 1, 5 * piece + 77, most - 1, most};
    CopyCrew crew;
    for (size_t bytes : sizes) {
        for (int rounds = 0; rounds < 4; rounds++) {
            if (!once(rounds & 1 ? &crew : nullptr, bytes, (unsigned)(bytes + rounds), -1) || !once(&crew, bytes, (unsigned)rounds, rounds)) return printf("%zu bytes\n", bytes), 1;
        }
    }
    std::vector<std::thread> threads;
    std::atomic<int> bad{0};
    for (unsigned t = 0; t < 4; t++) {
        threads.emplace_back([&, t] {
            for (unsigned i = 0; i < 12; i++) bad += !once(&crew, (i + 3) * piece + t, t * 100 + i, i % 5 == 4 ? (int)i : -1);
        });
    }
    for (std::thread &t : threads) t.join();
    if (bad) return printf("threads: %d\n", bad.load()), 1;
    puts("copied");
}
