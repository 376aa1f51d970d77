// Copies of a dispatch's host bindings to pinned memory, shared among a few threads.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace thip {

// The threads of a device that help a dispatch to copy; started by the first copy that is large enough, joined with the device.
//
// One thread copies 34 GB/s (4.8 MB from memory: 130 us) and the link to the GPU carries 53 (91 us), so alone it is the slower half; four
// copy the same in 23 us where they run and some 50 where they have to wake.  A dispatch finds them taken by another one: it copies by itself.
class CopyCrew {
public:
    static constexpr size_t kPiece = 256 * 1024;      // what a thread takes at a time
    static constexpr size_t kAlone = 1024 * 1024;     // up to here waking them takes as long as the copy
    static constexpr int kMaxPieces = 64;             // of a copy
    static constexpr unsigned kHelpers = 3;

    ~CopyCrew();

    // A copy of `bytes` (at most kMaxPieces pieces) that the calling thread takes part in.
    class Copy {
    public:
        // crew: null: the caller copies alone
        Copy(CopyCrew *crew, void *dst, const void *src, size_t bytes);
        ~Copy();  // all helpers have let go of it
        // Copies a piece, if one is left that nobody took; false: none.
        bool step();
        // Bytes from the start that are there.
        size_t ready();

    private:
        friend class CopyCrew;
        CopyCrew *crew = nullptr;  // whose helpers take part; null: nobody's
        uint8_t *dst;
        const uint8_t *src;
        size_t bytes;
        int pieces, first = 0;     // first: pieces before it are there
        std::atomic<int> next{0};
        std::atomic<bool> done[kMaxPieces];
    };

private:
    bool start();
    void help();
    std::mutex mutex;
    std::condition_variable wake;
    std::vector<std::thread> helpers;
    Copy *copy = nullptr;     // the one that is to be helped with
    uint64_t copies = 0;
    int inside = 0;           // helpers that work on it
    bool started = false, ending = false;
};

}  // namespace thip
