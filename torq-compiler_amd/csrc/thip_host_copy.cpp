#include "thip_host_copy.h"

#include <pthread.h>
#include <signal.h>
#include <string.h>

#include <algorithm>
#include <system_error>

namespace thip {

CopyCrew::~CopyCrew() {
    {
        std::lock_guard<std::mutex> lock(mutex);
        ending = true;
    }
    wake.notify_all();
    for (std::thread &t : helpers) t.join();
}

// With `mutex` held.  False: the system gives no threads.
bool CopyCrew::start() {
    if (started) return !helpers.empty();
    started = true;
    const unsigned cpus = std::thread::hardware_concurrency(), wanted = cpus > 1 ? std::min(cpus - 1, kHelpers) : 0;
    // the program's signals are not for these threads
    sigset_t all, before;
    sigfillset(&all);
    pthread_sigmask(SIG_SETMASK, &all, &before);
    try {
        helpers.reserve(wanted);
        for (unsigned i = 0; i < wanted; i++) helpers.emplace_back([this] { help(); });
    } catch (const std::exception &) {  // those that did start help
    }
    pthread_sigmask(SIG_SETMASK, &before, nullptr);
    return !helpers.empty();
}

void CopyCrew::help() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lock(mutex);
    for (;;) {
        wake.wait(lock, [&] { return ending || (copy && copies != seen); });
        if (ending) return;
        seen = copies;
        Copy *c = copy;
        inside++;
        lock.unlock();
        while (c->step()) {
        }
        lock.lock();
        inside--;
    }
}

CopyCrew::Copy::Copy(CopyCrew *of, void *dst_, const void *src_, size_t bytes_)
    : dst((uint8_t *)dst_), src((const uint8_t *)src_), bytes(bytes_), pieces((int)((bytes_ + kPiece - 1) / kPiece)) {
    for (int i = 0; i < pieces; i++) done[i].store(false, std::memory_order_relaxed);
    if (!of || bytes <= kAlone) return;
    {
        std::lock_guard<std::mutex> lock(of->mutex);
        if (of->copy || of->inside || !of->start()) return;  // taken
        of->copy = this;
        of->copies++;
        crew = of;
    }
    of->wake.notify_all();
}

CopyCrew::Copy::~Copy() {
    if (!crew) return;
    {
        std::lock_guard<std::mutex> lock(crew->mutex);
        next.store(pieces, std::memory_order_relaxed);  // also if the dispatch failed half-way
        crew->copy = nullptr;
    }
    // No piece is left, so whoever is inside is on its way out.  (Once the last one is, another copy may have the helpers.)
    for (;;) {
        {
            std::lock_guard<std::mutex> lock(crew->mutex);
            if (crew->inside == 0 || crew->copy) return;
        }
        std::this_thread::yield();
    }
}

bool CopyCrew::Copy::step() {
    const int i = next.fetch_add(1, std::memory_order_relaxed);
    if (i >= pieces) return false;
    const size_t at = (size_t)i * kPiece;
    memcpy(dst + at, src + at, std::min(kPiece, bytes - at));
    done[i].store(true, std::memory_order_release);
    return true;
}

size_t CopyCrew::Copy::ready() {
    while (first < pieces && done[first].load(std::memory_order_acquire)) first++;
    return std::min(bytes, (size_t)first * kPiece);
}

}  // namespace thip
