// oxr_copy.cpp -- the staged copies of oxr_copy.h.
#include "oxr_copy.h"
#include <algorithm>
#include <cstring>

namespace oxh {

CopyPool::~CopyPool() {
    {
        std::lock_guard<std::mutex> lk(mu_);
        stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
}

void CopyPool::begin() {
    if (!started_) {
        started_ = true;
        try {
            for (int k = 0; k < HELPERS; k++) threads_.emplace_back([this] { run(); });
        } catch (...) {   // no thread to be had: the caller copies alone (or with those that started)
        }
    }
    {
        std::lock_guard<std::mutex> lk(mu_);
        busy_ = true;
    }
    cv_.notify_all();
}

void CopyPool::end() { busy_ = false; }

void CopyPool::run() {
    unsigned seen = 0;
    for (;;) {
        {
            std::unique_lock<std::mutex> lk(mu_);
            cv_.wait(lk, [&] { return stop_ || busy_; });
            if (stop_) return;
        }
        while (busy_ && !stop_) {
            if (job_.load() == seen) {
                __builtin_ia32_pause();
                continue;
            }
            inside_.fetch_add(1);
            seen = job_.load();
            take_parts();
            inside_.fetch_sub(1);
        }
    }
}

// parts are claimed one by one, so a helper that wakes late finds none left
void CopyPool::take_parts() {
    for (;;) {
        const int k = next_.fetch_add(1), parts = parts_.load();
        if (k >= parts) return;
        const size_t step = (bytes_ / size_t(parts)) & ~size_t(63);
        const size_t at = step * size_t(k), n = k == parts - 1 ? bytes_ - at : step;
        std::memcpy(dst_ + at, src_ + at, n);
        left_.fetch_sub(1);
    }
}

void CopyPool::copy(char* dst, const char* src, size_t bytes) {
    if (!busy_ || threads_.empty() || bytes < (size_t(256) << 10)) {
        std::memcpy(dst, src, bytes);
        return;
    }
    // The fields are rewritten only when no helper reads them: all parts of the last job are
    // taken, and a helper that comes in meanwhile finds none until next_ starts again below.
    next_.store(1 << 20);
    while (inside_.load() != 0) {}
    dst_ = dst; src_ = src; bytes_ = bytes;
    const int parts = 2 * (int(threads_.size()) + 1);
    parts_.store(parts);
    left_.store(parts);
    next_.store(0);
    job_.fetch_add(1);
    take_parts();
    while (left_.load() > 0) {}
}

hipError_t Stager::ready(size_t bytes) {
    hipError_t e;
    for (int k = 0; k < SLOTS; k++)
        if (!done[k] && (e = hipEventCreateWithFlags(&done[k], hipEventDisableTiming)) != hipSuccess) return e;
    const size_t want = bytes > SLOT / 8 ? SLOT : SLOT / 8;
    if (slot_bytes >= want) return hipSuccess;
    for (int k = 0; k < SLOTS; k++) if ((e = wait(k)) != hipSuccess) return e;
    if (ring) (void)hipHostFree(ring);
    ring = nullptr;
    slot_bytes = 0;
    void* p = nullptr;
    if ((e = hipHostMalloc(&p, want * SLOTS, hipHostMallocDefault)) != hipSuccess) return e;
    ring = static_cast<char*>(p);
    slot_bytes = want;
    return hipSuccess;
}

// Halves above 1 MB and quarters above 2 MB: the host side of one runs beside another's crossing.
// A piece of its own costs 10 us and more, its event waited for, so there are no more of them
// (rays queried with 24 / 48 / 64 thousand, us: one piece 97 / 203 / 250, two 121 / 169 / 229,
// four - / - / 236, eight - / - / 340; a pageable hipMemcpy 104 / 203 / 225).
size_t Stager::piece(size_t bytes) {
    if (bytes <= SHORT) return SHORT;
    const size_t part = (bytes / (bytes > SLOT ? 4 : 2) + 0xffff) & ~size_t(0xffff);
    return std::min(SLOT, part);
}

hipError_t Stager::wait(int slot) {
    if (!pending[slot]) return hipSuccess;
    hipError_t e = marked[slot] ? hipEventSynchronize(done[slot]) : hipStreamSynchronize(on[slot]);
    if (e == hipSuccess) pending[slot] = false;
    return e;
}

hipError_t Stager::d2h(hipStream_t s, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    hipError_t e = ready(bytes);
    if (e != hipSuccess) return e;
    if (bytes <= SHORT) {
        // the stream is in order: an upload that may still read this slot comes before
        if ((e = hipMemcpyAsync(ring, src, bytes, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
        idle();
        std::memcpy(dst, ring, bytes);
        return e;
    }
    const size_t part = piece(bytes), n = (bytes + part - 1) / part;
    auto issue = [&](size_t i) -> hipError_t {
        const int k = int(i % SLOTS);
        const size_t at = i * part, len = std::min(part, bytes - at);
        hipError_t x = hipMemcpyAsync(ring + size_t(k) * slot_bytes, static_cast<const char*>(src) + at, len, hipMemcpyDeviceToHost, s);
        if (x == hipSuccess) x = hipEventRecord(done[k], s);
        if (x == hipSuccess) pending[k] = marked[k] = true;
        return x;
    };
    const bool helped = bytes > SLOT;
    if (helped) pool.begin();
    for (size_t i = 0; i < std::min<size_t>(n, SLOTS) && e == hipSuccess; i++) e = issue(i);
    for (size_t i = 0; i < n && e == hipSuccess; i++) {
        const int k = int(i % SLOTS);
        const size_t at = i * part, len = std::min(part, bytes - at);
        if ((e = wait(k)) != hipSuccess) break;
        pool.copy(static_cast<char*>(dst) + at, ring + size_t(k) * slot_bytes, len);
        if (i + SLOTS < n) e = issue(i + SLOTS);
    }
    if (helped) pool.end();
    return e;
}

hipError_t Stager::h2d(hipStream_t s, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    hipError_t e = ready(bytes);
    if (e != hipSuccess) return e;
    if (bytes <= SHORT) {
        int k = 0;   // a slot that is free, so that it need not wait for the copy before it
        while (k < SLOTS - 1 && pending[k]) k++;
        if ((e = wait(k)) != hipSuccess) return e;
        std::memcpy(ring + size_t(k) * slot_bytes, src, bytes);
        e = hipMemcpyAsync(dst, ring + size_t(k) * slot_bytes, bytes, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) { pending[k] = true; marked[k] = false; on[k] = s; }
        return e;
    }
    const size_t part = piece(bytes), n = (bytes + part - 1) / part;
    const bool helped = bytes > SLOT;
    if (helped) pool.begin();
    for (size_t i = 0; i < n && e == hipSuccess; i++) {
        const int k = int(i % SLOTS);
        const size_t at = i * part, len = std::min(part, bytes - at);
        if ((e = wait(k)) != hipSuccess) break;
        pool.copy(ring + size_t(k) * slot_bytes, static_cast<const char*>(src) + at, len);
        e = hipMemcpyAsync(static_cast<char*>(dst) + at, ring + size_t(k) * slot_bytes, len, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(done[k], s);
        if (e == hipSuccess) pending[k] = marked[k] = true;
    }
    if (helped) pool.end();
    return e;
}

void Stager::release() {
    for (int k = 0; k < SLOTS; k++) {
        (void)wait(k);
        if (done[k]) (void)hipEventDestroy(done[k]);
        done[k] = nullptr;
    }
    if (ring) (void)hipHostFree(ring);
    ring = nullptr;
    slot_bytes = 0;
}

} // namespace oxh
