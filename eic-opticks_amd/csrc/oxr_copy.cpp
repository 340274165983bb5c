// oxr_copy.cpp -- the staged copies of oxr_copy.h.
#include "oxr_copy.h"
#include <algorithm>
#include <cstring>

namespace oxh {

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
