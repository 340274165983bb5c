// oxr_dbuf.h -- device buffers, and the ones an engine keeps between calls.
#pragma once
#include <hip/hip_runtime_api.h>
#include <cstddef>

namespace oxh {

template <typename T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;     // capacity in elements
    hipError_t reserve(size_t want) {
        if (want <= n) return hipSuccess;
        if (p) { hipError_t e = hipFree(p); if (e != hipSuccess) return e; p = nullptr; n = 0; }
        hipError_t e = hipMalloc(reinterpret_cast<void**>(&p), want * sizeof(T));
        if (e == hipSuccess) n = want;
        return e;
    }
    void release() { if (p) (void)hipFree(p); p = nullptr; n = 0; }
};

} // namespace oxh

namespace oxl {

// Device buffers that a call (a merge, a query) uses and the engine keeps for the next:
// allocating and freeing them in every call cost a merge of 34k hits 60 of its 400 us and a
// query of 250k rays, with its pageable copies, 340 of 910. At most KEPT stays allocated
// between calls, nothing after a call that failed, and what stays is given back when an
// allocation of the engine finds no memory.
struct Workspace {
    static constexpr int N = 15;
    static constexpr size_t KEPT = size_t(512) << 20;
    oxh::DBuf<char> slot[N];
    unsigned in_use = 0;      // the slots of the call under way
    int used = 0;             // the slots a merge has taken
    size_t bytes() const { size_t b = 0; for (const auto& x : slot) b += x.n; return b; }
    // frees what no call is using; false if there was nothing
    bool give_back() {
        bool any = false;
        for (int k = 0; k < N; k++) {
            if ((in_use >> k & 1u) || !slot[k].p) continue;
            slot[k].release();
            any = true;
        }
        return any;
    }
    // slot k with at least so many bytes
    hipError_t get(int k, size_t want) {
        in_use |= 1u << k;
        return reserve(slot[k], want);
    }
    // b.reserve(n); the engine's other buffers too go before what is kept here
    template <typename T>
    hipError_t reserve(oxh::DBuf<T>& b, size_t n) {
        hipError_t e = b.reserve(n);
        if (e == hipErrorOutOfMemory && give_back()) {
            (void)hipGetLastError();   // of the first try, not the next launch's
            e = b.reserve(n);
        }
        return e;
    }
};

// One call's use of the work space, ended by its return
class WorkCall {
public:
    explicit WorkCall(Workspace& w) : w_(w) { w_.in_use = 0; w_.used = 0; }
    ~WorkCall() {
        w_.in_use = 0;
        if (!kept_ || w_.bytes() > Workspace::KEPT) (void)w_.give_back();
    }
    void keep() { kept_ = true; }      // the call succeeded
private:
    Workspace& w_;
    bool kept_ = false;
};

} // namespace oxl
