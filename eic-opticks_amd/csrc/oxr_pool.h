// oxr_pool.h -- helper threads for host copies.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>
#include <vector>

namespace oxh {

// Helper threads, started by the first large copy and joined with the owner. Several callers
// may copy at once: their jobs stand in a list, a helper joins the foremost and moves it to
// the back, and each caller works on its own job besides.
class CopyPool {
public:
    ~CopyPool();
    // memcpy split over the helpers and the caller
    void copy(char* dst, const char* src, size_t bytes);
    // Copies are to come: between begin and end the helpers are awake. One that finds no part for
    // SPIN_US sleeps until the next copy, so a window may hold a wait for the device (a kernel
    // ahead of a download). Windows may overlap. Spinning throughout instead, five threads took
    // 4.6 ms of processor time in a query of 250,000 rays of 0.9 ms, now 2.8; a query of
    // 2 million, whose kernel outlasts SPIN_US, takes 8.2 ms for 7.9.
    void begin();
    void end();
    // helper threads on this host: at most five, and one processor that the process may run on
    // is left to the caller (one processor: none)
    static int helpers_here();
private:
    // longer than a 2 MB piece takes to cross PCIe (40 us), about what two wakings take
    static constexpr int SPIN_US = 100;
    struct Job {
        char* dst;
        const char* src;
        size_t bytes;
        int parts;
        std::atomic<int> next{0};     // parts claimed
        std::atomic<int> left;        // parts not yet copied
        std::atomic<int> users{0};    // helpers that have joined
        Job* link = nullptr;
    };
    void run();
    bool help();                      // join a job until its parts are claimed; false if there is none
    void work(Job& job);
    std::vector<std::thread> threads_;
    std::mutex mu_;                   // threads_ and sleeping
    std::condition_variable cv_;
    bool started_ = false;
    std::atomic<int> helpers_{0};
    // what waiting helpers look at, in a cache line of its own
    alignas(64) std::atomic<int> waiting_{0};   // jobs with parts to claim
    std::atomic<int> open_{0};                  // windows
    std::atomic<unsigned> opened_{0};           // windows so far
    std::atomic<int> asleep_{0};                // helpers asleep within a window, which the next copy wakes
    std::atomic<bool> stop_{false};
    // The list of jobs is guarded by a flag to spin on: it is held for a few instructions, and a
    // thread put to sleep over it would wake after the copy's end.
    alignas(64) std::atomic_flag list_ = ATOMIC_FLAG_INIT;
    Job* first_ = nullptr;
    Job* last_ = nullptr;
};

} // namespace oxh
