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
// may copy at once: their jobs stand in a list, a helper takes one part of the foremost and
// moves it to the back, and each caller works on its own job besides.
class CopyPool {
public:
    ~CopyPool();
    // memcpy split over the helpers and the caller
    void copy(char* dst, const char* src, size_t bytes);
    // helpers spin for work between begin and end instead of sleeping; windows may overlap
    void begin();
    void end();
private:
    static constexpr int HELPERS = 5;
    struct Job {
        char* dst;
        const char* src;
        size_t bytes;
        int parts, next = 0;          // parts claimed so far, under mu_
        std::atomic<int> left;        // parts not yet copied
        Job* link = nullptr;
    };
    void run();
    bool take(Job* job);              // copy one part, of the job or of the foremost; false if there is none
    std::vector<std::thread> threads_;
    std::mutex mu_;                   // threads_, the list of jobs with parts to claim, and the claims
    std::condition_variable cv_;
    Job* first_ = nullptr;
    Job* last_ = nullptr;
    bool started_ = false;
    std::atomic<int> helpers_{0};
    std::atomic<int> open_{0};        // windows
    std::atomic<int> waiting_{0};     // parts to claim
    std::atomic<bool> stop_{false};
};

} // namespace oxh
