// oxr_pool.cpp -- the helper threads of oxr_pool.h.
#include "oxr_pool.h"
#include <algorithm>
#include <chrono>
#include <cstring>
#include <sched.h>

namespace oxh {

// One turn of a waiting loop: short waits stay on the processor, longer ones give it up to any
// thread that wants it, such as the one that is waited for.
static void relax(unsigned& turns) {
    if (++turns % 512 == 0) std::this_thread::yield();
    else __builtin_ia32_pause();
}

namespace {
struct Hold {
    std::atomic_flag& f;
    explicit Hold(std::atomic_flag& flag) : f(flag) {
        unsigned turns = 0;
        while (f.test_and_set(std::memory_order_acquire)) relax(turns);
    }
    ~Hold() { f.clear(std::memory_order_release); }
};
}

int CopyPool::helpers_here() {
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : int(std::thread::hardware_concurrency());
    return std::max(0, std::min(5, cpus - 1));
}

CopyPool::~CopyPool() {
    {
        std::lock_guard<std::mutex> lk(mu_);
        stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
}

void CopyPool::begin() {
    {
        std::lock_guard<std::mutex> lk(mu_);
        open_.fetch_add(1);
        opened_.fetch_add(1);
        if (!started_) {
            started_ = true;
            try {
                for (int k = helpers_here(); k > 0; k--) {
                    threads_.emplace_back([this] { run(); });
                    helpers_.fetch_add(1);
                }
            } catch (...) {   // no thread to be had: the caller copies alone (or with those that started)
            }
        }
    }
    cv_.notify_all();
}

void CopyPool::end() { open_.fetch_sub(1); }

void CopyPool::run() {
    using clock = std::chrono::steady_clock;
    unsigned seen = 0;     // the newest window it has been awake for
    bool tired = false;    // asleep within a window, for the next copy to wake
    for (;;) {
        {
            std::unique_lock<std::mutex> lk(mu_);
            if (tired) asleep_.fetch_add(1);
            cv_.wait(lk, [&] { return stop_ || (open_ > 0 && (opened_ != seen || waiting_ > 0)); });
            if (tired) asleep_.fetch_sub(1);
            if (stop_) return;
            seen = opened_;
        }
        tired = false;
        unsigned turns = 0;
        clock::time_point since = clock::now();
        while (open_ > 0 && !stop_) {
            if (waiting_ > 0 && help()) {
                turns = 0;
                since = clock::now();
                continue;
            }
            relax(turns);
            if (turns % 512 == 0 && clock::now() - since > std::chrono::microseconds(SPIN_US)) {
                tired = true;
                break;
            }
        }
    }
}

// claims and copies parts until none is left to claim
void CopyPool::work(Job& job) {
    const size_t step = (job.bytes / size_t(job.parts)) & ~size_t(63);
    for (int k; (k = job.next.fetch_add(1)) < job.parts;) {
        if (k == job.parts - 1) waiting_.fetch_sub(1);
        const size_t at = step * size_t(k), n = k == job.parts - 1 ? job.bytes - at : step;
        std::memcpy(job.dst + at, job.src + at, n);
        job.left.fetch_sub(1);
    }
}

bool CopyPool::help() {
    Job* job;
    {
        Hold hold(list_);
        job = first_;
        if (!job) return false;
        if (job != last_) {          // to the back
            first_ = job->link;
            job->link = nullptr;
            last_->link = job;
            last_ = job;
        }
        job->users.fetch_add(1);     // under the flag, so before its caller takes it off the list
    }
    work(*job);
    job->users.fetch_sub(1);         // the last use of the job: its caller may be gone after this
    return true;
}

void CopyPool::copy(char* dst, const char* src, size_t bytes) {
    const int helpers = helpers_;
    if (open_ <= 0 || helpers == 0 || bytes < (size_t(256) << 10)) {
        std::memcpy(dst, src, bytes);
        return;
    }
    Job job;
    job.dst = dst; job.src = src; job.bytes = bytes;
    job.parts = 2 * (helpers + 1);
    job.left = job.parts;
    {
        Hold hold(list_);
        (last_ ? last_->link : first_) = &job;
        last_ = &job;
        waiting_.fetch_add(1);
    }
    if (asleep_ > 0) {
        std::lock_guard<std::mutex> lk(mu_);   // one that counts as asleep waits already, or will see the job
        cv_.notify_all();
    }
    work(job);
    {
        Hold hold(list_);
        Job** at = &first_;
        Job* before = nullptr;
        while (*at != &job) { before = *at; at = &before->link; }
        *at = job.link;
        if (last_ == &job) last_ = before;
    }
    unsigned turns = 0;
    while (job.left > 0 || job.users > 0) relax(turns);
}

} // namespace oxh
