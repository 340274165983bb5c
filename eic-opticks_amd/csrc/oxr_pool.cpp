// oxr_pool.cpp -- the helper threads of oxr_pool.h.
#include "oxr_pool.h"
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
    {
        std::lock_guard<std::mutex> lk(mu_);
        open_.fetch_add(1);
        if (!started_) {
            started_ = true;
            try {
                for (int k = 0; k < HELPERS; k++) {
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
    for (;;) {
        {
            std::unique_lock<std::mutex> lk(mu_);
            cv_.wait(lk, [&] { return stop_ || open_ > 0; });
            if (stop_) return;
        }
        while (open_ > 0 && !stop_)
            if (waiting_ <= 0 || !take(nullptr)) __builtin_ia32_pause();
    }
}

bool CopyPool::take(Job* job) {
    int k;
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!job) job = first_;
        if (!job || job->next == job->parts) return false;
        k = job->next++;
        waiting_.fetch_sub(1);
        Job** at = &first_;          // out of the list, and to its back if parts are left
        Job* before = nullptr;
        while (*at != job) { before = *at; at = &before->link; }
        *at = job->link;
        if (last_ == job) last_ = before;
        job->link = nullptr;
        if (job->next < job->parts) {
            (last_ ? last_->link : first_) = job;
            last_ = job;
        }
    }
    const size_t step = (job->bytes / size_t(job->parts)) & ~size_t(63);
    const size_t at = step * size_t(k), n = k == job->parts - 1 ? job->bytes - at : step;
    std::memcpy(job->dst + at, job->src + at, n);
    job->left.fetch_sub(1);   // the last use of the job: its caller may be gone after this
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
        std::lock_guard<std::mutex> lk(mu_);
        (last_ ? last_->link : first_) = &job;
        last_ = &job;
        waiting_.fetch_add(job.parts);
    }
    while (take(&job)) {}
    while (job.left > 0) __builtin_ia32_pause();
}

} // namespace oxh
