/*
 * bp_parallel.cpp -- a small pool of host threads.
 *
 * Repacking a graph's arrays (rows of 10 floats, tables of 100) is bound by
 * memory latency and gains from every core, but a transfer of a few
 * megabytes takes less than starting 15 threads does (10-20 us each, one
 * after the other).  The threads are therefore kept between calls and woken;
 * a thread that finds nothing to do for a second ends, so that an idle
 * program holds none.
 */
#include "bp_parallel.h"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <deque>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

namespace {

struct Job {
    const std::function<void(unsigned)> *f;
    unsigned parts;
    std::atomic<unsigned> next{0}, done{0};

    bool left() const { return next.load(std::memory_order_relaxed) < parts; }

    /* takes parts until none is left */
    void work()
    {
        for (unsigned i; (i = next.fetch_add(1)) < parts;) {
            (*f)(i);
            done.fetch_add(1, std::memory_order_release);
        }
    }
};

struct Pool {
    std::mutex mu;
    std::condition_variable wake;
    std::deque<std::shared_ptr<Job>> jobs;
    unsigned threads = 0, idle = 0;
};

/* never destroyed: its threads may outlive main() */
Pool &pool()
{
    static Pool *p = new Pool;
    return *p;
}

void thread_main()
{
    Pool &p = pool();
    std::unique_lock<std::mutex> lock(p.mu);
    for (;;) {
        std::shared_ptr<Job> job;
        for (auto &j : p.jobs)
            if (j->left()) {
                job = j;
                break;
            }
        if (job) {
            lock.unlock();
            job->work();
            lock.lock();
            continue;
        }
        ++p.idle;
        const bool rest = p.wake.wait_for(lock, std::chrono::seconds(1)) == std::cv_status::timeout;
        --p.idle;
        if (rest && p.jobs.empty()) {
            --p.threads;
            return;
        }
    }
}

} // namespace

void bp_parallel(unsigned parts, const std::function<void(unsigned)> &f)
{
    const unsigned limit = std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
    if (parts < 2 || limit < 2) {
        for (unsigned i = 0; i < parts; ++i)
            f(i);
        return;
    }
    auto job = std::make_shared<Job>();
    job->f = &f;
    job->parts = parts;
    Pool &p = pool();
    {
        std::lock_guard<std::mutex> lock(p.mu);
        p.jobs.push_back(job);
        unsigned want = std::min(parts, limit) - 1;
        while (p.idle < want && p.threads < limit - 1) {
            try {
                std::thread(thread_main).detach();
            } catch (const std::system_error &) {
                break; /* the calling thread does the work */
            }
            ++p.threads;
            --want; /* this one comes by itself */
        }
    }
    p.wake.notify_all();
    job->work();
    while (job->done.load(std::memory_order_acquire) < parts)
        std::this_thread::yield();
    std::lock_guard<std::mutex> lock(p.mu);
    for (auto it = p.jobs.begin(); it != p.jobs.end(); ++it)
        if (*it == job) {
            p.jobs.erase(it);
            break;
        }
}
