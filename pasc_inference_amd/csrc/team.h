// Helper threads of the host copies (transfer.hip): parked between transfers, started when first
// needed, ended with the process's last context.  Host code only.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <deque>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace pasc {

class Team {
    struct Job {
        const std::function<void()> *fn = nullptr;
        int running = 0;
        bool closed = false;
    };
    std::mutex mu;
    std::condition_variable wake, done;
    std::deque<std::shared_ptr<Job>> queue;
    std::vector<std::thread> threads;
    int users = 0;
    // Threads of an earlier generation end.  It only grows, so no later open, run or close can take
    // back the end of threads that have not woken yet.  (A flag that the closer reset left them
    // asleep, and their closer waiting, when another context was opened and closed meanwhile.)
    uint64_t generation = 0;

    void loop(uint64_t mine) {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            wake.wait(lk, [&] { return generation != mine || !queue.empty(); });
            if (generation != mine) return;
            std::shared_ptr<Job> j = queue.front();
            queue.pop_front();
            if (j->closed) continue;
            j->running++;
            lk.unlock();
            (*j->fn)();
            lk.lock();
            if (--j->running == 0) done.notify_all();
        }
    }

  public:
    static constexpr int MOST = 7;

    static int helpers() {
        return std::min(MOST, std::max(1, (int)std::thread::hardware_concurrency() / 2) - 1);
    }
    void open() {
        std::lock_guard<std::mutex> lk(mu);
        users++;
    }
    void close() {
        std::vector<std::thread> gone;
        {
            std::lock_guard<std::mutex> lk(mu);
            if (--users > 0) return;
            generation++;
            gone.swap(threads);
        }
        wake.notify_all();
        for (auto &t : gone) t.join();
    }
    // fn on this thread and on up to n helpers; back when every helper that started has ended.
    // fn must not throw.
    void run(int n, const std::function<void()> &fn) {
        std::shared_ptr<Job> job;
        if (n > 0) {
            try {
                job = std::make_shared<Job>();
                job->fn = &fn;
                std::lock_guard<std::mutex> lk(mu);
                while ((int)threads.size() < std::min(n, helpers()))
                    threads.emplace_back([this, g = generation] { loop(g); });
                for (int i = 0; i < n; i++) queue.push_back(job);
            } catch (const std::exception &) {
                // fewer helpers: this thread does the rest
            }
            if (n == 1) wake.notify_one();
            else wake.notify_all();
        }
        fn();
        if (job) {
            std::unique_lock<std::mutex> lk(mu);
            job->closed = true;
            done.wait(lk, [&] { return job->running == 0; });
        }
    }
};

}  // namespace pasc
