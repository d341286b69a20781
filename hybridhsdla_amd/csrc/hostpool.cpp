#include "hostpool.h"

#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <exception>
#include <list>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace hsgen {

namespace {

constexpr unsigned kMaxThreads = 8;

struct Task {
    const void* group;
    std::function<void()> run;
};

}  // namespace

struct HostPool::State {
    std::mutex mu;
    std::condition_variable wake, done;
    std::list<Task> tasks;
    std::vector<const void*> current;     // per thread: the group it works for
    std::vector<std::thread> threads;
    bool quit = false;
    pid_t pid = getpid();

    void loop(int me)
    {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            wake.wait(lk, [this] { return quit || !tasks.empty(); });
            if (tasks.empty()) return;
            const Task t = std::move(tasks.front());
            tasks.pop_front();
            current[me] = t.group;
            lk.unlock();
            t.run();
            lk.lock();
            current[me] = nullptr;
            done.notify_all();
        }
    }
};

HostPool::HostPool() : s_(new State)
{
    const unsigned hw = std::thread::hardware_concurrency();
    State* s = s_;
    try {
        s->current.assign(kMaxThreads, nullptr);
        for (unsigned t = 0; t + 1 < hw && t < kMaxThreads; ++t) s->threads.emplace_back([s, t] { s->loop((int)t); });
    } catch (const std::exception&) {    // fewer threads, or none
    }
}

HostPool::~HostPool()
{
    if (getpid() != s_->pid) return;
    {
        std::lock_guard<std::mutex> lk(s_->mu);
        s_->quit = true;
    }
    s_->wake.notify_all();
    for (auto& t : s_->threads) t.join();
    delete s_;
}

size_t HostPool::size() const { return s_->threads.size(); }

void HostPool::post(const void* group, const std::function<void()>& run, size_t n)
{
    {
        std::lock_guard<std::mutex> lk(s_->mu);
        for (size_t i = 0; i < n; ++i) s_->tasks.push_back(Task{group, run});
    }
    s_->wake.notify_all();
}

void HostPool::finish(const void* group)
{
    std::unique_lock<std::mutex> lk(s_->mu);
    s_->tasks.remove_if([&](const Task& t) { return t.group == group; });
    s_->done.wait(lk, [&] { return std::find(s_->current.begin(), s_->current.end(), group) == s_->current.end(); });
}

}  // namespace hsgen
