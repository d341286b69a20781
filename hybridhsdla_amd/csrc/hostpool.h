// Threads that copy host memory (hostcopy.hip).
#pragma once

#include <cstddef>
#include <functional>

namespace hsgen {

// Threads of a context: started with its first large copy, at most 8, joined
// with the context.  Tasks run in the order they are posted; finish() withdraws
// a group's waiting tasks and waits for its running ones.
// A forked process has the object but none of the threads.  Its copy of what
// they wait on still counts them as waiting, and destroying that would wait for
// them for ever: there the destructor leaves the state as it is.
class HostPool {
public:
    HostPool();
    ~HostPool();
    HostPool(const HostPool&) = delete;
    HostPool& operator=(const HostPool&) = delete;
    size_t size() const;
    void post(const void* group, const std::function<void()>& run, size_t n);
    void finish(const void* group);

private:
    struct State;
    State* s_;
};

}  // namespace hsgen
