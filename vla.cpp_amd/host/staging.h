// Host work of a prefill in front of its uploads, shared out over threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <system_error>
#include <thread>
#include <vector>

#include "model.h"

namespace vla {

// Runs `work(task)` for every task of every group (group g: tasks first[g] .. first[g + 1] - 1) on up to `threads` threads,
// the calling one among them, in order; `ready(g)` is called on the calling thread, in order of g, as soon as it sees
// that the tasks of groups 0 .. g are done (an upload then overlaps the next groups' work).  The threads live for this
// call only: one start per call, where a start per group cost 27 observations 24 of them.  The first exception, of a task or
// of ready(), is thrown again when all threads are back: no further task starts, and ready() is not called for groups from there
// on (a task that throws never counts as done, so its group is not announced whoever looks at it when).
template <typename Work, typename Ready>
void run_staged(const std::vector<int>& first, int threads, Work work, Ready ready) {
    const int n_groups = (int)first.size() - 1, n_tasks = first.back();
    std::atomic<int> next{0};
    std::atomic<bool> failed{false};
    std::vector<std::atomic<int>> left(n_groups);
    for (int g = 0; g < n_groups; ++g) left[g] = first[g + 1] - first[g];
    std::exception_ptr error;
    std::atomic_flag has_error = ATOMIC_FLAG_INIT;
    auto fail = [&]() {
        if (!has_error.test_and_set()) error = std::current_exception();
        failed = true;
    };
    auto one = [&]() {  // false: no task left
        const int t = next.fetch_add(1);
        if (t >= n_tasks || failed) return false;
        try {
            work(t);
        } catch (...) {
            fail();
            return true;
        }
        const int g = (int)(std::upper_bound(first.begin(), first.end(), t) - first.begin()) - 1;
        left[g].fetch_sub(1, std::memory_order_release);
        return true;
    };
    std::vector<std::thread> pool;
    struct Join {
        std::vector<std::thread>& p;
        ~Join() { for (auto& t : p) t.join(); }
    };
    int done = 0;
    auto announce = [&]() {
        while (done < n_groups && left[done].load(std::memory_order_acquire) == 0) ready(done++);
    };
    {
        Join join{pool};
        try {
            for (int t = 1; t < std::min(threads, n_tasks); ++t) pool.emplace_back([&]() { while (one()) {} });
        } catch (const std::system_error&) {}  // no more threads to be had: the ones there are do the work
        try {
            while (one()) announce();
            while (done < n_groups && !failed) {  // the others' last tasks
                announce();
                std::this_thread::yield();
            }
        } catch (...) {
            fail();
        }
    }
    if (failed) std::rethrow_exception(error);
}

// Pieces of 1 MiB and more that an observation's `bytes` are cut into for run_staged, and the threads for a batch.  Up to four
// observations are left to the calling thread: the caller's next writes to lines that other cores have read take longer than the
// shares gain (three views of pi0, 6.3 MB: six threads made the call 0.2 ms shorter and the refill of the same buffer by the
// caller 4.5 ms longer; four observations of two views: two threads 0.6 and 6 ms).  Five to seven go to two threads (six
// observations of GR00T: three made the refill 5 ms longer), from there on a thread an observation; with text rows and a
// state encoder for each (`texts`) always.
inline int stage_pieces(size_t bytes) { return (int)std::max<size_t>(1, bytes >> 20); }
inline int stage_threads(int batch, bool texts) {
    return texts || batch >= 8 ? std::max(1, std::min(default_cpu_threads(), batch)) : batch < 5 ? 1 : std::min(default_cpu_threads(), 2);
}

}  // namespace vla
