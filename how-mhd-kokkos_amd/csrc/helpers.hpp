// Threads that help the calling thread with a task, and may come late.
//
// A new thread can wait milliseconds for a processor: the workers of an OpenMP
// region spin on every one of them for some time after it, and a slice of the
// scheduler is 3 ms.  So the calling thread waits only for helpers that have
// begun; one that comes when the task is done leaves without touching it.  (With
// a join of all, the upload after the host's initial state, 93,280 cells on 16
// processors with 16 OpenMP threads, took 3 to 5 ms instead of 0.5.)
#pragma once

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

namespace howmhd {

// Used by one thread at a time.  The threads end by themselves soon after they
// get a processor; the destructor waits for the late ones.
class Helpers {
public:
    Helpers() = default;
    Helpers(const Helpers&) = delete;
    Helpers& operator=(const Helpers&) = delete;
    ~Helpers() {
        for (auto& h : threads_) h.thread.join();
    }

    // work(false) on the calling thread and work(true) on up to n others, fewer
    // where the system gives no more; returns when every one that began has
    // ended.  work must do the whole task alone where no helper comes, and must
    // not throw.
    template <typename F>
    void run(int n, const F& work) {
        reap();
        std::shared_ptr<Task> task;
        try {
            if (n > 0) task = std::make_shared<Task>();
            // (late ones of earlier tasks count: a bound on the threads there are)
            while (n-- > 0 && threads_.size() < kMost) {
                threads_.emplace_back();
                threads_.back().task = task;
                threads_.back().thread = std::thread([task, &work] {
                    if (task->enter()) {
                        work(true);
                        task->leave();
                    }
                    task->gone.fetch_add(1);
                });
                ++task->made;
            }
        } catch (const std::system_error&) {
            threads_.pop_back();  // the one without a thread
        } catch (const std::bad_alloc&) {
            if (!threads_.empty() && !threads_.back().thread.joinable()) threads_.pop_back();
        }
        work(false);
        if (task) task->close();
    }

private:
    static constexpr size_t kMost = 32;

    struct Task {
        std::mutex mu;
        std::condition_variable idle;
        bool open = true;
        int inside = 0;
        int made = 0;              // threads of the task (calling thread only)
        std::atomic<int> gone{0};  // threads at their end
        bool enter() {
            std::lock_guard<std::mutex> lk(mu);
            inside += open ? 1 : 0;
            return open;
        }
        void leave() {
            std::lock_guard<std::mutex> lk(mu);
            if (--inside == 0) idle.notify_all();
        }
        void close() {
            std::unique_lock<std::mutex> lk(mu);
            open = false;
            idle.wait(lk, [this] { return inside == 0; });
        }
    };
    struct Helper {
        std::shared_ptr<Task> task;
        std::thread thread;
    };

    // Joins the threads of the tasks whose threads are all at their end.
    void reap() {
        for (auto& h : threads_)
            if (h.task->gone.load() == h.task->made) h.thread.join();
        threads_.erase(std::remove_if(threads_.begin(), threads_.end(), [](const Helper& h) { return !h.thread.joinable(); }),
                       threads_.end());
    }

    std::vector<Helper> threads_;
};

}  // namespace howmhd
