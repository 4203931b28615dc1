// The set-up passes' host threads (csrc/workers.hpp): all work is done once, an exception on any
// thread reaches the caller, and work goes on where the system gives no thread.
#include <sys/resource.h>

#include <atomic>
#include <cstdio>
#include <new>
#include <set>

#include "workers.hpp"

static int failed = 0;
#define CHECK(cond)                                                    \
    do {                                                               \
        if (!(cond)) {                                                 \
            std::printf("failed: %s (line %d)\n", #cond, __LINE__);    \
            ++failed;                                                  \
        }                                                              \
    } while (0)

// Runs n items on `most` threads, item `bad` throwing; returns whether the exception arrived.
// Every item starts only once `meet` threads have entered, so that each of them gets some.
static bool run(int most, int n, int bad, int meet, std::set<std::thread::id> *who = nullptr) {
    std::atomic<int> next{0}, done{0}, in{0};
    std::mutex mu;
    auto fn = [&] {
        ++in;
        while (in < meet) std::this_thread::yield();
        for (int i; (i = next++) < n;) {
            if (i == bad) throw std::bad_alloc();
            ++done;
            if (who) {
                std::lock_guard<std::mutex> lock(mu);
                who->insert(std::this_thread::get_id());
            }
        }
    };
    try {
        aphip::run_workers(most, fn);
    } catch (const std::bad_alloc &) {
        return true;
    }
    CHECK(done == n);
    return false;
}

int main() {
    // without room for a thread's stack no thread starts, and the caller does the work alone (first of
    // all: the stacks of ended threads are kept for later ones)
    struct rlimit old, none;
    getrlimit(RLIMIT_AS, &old);
    none = old;
    none.rlim_cur = 1;
    setrlimit(RLIMIT_AS, &none);
    std::thread t = aphip::try_thread([] {});
    const bool started = t.joinable();
    if (started) t.join();
    const bool threw = run(8, 100, -1, 1), thrown = run(8, 100, 7, 1);
    setrlimit(RLIMIT_AS, &old);
    CHECK(!started);
    CHECK(!threw && thrown);
    for (int most : {-1, 0, 1, 2, 8}) CHECK(!run(most, 100, -1, 1));
    CHECK(!run(4, 0, -1, 1));
    // thrown on the caller's thread or on another one
    for (int k = 0; k < 50; ++k) CHECK(run(8, 64, k, 8));
    CHECK(run(1, 3, 1, 1));
    std::set<std::thread::id> who;
    CHECK(!run(8, 100, -1, 8, &who) && !who.empty());
    std::printf(failed ? "%d checks failed\n" : "ok\n", failed);
    return failed != 0;
}
