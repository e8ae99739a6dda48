// Scenarios of transfer.hpp on the CPU; argv[1] names one.  Exit status 0: as it should be.
#include <pthread.h>
#include <sched.h>
#include <signal.h>
#include <time.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

// the clock of all threads but the main one may be made to run ahead
static const std::thread::id main_thread = std::this_thread::get_id();
static std::atomic<long> ahead_ns{0}, calls{0};  // calls: times read, one for each helper that is called
static int skewed_clock(clockid_t id, timespec* t) {
    const int r = clock_gettime(id, t);
    calls++;
    if (std::this_thread::get_id() == main_thread) return r;
    t->tv_nsec += ahead_ns;
    t->tv_sec += t->tv_nsec / 1000000000;
    t->tv_nsec %= 1000000000;
    return r;
}
#define clock_gettime skewed_clock
#include "transfer.hpp"

using gf::HostRing;

namespace {
constexpr size_t kUnit = 64 * 144;  // bytes of a unit, a group's links

// one download of `chunks` slots, chunk k filled with the byte 1 + k % 200; bytes of dst that hold neither that nor
// what was there before
long wrong_bytes(HostRing& r, long chunks, hipError_t& e) {
    const long per = (long)(r.slot / kUnit), units = chunks * per;
    std::vector<char> dst(units * kUnit, 0);
    e = r.pull(
        dst.data(), units, kUnit, [](long q) { return (size_t)q * kUnit; },
        [&](long q, long n, char* p) { return memset(p, (int)(1 + q / per % 200), n * kUnit), hipSuccess; }, nullptr);
    long wrong = 0;
    for (long k = 0; k < chunks; k++)
        for (size_t b = 0; b < per * kUnit; b++) {
            const int v = (unsigned char)dst[k * per * kUnit + b];
            wrong += v != (int)(1 + k % 200) && (v != 0 || e == hipSuccess);
        }
    return wrong;
}

// a whole transfer, and one whose wait for a chunk fails: an error, and nothing in the array that is not its own
int failed_wait() {
    HostRing r;
    r.shape(96 * kUnit, 0);  // several units a slot
    hipError_t e;
    if (wrong_bytes(r, 64, e) || e != hipSuccess) return printf("whole transfer: error %d\n", e), 1;
    long wrong = 0;
    for (int rep = 0; rep < 400; rep++) {
        fake.records = 0;
        fake.fail_wait_of = 16 + rep % 24;
        wrong += wrong_bytes(r, 64, e);
        if (e != hipErrorUnknown) return printf("the failed wait was not reported: %d\n", e), 1;
    }
    r.free();
    return wrong ? printf("%ld bytes of slots that were never filled\n", wrong), 1 : 0;
}

// every allocation that the device writes and the host reads is coherent whatever the environment's default
int coherent() {
    HostRing r;
    r.shape(96 * kUnit, 0);
    hipError_t e;
    if (wrong_bytes(r, 64, e) || e != hipSuccess) return 1;
    r.free();
    if (fake.host_allocs > 0 && (fake.host_flags & hipHostMallocCoherent)) return 0;
    return printf("flags %#x\n", fake.host_flags.load()), 1;
}

// pieces of 1 ms that helpers took
int by_helpers(HostRing& r) {
    std::atomic<int> others{0};
    gf::in_parts(r, 40, [&](long) {
        others += std::this_thread::get_id() != main_thread;
        usleep(1000);
    });
    return others;
}
// helpers that come 10 ms after they were called take nothing; the next ones that come at once do
int late_helper() {
    cpu_set_t set;
    if (sched_getaffinity(0, sizeof set, &set) == 0 && CPU_COUNT(&set) < 2) return 0;  // no helpers
    HostRing r;
    r.shape(96 * kUnit, 0);
    ahead_ns = 10000000;
    const int late = by_helpers(r);
    ahead_ns = 0;
    const int in_time = by_helpers(r);
    r.free();
    return late == 0 && in_time > 0 ? 0 : (printf("pieces taken late %d, in time %d\n", late, in_time), 1);
}

// a transfer too small to share calls no helper, also where another context has some waiting
int small_transfer() {
    HostRing helped, r;
    helped.shape(96 * kUnit, 0);
    r.shape(96 * kUnit, 0);
    (void)by_helpers(helped);
    usleep(20000);
    calls = 0;
    hipError_t e;
    const long wrong = wrong_bytes(r, 2, e);
    r.free();
    helped.free();
    return wrong == 0 && calls == 0 ? 0 : (printf("wrong %ld, helpers called %ld\n", wrong, calls.load()), 1);
}
// contexts on several threads, helpers started and ended all the while
int several_threads() {
    std::atomic<long> wrong{0};
    std::vector<std::thread> threads;
    for (int id = 0; id < 4; id++)
        threads.emplace_back([&wrong, id] {
            for (int rep = 0; rep < 40; rep++) {
                HostRing r;
                r.shape(96 * kUnit * (1 + rep % 3), 0);
                const long units = (long)(r.slot / kUnit) * (2 + (rep * 7 + id) % 40);
                std::vector<char> dev(units * kUnit), host(dev.size()), back(dev.size());
                for (size_t k = 0; k < dev.size(); k += 61) dev[k] = (char)(k * 31 + id + rep);
                auto off = [](long q) { return (size_t)q * kUnit; };
                hipError_t e = r.pull(host.data(), units, kUnit, off, [&](long q, long n, char* p) {
                    return memcpy(p, &dev[q * kUnit], n * kUnit), hipSuccess;
                }, nullptr);
                wrong += e != hipSuccess || host != dev;
                e = r.push(host.data(), units, kUnit, off, [&](long q, long n, const char* p) {
                    return memcpy(&back[q * kUnit], p, n * kUnit), hipSuccess;
                }, nullptr);
                wrong += e != hipSuccess || back != dev;
                std::vector<int> seen(50, 0);
                gf::in_parts(r, 50, [&](long k) { seen[k]++; });
                for (const int n : seen) wrong += n != 1;
                r.free();
            }
        });
    for (std::thread& t : threads) t.join();
    return wrong ? printf("%ld wrong\n", wrong.load()), 1 : 0;
}
// a signal to the process that the program has blocked stays pending: no helper takes it
int blocked_signal() {
    HostRing r;
    r.shape(96 * kUnit, 0);
    (void)by_helpers(r);
    sigset_t set;
    sigemptyset(&set);
    sigaddset(&set, SIGUSR1);
    pthread_sigmask(SIG_BLOCK, &set, nullptr);
    kill(getpid(), SIGUSR1);
    usleep(100000);
    sigpending(&set);
    r.free();
    return sigismember(&set, SIGUSR1) ? 0 : 1;
}
}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "failed_wait") return failed_wait();
    if (what == "coherent") return coherent();
    if (what == "late_helper") return late_helper();
    if (what == "blocked_signal") return blocked_signal();
    if (what == "small_transfer") return small_transfer();
    if (what == "several_threads") return several_threads();
    return printf("no scenario %s\n", what.c_str()), 2;
}
