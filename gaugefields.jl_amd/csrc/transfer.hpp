// transfer.hpp -- host arrays in and out of the device through a ring of pinned slots.
//
// A copy between the device and ordinary (pageable) memory runs at 10 GB/s where the array has just been
// allocated, as every array that is handed out has: the runtime's own staging is one thread's, and so are the
// page faults.  Here the layout kernels write to (read from) pinned memory across the link themselves, so nothing
// is staged on the device, and several threads copy between the slots and the caller's array while the kernels go
// on.  Download of the links, FP64 32^4 (604 MB) 58 -> 13 ms, 24^3x48 37 -> 8.6, 16^4 3.6 -> 1.0, 8^4 0.17 -> 0.13.
#pragma once
#include <pthread.h>
#include <sched.h>
#include <signal.h>
#include <time.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>

#include <hip/hip_runtime.h>

namespace gf {

// Pieces 0 .. total of one call's work; those below `limit` may be claimed, in order, by whoever is running.
struct Job {
    long total = 0, next = 0, limit = 0, active = 0;
    bool offered = false;  // to the helpers
    virtual void run(long i) = 0;       // outside the lock
    virtual void ran(long) {}           // inside it
    virtual ~Job() = default;
};

// Helper threads of the process, for the copies and checks of all contexts.  A call never waits for a helper to start:
// its own thread takes pieces like any other, and a helper that comes too late finds nothing to claim.  It does wait for
// a piece that a helper has claimed, and where the processors are taken (behind an OpenMP loop its threads go on
// spinning) the scheduler may take a helper off in the middle of one, or the caller off for a helper, for 3 ms.  So
// helpers are called one at a time, each by the one before it, and one that the scheduler brought late (kLate) takes
// nothing: where the processors are taken the call is mostly its own thread's.
// Links down behind an OpenMP loop of 16 threads on 16 processors, mean and 99th percentile in us, all seven called at
// once / one by one: 8^4 211-256, 2725-4028 / 132-151, 306-377 (without helpers, by the runtime's copy, 190, 697); 12^4
// 665-697, 4288-4419 / 569-663, 1261-1634 (725, 1349); 16^4 and larger means within 6 %.  What is computed and not only
// copied (the SU(3) check) gets less help there: links up 24^4 8.5 / 10.3 ms (19.8).  With the processors free the same:
// down 8^4 177 / 142 us, 12^4 423 / 430, 16^4 908 / 923, 24^4 4453 / 4368, 32^4 13.4 / 13.3 ms.  As SCHED_BATCH, which never
// takes the caller off for a helper: means 10-20 % longer from 16^4 on.
// (Threads started and joined by each call waited for the processors as well.)  Started when the first large array
// comes, ended when the last context that has used them is destroyed; none in a forked child, which has only the
// thread that forked.
class Helpers {
  public:
    static constexpr int kMax = 7;  // and the caller: 32^4 links with 8 threads 15.0 ms, four 15.4, two 25
    static constexpr long long kLate = 200 * 1000;  // ns from the call
    static Helpers& get() {
        static Helpers* const h = new Helpers;  // outlives every static destructor
        return *h;
    }
    void retain() {
        if (getpid() != pid_) return;
        std::lock_guard<std::mutex> start(life_);
        if (users_++ > 0) return;
        cpu_set_t set;
        const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
        pthread_attr_t at;
        if (pthread_attr_init(&at) != 0) return;
        (void)pthread_attr_setstacksize(&at, 2 << 20);
        sigset_t all, mask;  // the program's signals are for its own threads
        sigfillset(&all);
        for (const int own : {SIGSEGV, SIGBUS, SIGFPE, SIGILL, SIGTRAP}) sigdelset(&all, own);
        (void)pthread_sigmask(SIG_SETMASK, &all, &mask);
        while (n_ < std::min(kMax, cpus - 1) && pthread_create(&one_[n_].thread, &at, loop, &one_[n_]) == 0) n_++;
        (void)pthread_sigmask(SIG_SETMASK, &mask, nullptr);
        pthread_attr_destroy(&at);
    }
    void release() {
        if (getpid() != pid_) return;
        std::lock_guard<std::mutex> end(life_);
        if (--users_ > 0) return;
        {
            std::lock_guard<std::mutex> lk(m_);
            stop_ = true;
            for (One& o : one_) o.work.notify_one();
        }
        for (; n_ > 0; n_--) pthread_join(one_[n_ - 1].thread, nullptr);
        std::lock_guard<std::mutex> lk(m_);
        for (One& o : one_) o.called = 0;
        idle_ = 0;
        calling_ = stop_ = false;
    }

    // offers the job to the helpers (if there is room: a job that is not offered is its caller's alone)
    void open(Job& j) {
        std::lock_guard<std::mutex> lk(m_);
        for (Job*& p : jobs_)
            if (!p) {
                p = &j;
                j.offered = true;
                break;
            }
        call(j);
    }
    void allow(Job& j, long limit) {
        std::lock_guard<std::mutex> lk(m_);
        j.limit = limit;
        call(j);
    }
    // the calling thread takes a piece; false if there is none to claim
    bool step(Job& j) {
        std::unique_lock<std::mutex> lk(m_);
        return one(j, lk);
    }
    // waits until cond() holds, which the end of a piece of another thread may make true
    template <typename F>
    void wait(F cond) {
        std::unique_lock<std::mutex> lk(m_);
        done_.wait(lk, cond);
    }
    template <typename F>
    bool check(F cond) {
        std::lock_guard<std::mutex> lk(m_);
        return cond();
    }
    // no piece of the job is running or will be
    void close(Job& j) {
        std::unique_lock<std::mutex> lk(m_);
        for (Job*& p : jobs_)
            if (p == &j) p = nullptr;
        done_.wait(lk, [&] { return j.active == 0; });
    }

  private:
    struct One {
        pthread_t thread;
        std::condition_variable work;
        long long called = 0;  // when; 0: not
    };
    static long long now() {
        timespec t;
        clock_gettime(CLOCK_MONOTONIC, &t);
        return t.tv_sec * 1000000000ll + t.tv_nsec;
    }
    static bool claimable(const Job& j) { return j.next < std::min(j.limit, j.total); }
    // a helper, if there is a piece for it and none is on its way
    void call(const Job& j) {
        if (!j.offered || !claimable(j) || calling_ || idle_ == 0) return;
        One& o = *idle_at_[--idle_];
        o.called = now();
        calling_ = true;
        o.work.notify_one();
    }
    bool one(Job& j, std::unique_lock<std::mutex>& lk) {
        if (!claimable(j)) return false;
        const long i = j.next++;
        j.active++;
        call(j);
        lk.unlock();
        j.run(i);
        lk.lock();
        j.ran(i);
        j.active--;
        done_.notify_all();
        return true;
    }
    static void* loop(void* p) {
        Helpers& h = get();
        One& me = *(One*)p;
        std::unique_lock<std::mutex> lk(h.m_);
        while (!h.stop_) {
            h.idle_at_[h.idle_++] = &me;
            me.work.wait(lk, [&] { return h.stop_ || me.called != 0; });
            if (h.stop_) break;
            bool any = now() - me.called <= kLate;
            me.called = 0;
            h.calling_ = false;
            while (any) {
                any = false;
                for (Job*& j : h.jobs_)
                    if (j && h.one(*j, lk)) {
                        any = true;
                        break;
                    }
            }
        }
        return nullptr;
    }

    const pid_t pid_ = getpid();
    std::mutex life_, m_;
    std::condition_variable done_;
    Job* jobs_[8] = {};
    One one_[kMax];
    One* idle_at_[kMax];
    int idle_ = 0;
    bool calling_ = false;  // a helper that has been called has not come yet
    int n_ = 0, users_ = 0;
    bool stop_ = false;
};

// Host memory that kernels write and the host reads behind an event or a wait: coherent by name, as the default for
// it is the environment's (HIP_HOST_COHERENT).
inline hipError_t pin_alloc(void** p, size_t bytes) { return hipHostMalloc(p, bytes, hipHostMallocCoherent); }

constexpr int kSlots = 16;
constexpr size_t kSlotMin = 256 << 10, kSlotMax = 2 << 20, kUnitMax = 64 * 144;  // a group's links

struct HostRing {
    char* slot_at[kSlots] = {};  // pinned, as transfers come to need them
    char* piece[kSlots] = {};    // the allocations they lie in
    hipEvent_t ev[kSlots] = {};
    size_t slot = 0;  // bytes
    int device = 0;
    bool helped = false;

    // `most`: the largest transfer of the context.  A slot holds 1/32 of it, 256 KB to 2 MB: each costs a launch and
    // an event, 4 us during which the link is idle (512 KB slots 29 GB/s, 1 MB 43, 2 MB 48, 4 MB 50).
    void shape(size_t most, int dev) {
        device = dev;
        slot = most <= kSlotMin ? std::max(most, kUnitMax) : std::min(std::max(most / 32, kSlotMin), kSlotMax);
        slot = (slot + 4095) / 4096 * 4096;
    }
    // Slots that the context pins with its other host memory: all that a small lattice needs (up to 1 MB)
    int slots_at_hand(size_t most) const { return slot <= kSlotMin ? (int)std::min<size_t>(4, (most + slot - 1) / slot) : 0; }
    void adopt(char* p, int n) {
        for (int k = 0; k < n; k++) slot_at[k] = p + slot * k;
    }
    // Slots for a transfer of `chunks` slots: half of them, 4 to 16, as pinning takes about as long as copying,
    // and in one piece, as pinning any piece takes 0.3 ms; what there is if there is no more pinned memory, and 0 if
    // there is none at all (err).
    int slots_for(long chunks, hipError_t& err) {
        const int n = (int)std::min<long>(chunks, std::min<long>(std::max(chunks / 2, 4L), kSlots));
        int have = 0;
        while (have < kSlots && slot_at[have]) have++;
        for (int more = n - have; more > 0 && have < n; more = std::min(more / 2, n - have)) {
            char* p = nullptr;
            err = pin_alloc((void**)&p, slot * more);
            if (err != hipSuccess) {
                (void)hipGetLastError();
                continue;
            }
            piece[have] = p;
            for (int k = 0; k < more; k++) slot_at[have + k] = p + slot * k;
            have += more;
        }
        for (int k = 0; k < std::min(n, have); k++) {
            if (!ev[k]) err = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
            if (!ev[k]) return k;
        }
        return std::min(n, have);
    }
    void need_helpers() {
        if (!helped) Helpers::get().retain();
        helped = true;
    }
    void free() {
        if (helped) Helpers::get().release();
        helped = false;
        for (char*& p : piece) {
            if (p) (void)hipHostFree(p);
            p = nullptr;
        }
        for (char*& p : slot_at) p = nullptr;
        for (hipEvent_t& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    // One transfer: chunk i of `per` units goes through slot i % slots.
    template <typename O>
    struct Transfer : Job {
        HostRing& r;
        const O& offset;
        char* const host;
        const bool down;
        const long units, per;
        hipError_t err = hipSuccess;
        int slots;
        long last[kSlots];  // last chunk copied between the slot and the host array
        Transfer(HostRing& ring, char* h, bool d, long n, size_t unit_bytes, const O& o)
            : r(ring), offset(o), host(h), down(d), units(n), per((long)(ring.slot / unit_bytes)) {
            total = (units + per - 1) / per;
            slots = ring.slots_for(total, err);
            if (slots > 0) err = hipSuccess;
            for (long& k : last) k = -1;
        }
        char* at(long i) const { return r.slot_at[i % slots]; }
        bool copied(long i) const { return last[i % slots] == i; }
        void run(long i) override {
            if (down) {
                (void)hipSetDevice(r.device);
                const hipError_t e = hipEventSynchronize(r.ev[i % slots]);
                if (e != hipSuccess) {
                    Helpers::get().check([&] { return err = e, true; });
                    return;
                }
            }
            const size_t a = offset(i * per), b = offset(std::min(units, (i + 1) * per));
            if (down)
                memcpy(host + a, at(i), b - a);
            else
                memcpy(at(i), host + a, b - a);
        }
        void ran(long i) override { last[i % slots] = i; }
        template <typename F>
        hipError_t launch(long i, F f, hipStream_t st) {
            const hipError_t e = f(i * per, std::min(per, units - i * per), at(i));
            return e == hipSuccess ? hipEventRecord(r.ev[i % slots], st) : e;
        }
    };

    // Device to dst: `units` units, offset(q) = byte at which unit q starts (offset(units) the total), none longer
    // than unit_bytes <= slot.  fill(q0, n, p) puts the work on `st` that writes units q0 .. q0 + n to p.
    template <typename O, typename F>
    hipError_t pull(char* dst, long units, size_t unit_bytes, const O& offset, F fill, hipStream_t st) {
        Helpers& h = Helpers::get();
        Transfer<O> t(*this, dst, true, units, unit_bytes, offset);
        if (t.slots == 0) return t.err;
        const int slots = t.slots;
        const bool share = t.total >= 4;
        if (share) need_helpers();
        hipError_t e = hipSuccess;
        long issued = 0;
        bool open = false;
        for (;;) {
            // what has a free slot goes to the device
            while (e == hipSuccess && issued < t.total &&
                   (issued < slots || h.check([&] { return t.copied(issued - slots); })))
                e = t.launch(issued, fill, st), issued += e == hipSuccess;
            if (e != hipSuccess) break;
            if (!open && share) {
                // helpers come when there is something to copy; until then what was on the stream may take long
                e = hipEventSynchronize(ev[0]);
                if (e != hipSuccess) break;
                h.open(t);
                open = true;
            }
            h.allow(t, issued);
            if (h.check([&] { return t.err != hipSuccess; })) break;
            if (h.step(t)) continue;
            if (issued == t.total) break;
            h.wait([&] { return t.err != hipSuccess || t.copied(issued - slots); });
        }
        // after an error no chunk is claimed any more: what the slots hold is not its own
        h.check([&] {
            if (e == hipSuccess) e = t.err;
            if (e != hipSuccess) t.limit = 0;
            return true;
        });
        h.close(t);
        if (e == hipSuccess) e = t.err;
        if (e != hipSuccess) (void)hipStreamSynchronize(st);  // nothing writes to the slots any more
        return e;
    }

    // src to the device: drain(q0, n, p) puts the work on `st` that reads units q0 .. q0 + n from p.
    template <typename O, typename F>
    hipError_t push(const char* src, long units, size_t unit_bytes, const O& offset, F drain, hipStream_t st) {
        Helpers& h = Helpers::get();
        Transfer<O> t(*this, const_cast<char*>(src), false, units, unit_bytes, offset);
        if (t.slots == 0) return t.err;
        const int slots = t.slots;
        hipError_t e = hipSuccess;
        long issued = 0, freed = 0;  // chunks on the device's side, and those it has read
        t.limit = slots;
        if (t.total >= 4) {
            need_helpers();
            h.open(t);
        }
        while (issued < t.total) {
            if (h.check([&] { return t.copied(issued); })) {
                e = t.launch(issued, drain, st);
                if (e != hipSuccess) break;
                issued++;
                continue;
            }
            if (freed < issued && freed + slots < t.total) {
                e = hipEventQuery(ev[freed % slots]);
                if (e == hipErrorNotReady) {
                    (void)hipGetLastError();
                    if (h.step(t)) continue;
                    e = hipEventSynchronize(ev[freed % slots]);
                }
                if (e != hipSuccess) break;
                freed++;
                h.allow(t, freed + slots);
                continue;
            }
            if (!h.step(t)) h.wait([&] { return t.copied(issued); });
        }
        h.allow(t, 0);
        h.close(t);
        const hipError_t s = hipStreamSynchronize(st);
        return e != hipSuccess ? e : s;
    }
};

// f(k) for k = 0 .. parts - 1, by the caller and the helpers that ring `r` has
template <typename F>
void in_parts(HostRing& r, long parts, F f) {
    struct Parts : Job {
        F& f;
        explicit Parts(F& g) : f(g) {}
        void run(long i) override { f(i); }
    } j(f);
    j.total = j.limit = parts;
    Helpers& h = Helpers::get();
    if (parts > 1) {
        r.need_helpers();
        h.open(j);
    }
    while (h.step(j)) {
    }
    h.close(j);
}

}  // namespace gf
