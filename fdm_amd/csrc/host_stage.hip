// Host arrays to and from the device through pinned memory.
//
// The drop-in classes solve on the caller's host arrays, which are pageable.
// The runtime's own copies of such memory run far below the link: 16 MiB takes
// 452 us in and 941 us out against 302 us for pinned memory, and a 127^3 FP64
// solve between them 50 us.  What holds them back is the host side, one thread
// moving pages in step with the link.  Here a few threads move 512 KiB pieces
// between the caller's array and pinned memory while the copy engine moves what
// is ready: a 127^3 FP64 host solve 1500 -> 870 us.  Arrays the caller has pinned
// do not come here: the runtime copies them at the link's rate (the same solve 658
// us by its copies, 860 through the stage).
// A copy of the engine costs about 9 us beside its bytes (16 copies of 1 MiB 440
// us, one of 16 MiB 293), so its copies are few and grow from 1 MiB (in: it starts
// early) or shrink to 1 MiB (out: little is left to move when it ends).
//
// One stage per device, shared by the plans that use it: 32 MiB of pinned
// memory, in two halves that alternate in longer copies, and kWorkers threads
// that sleep between copies (a thread spins for kSpin before it sleeps, which
// covers the time between a solve's two copies).  A stage serves one copy at a
// time; a second thread's copy is refused and goes the runtime's way.
#include "host_stage.hpp"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace fdmgpu {

namespace {
constexpr size_t kMiB = (size_t)1 << 20;
constexpr size_t kPiece = kMiB / 2;         // a thread's share
constexpr size_t kHalf = 16 * kMiB;         // pinned bytes of one half: the longest part of a copy
constexpr int kGroups = 5, kWorkers = 6;
constexpr size_t kGroupEnd[2][kGroups] = {  // the engine's copies of a part, in and out
    {1 * kMiB, 2 * kMiB, 4 * kMiB, 8 * kMiB, 16 * kMiB},
    {8 * kMiB, 12 * kMiB, 14 * kMiB, 15 * kMiB, 16 * kMiB}};
constexpr std::chrono::microseconds kSpin{200};

int group_of(int dir, size_t off) {
    int g = 0;
    while (off >= kGroupEnd[dir][g]) ++g;
    return g;
}
size_t group_begin(int dir, int g) { return g ? kGroupEnd[dir][g - 1] : 0; }
}  // namespace

class HostStage {
  public:
    explicit HostStage(int device) : device_(device) {}
    ~HostStage() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
            job_no_.fetch_add(1);
        }
        cv_.notify_all();
        for (std::thread& t : workers_) t.join();
        (void)hipSetDevice(device_);
        // (whoever drops the last reference has synchronized the device: no copy
        // is in flight)
        for (Half& h : half_) {
            for (hipEvent_t e : h.ev)
                if (e) (void)hipEventDestroy(e);
            if (h.mem) (void)hipHostFree(h.mem);
        }
    }

    bool init() {
        // allocating is no offence to a capture that another thread has open
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return false;
        const bool ok = allocate();
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (!ok) return false;
        try {
            for (int i = 0; i < kWorkers; ++i) workers_.emplace_back([this] { work(); });
        } catch (...) {
            return false;   // the destructor joins those that started
        }
        return true;
    }

    hipError_t in(char* dst, const char* src, size_t bytes, hipStream_t s) {
        std::unique_lock<std::mutex> busy(busy_, std::try_to_lock);
        if (!busy) return hipErrorNotReady;
        for (size_t at = 0; at < bytes; at += kHalf) {
            Half& h = half_[(at / kHalf) & 1];
            const size_t n = bytes - at < kHalf ? bytes - at : kHalf;
            hipError_t e = settle(h, kGroups - 1);   // its last part has left
            if (e != hipSuccess) return e;
            std::atomic<size_t> left[kGroups];
            for (int g = 0; g < kGroups; ++g) {
                const size_t lo = group_begin(0, g), hi = kGroupEnd[0][g] < n ? kGroupEnd[0][g] : n;
                left[g].store(hi > lo ? hi - lo : 0);
            }
            e = run(n, [&](size_t off, size_t len) {
                std::memcpy(h.mem + off, src + at + off, len);
                const int g = group_of(0, off);
                if (left[g].fetch_sub(len) != len) return hipSuccess;
                // the group's last piece: off it goes
                const size_t lo = group_begin(0, g), hi = kGroupEnd[0][g] < n ? kGroupEnd[0][g] : n;
                return hipMemcpyAsync(dst + at + lo, h.mem + lo, hi - lo, hipMemcpyHostToDevice, s);
            });
            const hipError_t m = mark(h, kGroups - 1, s);   // also after a failure: some copies may be under way
            if (e != hipSuccess || m != hipSuccess) return e != hipSuccess ? e : m;
        }
        return hipSuccess;
    }

    hipError_t out(char* dst, const char* src, size_t bytes, hipStream_t s) {
        std::unique_lock<std::mutex> busy(busy_, std::try_to_lock);
        if (!busy) return hipErrorNotReady;
        auto part = [&](size_t at) { return bytes - at < kHalf ? bytes - at : kHalf; };
        auto fetch = [&](size_t at) -> hipError_t {
            if (at >= bytes) return hipSuccess;
            Half& h = half_[(at / kHalf) & 1];
            const size_t n = part(at);
            hipError_t e = settle(h, kGroups - 1);
            for (int g = 0; g < kGroups && e == hipSuccess; ++g) {
                const size_t lo = group_begin(1, g), hi = kGroupEnd[1][g] < n ? kGroupEnd[1][g] : n;
                if (hi > lo) e = hipMemcpyAsync(h.mem + lo, src + at + lo, hi - lo, hipMemcpyDeviceToHost, s);
                if (e == hipSuccess && (hi > lo || g == kGroups - 1)) e = mark(h, g, s);
            }
            return e;
        };
        hipError_t e = fetch(0);
        if (e == hipSuccess) e = fetch(kHalf);
        for (size_t at = 0; at < bytes && e == hipSuccess; at += kHalf) {
            Half& h = half_[(at / kHalf) & 1];
            e = run(part(at), [&](size_t off, size_t len) {
                const hipError_t w = settle(h, group_of(1, off));
                if (w == hipSuccess) std::memcpy(dst + at + off, h.mem + off, len);
                return w;
            });
            if (e == hipSuccess) e = fetch(at + 2 * kHalf);
        }
        return e;
    }

  private:
    struct Half {
        char* mem = nullptr;
        hipEvent_t ev[kGroups] = {};   // group g's copy; the last: the whole part's
        bool used[kGroups] = {};
    };

    bool allocate() {
        if (hipSetDevice(device_) != hipSuccess) return false;
        for (Half& h : half_) {
            if (hipHostMalloc((void**)&h.mem, kHalf, hipHostMallocDefault) != hipSuccess) {
                h.mem = nullptr;
                return false;
            }
            for (hipEvent_t& e : h.ev)
                if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                    e = nullptr;
                    return false;
                }
        }
        return true;
    }

    // The copies enqueued so far (mark) are complete (settle).  Marks are made by
    // the calling thread between runs only.
    static hipError_t mark(Half& h, int g, hipStream_t s) {
        h.used[g] = true;
        return hipEventRecord(h.ev[g], s);
    }
    static hipError_t settle(const Half& h, int g) { return h.used[g] ? hipEventSynchronize(h.ev[g]) : hipSuccess; }

    using Step = std::function<hipError_t(size_t offset, size_t bytes)>;

    void drain() {
        for (;;) {
            const size_t off = next_.fetch_add(kPiece), all = bytes_.load();
            if (off >= all) return;
            if (error_.load() == hipSuccess) {   // after a failure the pieces are only counted
                const size_t n = all - off < kPiece ? all - off : kPiece;
                const hipError_t e = step_(off, n);
                if (e != hipSuccess) error_.store(e);
            }
            left_.fetch_sub(1);
        }
    }

    // step(off, n) for every piece of `bytes`, by the workers and this thread
    hipError_t run(size_t bytes, Step step) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            step_ = std::move(step);
            error_.store(hipSuccess);
            left_.store((bytes + kPiece - 1) / kPiece);
            next_.store(0);
            bytes_.store(bytes);
            job_no_.fetch_add(1);
        }
        cv_.notify_all();
        drain();
        // every worker is out of the job before its description goes: those in
        // it, and one that saw it just before it was closed
        while (left_.load() > 0) std::this_thread::yield();
        {
            std::lock_guard<std::mutex> lk(mu_);
            bytes_.store(0);
        }
        while (in_job_.load() > 0) std::this_thread::yield();
        return error_.load();
    }

    void work() {
        (void)hipSetDevice(device_);
        unsigned long seen = 0;
        for (;;) {
            const auto until = std::chrono::steady_clock::now() + kSpin;
            while (job_no_.load() == seen && std::chrono::steady_clock::now() < until) std::this_thread::yield();
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return job_no_.load() != seen; });
                if (stop_) return;
                seen = job_no_.load();
                if (bytes_.load() == 0) continue;   // the job is over
                in_job_.fetch_add(1);
            }
            drain();
            in_job_.fetch_sub(1);
        }
    }

    const int device_;
    Half half_[2];
    std::vector<std::thread> workers_;
    std::mutex busy_;   // one copy at a time
    std::mutex mu_;     // the job's description
    std::condition_variable cv_;
    bool stop_ = false;
    std::atomic<unsigned long> job_no_{0};
    Step step_;
    std::atomic<size_t> bytes_{0}, next_{0}, left_{0};
    std::atomic<int> in_job_{0};
    std::atomic<hipError_t> error_{hipSuccess};
};

std::shared_ptr<HostStage> host_stage(int device, bool create) {
    constexpr int kDevices = 64;
    static std::mutex mu;
    static std::weak_ptr<HostStage> stages[kDevices];
    if (device < 0 || device >= kDevices) return nullptr;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<HostStage> st = stages[device].lock();
    if (st || !create) return st;
    try {
        st = std::make_shared<HostStage>(device);
        if (!st->init()) return nullptr;
    } catch (...) {
        return nullptr;
    }
    stages[device] = st;
    return st;
}

// (the job's description may allocate: out of memory, the copy goes the runtime's way)
hipError_t stage_in(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s) {
    try {
        return st.in((char*)dst, (const char*)src, bytes, s);
    } catch (...) {
        return hipErrorNotReady;
    }
}
hipError_t stage_out(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s) {
    try {
        return st.out((char*)dst, (const char*)src, bytes, s);
    } catch (...) {
        return hipErrorNotReady;
    }
}

}  // namespace fdmgpu
