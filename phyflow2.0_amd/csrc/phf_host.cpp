// phf_host.cpp -- host arrays in and out of a call (see phf_host.hpp).
//
// Results go to pageable arrays that the caller has just allocated.  The
// runtime's own copy to such memory moves 17 GB/s on the MI355X host, while
// the link does 55 GB/s into pinned memory: what is slow is one thread
// copying (and faulting in) the destination.  copy_out therefore lets the
// device write pinned slots and has up to kWorkers + 1 threads empty them.
#include "phf_host.hpp"

#include <atomic>
#include <chrono>
#include <cmath>
#include <memory>
#include <thread>

namespace phf {

// ---------------------------------------------------------------- workers --
namespace {

constexpr int kWorkers = 6;

struct Job {
    void (*fn)(void *, int);
    void *ctx;
    int n;
    std::atomic<int> next{0}, done{0};
    // takes tasks until none is left
    void work()
    {
        int mine = 0;
        for (int i; (i = next.fetch_add(1, std::memory_order_relaxed)) < n; ++mine) fn(ctx, i);
        if (mine) done.fetch_add(mine, std::memory_order_release);
    }
};

// Worker threads, started by the first job that can use them.  They look for
// jobs for some 100 us after one (calls come in bursts) and then sleep.  Never
// destroyed: they sleep until the process ends.
class Workers {
  public:
    static Workers &get()
    {
        static Workers *w = new Workers();
        return *w;
    }
    void add(const std::shared_ptr<Job> &job)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (!started_) start();
            jobs_.push_back(job);
            pending_.fetch_add(1, std::memory_order_release);
        }
        cv_.notify_all();
    }
    // takes the job, whose tasks are all taken, off the list and waits for them
    void finish(const std::shared_ptr<Job> &job)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (size_t i = 0; i < jobs_.size(); ++i)
                if (jobs_[i] == job) {
                    jobs_.erase(jobs_.begin() + (long)i);
                    break;
                }
            pending_.fetch_sub(1, std::memory_order_release);
        }
        while (job->done.load(std::memory_order_acquire) < job->n) std::this_thread::yield();
    }

  private:
    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<std::shared_ptr<Job>> jobs_;
    std::atomic<int> pending_{0};
    bool started_ = false;

    void start()
    {
        started_ = true;
        const unsigned hw = std::thread::hardware_concurrency();
        const int n = hw > 2 ? std::min<int>(kWorkers, (int)hw / 2) : 0;
        for (int i = 0; i < n; ++i) {
            try {
                std::thread([this] { loop(); }).detach();
            } catch (...) {
                break;  // the caller works alone
            }
        }
    }
    std::shared_ptr<Job> take()
    {
        std::lock_guard<std::mutex> lk(mu_);
        for (auto &j : jobs_)
            if (j->next.load(std::memory_order_relaxed) < j->n) return j;
        return nullptr;
    }
    void loop()
    {
        using clock = std::chrono::steady_clock;
        auto last = clock::now();
        for (;;) {
            std::shared_ptr<Job> j;
            if (pending_.load(std::memory_order_acquire) > 0) j = take();
            if (j) {
                j->work();
                last = clock::now();
            } else if (clock::now() - last < std::chrono::microseconds(100)) {
                std::this_thread::yield();
            } else {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [this] {
                    for (auto &q : jobs_)
                        if (q->next.load(std::memory_order_relaxed) < q->n) return true;
                    return false;
                });
                last = clock::now();
            }
        }
    }
};

}  // namespace

void host_parallel(int n, void (*fn)(void *, int), void *ctx)
{
    if (n <= 1) {
        if (n == 1) fn(ctx, 0);
        return;
    }
    std::shared_ptr<Job> job;
    try {
        job = std::make_shared<Job>();
        job->fn = fn;
        job->ctx = ctx;
        job->n = n;
        Workers::get().add(job);
    } catch (...) {  // no memory for it: the caller works alone
        for (int i = 0; i < n; ++i) fn(ctx, i);
        return;
    }
    job->work();
    Workers::get().finish(job);
}

// ------------------------------------------------------------- validation --
// Whether all of p[0..n) are finite: adding one to the exponent field carries
// into the sign place exactly for infinities and NaN, so the loop is three
// integer operations that vectorise.
static bool all_finite(const double *p, int64_t n)
{
    uint64_t acc = 0;
    for (int64_t i = 0; i < n; ++i) {
        uint64_t b;
        std::memcpy(&b, p + i, sizeof(b));
        acc |= (b & 0x7fffffffffffffffull) + 0x0010000000000000ull;
    }
    return (acc >> 63) == 0;
}

int check_host_array(const double *p, int64_t n, const char *name, bool finite)
{
    if (n > 0 && p == nullptr) {
        set_error("%s is NULL but has %lld entries", name, (long long)n);
        return PHF_ERR_INVALID;
    }
    if (!finite || n <= 0) return PHF_OK;
    constexpr int64_t kPart = 1 << 16;
    const int parts = (int)((n + kPart - 1) / kPart);
    std::atomic<bool> ok{true};
    auto part = [&](int k) {
        const int64_t lo = (int64_t)k * kPart;
        if (!all_finite(p + lo, std::min(kPart, n - lo))) ok = false;
    };
    if (parts <= 2)  // less than waking a thread costs
        for (int k = 0; k < parts; ++k) part(k);
    else
        host_parallel(parts, part);
    if (ok) return PHF_OK;
    for (int64_t i = 0; i < n; ++i)
        if (!std::isfinite(p[i])) {
            set_error("%s[%lld] is not finite", name, (long long)i);
            return PHF_ERR_INVALID;
        }
    return PHF_OK;
}

// ----------------------------------------------------------------- inputs --
// Largest total that is packed: a transfer costs some 8 us whatever its size,
// and the pack is one thread's copy.
static constexpr int64_t kPackBytes = 128 << 10;

// whether the lane has its staging (no memory left to pin: the runtime's copies)
static bool have_pin(Lane *L)
{
    if (L->pin.ensure(kPackBytes) == PHF_OK) return true;
    (void)hipGetLastError();
    clear_error();
    return false;
}

int copy_in(Lane *L, std::initializer_list<HostIn> in)
{
    int64_t total = 0;
    for (const HostIn &a : in) total += a.n > 0 ? a.n : 1;
    double *d;
    PHF_ALLOC(d, L->arena, double, (size_t)total);
    const bool pack = total * (int64_t)sizeof(double) <= kPackBytes && have_pin(L);
    double *pin = reinterpret_cast<double *>(L->pin.ptr);
    int64_t at = 0;
    for (const HostIn &a : in) {
        *a.dev = d + at;
        if (a.n > 0) {
            if (pack)
                std::memcpy(pin + at, a.host, sizeof(double) * a.n);
            else
                PHF_HIP(hipMemcpyAsync(d + at, a.host, sizeof(double) * a.n,
                                       hipMemcpyHostToDevice, L->stream));
        }
        at += a.n > 0 ? a.n : 1;
    }
    if (pack) {
        PHF_HIP(hipMemcpyAsync(d, pin, sizeof(double) * total, hipMemcpyHostToDevice, L->stream));
        PHF_TRY(L->pin.mark(L->stream));
    }
    return PHF_OK;
}

int copy_points_in(Lane *L, const double *xb, const double *yb, const double *wb, int64_t nb,
                   const double *xt, const double *yt, int64_t nt, double **dxb, double **dyb,
                   double **dwb, double **dxt, double **dyt)
{
    if (xt != xb || yt != yb || nt != nb)
        return copy_in(L, {{xb, nb, dxb}, {yb, nb, dyb}, {wb, nb, dwb}, {xt, nt, dxt}, {yt, nt, dyt}});
    PHF_TRY(copy_in(L, {{xb, nb, dxb}, {yb, nb, dyb}, {wb, nb, dwb}}));
    *dxt = *dxb;
    *dyt = *dyb;
    return PHF_OK;
}

// ---------------------------------------------------------------- results --
namespace {

constexpr size_t kSlot = size_t(1) << 20;  // bytes per transfer at most
constexpr int kSlots = 16;
constexpr size_t kTask = size_t(128) << 10;  // bytes per thread's copy
// Totals from which results go through a ring; the runtime's own copies are
// quicker below (three arrays of 720 KB in all: 59 against 70 us; 1.4 MB 89
// against 95; 2.9 MB 148 against 129; 24 MB 1,405 against 821 us, or 2,767
// against 980 into fresh memory).
constexpr size_t kRingBytes = size_t(2) << 20;

// Pinned slots with the events that end their transfers.  One ring exists in
// the process (16 MiB), made when first needed and kept.
struct Ring {
    char *ptr = nullptr;
    hipEvent_t ev[kSlots] = {};
    bool make()
    {
        bool ok = hipHostMalloc(reinterpret_cast<void **>(&ptr), kSlot * kSlots,
                                hipHostMallocDefault) == hipSuccess;
        for (int i = 0; ok && i < kSlots; ++i)
            ok = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            drop();
        }
        return ok;
    }
    void drop()
    {
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        if (ptr) (void)hipHostFree(ptr);
        *this = Ring();
    }
};

Ring g_ring;
std::atomic<int> g_fetches{0};  // results of kRingBytes or more under way

// The ring is for a fetch that is alone when it begins.  Threads that fetch at
// the same time have the runtime's copies side by side, each on its own core,
// and the workers only get in their way (four threads, 24 MB each: 2.4 ms a
// fetch by the runtime, 3.1 ms with a ring each, 3.0 with one ring for the
// first of them).
struct Fetch {
    const bool alone = g_fetches.fetch_add(1, std::memory_order_acq_rel) == 0;
    ~Fetch() { g_fetches.fetch_sub(1, std::memory_order_acq_rel); }
};

struct Piece {  // one transfer into a slot
    char *host;
    const char *dev;
    size_t bytes;
    int task0;  // first of its tasks
};

}  // namespace

int copy_out(Lane *L, std::initializer_list<HostOut> out)
{
    // events are made and recorded below, which takes the stream's own device
    DeviceScope ds;
    PHF_HIP(ds.err);
    size_t total = 0;
    for (const HostOut &o : out) total += o.bytes;
    auto plain = [&]() -> int {
        for (const HostOut &o : out)
            if (o.bytes)
                PHF_HIP(hipMemcpyAsync(o.host, o.dev, o.bytes, hipMemcpyDeviceToHost, L->stream));
        PHF_HIP(hipStreamSynchronize(L->stream));
        return PHF_OK;
    };
    if (total <= size_t(kPackBytes)) {
        if (!have_pin(L)) return plain();
        // neighbours in the arena come in one transfer; arrays that touch but are
        // allocations of their own must not
        size_t at = 0, run = 0;
        const char *from = nullptr;
        for (const HostOut &o : out) {
            const char *d = static_cast<const char *>(o.dev);
            if (run > 0 && (d != from + run || !L->arena.within_block(from, run + o.bytes))) {
                PHF_HIP(hipMemcpyAsync(L->pin.ptr + at, from, run, hipMemcpyDeviceToHost,
                                       L->stream));
                at += run;
                run = 0;
            }
            if (run == 0) from = d;
            run += o.bytes;
        }
        if (run > 0)
            PHF_HIP(hipMemcpyAsync(L->pin.ptr + at, from, run, hipMemcpyDeviceToHost, L->stream));
        PHF_HIP(hipStreamSynchronize(L->stream));
        at = 0;
        for (const HostOut &o : out) {
            if (o.bytes) std::memcpy(o.host, L->pin.ptr + at, o.bytes);
            at += o.bytes;
        }
        return PHF_OK;
    }
    if (total < kRingBytes) return plain();
    Fetch fetch;
    if (!fetch.alone || !(g_ring.ptr || g_ring.make())) return plain();
    const Ring ring = g_ring;
    std::vector<Piece> pc;
    std::vector<int> piece_of;  // of every task
    std::unique_ptr<std::atomic<int>[]> left;
    std::unique_ptr<std::atomic<bool>[]> sent;
    int ntask = 0;
    try {
        for (const HostOut &o : out)
            for (size_t at = 0; at < o.bytes; at += kSlot) {
                const size_t b = std::min(kSlot, o.bytes - at);
                pc.push_back({static_cast<char *>(o.host) + at,
                              static_cast<const char *>(o.dev) + at, b, ntask});
                ntask += (int)((b + kTask - 1) / kTask);
                piece_of.resize((size_t)ntask, (int)pc.size() - 1);
            }
        left.reset(new std::atomic<int>[pc.size()]);
        sent.reset(new std::atomic<bool>[pc.size()]);
    } catch (...) {  // no memory for the bookkeeping
        return plain();
    }
    const int np = (int)pc.size();
    std::atomic<int> err{(int)hipSuccess};
    auto send = [&](int p) {
        const Piece &q = pc[(size_t)p];
        hipError_t e = hipMemcpyAsync(ring.ptr + kSlot * (size_t)(p % kSlots), q.dev, q.bytes,
                                      hipMemcpyDeviceToHost, L->stream);
        if (e == hipSuccess) e = hipEventRecord(ring.ev[p % kSlots], L->stream);
        if (e != hipSuccess) err = (int)e;
        sent[(size_t)p].store(true, std::memory_order_release);
    };
    for (int p = 0; p < np; ++p) {
        left[(size_t)p] = (p + 1 < np ? pc[(size_t)p + 1].task0 : ntask) - pc[(size_t)p].task0;
        sent[(size_t)p] = false;
    }
    for (int p = 0; p < std::min(np, kSlots); ++p) send(p);
    const int dev = Context::get().device();
    // tasks are taken in order, so the ones that free a slot are always at
    // work before the ones that wait for it
    host_parallel(ntask, [&](int t) {
        const int p = piece_of[(size_t)t];
        const Piece &q = pc[(size_t)p];
        while (!sent[(size_t)p].load(std::memory_order_acquire)) std::this_thread::yield();
        if (err.load() == (int)hipSuccess) {
            const hipError_t e = hipEventSynchronize(ring.ev[p % kSlots]);
            if (e != hipSuccess) err = (int)e;
        }
        if (err.load() == (int)hipSuccess) {
            const size_t at = (size_t)(t - q.task0) * kTask;
            std::memcpy(q.host + at, ring.ptr + kSlot * (size_t)(p % kSlots) + at,
                        std::min(kTask, q.bytes - at));
        }
        if (left[(size_t)p].fetch_sub(1, std::memory_order_acq_rel) == 1 && p + kSlots < np) {
            (void)hipSetDevice(dev);
            send(p + kSlots);
        }
    });
    // nothing of the ring is in use afterwards, also after an error
    const hipError_t se = hipStreamSynchronize(L->stream);
    PHF_HIP((hipError_t)err.load());
    PHF_HIP(se);
    return PHF_OK;
}

}  // namespace phf
