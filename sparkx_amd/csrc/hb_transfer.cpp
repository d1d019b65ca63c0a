// hb_transfer.cpp -- copies between pageable host memory and the device.
//
// hipMemcpy of pageable memory touches every page of it from one thread; a result array
// fresh from the allocator is faulted in and zeroed page by page on the way, which takes
// longer than the bus: 134 MB of results of a 16.7M-node graph took 13.5 ms (10 GB/s).  Here
// the bytes pass through pinned slots: while the bus fills or empties some of them, a pool of
// host threads copies the others, each thread touching its own pages (the same 134 MB:
// 4.2 ms).  A call that finds the slots taken by another thread, a buffer that HIP knows
// (pinned, managed, device) and a short copy go straight to hipMemcpyAsync.
#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

#include "hb_kernels.h"

namespace hb {
namespace {

// Worker threads that run one job at a time, part k of it on worker k; kept for the life
// of the process.  A child of fork() has none of them and runs every part itself.
class Pool {
public:
    static Pool &get()
    {
        static Pool *p = new Pool();  // never destroyed: its threads may outlive static objects
        return *p;
    }
    unsigned parts() const { return getpid() == pid_ ? (unsigned)workers_ + 1 : 1; }
    // fn(k) for k < parts(), the last part on this thread; one caller at a time (the slots' lock)
    void run(const std::function<void(unsigned)> &fn)
    {
        const unsigned n = parts();
        if (n > 1) {
            std::lock_guard<std::mutex> lk(mu_);
            job_ = &fn;
            left_ = n - 1;
            ++round_;
        }
        if (n > 1) start_.notify_all();
        fn(n - 1);
        if (n > 1) {
            std::unique_lock<std::mutex> lk(mu_);
            done_.wait(lk, [&] { return left_ == 0; });
            job_ = nullptr;
        }
    }

private:
    Pool() : pid_(getpid())
    {
        const unsigned hw = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
        for (unsigned k = 0; k + 1 < hw; ++k) {
            try {
                std::thread([this, k] { work(k); }).detach();
            } catch (const std::system_error &) {
                break;  // as many as the system gives
            }
            ++workers_;
        }
    }
    void work(unsigned k)
    {
        uint64_t seen = 0;
        for (;;) {
            const std::function<void(unsigned)> *job;
            {
                std::unique_lock<std::mutex> lk(mu_);
                start_.wait(lk, [&] { return round_ != seen; });
                seen = round_;
                job = job_;
            }
            (*job)(k);
            std::lock_guard<std::mutex> lk(mu_);
            if (--left_ == 0) done_.notify_one();
        }
    }
    const pid_t pid_;
    unsigned workers_ = 0;
    std::mutex mu_;
    std::condition_variable start_, done_;
    const std::function<void(unsigned)> *job_ = nullptr;
    unsigned left_ = 0;
    uint64_t round_ = 0;
};

// Pinned slots shared by every transfer of the process, allocated on first use and kept to
// the end (pinning host pages costs milliseconds).
constexpr size_t kSlot = size_t(8) << 20;
constexpr int kSlots = 4;
std::mutex g_slots_mu;
char *g_slots = nullptr;

struct Slots {
    std::unique_lock<std::mutex> lock;
    hipEvent_t ev[kSlots] = {};
    bool ok = false;

    // events: whether slots will be reused or copied out of while others fill
    Slots(bool wait, bool events) : lock(g_slots_mu, std::defer_lock)
    {
        if (wait) lock.lock();
        else if (!lock.try_lock()) return;
        if (!g_slots && hipHostMalloc((void **)&g_slots, kSlot * kSlots, hipHostMallocPortable) != hipSuccess) {
            g_slots = nullptr;
            (void)hipGetLastError();
            return;
        }
        for (auto &e : ev)
            if (events && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return;
        ok = true;
    }
    ~Slots()
    {
        for (auto e : ev)
            if (e) (void)hipEventDestroy(e);
    }
    char *at(uint64_t k) const { return g_slots + (k % kSlots) * kSlot; }
};

// memory HIP allocated, which the bus reaches by itself
bool known_to_hip(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// [0, n) in parts, cut at multiples of `align`
std::pair<size_t, size_t> part_of(size_t n, unsigned k, unsigned parts, size_t align)
{
    const size_t per = ((n + parts - 1) / parts + align - 1) / align * align;
    const size_t a = std::min(n, per * k);
    return {a, std::min(n, a + per)};
}

// below this one hipMemcpyAsync is as fast: waking the pool four times takes some 0.1 ms (the
// accumulators of a 32-graph batch, up to 2 MiB each: 11.7 ms a pass through the pool, 10.5
// without; an 8 MiB array 0.40 ms, 0.64 without)
constexpr size_t kShort = size_t(4) << 20;

// count elements of `in` device bytes each, delivered to the host by put(slot, first, last)
hipError_t pull(Slots &sl, const void *src, size_t count, size_t in, hipStream_t s,
                const std::function<void(const char *, size_t, size_t)> &put)
{
    // at least four chunks, so that the bus and the threads overlap
    const size_t per = std::max<size_t>(1, std::min(kSlot / in, (count + 3) / 4));
    const size_t chunks = (count + per - 1) / per;
    auto fill = [&](size_t k) -> hipError_t {
        const size_t a = k * per, len = std::min(per, count - a);
        const hipError_t e = hipMemcpyAsync(sl.at(k), (const char *)src + a * in, len * in, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipEventRecord(sl.ev[k % kSlots], s);
    };
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < std::min<size_t>(chunks, kSlots) && e == hipSuccess; ++k) e = fill(k);
    Pool &pool = Pool::get();
    for (size_t k = 0; k < chunks && e == hipSuccess; ++k) {
        e = hipEventSynchronize(sl.ev[k % kSlots]);
        if (e != hipSuccess) break;
        const size_t a = k * per, len = std::min(per, count - a);
        const unsigned parts = pool.parts();
        pool.run([&](unsigned p) {
            const auto r = part_of(len, p, parts, 4096 / in);
            if (r.first < r.second) put(sl.at(k) + r.first * in, a + r.first, a + r.second);
        });
        if (k + kSlots < chunks) e = fill(k + kSlots);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing still writes the slots
    return e;
}

}  // namespace

hipError_t read_back(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    if (bytes >= kShort && !known_to_hip(dst)) {
        Slots sl(false, true);
        if (sl.ok)
            return pull(sl, src, bytes, 1, s, [&](const char *from, size_t a, size_t b) {
                memcpy((char *)dst + a, from, b - a);
            });
    }
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipStreamSynchronize(s);
}

hipError_t read_back_u64(uint64_t *dst, const uint32_t *src, size_t count, hipStream_t s)
{
    Slots sl(true, true);
    if (!sl.ok) {  // no pinned memory: through an ordinary buffer
        std::vector<uint32_t> tmp(count);
        hipError_t e = hipMemcpyAsync(tmp.data(), src, count * 4, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess)
            for (size_t i = 0; i < count; ++i) dst[i] = tmp[i];
        return e;
    }
    return pull(sl, src, count, 4, s, [&](const char *from, size_t a, size_t b) {
        const uint32_t *f = (const uint32_t *)from;
        for (size_t i = a; i < b; ++i) dst[i] = f[i - a];
    });
}

hipError_t upload_by(void *dst, size_t count, size_t out, hipStream_t s,
                     const std::function<bool(char *, size_t, size_t)> &get, bool *refused)
{
    *refused = false;
    const bool small = count * out < kShort;  // one slot, not worth waking the pool
    Slots sl(true, !small);
    if (!sl.ok) return hipErrorOutOfMemory;
    const size_t per = std::max<size_t>(1, small ? count : std::min(kSlot / out, (count + 3) / 4));
    const size_t chunks = (count + per - 1) / per;
    Pool &pool = Pool::get();
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < chunks && e == hipSuccess && !*refused; ++k) {
        if (k >= kSlots) e = hipEventSynchronize(sl.ev[k % kSlots]);
        if (e != hipSuccess) break;
        const size_t a = k * per, len = std::min(per, count - a);
        const unsigned parts = small ? 1 : pool.parts();
        std::vector<char> bad(parts, 0);
        const std::function<void(unsigned)> job = [&](unsigned p) {
            const auto r = part_of(len, p, parts, 64);
            if (r.first < r.second) bad[p] = !get(sl.at(k) + r.first * out, a + r.first, a + r.second);
        };
        if (small) job(0);
        else pool.run(job);
        for (char b : bad) *refused = *refused || b;
        if (*refused) break;
        e = hipMemcpyAsync((char *)dst + a * out, sl.at(k), len * out, hipMemcpyHostToDevice, s);
        if (e == hipSuccess && !small) e = hipEventRecord(sl.ev[k % kSlots], s);
    }
    const hipError_t w = hipStreamSynchronize(s);  // no copy still reads the slots
    return e != hipSuccess ? e : w;
}

hipError_t upload(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    if (bytes >= kShort && !known_to_hip(src)) {
        bool refused;
        const hipError_t e = upload_by(
            dst, bytes, 1, s,
            [&](char *to, size_t a, size_t b) {
                memcpy(to, (const char *)src + a, b - a);
                return true;
            },
            &refused);
        if (e != hipErrorOutOfMemory) return e;
    }
    return bytes ? hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, s) : hipSuccess;
}

void host_parallel(size_t count, const std::function<void(size_t, size_t)> &fn)
{
    if (count < (size_t(1) << 16)) return fn(0, count);
    std::lock_guard<std::mutex> lock(g_slots_mu);  // the pool's one job at a time
    Pool &pool = Pool::get();
    const unsigned parts = pool.parts();
    pool.run([&](unsigned p) {
        const auto r = part_of(count, p, parts, 512);
        if (r.first < r.second) fn(r.first, r.second);
    });
}

}  // namespace hb
