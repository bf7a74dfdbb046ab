// Page-locked host memory pool and host-polled completion words.
#include "host_io.h"

#include <immintrin.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "engine.h"

namespace fynhip {

namespace {
struct Block {
    size_t bytes;
    bool lent;
    const unsigned* flag;   // lent until this word reads `value`, null: until it is given back
    unsigned value;
    bool filled_by_host;    // what it was used for last
};
bool told(const unsigned* flag, unsigned value) {   // (values pass in rising order; the difference survives the wrap-around)
    return (int)(__atomic_load_n(flag, __ATOMIC_ACQUIRE) - value) >= 0;
}
bool idle(Block& b) {
    if (b.flag && told(b.flag, b.value)) {
        b.flag = nullptr;
        b.lent = false;
    }
    return !b.lent;
}
std::mutex g_pool_mu;
std::map<char*, Block> g_blocks;   // by address
size_t g_pool_bytes = 0;
int g_networks = 0;

size_t size_class(size_t bytes) {   // sizes in steps of an eighth of the next power of two, so that like sizes share blocks
    size_t step = 4096;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}
// The pool's lock.  The runtime is not called under it: locking and releasing memory may wait for the GPU, and what the
// GPU waits for (a frame that another thread is copying) may need the lock.
class PoolLock {
  public:
    PoolLock() { g_pool_mu.lock(); }
    ~PoolLock() { unlock(); }
    PoolLock(const PoolLock&) = delete;
    PoolLock& operator=(const PoolLock&) = delete;
    void give_back_idle() {   // (when the lock is left)
        for (auto it = g_blocks.begin(); it != g_blocks.end();) {
            if (!idle(it->second)) {
                ++it;
                continue;
            }
            g_pool_bytes -= it->second.bytes;
            freed_.push_back(it->first);
            it = g_blocks.erase(it);
        }
    }
    void lock() { g_pool_mu.lock(); }
    void unlock() {
        g_pool_mu.unlock();
        for (char* p : freed_) (void)hipHostFree(p);
        freed_.clear();
    }

  private:
    std::vector<char*> freed_;
};
}  // namespace

void* HostPool::acquire(size_t bytes, bool bounded, bool filled_by_host) {
    const size_t want = size_class(bytes ? bytes : 1);
    PoolLock lk;
    // (a block that served the same purpose before: the host's copy into one that the host has written lately finds its
    // lines in the caches -- 3.8 MB in 60 us, against 90 into one that the GPU has written)
    std::pair<char* const, Block>* pick = nullptr;
    for (auto& kv : g_blocks)
        if (kv.second.bytes == want && idle(kv.second) && (!pick || pick->second.filled_by_host != filled_by_host)) pick = &kv;
    if (pick) {
        pick->second.lent = true;
        pick->second.filled_by_host = filled_by_host;
        return pick->first;
    }
    if (bounded && g_networks == 0) return nullptr;
    if (g_pool_bytes + want > kBytes) {
        lk.give_back_idle();
        if (bounded && g_pool_bytes + want > kBytes) return nullptr;
    }
    g_pool_bytes += want;   // (taken before the lock is left)
    lk.unlock();
    void* p = nullptr;
    const hipError_t e = hipHostMalloc(&p, want, hipHostMallocPortable);
    lk.lock();
    if (e != hipSuccess) {
        (void)hipGetLastError();
        g_pool_bytes -= want;
        if (bounded) return nullptr;
        fail(FYN_ERR_DEVICE, "no page-locked memory (%zu bytes): %s", want, hipGetErrorString(e));
    }
    g_blocks[static_cast<char*>(p)] = Block{want, true, nullptr, 0, filled_by_host};
    return p;
}

void HostPool::release(void* p) {
    if (!p) return;
    PoolLock lk;
    auto it = g_blocks.find(static_cast<char*>(p));
    if (it == g_blocks.end() || !it->second.lent) return;
    it->second.lent = false;
    if (g_networks == 0 || g_pool_bytes > kBytes) lk.give_back_idle();
}

void HostPool::release_then(void* p, const unsigned* flag, unsigned value) {
    PoolLock lk;
    auto it = g_blocks.find(static_cast<char*>(p));
    if (it == g_blocks.end()) return;
    it->second.flag = flag;
    it->second.value = value;
}

void HostPool::forget(const unsigned* flag) {
    PoolLock lk;
    for (auto& kv : g_blocks)
        if (kv.second.flag == flag) {
            kv.second.flag = nullptr;
            kv.second.lent = false;
        }
}

bool HostPool::contains(const void* p, size_t bytes) {
    PoolLock lk;
    char* c = const_cast<char*>(static_cast<const char*>(p));
    auto it = g_blocks.upper_bound(c);
    if (it == g_blocks.begin()) return false;
    --it;
    return it->second.lent && c + bytes <= it->first + it->second.bytes;
}

void HostPool::network_created() {
    PoolLock lk;
    g_networks++;
}
void HostPool::network_gone() {
    PoolLock lk;
    if (--g_networks == 0) lk.give_back_idle();
}

void HostSignal::create(unsigned* counter) {
    counter_ = counter;
    flag_ = static_cast<unsigned*>(HostPool::acquire(kFeed + sizeof(FeedWord), false));
    *flag_ = value_ = 0;
    *feed() = FeedWord{};
}
void HostSignal::destroy() {
    if (flag_) HostPool::forget(flag_);
    HostPool::release(flag_);
    flag_ = nullptr;
}
HostDone HostSignal::next() { return HostDone{counter_, flag_, ++value_}; }

bool HostSignal::reached(unsigned value) const {
    return told(flag_, value);
}

void HostSignal::wait(unsigned value, hipStream_t s) const {
    auto done = [&] { return reached(value); };
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 1; !done(); i++) {
        _mm_pause();
        if (i % 256 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2)) {
            FYN_HIP(hipStreamSynchronize(s));
            if (!done()) fail(FYN_ERR_DEVICE, "a launch ended without telling so");
            return;
        }
    }
}

// ---- copies ----
struct HostCopy::Job {
    struct Slice {
        char* dst;
        const char* src;
        size_t bytes;
    };
    std::vector<Slice> slices;
    size_t bytes = 0;
    std::unique_ptr<std::atomic<char>[]> made;
    std::atomic<size_t> next{0};
    bool one() {   // makes the next copy; false: all have been taken
        const size_t i = next.fetch_add(1, std::memory_order_relaxed);
        if (i >= slices.size()) return false;
        memcpy(slices[i].dst, slices[i].src, slices[i].bytes);
        made[i].store(1, std::memory_order_release);
        return true;
    }
};

// The helper threads.  They sleep while there is nothing to copy; the object is never destroyed, so that they may be
// asleep in it when the process ends.
struct HostCopyHelpers {
    static constexpr size_t kSlice = 256u << 10;
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::shared_ptr<HostCopy::Job>> jobs;
    const unsigned count = std::min(3u, std::thread::hardware_concurrency() / 4);
    HostCopyHelpers() {
        for (unsigned i = 0; i < count; i++) std::thread([this] { work(); }).detach();
    }
    static HostCopyHelpers& get() {
        static HostCopyHelpers* h = new HostCopyHelpers;
        return *h;
    }
    void offer(const std::shared_ptr<HostCopy::Job>& job) {
        if (!count) return;   // (few CPUs: nobody would take it from the queue)
        {
            std::lock_guard<std::mutex> lk(mu);
            jobs.push_back(job);
        }
        cv.notify_all();
    }
    void work() {
        for (;;) {
            std::shared_ptr<HostCopy::Job> job;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [this] { return !jobs.empty(); });
                job = jobs.front();
                if (job->next.load(std::memory_order_relaxed) >= job->slices.size()) {
                    jobs.pop_front();
                    continue;
                }
            }
            while (job->one()) {
            }
        }
    }
};

HostCopy::HostCopy() : job_(std::make_shared<Job>()) {}
HostCopy::~HostCopy() {
    if (job_->made) upto(mark());
}
void HostCopy::add(void* dst, const void* src, size_t bytes) {
    for (size_t o = 0; o < bytes; o += HostCopyHelpers::kSlice)
        job_->slices.push_back({static_cast<char*>(dst) + o, static_cast<const char*>(src) + o, std::min(HostCopyHelpers::kSlice, bytes - o)});
    job_->bytes += bytes;
}
size_t HostCopy::mark() const { return job_->slices.size(); }
char* HostCopy::end_of(size_t mark) const { return job_->slices[mark - 1].dst + job_->slices[mark - 1].bytes; }
void HostCopy::start(size_t alone) {
    job_->made.reset(new std::atomic<char>[job_->slices.size()]());
    if (job_->bytes >= alone) HostCopyHelpers::get().offer(job_);
}
void HostCopy::upto(size_t mark) {
    for (;;) {
        while (seen_ < mark && job_->made[seen_].load(std::memory_order_acquire)) seen_++;
        if (seen_ >= mark) return;
        if (!job_->one()) _mm_pause();
    }
}

Memory memory_of(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return Memory::Pageable;
    }
    if (a.type == hipMemoryTypeDevice) return Memory::Device;
    return a.type == hipMemoryTypeUnregistered ? Memory::Pageable : Memory::PageLocked;
}

}  // namespace fynhip
