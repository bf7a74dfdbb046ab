// Page-locked host memory and the words in it through which launches tell the host that they are done.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <memory>

#include "kernels.h"

namespace fynhip {

// Blocks of page-locked memory, kept for the next user instead of being locked and released every time (locking 25 MB
// takes milliseconds, a transfer of them half of one).  Shared by all networks and threads of the process.  Results are
// put into it only while less than kBytes are locked (networks' own staging areas are not refused), and what nobody has
// on loan goes back to the system when room is needed and with the last network.
class HostPool {
  public:
    static constexpr size_t kBytes = size_t(512) << 20;
    static void* acquire(size_t bytes, bool bounded, bool filled_by_host = false);   // bounded: null when the pool is full or there is no GPU; else throws when memory cannot be had
    static void release(void* p);                       // null is nothing
    static void release_then(void* p, const unsigned* flag, unsigned value);   // when the word `flag` reads `value` (HostSignal); nothing else may use the block any more by now
    static void forget(const unsigned* flag);           // the word goes away: blocks that wait for it are free
    static bool contains(const void* p, size_t bytes);  // whether the range lies inside a block on loan
    static void network_created();
    static void network_gone();
};


// Copies between host buffers, shared with a few helper threads of the process when they are large: one core moves 20 to
// 40 GB/s of memory that no cache holds, less than the link to the GPU takes (55 GB/s); four move 100.  The copies are
// done in the order in which they were added, so that what depends on the first ones can start early.  Waking a helper
// takes 20 to 50 us and pulls the caller's buffer into another core's cache: a single call shares 8 MB and more, a
// pipeline, where the copies are what the frames wait for, 1 MB.
class HostCopy {
  public:
    HostCopy();
    ~HostCopy();   // (all copies have been made then)
    void add(void* dst, const void* src, size_t bytes);
    size_t mark() const;       // for upto(): the copies added so far
    char* end_of(size_t mark) const;   // where the last of these copies ends in its target
    void start(size_t alone = 8u << 20);   // all copies have been added; fewer bytes than `alone` are not shared
    void upto(size_t mark);    // returns when these copies have been made, having done its share

  private:
    struct Job;
    std::shared_ptr<Job> job_;
    size_t seen_ = 0;
    friend struct HostCopyHelpers;
};

// One stream's word.
class HostSignal {
  public:
    void create(unsigned* counter);   // a word of device memory that is zero
    void destroy();
    HostDone next();                           // for the next launch on the stream
    // Returns when the launch that was given `value`, and so everything in front of it on the stream, has been carried
    // out.  Polls for a while, then leaves the waiting to the runtime, which also reports a failed launch.
    void wait(unsigned value, hipStream_t s) const;
    bool reached(unsigned value) const;   // whether that is so already (any thread)
    unsigned last() const { return value_; }
    FeedWord* feed() const { return reinterpret_cast<FeedWord*>(reinterpret_cast<char*>(flag_) + kFeed); }   // another word beside it, zero at first
    void release_then(void* block, unsigned value) const { HostPool::release_then(block, flag_, value); }

  private:
    static constexpr size_t kFeed = 128;   // (words that the GPU and the host write lie in lines of their own)
    unsigned* flag_ = nullptr;
    unsigned* counter_ = nullptr;
    unsigned value_ = 0;
};

// A block on loan for a scope.  Where launches read or write it, the scope ends the host's use of it and the last of them
// the GPU's: the block is the pool's again when both have.
class HostLoan {
  public:
    HostLoan() = default;
    explicit HostLoan(size_t bytes, bool filled_by_host = false) : p_(HostPool::acquire(bytes, false, filled_by_host)), frame_(filled_by_host) {}
    HostLoan(HostLoan&& o) noexcept : p_(o.p_), frame_(o.frame_), signal_(o.signal_), value_(o.value_) { o.p_ = nullptr; }
    HostLoan(const HostLoan&) = delete;
    HostLoan& operator=(const HostLoan&) = delete;
    ~HostLoan() {
        // (the area of a frame waits for the next one: it does not go back to the system here, however full the pool is)
        if (signal_ && (frame_ || !signal_->reached(value_))) signal_->release_then(p_, value_);
        else HostPool::release(p_);
    }
    void used_until(const HostSignal& s, unsigned value) { signal_ = &s; value_ = value; }   // by the launch that was given `value`
    float* floats() const { return static_cast<float*>(p_); }

  private:
    void* p_ = nullptr;
    bool frame_ = false;
    const HostSignal* signal_ = nullptr;
    unsigned value_ = 0;
};

// What HIP knows of a buffer of the caller's: memory of the host's that it knows nothing of, page-locked or managed memory
// (which work on a stream may be using), device memory.
enum class Memory { Pageable, PageLocked, Device };
Memory memory_of(const void* p);
inline bool host_memory(const void* p) { return memory_of(p) != Memory::Device; }   // the host can read and write it itself

}  // namespace fynhip
