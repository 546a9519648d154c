#include "staging.h"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <stdexcept>
#include <string>

namespace bnn {

static void hip_check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

namespace {
// Another device is the calling thread's current one for a while.
class OnDevice {
   public:
    explicit OnDevice(int device) {
        hip_check(hipGetDevice(&before_), "hipGetDevice");
        if (before_ == device) return;
        hip_check(hipSetDevice(device), "hipSetDevice");
        changed_ = true;
    }
    ~OnDevice() {
        if (changed_) (void)hipSetDevice(before_);
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;

   private:
    int before_ = 0;
    bool changed_ = false;
};
}  // namespace

void *copy_stream(int device) {
    static std::mutex mutex;
    static auto &streams = *new std::map<int, hipStream_t>;  // never destroyed: a blob may be read while the process ends
    std::lock_guard<std::mutex> lock(mutex);
    hipStream_t &s = streams[device];
    if (!s) {
        const OnDevice on(device);
        hip_check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
    }
    return s;
}

void *ShareStreams::begin(size_t most) {
    share_ = 0;
    const OnDevice on(device_);
    for (void *&s : streams_) {
        if (s) continue;
        hipStream_t made;
        hip_check(hipStreamCreateWithFlags(&made, hipStreamNonBlocking), "hipStreamCreate");
        s = made;
    }
    while (events_.size() < most) {
        hipEvent_t e;
        hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        events_.push_back(e);
    }
    return at_hand();
}

void *ShareStreams::pass(void *behind) {
    hipEvent_t e = static_cast<hipEvent_t>(events_.at(share_));
    hip_check(hipEventRecord(e, static_cast<hipStream_t>(at_hand())), "hipEventRecord");
    hip_check(hipStreamWaitEvent(static_cast<hipStream_t>(behind), e, 0), "hipStreamWaitEvent");
    ++share_;
    return at_hand();
}

void ShareStreams::synchronize() {
    for (void *s : streams_)
        if (s) (void)hipStreamSynchronize(static_cast<hipStream_t>(s));
}

ShareStreams::~ShareStreams() {
    for (void *e : events_) (void)hipEventDestroy(static_cast<hipEvent_t>(e));
    for (void *s : streams_)
        if (s) (void)hipStreamDestroy(static_cast<hipStream_t>(s));
}

Staging::Staging(size_t bytes) {
    bytes_ = std::min(std::max(bytes, kPiece), kSmall);
    hip_check(hipGetDevice(&device_), "hipGetDevice");
    void *p = nullptr;
    hip_check(hipHostMalloc(&p, bytes_, 0), "hipHostMalloc");
    memory_ = static_cast<unsigned char *>(p);
    for (size_t i = 0; i < kEvents; ++i) {
        hipEvent_t e;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            for (void *made : events_) (void)hipEventDestroy(static_cast<hipEvent_t>(made));
            (void)hipHostFree(memory_);
            throw std::runtime_error("hipEventCreate failed");
        }
        events_.push_back(e);
    }
}

Staging::~Staging() {
    {
        std::lock_guard<std::mutex> lock(mutex_);
        stop_ = true;
    }
    wake_.notify_all();
    for (auto &t : helpers_) t.join();
    for (void *e : events_) (void)hipEventDestroy(static_cast<hipEvent_t>(e));
    (void)hipHostFree(memory_);
}

void Staging::grow(size_t bytes) {
    std::lock_guard<std::mutex> one(use_);
    const size_t want = std::min(bytes, kMost);
    if (want <= bytes_) return;
    void *p = nullptr;
    hip_check(hipHostMalloc(&p, want, 0), "hipHostMalloc");
    (void)hipHostFree(memory_);
    memory_ = static_cast<unsigned char *>(p), bytes_ = want;
}

void Staging::wait_for_room(size_t block) {
    if (block < ring_) return;
    const size_t transfer = transfer_of_[block - ring_];
    while (issued_.load(std::memory_order_acquire) <= transfer) {
        if (failed_.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
    }
    // (the event may be that of a later transfer by now, which took it over when this one had ended)
    hip_check(hipEventSynchronize(static_cast<hipEvent_t>(events_[transfer % kEvents])), "hipEventSynchronize");
}

void Staging::copy_block(size_t block) {
    std::memcpy(memory_ + (block % ring_) * kBlock, src_ + block * kBlock, std::min(kBlock, size_ - block * kBlock));
    done_[block].store(true, std::memory_order_release);
}

void Staging::copy_blocks() {
    for (;;) {
        const size_t b = next_.fetch_add(1, std::memory_order_relaxed);
        if (b >= blocks_ || failed_.load(std::memory_order_relaxed)) return;
        wait_for_room(b);
        if (failed_.load(std::memory_order_relaxed)) return;
        copy_block(b);
    }
}

void Staging::helper() {
    (void)hipSetDevice(device_);
    size_t seen = 0;
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
        wake_.wait(lock, [&] { return stop_ || generation_ != seen; });
        if (stop_) return;
        seen = generation_;
        if (!open_) continue;  // woken after the end
        ++busy_;
        lock.unlock();
        try {
            copy_blocks();
        } catch (...) {
            failed_.store(true);
        }
        lock.lock();
        if (--busy_ == 0) idle_.notify_one();
    }
}

void Staging::start_helpers() {
    if (!helpers_.empty()) return;
    const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
    try {
        for (unsigned i = 0; i < std::min(3u, cores - 1); ++i) helpers_.emplace_back([this] { helper(); });
    } catch (const std::system_error &) {
        // fewer then; the calling thread copies too
    }
}

void Staging::upload(void *dst, const void *src, size_t bytes, void *stream, const std::function<void *(size_t)> &arriving) {
    if (bytes == 0) return;
    std::lock_guard<std::mutex> one(use_);
    hipStream_t s = static_cast<hipStream_t>(stream);
    start_helpers();
    dst_ = static_cast<unsigned char *>(dst), src_ = static_cast<const unsigned char *>(src);
    size_ = bytes, blocks_ = (bytes + kBlock - 1) / kBlock;
    // a whole input that fits lies in one piece; a longer one goes round in whole blocks
    ring_ = bytes <= bytes_ ? blocks_ : bytes_ / kBlock;
    transfers_.clear(), transfer_of_.clear();
    for (size_t first = 0, most = 4; first < blocks_; most = std::min(2 * most, kLargest / kBlock)) {
        const size_t left_in_ring = ring_ - first % ring_, n = std::min({most, blocks_ - first, left_in_ring});
        transfer_of_.insert(transfer_of_.end(), n, transfers_.size());
        transfers_.push_back(Transfer{first, n});
        first += n;
    }
    next_.store(0), issued_.store(0), failed_.store(false);
    if (done_.size() < blocks_) done_ = std::vector<std::atomic<bool>>(blocks_);
    for (size_t b = 0; b < blocks_; ++b) done_[b].store(false, std::memory_order_relaxed);
    {
        std::lock_guard<std::mutex> lock(mutex_);
        open_ = true;
        ++generation_;
    }
    wake_.notify_all();

    // starts the transfers whose blocks are there, in order
    size_t ready = 0;  // blocks from the first on that are
    auto issue = [&] {
        while (ready < blocks_ && done_[ready].load(std::memory_order_acquire)) ++ready;
        size_t t = issued_.load(std::memory_order_relaxed);
        for (; t < transfers_.size() && transfers_[t].first + transfers_[t].blocks <= ready; ++t) {
            const size_t at = transfers_[t].first * kBlock, n = std::min(transfers_[t].blocks * kBlock, size_ - at);
            hip_check(hipMemcpyAsync(dst_ + at, memory_ + (transfers_[t].first % ring_) * kBlock, n, hipMemcpyHostToDevice, s), "hipMemcpyAsync");
            if (ring_ < blocks_) {
                hipEvent_t e = static_cast<hipEvent_t>(events_[t % kEvents]);
                // whoever waits for the transfer that had it before -- of another stream, perhaps -- may find this one's record
                if (t >= kEvents) hip_check(hipEventSynchronize(e), "hipEventSynchronize");
                hip_check(hipEventRecord(e, s), "hipEventRecord");
            }
            issued_.store(t + 1, std::memory_order_release);
            if (arriving) s = static_cast<hipStream_t>(arriving(at + n));
        }
        if (failed_.load(std::memory_order_relaxed)) throw std::runtime_error("the input's copy failed");
    };
    auto wait_for_helpers = [&] {
        std::unique_lock<std::mutex> lock(mutex_);
        open_ = false;
        idle_.wait(lock, [&] { return busy_ == 0; });
    };
    try {
        for (;;) {
            issue();
            const size_t b = next_.fetch_add(1, std::memory_order_relaxed);
            if (b >= blocks_) break;
            while (b >= ring_ && issued_.load(std::memory_order_relaxed) <= transfer_of_[b - ring_]) issue();
            wait_for_room(b);
            copy_block(b);
        }
        while (issued_.load(std::memory_order_relaxed) < transfers_.size()) issue();
    } catch (...) {
        failed_.store(true);
        wait_for_helpers();
        (void)hipStreamSynchronize(s);
        throw;
    }
    wait_for_helpers();
}

void Staging::download(void *dst, const void *src, size_t bytes) {
    std::lock_guard<std::mutex> one(use_);
    hipStream_t s = static_cast<hipStream_t>(copy_stream(device_));
    const size_t pieces = (bytes + kPiece - 1) / kPiece, window = std::min(kEvents, bytes_ / kPiece);  // (an event each)
    try {
        for (size_t i = 0; i < pieces + window; ++i) {
            if (i >= window) {
                const size_t c = i - window;
                hip_check(hipEventSynchronize(static_cast<hipEvent_t>(events_[c % window])), "hipEventSynchronize");
                std::memcpy(static_cast<unsigned char *>(dst) + c * kPiece, memory_ + (c % window) * kPiece, std::min(kPiece, bytes - c * kPiece));
            }
            if (i < pieces) {
                hip_check(hipMemcpyAsync(memory_ + (i % window) * kPiece, static_cast<const unsigned char *>(src) + i * kPiece,
                                         std::min(kPiece, bytes - i * kPiece), hipMemcpyDeviceToHost, s),
                          "hipMemcpyAsync D2H");
                hip_check(hipEventRecord(static_cast<hipEvent_t>(events_[i % window]), s), "hipEventRecord");
            }
        }
    } catch (...) {
        (void)hipStreamSynchronize(s);
        throw;
    }
}

}  // namespace bnn
