// Pinned host memory between a Net and its callers' pageable buffers.
//
// A copy from or to pageable memory goes through the runtime's own small staging or pins the caller's pages for the call: 24 MB
// to the device took 650 to 890 us (430 from pinned memory), 256 KB either way 106 us (13), 160 KB from the device 70.
// A Staging holds 512 KB to 1 MB of pinned memory for the life of its Net, and up to 32 MB from the second large input on: memory
// that is pinned for the first time is mapped page by page as it is first written, 0.4 ms for 2 MB and 2.5 for 24, which pays after ten
// to twenty runs (batch 40 of 224 x 224 images: 1.01 ms a run without, 0.87 with it, 3.8 the run that writes it first; 0.92 with 8 MB,
// 1.06 with 4).  Large inputs run through it in blocks of 256 KB that the
// calling thread and up to three helpers copy in, and leave it in transfers of 1, 2, 4 and then 8 MB, each started as soon
// as its blocks are there: one transfer costs 15 us beside its bytes, and the first should not wait long (24 MB in equal
// transfers of 512 KB, 2 MB and 4 MB: 960, 675 and 720 us; the link alone takes 430).
#pragma once

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace bnn {

// The stream (a hipStream_t) for copies between host and device memory that belong to no net's own stream: one per device, for the
// life of the process (making one takes 150 to 200 us), and one that does not synchronise with the null stream.  A plain hipMemcpy works
// on the null stream, and a null-stream operation issued by one thread while another thread's Net captures its HIP graph fails and
// invalidates that capture.
void *copy_stream(int device);

class Staging {
   public:
    static constexpr size_t kBlock = 256u << 10, kSmall = 1u << 20, kMost = 32u << 20, kLargest = 8u << 20;
    static constexpr size_t kPiece = 512u << 10;  // of a download: its first piece is copied out while the next ones arrive

    // Room for `bytes`, 512 KB at least and 1 MB at most; allocates, and so does grow: up to 32 MB (memory() is another then).
    explicit Staging(size_t bytes);
    ~Staging();
    void grow(size_t bytes);
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;

    unsigned char *memory() const { return memory_; }
    size_t bytes() const { return bytes_; }
    int device() const { return device_; }

    // Copies host memory to the device on `stream`; `src` may change once the call returns.  The caller synchronises the
    // stream before the next call (a Net's runs do).  `arriving`, if given, is told how many bytes have been asked for, from the
    // front on, each time that grows, and says which stream brings the next (the caller synchronises all of them).
    void upload(void *dst, const void *src, size_t bytes, void *stream, const std::function<void *(size_t)> &arriving = nullptr);
    // Copies device memory to the host and waits, over the copy stream of the device that the Staging's events are of: the runtime
    // records no event of one device on a stream of another.
    void download(void *dst, const void *src, size_t bytes);

   private:
    struct Transfer {
        size_t first, blocks;
    };
    void wait_for_room(size_t block);  // what the block is about to overwrite has been transferred
    void copy_block(size_t block);
    void copy_blocks();  // takes blocks until there are none left (a helper's share of an upload)
    void helper();
    void start_helpers();

    unsigned char *memory_ = nullptr;
    size_t bytes_ = 0;
    int device_ = 0;
    static constexpr size_t kEvents = 16;
    std::vector<void *> events_;  // of transfer i: i % kEvents

    // the upload at hand
    unsigned char *dst_ = nullptr;
    const unsigned char *src_ = nullptr;
    size_t size_ = 0, blocks_ = 0, ring_ = 0;  // ring_: blocks in the pinned memory
    std::vector<Transfer> transfers_;
    std::vector<size_t> transfer_of_;  // a block's
    std::atomic<size_t> next_{0}, issued_{0};
    std::atomic<bool> failed_{false};
    std::vector<std::atomic<bool>> done_;

    std::vector<std::thread> helpers_;
    std::mutex mutex_;
    std::condition_variable wake_, idle_;
    size_t generation_ = 0;
    bool open_ = false;  // the upload at hand takes helpers
    int busy_ = 0;       // and has this many
    bool stop_ = false;
    std::mutex use_;  // one upload or download at a time
};

// The streams that bring the shares of an input in turn, and an event for each share, on a device of the caller's choice -- that of the
// stream behind them -- whichever is current for the calling thread: the runtime records no event of one device on a stream of another.
class ShareStreams {
   public:
    explicit ShareStreams(int device) : device_(device) {}
    ~ShareStreams();
    ShareStreams(const ShareStreams &) = delete;
    ShareStreams &operator=(const ShareStreams &) = delete;

    // The stream of the first of at most so many shares; what that takes and is not there yet is made here.
    void *begin(size_t most);
    // `behind` waits for what the share's stream has been given; the next share's stream.
    void *pass(void *behind);
    void *at_hand() const { return streams_[share_ % 2]; }
    void synchronize();

   private:
    int device_;
    void *streams_[2] = {};
    std::vector<void *> events_;
    size_t share_ = 0;
};

}  // namespace bnn
