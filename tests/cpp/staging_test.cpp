// Staging and Mat's copies through it over a runtime of two devices that lives in host memory: what the real one refuses -- an event
// of one device on a stream of another -- is refused here too, and a stream does its copies as late as it may, when somebody waits for
// it or for an event behind them.  Run by tests/test_staging.py, without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <vector>

#include "../../dabnn_amd/host/mat.h"
#include "../../dabnn_amd/host/staging.h"

static thread_local int current = 0;
static int pinned = 0, streams = 0, events = 0;  // alive
struct Stream {
    int device;
    std::deque<std::function<void()>> waiting;
    size_t asked = 0, done = 0;
    void run_until(size_t n) {
        for (; done < n; ++done) waiting.front()(), waiting.pop_front();
    }
};
struct Event {
    int device;
    Stream *stream = nullptr;
    size_t behind = 0;  // so many operations of the stream
};
static std::mutex runtime;  // copies of several threads
static Stream &of(hipStream_t s) { return *reinterpret_cast<Stream *>(s); }
static Event &of(hipEvent_t e) { return *reinterpret_cast<Event *>(e); }
static hipError_t ask(hipStream_t s, std::function<void()> operation) {
    std::lock_guard<std::mutex> lock(runtime);
    of(s).waiting.push_back(std::move(operation)), ++of(s).asked;
    return hipSuccess;
}

extern "C" {
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "refused"; }
hipError_t hipGetDevice(int *d) { return *d = current, hipSuccess; }
hipError_t hipSetDevice(int d) { return current = d, hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return *p = malloc(n), hipSuccess; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return ++pinned, *p = malloc(n), hipSuccess; }
hipError_t hipHostFree(void *p) { return --pinned, free(p), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return ++streams, *s = reinterpret_cast<hipStream_t>(new Stream{current, {}}), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::mutex> lock(runtime);
    return of(s).run_until(of(s).asked), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return hipStreamSynchronize(s), --streams, delete &of(s), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return ++events, *e = reinterpret_cast<hipEvent_t>(new Event{current}), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return --events, delete &of(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> lock(runtime);
    if (of(e).device != of(s).device) return hipErrorInvalidHandle;
    return of(e).stream = &of(s), of(e).behind = of(s).asked, hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }  // (of any device)
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> lock(runtime);
    if (of(e).stream) of(e).stream->run_until(of(e).behind);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t stream) {
    return ask(stream, [=] { memcpy(d, s, n); });
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t stream) {
    return ask(stream, [=] {
        for (size_t y = 0; y < h; ++y) memcpy(static_cast<char *>(d) + y * dp, static_cast<const char *>(s) + y * sp, w);
    });
}
}

#define CHECK(x)                                               \
    do {                                                       \
        if (!(x)) {                                            \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #x);     \
            return 1;                                          \
        }                                                      \
    } while (0)

static int round_trip(bnn::Staging &staging, int device, size_t floats) {
    current = device;
    std::vector<float> in(floats), out(floats, -1.f);
    for (size_t i = 0; i < floats; ++i) in[i] = (float)(i % 1000003);
    auto m = bnn::Mat::planned(1, 1, 1, (int)floats, bnn::DataType::Float, "m");
    m->allocate();
    hipStream_t s;
    (void)hipStreamCreateWithFlags(&s, 0);
    staging.upload(m->dev, in.data(), floats * 4, s);
    (void)hipStreamDestroy(s);
    m->download(out.data(), floats * 4, &staging);
    CHECK(out == in);
    return 0;
}

// An input in shares, as a net takes a large one: the streams and events are of the net's device, whichever is current for the thread
// that runs it.
static int shares_of_an_input(int device, size_t floats) {
    current = device;
    bnn::Staging staging(floats * 4);
    staging.grow(floats * 4);
    bnn::ShareStreams shares(staging.device());
    hipStream_t behind;
    (void)hipStreamCreateWithFlags(&behind, 0);
    current = 1 - device;
    const int events_before = events;
    for (int run = 0; run < 3; ++run) {
        std::vector<float> in(floats), out(floats, -1.f);
        for (size_t i = 0; i < floats; ++i) in[i] = (float)((i + run) % 1000003);
        size_t done = 0, told = 0;
        staging.upload(out.data(), in.data(), floats * 4, shares.begin(floats * 4 / (8u << 20) + 1), [&](size_t bytes) -> void * {
            told = bytes;
            if (bytes < floats * 4 && bytes - done < (8u << 20)) return shares.at_hand();
            done = bytes;
            void *before = shares.at_hand(), *next = shares.pass(behind);
            if (next == before) throw std::runtime_error("the next share is on the same stream");
            return next;
        });
        shares.synchronize();
        CHECK(out == in && told == floats * 4 && current == 1 - device);
    }
    CHECK(events - events_before == (int)(floats * 4 / (8u << 20) + 1));  // made once
    (void)hipStreamDestroy(behind);
    return 0;
}

int main() {
    try {
        {
            // a copy without a Staging first: Mat's own stream is of device 0
            std::vector<float> some(64, 3.f);
            auto plain = bnn::Mat::planned(1, 1, 1, 64, bnn::DataType::Float, "plain");
            plain->allocate();
            plain->upload(some.data(), 256);
            plain->download(some.data(), 256);
        }
        for (int device : {0, 1}) {
            current = device;
            bnn::Staging staging(10 << 20);
            CHECK(staging.bytes() == 1 << 20);
            for (size_t floats : {1000, 400000}) CHECK(round_trip(staging, device, floats) == 0);  // one piece, longer than the pinned memory
            staging.grow(10 << 20);
            staging.grow(5 << 20);
            CHECK(staging.bytes() == 10 << 20 && pinned == 1);
            for (size_t floats : {1000, 400000, 2000001, 21000000}) {  // pieces, a round of the events, longer than the pinned memory
                CHECK(round_trip(staging, device, floats) == 0);
            }
            staging.grow(100 << 20);
            CHECK(staging.bytes() == 32 << 20 && round_trip(staging, device, 21000000) == 0);
            // asked for from a thread whose current device is another one, which stays what it was
            current = 1 - device;
            std::vector<float> in(200000, 2.f), out(200000);
            staging.download(out.data(), in.data(), in.size() * 4);
            CHECK(out == in && current == 1 - device);
        }
        for (int device : {0, 1})
            for (size_t floats : {4500000, 12000000, 30000000}) CHECK(shares_of_an_input(device, floats) == 0);  // below and above the pinned memory's 32 MB
        CHECK(pinned == 0 && events == 0 && streams == 2);  // one copy stream per device
    } catch (const std::exception &e) {
        printf("exception: %s\n", e.what());
        return 1;
    }
    puts("ok");
    return 0;
}
