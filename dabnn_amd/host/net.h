// bnn::Net (dabnn/net.h:22-68): loads a .dab model, owns the blobs, runs the
// layers in order.  Public surface as in the reference -- create / read /
// read_buf / run / get_blob and the flags optimize / run_fconv / strict --
// plus a batch size, which the reference does not have (dabnn/net.cpp:64-65).
//
// All blobs live in device memory; run() takes a HOST pointer to
// batch x H x W x C floats (NHWC) like the reference's run(void*), uploads it,
// enqueues every layer on the net's stream and waits.  run_device() takes a
// device pointer and reads the input in place (as the reference's run wraps
// its host pointer without a copy).
#pragma once

#include <map>
#include <memory>
#include <string>
#include <vector>

#include "layer.h"
#include "mat.h"

namespace bnn {

class BinConv;
class Staging;
class ShareStreams;

class FloatConv;

class BNN_API Net : public std::enable_shared_from_this<Net> {
   public:
    static std::shared_ptr<Net> create();
    ~Net();

    void set_batch(int batch);  // before read(); default 1
    int batch() const { return batch_; }
    const std::string &input_name() const { return input_name_; }
    void read(const std::string &path);
    void read_buf(const void *ptr);
    void read_buf(const void *ptr, size_t len);  // the same, with every offset of the model checked against len
    void run(const void *host_input);
    // The layers read device_input where it lies, which must stay valid and unchanged until the call returns (256-byte
    // aligned, as hipMalloc gives it; anything else is copied into the net's own input blob).  The HIP graph holds
    // the address it was captured with: the same buffer run after run replays it, another buffer makes the net
    // capture again, and from the third such change on the net copies every input into its own blob instead.
    // nullptr: the input blob already holds the input.
    void run_device(const void *device_input);
    // The blob with its host mirror up to date (dabnn/net.cpp:288-290): `data`, operator[] ... read what the last
    // run left on the device.
    std::shared_ptr<Mat> get_blob(const std::string &name);
    // The same blob without the device-to-host copy (what the layers and the C ABI use).  A blob that the net keeps as
    // channels of a wider one comes as a contiguous copy, which every later run brings up to date.
    std::shared_ptr<Mat> blob(const std::string &name);
    // The blob as the layers hold it, slice or not; Mat::download and the host accessors work on both.
    std::shared_ptr<Mat> stored_blob(const std::string &name);
    // The blob's device memory to the host, contiguous, at most `bytes` of it (what dabnet_get_blob does): outputs of the last
    // run that are asked for run after run are in pinned memory already.
    void download(const std::shared_ptr<Mat> &m, void *host, size_t bytes);
    // If `m` is the column matrix of a layer that convolves without one, or a blob inside two layers' one pass: makes it, and
    // keeps it up to date from now on.
    void make_columns(const std::shared_ptr<Mat> &m);
    bool has_blob(const std::string &name) const { return mat_map_.count(name) != 0; }
    std::vector<std::string> layer_descriptions() const;

    // optimize: true picks the direct 3x3 kernel where it applies, false sends every
    // BinConv through im2col + bgemm (the reference's switch between its optimised and
    // plain kernels; both settings give identical outputs).
    bool optimize = true;
    bool run_fconv = true;
    bool strict = true;

    // Replay the layer sequence as one HIP graph from the third run on (the first two run eagerly so that every
    // kernel has been launched once outside capture).  Launch overhead dominates at batch 1; switch off to
    // debug or when layers are added between runs.
    bool use_graph = true;

    // per-layer-type milliseconds of the last runs when profiling (BNN_BENCHMARK of the reference)
    bool profile = false;
    std::map<std::string, double> layer_time_;
    std::string time_report() const;

    void *stream() const { return stream_; }
    void add_mat(const std::string &name, std::shared_ptr<Mat> mat);
    std::map<std::string, std::shared_ptr<Mat>> mat_map_;
    // blobs of the model that the optimized layer list never writes (name -> why); get_blob names the reason
    std::map<std::string, std::string> elided_;

   private:
    Net();
    void prepare(const void *model_buf, size_t len);
    void fuse_binconv_epilogues();
    void fuse_prelu();
    void allocate_blobs();
    void store_concats_in_place();
    void pool_inside_convs();
    void pair_residual_layers();
    void branches_inside_binconvs();
    void pool_inside_pairs();
    std::weak_ptr<Net> get_weak() { return shared_from_this(); }
    std::vector<std::shared_ptr<Layer>> layers;
    std::map<std::string, std::vector<uint32_t>> shapes_;  // NHWC with N = 1, as stored in the model
    std::string input_name_;
    std::vector<uint8_t> file_;  // owns the model bytes when read from a path
    int batch_ = 1;
    void *stream_ = nullptr;
    bool prepared_ = false;
    std::map<const Mat *, std::shared_ptr<Mat>> contiguous_;  // slice -> the copy that blob() handed out
    std::vector<std::shared_ptr<const BinConv>> columns_;  // layers whose column matrix somebody asked for
    std::vector<std::shared_ptr<const Layer>> alone_;      // and those inside another's pass whose own results somebody did
    int runs_ = 0;
    // The captured layers and the input address that their kernels hold: all of them, all of them behind the copy of a small host
    // input from staging_, or those behind the head.
    enum Kind { kLayers, kStagedLayers, kBehindHead, kKinds };
    struct Graph {
        void *exec = nullptr;
        const void *input = nullptr;
        int copies = 0;  // of mirrors
    } graphs_[kKinds];
    void *input_own_dev_ = nullptr;       // the input blob's own allocation
    int input_rebinds_ = 0;               // captures thrown away because the caller's buffer changed
    bool copy_input_ = false;             // the caller's buffers keep changing: copy into the own blob
    void bind_input(const void *device_input, Kind kind);
    bool layers_write_input();
    void launch_layers(Kind kind);
    void enqueue_layers(Kind kind);
    // How many layers at the front run on the first images of a large host input while the others are still on their way, and the
    // streams that bring its shares.
    size_t head_ = 0;
    std::unique_ptr<ShareStreams> shares_;
    void find_head();
    void run_head(int first, int count);
    void upload_and_run_head(const void *host_input, bool pageable);
    std::unique_ptr<Staging> staging_;    // pinned memory for inputs, and for blobs that are asked for
    bool uploaded_ = false;               // a large input from pageable memory
    // Small blobs that no layer reads are copied to pinned memory behind the layers of the first two runs, and of every run once they
    // have been asked for.
    struct Mirror {
        std::shared_ptr<Mat> mat;
        float *host;
        std::shared_ptr<FloatConv> writer;  // the layer that writes it last, where that can write the copy too
        bool asked = false;
        bool copied = false;  // by the run at hand
        bool valid = false;   // holds what the last run left
    };
    std::vector<Mirror> mirrors_;
    void *mirror_memory_ = nullptr;
    void plan_mirrors();
};

}  // namespace bnn
