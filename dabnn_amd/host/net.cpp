#include "net.h"

#include <algorithm>
#include <cstring>

#include <hip/hip_runtime_api.h>

#include <fstream>
#include <mutex>
#include <set>
#include <sstream>
#include <stdexcept>

#include "../../include/dabnn_hip_tuning.h"
#include "layers.h"
#include "model.h"
#include "staging.h"

namespace bnn {

namespace {

void hip_check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace

// ---------------------------------------------------------------- Layer::forward with optional timing
void Layer::forward() {
    auto net = net_.lock();
    if (!net->profile) {
        forward_impl();
        return;
    }
    hipStream_t s = static_cast<hipStream_t>(net->stream());
    hipEvent_t e0, e1;
    hip_check(hipEventCreate(&e0), "hipEventCreate");
    hip_check(hipEventCreate(&e1), "hipEventCreate");
    hip_check(hipEventRecord(e0, s), "hipEventRecord");
    forward_impl();
    hip_check(hipEventRecord(e1, s), "hipEventRecord");
    hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
    float ms = 0.f;
    hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
    net->layer_time_[type_] += ms;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
}

// ---------------------------------------------------------------- Net
// Nets of one process may run on host threads of their own.  A net captures its HIP graph on its third run; device
// allocations and frees of other threads (a net being read or destroyed) and a second capture stay out of that
// window.  Kernel launches and copies of other nets do not take the lock.
static std::mutex &capture_mutex() {
    static std::mutex m;
    return m;
}

Net::Net() {
    hipStream_t s;
    hip_check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
    stream_ = s;
}

Net::~Net() {
    std::lock_guard<std::mutex> lock(capture_mutex());
    for (const Graph &g : graphs_)
        if (g.exec) (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(g.exec));
    if (input_own_dev_ && mat_map_.count(input_name_)) mat_map_[input_name_]->dev = input_own_dev_;  // freed by its Mat
    layers.clear();
    columns_.clear();
    alone_.clear();
    contiguous_.clear();
    mirrors_.clear();
    mat_map_.clear();
    staging_.reset();
    shares_.reset();
    if (mirror_memory_) (void)hipHostFree(mirror_memory_);
    if (stream_) (void)hipStreamDestroy(static_cast<hipStream_t>(stream_));
}

std::shared_ptr<Net> Net::create() {
    struct make_shared_enabler : public Net {};
    return std::make_shared<make_shared_enabler>();
}

void Net::set_batch(int batch) {
    BNN_ASSERT(!prepared_, "set_batch must be called before the model is read");
    BNN_ASSERT(batch > 0, "batch must be positive");
    batch_ = batch;
}

void Net::read(const std::string &path) {
    // dabnn/net.cpp:32-44 maps the file; here the bytes are copied once and the
    // tensors uploaded to the device, so the file buffer can go afterwards.
    std::ifstream f(path, std::ios::binary | std::ios::ate);
    if (!f) throw std::invalid_argument("Open file error " + path);
    const std::streamsize size = f.tellg();
    if (size < 8) throw std::invalid_argument("Not a dabnn model: " + path);
    f.seekg(0);
    file_.resize((size_t)size);
    if (!f.read(reinterpret_cast<char *>(file_.data()), size)) throw std::invalid_argument("Read file error " + path);
    prepare(file_.data(), file_.size());
    file_.clear();
    file_.shrink_to_fit();
}

void Net::read_buf(const void *ptr) {
    // the reference's signature (dabnn/net.cpp:46): the extent of the buffer is unknown, so offsets are only kept
    // from wrapping around; callers that know the size use read_buf(ptr, len)
    BNN_ASSERT(ptr != nullptr, "read_buf: null model buffer");
    prepare(ptr, SIZE_MAX);
}

void Net::read_buf(const void *ptr, size_t len) {
    BNN_ASSERT(ptr != nullptr, "read_buf: null model buffer");
    prepare(ptr, len);
}

void Net::add_mat(const std::string &name, std::shared_ptr<Mat> mat) { mat_map_[name] = mat; }

std::shared_ptr<Mat> Net::get_blob(const std::string &name) {
    auto m = blob(name);
    m->sync_to_host(staging_.get());
    return m;
}

void Net::download(const std::shared_ptr<Mat> &m, void *host, size_t bytes) {
    for (Mirror &mirror : mirrors_) {
        if (mirror.mat != m || bytes > m->bytes()) continue;
        mirror.asked = true;
        if (!mirror.valid) break;
        std::memcpy(host, mirror.host, bytes);
        return;
    }
    m->download(host, bytes, staging_.get());
}

std::shared_ptr<Mat> Net::blob(const std::string &name) {
    auto m = stored_blob(name);
    make_columns(m);
    if (!m->ld) return m;
    auto it = contiguous_.find(m.get());
    if (it != contiguous_.end()) return it->second;
    std::lock_guard<std::mutex> lock(capture_mutex());
    auto copy = std::make_shared<Mat>(m->n, m->h, m->w, m->elem_c, m->data_type, m->name);
    m->gather_to(copy->dev, stream_);
    hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
    contiguous_[m.get()] = copy;
    return copy;
}

void Net::make_columns(const std::shared_ptr<Mat> &m) {
    if (!prepared_ || m->dev || m->external_memory) return;
    for (const auto &l : layers) {
        auto bc = std::dynamic_pointer_cast<BinConv>(l);
        auto pool = std::dynamic_pointer_cast<MaxPool>(l);
        if (pool && pool->inside_conv && pool->output_mat == m) {
            std::lock_guard<std::mutex> lock(capture_mutex());
            m->allocate();
            pool->forward_alone();
            hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
            alone_.push_back(pool);
            return;
        }
        if (bc && bc->branch && bc->branch->output_mat == m) {
            std::lock_guard<std::mutex> lock(capture_mutex());
            m->allocate();
            bc->branch->forward_alone();
            hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
            alone_.push_back(bc->branch);
            return;
        }
        if (bc && bc->pooled_in_pass && bc->output_mat == m) {
            std::lock_guard<std::mutex> lock(capture_mutex());
            m->allocate();
            bc->forward_alone();
            hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
            alone_.push_back(bc);
            return;
        }
        if (bc && bc->next_in_pass && (bc->output_mat == m || bc->fused_sign_out == m)) {
            std::lock_guard<std::mutex> lock(capture_mutex());
            bc->output_mat->allocate();
            bc->fused_sign_out->allocate();
            bc->forward_alone();
            hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
            alone_.push_back(bc);
            return;
        }
        if (!bc || bc->col_mat != m) continue;
        if (bc->inside_pass) make_columns(bc->binarized_mat);  // what the matrix is made from
        std::lock_guard<std::mutex> lock(capture_mutex());
        m->allocate();
        bc->fill_columns();
        hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
        columns_.push_back(bc);
        return;
    }
}

std::shared_ptr<Mat> Net::stored_blob(const std::string &name) {
    auto it = mat_map_.find(name);
    if (it == mat_map_.end()) {
        auto gone = elided_.find(name);
        if (gone != elided_.end())
            throw std::runtime_error("blob " + name + " is not produced: " + gone->second + "; read the model with optimize = false to get it");
        throw std::out_of_range("Key " + name + " not found.");  // StrKeyMap::at, common/StrKeyMap.h
    }
    return it->second;
}

void Net::prepare(const void *buf, size_t len) {
    std::lock_guard<std::mutex> lock(capture_mutex());
    BNN_ASSERT(!prepared_, "a Net can be read once");
    BNN_ASSERT(!(strict && !run_fconv), "fconv must be run in strict mode");
    // parse (bounds-checked) and check the whole model on the host before anything is allocated on the device
    ModelDesc model = parse_model(buf, len);
    check_model(model, run_fconv);
    for (const auto &kv : model.shapes) shapes_[kv.first] = kv.second;
    // every blob of the batch must stay within the int extents of Mat and of the kernels' pixel counts
    for (const auto &kv : model.shapes) {
        if (kv.second.size() != 4) continue;
        const uint64_t per_image = (uint64_t)kv.second[1] * kv.second[2] * kv.second[3];
        BNN_ASSERT(per_image * (uint64_t)batch_ < (1ull << 31), "blob " + kv.first + " is too large at batch " + std::to_string(batch_));
    }

    // inputs: the first one only (dabnn/net.cpp:59-70)
    {
        const InputDesc &in = model.inputs[0];
        input_name_ = in.name;
        add_mat(input_name_, std::make_shared<Mat>(batch_, in.shape[1], in.shape[2], in.shape[3], DataType::Float, input_name_));
        input_own_dev_ = mat_map_[input_name_]->dev;
    }

    // initializers (dabnn/net.cpp:72-138), uploaded to the device
    for (const TensorDesc &t : model.initializers) {
        std::shared_ptr<Mat> m;
        if (t.is_bit) {
            // shape is [n][kh][kw][c]; the word count per filter may include the padding to 128 bits
            m = std::make_shared<Mat>(t.len, DataType::Bit, t.name);
            m->n = t.shape[0], m->h = t.shape[1], m->w = t.shape[2], m->c = t.shape[3] / 64, m->elem_c = t.shape[3];
            m->upload(t.data, t.len * 8);
        } else {
            if (t.shape.size() == 4)
                m = std::make_shared<Mat>((int)t.shape[0], (int)t.shape[1], (int)t.shape[2], (int)t.shape[3], DataType::Float, t.name);
            else
                m = std::make_shared<Mat>((size_t)t.shape[0], DataType::Float, t.name);
            m->upload(t.data, t.len * 4);
        }
        add_mat(t.name, m);
    }

    auto new_output = [&](const std::string &name, DataType type = DataType::Float, int images = 0) {
        const auto &s = model.shapes.at(name);
        if (!has_blob(name))
            add_mat(name, Mat::planned(images ? images : batch_, (int)s[1], (int)s[2], (int)s[3], type, name));
    };
    auto alias_output = [&](const std::string &output, const std::string &input) {  // ADD_INPLACE_LAYER
        add_mat(output, blob(input));
    };

    for (const LayerDesc &l : model.layers) {
        switch (l.type) {
            case kFpConv2D:
            case kBinConv2D: {
                new_output(l.outputs[0]);
                if (l.type == kBinConv2D) {
                    layers.push_back(std::make_shared<BinConv>(get_weak(), l.name, l.inputs[0], l.weight, l.outputs[0], l.pad_h,
                                                               l.pad_w, l.stride_h, l.stride_w));
                } else if (run_fconv) {
                    if (!l.bias.empty())
                        layers.push_back(std::make_shared<FloatConv>(get_weak(), l.name, l.inputs[0], l.weight, l.bias, l.outputs[0],
                                                                     l.pad_h, l.pad_w, l.stride_h, l.stride_w, l.dil_h));
                    else
                        layers.push_back(std::make_shared<FloatConv>(get_weak(), l.name, l.inputs[0], l.weight, l.outputs[0], l.pad_h,
                                                                     l.pad_w, l.stride_h, l.stride_w, l.dil_h));
                }
                break;
            }
            case kAffine:
                alias_output(l.outputs[0], l.inputs[0]);
                layers.push_back(std::make_shared<Affine>(get_weak(), l.name, l.inputs[0], l.a, l.b));
                break;
            case kAdd:
                alias_output(l.outputs[0], l.inputs[0]);
                layers.push_back(std::make_shared<Add>(get_weak(), l.name, l.inputs[0], l.inputs[1]));
                break;
            case kRelu:
                alias_output(l.outputs[0], l.inputs[0]);
                layers.push_back(std::make_shared<Relu>(get_weak(), l.name, l.inputs[0]));
                break;
            case kMaxPool:
            case kAvePool:
                new_output(l.outputs[0]);
                if (l.type == kMaxPool)
                    layers.push_back(std::make_shared<MaxPool>(get_weak(), l.name, l.inputs[0], l.outputs[0], l.kernel_shape[0],
                                                               l.kernel_shape[1], l.pad_h, l.pad_w, l.stride_h, l.stride_w));
                else
                    layers.push_back(std::make_shared<AvePool>(get_weak(), l.name, l.inputs[0], l.outputs[0], l.kernel_shape[0],
                                                               l.kernel_shape[1], l.pad_h, l.pad_w, l.stride_h, l.stride_w));
                break;
            case kPRelu:
                alias_output(l.outputs[0], l.inputs[0]);
                layers.push_back(std::make_shared<PRelu>(get_weak(), l.name, l.inputs[0], l.slope));
                break;
            case kConcat:
                new_output(l.outputs[0]);
                layers.push_back(std::make_shared<Concat>(get_weak(), l.name, l.inputs[0], l.inputs[1], l.outputs[0]));
                break;
            case kSplit: {  // dabnn/net.cpp:245-250: the outputs take the input's type and image count
                const int images = blob(l.inputs[0])->n;
                new_output(l.outputs[0], DataType::Bit, images);
                new_output(l.outputs[1], DataType::Bit, images);
                layers.push_back(std::make_shared<Split>(get_weak(), l.name, l.inputs[0], l.outputs[0], l.outputs[1]));
                break;
            }
            case kShuffle:
                alias_output(l.outputs[0], l.inputs[0]);
                layers.push_back(std::make_shared<Shuffle>(get_weak(), l.name, l.inputs[0]));
                break;
            default:
                throw std::runtime_error(std::string("Not supported op ") + layer_type_name(l.type));
        }
    }
    if (optimize) {
        fuse_binconv_epilogues();
        fuse_prelu();
        store_concats_in_place();
        pool_inside_convs();
        pair_residual_layers();
        branches_inside_binconvs();
        pool_inside_pairs();
    }
    allocate_blobs();
    // an in-place layer on the input blob would write into a caller's buffer that is read in place
    copy_input_ = layers_write_input();
    find_head();
    staging_ = std::make_unique<Staging>(blob(input_name_)->bytes());
    if (head_) shares_ = std::make_unique<ShareStreams>(staging_->device());
    plan_mirrors();
    hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "hipStreamSynchronize");
    prepared_ = true;
}

// Blobs a layer reads and writes (in-place layers do both).
static void layer_io(const std::shared_ptr<Layer> &l, std::vector<const Mat *> &reads, std::vector<const Mat *> &writes) {
    reads.clear(), writes.clear();
    if (auto bc = std::dynamic_pointer_cast<BinConv>(l)) {
        if (bc->inside_pass) return;
        reads = {(bc->branch_pooled ? bc->branch_pooled : bc->input_mat).get()};
        if (bc->next_in_pass) {
            const auto &pooled = bc->next_in_pass->pooled_in_pass;
            writes = {(pooled ? pooled : bc->next_in_pass->output_mat).get(), bc->binarized_mat.get()};
            if (bc->next_in_pass->fused_sign_out) writes.push_back(bc->next_in_pass->fused_sign_out.get());
            return;
        }
        if (bc->fused_shortcut && !bc->branch) reads.push_back(bc->fused_shortcut.get());
        writes = {bc->output_mat.get(), bc->binarized_mat.get()};
        if (!bc->reads_packed()) writes.push_back(bc->col_mat.get());
    } else if (auto fc = std::dynamic_pointer_cast<FloatConv>(l)) {
        if (fc->inside_block) return;
        reads = {fc->fused_pool_input ? fc->fused_pool_input.get() : fc->input_mat.get()};
        writes = {fc->output_mat ? fc->output_mat.get() : fc->fused_maxpool_out.get()};
        if (fc->fused_maxpool_sign) writes.push_back(fc->fused_maxpool_sign.get());
        if (fc->fused_sign_out) writes.push_back(fc->fused_sign_out.get());
        if (fc->fused_pool_input && !fc->fused_pool_max && !fc->input_mat->external_memory) writes.push_back(fc->input_mat.get());  // the pooled blob, a side product
    } else if (auto af = std::dynamic_pointer_cast<Affine>(l)) {
        reads = writes = {af->data_mat.get()};
    } else if (auto ad = std::dynamic_pointer_cast<Add>(l)) {
        reads = {ad->input1_mat.get(), ad->input2_mat.get()};
        writes = {ad->input1_mat.get()};
    } else if (auto re = std::dynamic_pointer_cast<Relu>(l)) {
        reads = writes = {re->data_mat.get()};
    } else if (auto pr = std::dynamic_pointer_cast<PRelu>(l)) {
        if (!pr->inside_conv) reads = writes = {pr->data_mat.get()};
    } else if (auto cc = std::dynamic_pointer_cast<Concat>(l)) {
        reads = {cc->input1_mat.get(), cc->input2_mat.get()};
        writes = {cc->output_mat.get()};
    } else if (auto ap = std::dynamic_pointer_cast<AvePool>(l)) {
        reads = {ap->input_mat.get()};
        writes = {ap->output_mat.get()};
    } else if (auto mp = std::dynamic_pointer_cast<MaxPool>(l)) {
        if (mp->inside_conv) return;
        reads = {mp->input_mat.get()};
        writes = {mp->output_mat.get()};
    } else if (auto sp = std::dynamic_pointer_cast<Split>(l)) {
        reads = {sp->input_mat.get()};
        writes = {sp->output_mat1.get(), sp->output_mat2.get()};
    } else if (auto sh = std::dynamic_pointer_cast<Shuffle>(l)) {
        reads = writes = {sh->data_mat.get()};
    }
}

// Memory for the planned blobs that are left, but for the column matrices of layers that convolve without one and the
// blobs inside one pass of two layers (make_columns).  A blob whose name a later layer took over is only known to its layers.
void Net::allocate_blobs() {
    std::vector<const Mat *> rd, wr;
    std::set<const Mat *> on_demand;
    for (const auto &l : layers) {
        auto bc = std::dynamic_pointer_cast<BinConv>(l);
        if (bc && bc->reads_packed()) on_demand.insert(bc->col_mat.get());
        if (bc && bc->next_in_pass) on_demand.insert({bc->output_mat.get(), bc->fused_sign_out.get()});
        if (bc && bc->branch) on_demand.insert(bc->branch->output_mat.get());
        if (bc && bc->pooled_in_pass) on_demand.insert(bc->output_mat.get());
        auto mp = std::dynamic_pointer_cast<MaxPool>(l);
        if (mp && mp->inside_conv) on_demand.insert(mp->output_mat.get());
    }
    for (const auto &kv : mat_map_)
        if (!on_demand.count(kv.second.get())) kv.second->allocate();
    for (const auto &l : layers) {
        layer_io(l, rd, wr);
        for (const auto *list : {&rd, &wr})
            for (const Mat *m : *list) const_cast<Mat *>(m)->allocate();
    }
}

bool Net::layers_write_input() {
    std::vector<const Mat *> rd, wr;
    const Mat *in = blob(input_name_).get();
    for (const auto &l : layers) {
        layer_io(l, rd, wr);
        for (const Mat *m : wr)
            if (m == in) return true;
    }
    return false;
}

// Float blobs of up to 2 MB in all that layers write and none but in-place ones read: the net's outputs.  A copy of its own
// takes 20 to 100 us of a call (from the device to pageable memory, and a second synchronisation); behind the layers it
// takes 2 (4 KB) to 20 us (1 MB: 66 us of a call before).  Above that size the link would hold up callers who ask for another blob.
// Who never asks should not pay it either (batch 1 from device memory 96 -> 101 us, batch 256 20 of 1030): a blob that nobody asked for
// after the first two runs, which are not captured, is left out until somebody does.  A FloatConv that makes such a blob writes the copy
// itself (batch 1 and 6: 3 us of a run less, a launch; batch 256, whose megabyte then leaves while the classifier runs: 10).
void Net::plan_mirrors() {
    constexpr size_t kMost = 2u << 20;
    std::vector<const Mat *> rd, wr;
    std::set<const Mat *> read, written;
    for (const auto &l : layers) {
        layer_io(l, rd, wr);
        for (const Mat *m : wr) written.insert(m);
        for (const Mat *m : rd)
            if (std::find(wr.begin(), wr.end(), m) == wr.end()) read.insert(m);
    }
    size_t total = 0;
    for (const auto &kv : mat_map_) {
        const auto &m = kv.second;
        const bool known = std::any_of(mirrors_.begin(), mirrors_.end(), [&](const Mirror &x) { return x.mat == m; });
        if (known || m->data_type != DataType::Float || m->ld || !m->dev || !written.count(m.get()) || read.count(m.get()) ||
            m->bytes() == 0 || total + m->bytes() > kMost)
            continue;
        std::shared_ptr<FloatConv> writer;
        for (const auto &l : layers) {
            layer_io(l, rd, wr);
            if (std::find(wr.begin(), wr.end(), m.get()) != wr.end()) writer = std::dynamic_pointer_cast<FloatConv>(l);
        }
        if (writer && (writer->output_mat != m || !writer->can_copy())) writer = nullptr;
        mirrors_.emplace_back(Mirror{m, nullptr, writer});
        total += (m->bytes() + 255) / 256 * 256;
    }
    if (mirrors_.empty()) return;
    hip_check(hipHostMalloc(&mirror_memory_, total, 0), "hipHostMalloc");
    auto *at = static_cast<unsigned char *>(mirror_memory_);
    for (Mirror &x : mirrors_) {
        x.host = reinterpret_cast<float *>(at);
        at += (x.mat->bytes() + 255) / 256 * 256;
    }
}

static bool contains(const std::vector<const Mat *> &v, const Mat *m) {
    for (const Mat *x : v)
        if (x == m) return true;
    return false;
}

// Three rewrites of the layer list; blob names and contents after run() are unchanged, because the in-place layers
// wrote into the convolution's output blob anyway.
//  1. In a down-sampling block the converter emits BinConv, Affine, [AvePool, FpConv2D, Affine], Add: the shortcut
//     branch in brackets neither reads nor writes the BinConv's blobs, so BinConv and Affine move behind it, next to
//     their Add.
//  2. BinConv -> Affine (-> Add) on the same blob becomes one pass of its kernel, FloatConv -> Affine (-> Relu) one
//     pass of the float convolution.
//  3. When the blob such a fused BinConv completes is the input of a later BinConv, the pass also writes that
//     layer's packed input and the later layer skips its pack_mat.
//  4. AvePool 2x2 stride 2 -> 1x1 FloatConv (the shortcut branch of a down-sampling block), the convolution being
//     the only reader of the pooled blob, becomes one launch that does not write that blob: it leaves the net
//     (get_blob says why).  With eight pooled pixels or fewer the blob stays and is written.
//  5. FloatConv (-> Affine -> Relu) -> MaxPool 3x3 stride 2 pad 1, the pool being the only reader of the convolution's
//     blob (the stem), becomes one pass that never writes that blob when the library says the pass pays for these
//     shapes; the blob leaves the net (get_blob says why) and its memory, four times the pooled blob's, is freed.
void Net::fuse_binconv_epilogues() {
    std::vector<const Mat *> rd, wr;
    for (size_t i = 0; i + 2 < layers.size(); ++i) {
        auto bc = std::dynamic_pointer_cast<BinConv>(layers[i]);
        auto af = std::dynamic_pointer_cast<Affine>(layers[i + 1]);
        if (!bc || !af || af->data_mat != bc->output_mat) continue;
        size_t j = i + 2;
        bool movable = true;
        for (; j < layers.size(); ++j) {
            layer_io(layers[j], rd, wr);
            if (contains(rd, bc->output_mat.get()) || contains(wr, bc->output_mat.get())) break;
            // the branch must not disturb what the BinConv reads, nor use its scratch
            if (contains(wr, bc->input_mat.get()) || contains(rd, bc->binarized_mat.get()) ||
                contains(wr, bc->binarized_mat.get()) || rd.empty())
                movable = false;
        }
        auto ad = j < layers.size() ? std::dynamic_pointer_cast<Add>(layers[j]) : nullptr;
        if (!movable || j == i + 2 || !ad || ad->input1_mat != bc->output_mat || ad->input2_mat == bc->output_mat) continue;
        std::rotate(layers.begin() + i, layers.begin() + i + 2, layers.begin() + j);  // [bc, af, branch...] -> [branch..., bc, af]
        i = j;  // continue behind the Add
    }

    std::vector<std::shared_ptr<Layer>> out;
    for (size_t i = 0; i < layers.size(); ++i) {
        auto bc = std::dynamic_pointer_cast<BinConv>(layers[i]);
        auto af = i + 1 < layers.size() ? std::dynamic_pointer_cast<Affine>(layers[i + 1]) : nullptr;
        // (1024 input channels: the direct kernel has no fused epilogue)
        if (bc && af && bc->reads_packed() && (bc->method() == BinConv::BGEMM || (bc->input_mat->elem_c <= 512 && bc->output_mat->c % 4 == 0)) &&
            af->data_mat == bc->output_mat) {
            bc->fused_a = af->a_mat;
            bc->fused_b = af->b_mat;
            size_t skip = 1;
            auto ad = i + 2 < layers.size() ? std::dynamic_pointer_cast<Add>(layers[i + 2]) : nullptr;
            if (ad && ad->input1_mat == bc->output_mat && ad->input2_mat != bc->output_mat) {
                bc->fused_shortcut = ad->input2_mat;
                skip = 2;
            }
            out.push_back(bc);
            i += skip;
        } else if (auto fc = std::dynamic_pointer_cast<FloatConv>(layers[i])) {
            // FloatConv -> Affine (-> Relu), all on the convolution's output blob
            size_t skip = 0;
            if (af && af->data_mat == fc->output_mat) {
                fc->fused_a = af->a_mat;
                fc->fused_b = af->b_mat;
                skip = 1;
            }
            auto re = i + skip + 1 < layers.size() ? std::dynamic_pointer_cast<Relu>(layers[i + skip + 1]) : nullptr;
            if (re && re->data_mat == fc->output_mat) {
                fc->fused_relu = true;
                ++skip;
            }
            out.push_back(fc);
            i += skip;
        } else {
            out.push_back(layers[i]);
        }
    }
    layers.swap(out);

    // the same for a MaxPool whose output a BinConv packs (the first block of a Bi-Real net)
    for (size_t i = 0; i < layers.size(); ++i) {
        auto pool = std::dynamic_pointer_cast<MaxPool>(layers[i]);
        if (!pool || pool->output_mat->c % 64 != 0) continue;
        for (size_t j = i + 1; j < layers.size(); ++j) {
            auto consumer = std::dynamic_pointer_cast<BinConv>(layers[j]);
            if (consumer && consumer->input_mat == pool->output_mat) {
                if (consumer->reads_packed() && !consumer->input_prepacked) {
                    pool->fused_sign_out = consumer->binarized_mat;
                    consumer->input_prepacked = true;
                }
                break;
            }
            layer_io(layers[j], rd, wr);
            if (contains(wr, pool->output_mat.get())) break;
        }
    }
    for (size_t i = 0; i < layers.size(); ++i) {
        auto producer = std::dynamic_pointer_cast<BinConv>(layers[i]);
        if (!producer || !producer->fused_a || producer->output_mat->c % 64 != 0) continue;
        // with 512 input channels only in the size classes 0 and 3 (dabnn_hip_tuning.h): large problems there leave the
        // packing to the layer that reads the blob
        if (producer->method() == BinConv::DIRECT_CONV && producer->input_mat->elem_c >= 512) {
            const int64_t pixels = (int64_t)producer->output_mat->n * producer->output_mat->h * producer->output_mat->w;
            if (!dab_bconv3x3_splits_depth(pixels, producer->input_mat->elem_c, producer->output_mat->c) &&
                dab_bconv3x3_epilogue_build(pixels, producer->input_mat->elem_c, producer->output_mat->c, producer->stride_h, 1) != 3)
                continue;
        }
        for (size_t j = i + 1; j < layers.size(); ++j) {
            auto consumer = std::dynamic_pointer_cast<BinConv>(layers[j]);
            if (consumer && consumer->input_mat == producer->output_mat) {
                if (consumer->reads_packed()) {
                    producer->fused_sign_out = consumer->binarized_mat;
                    consumer->input_prepacked = true;
                }
                break;
            }
            layer_io(layers[j], rd, wr);
            if (contains(wr, producer->output_mat.get())) break;  // the blob changes again before anyone packs it
        }
    }

    for (size_t i = 0; i + 1 < layers.size(); ++i) {
        auto pool = std::dynamic_pointer_cast<AvePool>(layers[i]);
        if (!pool || pool->pad_h != 0 || pool->pad_w != 0 || pool->input_mat->c % 4 != 0) continue;
        const bool two_by_two = pool->kernel_h == 2 && pool->kernel_w == 2 && pool->stride_h == 2 && pool->stride_w == 2 &&
                                pool->input_mat->h >= 2 && pool->input_mat->w >= 2;
        // one window over the whole image (the pool before a classifier); whether the one-launch form covers the shapes
        // is asked below, when the convolution is known
        const bool global = !two_by_two && pool->kernel_h == pool->input_mat->h && pool->kernel_w == pool->input_mat->w;
        if (!two_by_two && !global) continue;
        // the one reader of the pooled blob must be a 1x1 FloatConv, with nothing in between that rewrites the pool's input
        size_t j = i + 1;
        bool ok = true;
        for (; j < layers.size(); ++j) {
            layer_io(layers[j], rd, wr);
            if (contains(rd, pool->output_mat.get())) break;
            if (contains(wr, pool->input_mat.get()) || contains(wr, pool->output_mat.get())) ok = false;
        }
        auto fc = j < layers.size() ? std::dynamic_pointer_cast<FloatConv>(layers[j]) : nullptr;
        if (!ok || !fc || fc->input_mat != pool->output_mat || fc->weight_mat->h != 1 || fc->weight_mat->w != 1 ||
            fc->pad_h != 0 || fc->pad_w != 0 || fc->stride_h != 1 || fc->stride_w != 1 || fc->dilation != 1)
            continue;
        for (size_t k = j + 1; k < layers.size() && ok; ++k) {
            layer_io(layers[k], rd, wr);
            if (contains(rd, pool->output_mat.get())) ok = false;  // someone else wants the pooled blob at its own time
        }
        if (!ok) continue;
        if (global && !dab_global_ave_pool_fconv1x1_takes(pool->input_mat->n, pool->input_mat->h, pool->input_mat->w,
                                                          pool->input_mat->c, fc->output_mat->c))
            continue;
        fc->fused_pool_input = pool->input_mat;
        fc->fused_pool_global = global;
        // Nobody but this convolution reads the pooled blob, so the 2x2 form does not write it: the blob leaves the
        // net (get_blob says why) and a Mat without memory keeps its shape for the layer.  Eight pooled pixels or
        // fewer run as the two launches and keep the blob.
        const Mat &pooled = *pool->output_mat;
        if (!global && (long long)pooled.n * pooled.h * pooled.w > 8) {
            for (auto it = mat_map_.begin(); it != mat_map_.end();) {
                if (it->second == pool->output_mat) {
                    elided_[it->first] = "the AvePool runs inside the convolution that reads it";
                    it = mat_map_.erase(it);
                } else {
                    ++it;
                }
            }
            fc->input_mat = std::make_shared<Mat>(pooled.n, pooled.h, pooled.w, pooled.c, nullptr, DataType::Float);
        }
        layers.erase(layers.begin() + i);
        --i;
    }

    for (size_t i = 0; i + 1 < layers.size(); ++i) {
        auto fc = std::dynamic_pointer_cast<FloatConv>(layers[i]);
        auto pool = std::dynamic_pointer_cast<MaxPool>(layers[i + 1]);
        if (!fc || !pool || fc->fused_pool_input || pool->input_mat != fc->output_mat || pool->kernel_h != 3 ||
            pool->kernel_w != 3 || pool->stride_h != 2 || pool->stride_w != 2 || pool->pad_h != 1 || pool->pad_w != 1)
            continue;
        bool only_reader = true;
        for (size_t j = 0; j < layers.size() && only_reader; ++j) {
            if (j == i || j == i + 1) continue;
            layer_io(layers[j], rd, wr);
            if (contains(rd, fc->output_mat.get()) || contains(wr, fc->output_mat.get())) only_reader = false;
        }
        const Mat &in = *fc->input_mat;
        const Mat &wt = *fc->weight_mat;
        if (!only_reader || !dab_fconv_maxpool_pays(in.n, in.h, in.w, in.c, wt.h, wt.w, fc->pad_h, fc->pad_w, fc->stride_h,
                                                    fc->stride_w, fc->dilation, fc->dilation, wt.n))
            continue;
        const int64_t carry = dab_fconv_maxpool_carry_floats(in.n, in.h, in.w, in.c, wt.h, wt.w, fc->pad_h, fc->pad_w,
                                                             fc->stride_h, fc->stride_w, fc->dilation, fc->dilation, wt.n);
        fc->fused_maxpool_out = pool->output_mat;
        fc->fused_maxpool_sign = pool->fused_sign_out;
        fc->fused_maxpool_carry = std::make_shared<Mat>((size_t)carry, DataType::Float, fc->name_ + "_carry");
        for (auto it = mat_map_.begin(); it != mat_map_.end();) {
            if (it->second == fc->output_mat) {
                elided_[it->first] = "the convolution and the MaxPool behind it run as one pass";
                it = mat_map_.erase(it);
            } else {
                ++it;
            }
        }
        fc->output_mat.reset();
        layers.erase(layers.begin() + i + 1);
    }
}

// FloatConv (-> Affine) -> PRelu on the convolution's blob: the convolution's epilogue applies the slopes.  Convolutions
// that already run as one pass with a pool, with a Relu, or on the kernel for 32 input channels (3x3, stride 1), which has
// no such epilogue, keep the layer.
void Net::fuse_prelu() {
    for (size_t i = 0; i + 1 < layers.size(); ++i) {
        auto fc = std::dynamic_pointer_cast<FloatConv>(layers[i]);
        auto pr = std::dynamic_pointer_cast<PRelu>(layers[i + 1]);
        if (!fc || !pr || !fc->output_mat || pr->data_mat != fc->output_mat || fc->fused_relu || fc->fused_pool_input || fc->fused_maxpool_out) continue;
        if (fc->input_mat->c == 32 && fc->weight_mat->h == 3 && fc->weight_mat->w == 3 && fc->stride_h == 1 && fc->stride_w == 1) continue;
        if (fc->input_mat == fc->output_mat || (long long)fc->output_mat->n * fc->output_mat->h * fc->output_mat->w <= 8) continue;
        fc->fused_slope = pr->slope_mat;
        pr->inside_conv = true;
    }
}

// A Concat whose inputs are made for it copies nothing: the inputs become slices of the output, their producers write
// them there, and the BinConvs that read an input, or the output, read its packed copy as a slice of the output's.  The
// condition on each input: one producer, a BinConv or FloatConv whose epilogue writes slices and sign bits (or a Concat
// that is itself stored this way), no layer that rewrites it, and no reader but this Concat and BinConvs; on the output:
// no layer that rewrites it (its inputs keep their values).  DenseNet blocks nest: features, then the concatenation of
// features and new channels, are slices of the last concatenation of the block.
void Net::store_concats_in_place() {
    using MatP = std::shared_ptr<Mat>;
    std::vector<const Mat *> rd, wr;
    std::map<const Mat *, std::shared_ptr<Concat>> parent;  // slice -> the Concat whose output holds it
    // whether a layer may write `m` as a slice, with its sign bits
    auto writes_slices = [&](const std::shared_ptr<Layer> &l, const MatP &m) {
        if (auto cc = std::dynamic_pointer_cast<Concat>(l)) return cc->in_place;
        if (m->c % 64 != 0 || m->data_type != DataType::Float) return false;
        if (auto bc = std::dynamic_pointer_cast<BinConv>(l)) return bc->output_mat == m && bc->fused_a && !bc->fused_shortcut && bc->reads_packed();
        if (auto fc = std::dynamic_pointer_cast<FloatConv>(l)) return fc->output_mat == m && fc->fused_slope != nullptr;
        return false;
    };
    for (const auto &layer : layers) {
        auto cc = std::dynamic_pointer_cast<Concat>(layer);
        if (!cc || cc->input1_mat == cc->input2_mat) continue;
        // offsets of dab_bconv and of the float convolution's tiles: 32 bits over the packed and 2^30 bytes over 128 rows
        const Mat &whole = *cc->output_mat;
        bool ok = whole.c % 64 == 0 && whole.c < (1 << 20) && (long long)whole.n * whole.h * whole.w * (whole.c / 64) * 8 < (1ll << 31);
        for (const MatP &m : {cc->input1_mat, cc->input2_mat, cc->output_mat}) {
            const bool is_output = m == cc->output_mat;
            if (m == stored_blob(input_name_) || parent.count(m.get())) ok = false;
            for (const auto &l : layers) {
                if (!ok) break;
                layer_io(l, rd, wr);
                if (contains(wr, m.get()) && l != layer && (is_output || !writes_slices(l, m))) ok = false;
                auto bc = std::dynamic_pointer_cast<BinConv>(l);
                if (bc && bc->input_mat == m && !bc->reads_packed()) ok = false;
                if (!is_output && bc && bc->fused_shortcut == m) ok = false;
                if (!is_output && contains(rd, m.get()) && l != layer && !bc) ok = false;
                // (a layer with a slice runs in dab_bconv, the direct 3x3 ones too)
                if (bc && (bc->input_mat == m || bc->output_mat == m) &&
                    ((long long)bc->weight_mat->total() * 8 >= (1ll << 31) || bc->weight_mat->n >= (1 << 22)))
                    ok = false;
            }
            if (!is_output && ok) {
                int writers = 0;
                for (const auto &l : layers) {
                    layer_io(l, rd, wr);
                    writers += contains(wr, m.get());
                }
                ok = ok && writers == 1;
            }
        }
        if (!ok) continue;
        cc->in_place = true;
        parent[cc->input1_mat.get()] = parent[cc->input2_mat.get()] = cc;
    }
    if (parent.empty()) return;

    // the outermost Concat output that holds `m`, and where
    auto locate = [&](MatP m) {
        int first = 0;
        for (auto it = parent.find(m.get()); it != parent.end(); it = parent.find(m.get())) {
            if (m == it->second->input2_mat) first += it->second->input1_mat->c;
            m = it->second->output_mat;
        }
        return std::make_pair(m, first);
    };
    auto held = [&](const MatP &m) {  // in the family of an in-place Concat
        if (parent.count(m.get())) return true;
        for (const auto &kv : parent)
            if (kv.second->output_mat == m) return true;
        return false;
    };
    // packed copies: one for each outermost output that a BinConv reads any part of
    std::map<const Mat *, MatP> packed;
    for (const auto &l : layers) {
        auto bc = std::dynamic_pointer_cast<BinConv>(l);
        if (!bc || !held(bc->input_mat)) continue;
        const auto at = locate(bc->input_mat);
        MatP &bits = packed[at.first.get()];
        if (!bits) bits = Mat::planned(at.first->n, at.first->h, at.first->w, at.first->c, DataType::Bit, "packed_" + at.first->name);
        bc->binarized_mat->become_slice(bits, at.second / 64);
        bc->input_prepacked = true;
    }
    for (const auto &l : layers) {
        auto bc = std::dynamic_pointer_cast<BinConv>(l);
        auto fc = std::dynamic_pointer_cast<FloatConv>(l);
        MatP out = bc ? bc->output_mat : fc ? fc->output_mat : nullptr;
        if (!out || !parent.count(out.get())) continue;
        const auto at = locate(out);
        MatP sign;
        if (packed.count(at.first.get())) {
            sign = std::make_shared<Mat>(out->n, out->h, out->w, out->c, nullptr, DataType::Bit);
            sign->become_slice(packed[at.first.get()], at.second / 64);
        }
        (bc ? bc->fused_sign_out : fc->fused_sign_out) = sign;
    }
    for (const auto &kv : mat_map_) {
        const auto at = locate(kv.second);
        if (at.first != kv.second && !kv.second->ld) kv.second->become_slice(at.first, at.second);
    }
}

// MaxPool 2x2 stride 2 whose one reader is a 1x1 FloatConv (the transition of a dense block): the convolution's loader takes the
// maxima where the library has that in one launch and one tile holds all output channels, so that the maxima are taken once.  Two
// launches / one, us: 10 240 pixels x 256 -> 128 23.2 / 19.1, 32 768 x 256 -> 128 47.9 / 30.7 (134 MB read, 4.4 TB/s), 131 072 x 128 ->
// 64 84 / 54, 65 536 x 64 -> 128 30.5 / 25.1; all of 40 problems of up to 131 072 pixels 1.14 to 1.78 times as fast.  With 160 to 256
// channels 0.65 to 1.3 (34 816 x 256 -> 160 61 / 76), with more 0.6 to 1.1.  Nothing may rewrite what the pool reads, so that the
// pooled blob can still be made for who asks for it.
void Net::pool_inside_convs() {
    std::vector<const Mat *> rd, wr;
    for (size_t i = 0; i + 1 < layers.size(); ++i) {
        auto pool = std::dynamic_pointer_cast<MaxPool>(layers[i]);
        if (!pool || pool->fused_sign_out || pool->kernel_h != 2 || pool->kernel_w != 2 || pool->stride_h != 2 || pool->stride_w != 2 || pool->pad_h != 0 ||
            pool->pad_w != 0 || pool->input_mat->ld || pool->output_mat->ld || pool->input_mat == stored_blob(input_name_))
            continue;
        const Mat &in = *pool->input_mat;
        std::shared_ptr<FloatConv> reader;
        bool ok = true;
        for (size_t j = 0; j < layers.size() && ok; ++j) {
            if (j == i) continue;
            layer_io(layers[j], rd, wr);
            if (contains(wr, pool->output_mat.get()) || (j > i && contains(wr, pool->input_mat.get()))) ok = false;
            if (!contains(rd, pool->output_mat.get())) continue;
            ok = ok && j > i && !reader;
            reader = std::dynamic_pointer_cast<FloatConv>(layers[j]);
            ok = ok && reader;
        }
        if (!ok || !reader || reader->input_mat != pool->output_mat || reader->fused_pool_input || reader->fused_maxpool_out || reader->weight_mat->h != 1 ||
            reader->weight_mat->w != 1 || reader->pad_h != 0 || reader->pad_w != 0 || reader->stride_h != 1 || reader->stride_w != 1 || reader->dilation != 1 ||
            reader->output_mat->c > 128 || !dab_max_pool2_fconv1x1_takes(in.n, in.h, in.w, in.c, reader->output_mat->c))
            continue;
        reader->fused_pool_input = pool->input_mat;
        reader->fused_pool_max = true;
        pool->inside_conv = true;
    }
}

// Two residual layers over 64 channels that follow each other (BinConv + Affine + Add of its own input, at stride 1) run as one
// pass that keeps the blob between them on the chip, where that blob and its packed copy have no other reader and nothing
// rewrites what the first layer reads (who asks for them has that layer run again).  Pays from 48 000 pixels on, where the
// layers are bound by memory, two launches / one pass, by themselves in a graph: 56 x 56 at 12 images 12.0 / 11.3 us, 16 12.5 / 11.5, 24 20.8 / 13.4, 64
// 43 / 21, 256 158 / 90; 28 x 28 at 40 images 9.7 / 12.1, 64 12.2 / 9.8.  Up to 64 columns: a strip of wider rows is so low
// that its neighbours' rows are most of the work.
void Net::pair_residual_layers() {
    std::vector<const Mat *> rd, wr;
    auto residual = [&](const std::shared_ptr<BinConv> &bc) {
        const Mat &in = *bc->input_mat;
        return bc->method() == BinConv::DIRECT_CONV && in.elem_c == 64 && bc->weight_mat->n == 64 && bc->stride_h == 1 && bc->pad_h == 1 && bc->fused_a &&
               bc->fused_shortcut == bc->input_mat && !bc->has_slices() && !in.ld && bc->output_mat != bc->input_mat && in.w <= 64 &&
               (long long)in.n * in.h * in.w >= 48000 && dab_bconv3x3_pair_takes(in.n, in.h, in.w);
    };
    for (size_t i = 0; i + 1 < layers.size(); ++i) {
        auto first = std::dynamic_pointer_cast<BinConv>(layers[i]), second = std::dynamic_pointer_cast<BinConv>(layers[i + 1]);
        if (!first || !second || !residual(first) || !residual(second) || second->input_mat != first->output_mat || !second->input_prepacked ||
            first->fused_sign_out != second->binarized_mat || second->output_mat == first->input_mat || second->fused_sign_out == first->binarized_mat)
            continue;
        bool ok = true;
        for (size_t j = 0; j < layers.size() && ok; ++j) {
            if (j == i || j == i + 1) continue;
            layer_io(layers[j], rd, wr);
            auto bc = std::dynamic_pointer_cast<BinConv>(layers[j]);
            for (const auto &m : {first->output_mat, second->binarized_mat})
                if (contains(rd, m.get()) || contains(wr, m.get()) || (bc && (bc->binarized_mat == m || bc->fused_sign_out == m))) ok = false;
            if (j > i && (contains(wr, first->input_mat.get()) || contains(wr, first->binarized_mat.get()) || (bc && bc->fused_sign_out == first->binarized_mat)))
                ok = false;
        }
        // (the net's input may be a buffer of the caller's, gone after the run)
        if (!ok || first->input_mat == stored_blob(input_name_)) continue;
        first->next_in_pass = second;
        second->first_in_pass = first.get();
        second->inside_pass = true;
        ++i;
    }
}

// The shortcut branch of a down-sampling block -- AvePool 2x2 inside a 1x1 FloatConv (+ Affine) that reads what the block's first
// BinConv reads and whose result only that layer adds -- runs in the BinConv's pass, which keeps the branch's result on the chip; who
// asks for its blob has the pass run again with that output.  So nothing may rewrite, later, what the pass reads or writes, nor read
// or write the branch's blob.  Two launches against one: bconv_down.hip; 256 input channels gain least in large nets, whose clock is lower
// (Bi-Real-18, a run with that block in two / one: 100 images 549 / 539 us, 200 916 / 904, 256 1108 / 1107, 300 1273 / 1278).
void Net::branches_inside_binconvs() {
    std::vector<const Mat *> rd, wr;
    for (size_t i = 1; i < layers.size(); ++i) {
        auto bc = std::dynamic_pointer_cast<BinConv>(layers[i]);
        if (!bc || bc->method() != BinConv::DIRECT_CONV || bc->stride_h != 2 || bc->pad_h != 1 || !bc->fused_a || !bc->fused_shortcut || bc->has_slices() ||
            bc->input_mat->ld || bc->input_mat == stored_blob(input_name_) || bc->output_mat == bc->input_mat)
            continue;
        const Mat &in = *bc->input_mat;
        const int cout = bc->weight_mat->n;
        if (!dab_bconv3x3_down_takes(in.n, in.h, in.w, in.elem_c, cout)) continue;
        std::shared_ptr<FloatConv> branch;
        size_t at = 0;
        for (size_t j = 0; j < i; ++j) {
            auto fc = std::dynamic_pointer_cast<FloatConv>(layers[j]);
            if (fc && fc->output_mat == bc->fused_shortcut) branch = fc, at = j;
        }
        // (the pooled blob has no memory: nobody else reads it)
        if (!branch || branch->fused_pool_input != bc->input_mat || branch->fused_pool_global || branch->fused_pool_max || branch->fused_relu || branch->fused_slope ||
            branch->fused_sign_out || branch->output_mat->ld || !branch->input_mat->external_memory || branch->output_mat == stored_blob(input_name_))
            continue;
        bool ok = true;
        for (size_t j = 0; j < layers.size() && ok; ++j) {
            if (j == at || j == i) continue;
            layer_io(layers[j], rd, wr);
            const Mat *sum = branch->output_mat.get();
            if (contains(rd, sum) || contains(wr, sum)) ok = false;
            if (j < at) continue;
            auto other = std::dynamic_pointer_cast<BinConv>(layers[j]);
            for (const auto &m : {bc->input_mat, bc->binarized_mat})
                if (contains(wr, m.get()) || (other && (other->fused_sign_out == m || (other->next_in_pass && other->next_in_pass->fused_sign_out == m)))) ok = false;
            for (const auto &m : {bc->output_mat, bc->fused_sign_out})
                if (j > i && m && contains(wr, m.get()) && !(other && other->binarized_mat == m)) ok = false;
        }
        if (!ok) continue;
        bc->branch = branch;
        branch->inside_block = bc.get();
    }
}

// Two residual layers in one pass, in front of a down-sampling block whose branch runs in its BinConv's pass: where nobody else reads
// the second layer's result, the pass writes it pooled (and its sign bits), a quarter of the bytes, and the block's pass reads that; who
// asks for the result has the unpooled pass run.  56 x 56, the two passes one behind the other in a graph, us: 17 images 21.0 -> 18.7, 40
// 33.5 -> 32.0, 100 65.6 -> 56.2, 256 159 -> 125.
void Net::pool_inside_pairs() {
    std::vector<const Mat *> rd, wr;
    for (const auto &l : layers) {
        auto reader = std::dynamic_pointer_cast<BinConv>(l);
        if (!reader || !reader->branch) continue;
        const auto &m = reader->input_mat;
        std::shared_ptr<BinConv> second;
        bool ok = dab_bconv3x3_pair_pool_takes(m->n, m->h, m->w);
        for (const auto &other : layers) {
            layer_io(other, rd, wr);
            if (other != l && contains(rd, m.get())) ok = false;
            if (!contains(wr, m.get())) continue;
            auto first = std::dynamic_pointer_cast<BinConv>(other);
            ok = ok && first && first->next_in_pass && !second;
            second = ok ? first->next_in_pass : nullptr;
        }
        if (!ok || !second || second->output_mat != m || second->fused_sign_out != reader->binarized_mat || !reader->input_prepacked) continue;
        second->pooled_in_pass = Mat::planned(m->n, m->h / 2, m->w / 2, m->c, DataType::Float, "pooled_" + m->name);
        reader->branch_pooled = second->pooled_in_pass;
    }
}

// Host inputs of up to a megabyte are put into pinned memory, from where the layers' first kernel takes them; larger ones
// go through it in blocks from the second on, and memory that the caller has pinned is copied from where it lies.
void Net::run(const void *host_input) {
    BNN_ASSERT(prepared_, "run before read");
    BNN_ASSERT(host_input != nullptr, "run: null input");
    auto in = blob(input_name_);
    hipPointerAttribute_t where;
    bool pageable = true;
    if (hipPointerGetAttributes(&where, host_input) == hipSuccess)
        pageable = where.type == hipMemoryTypeUnregistered;
    else
        (void)hipGetLastError();
    const bool staged = pageable && in->bytes() <= (1u << 20);  // (staging_ holds that much)
    if (!staged && head_ && !profile && (!pageable || uploaded_)) {
        BNN_ASSERT(!(strict && !run_fconv), "fconv must be run in strict mode");
        bind_input(nullptr, kBehindHead);
        upload_and_run_head(host_input, pageable);
        launch_layers(kBehindHead);
        return;
    }
    bind_input(nullptr, staged ? kStagedLayers : kLayers);
    if (staged)
        std::memcpy(staging_->memory(), host_input, in->bytes());
    else if (pageable && uploaded_) {
        {
            std::lock_guard<std::mutex> lock(capture_mutex());
            staging_->grow(in->bytes());
        }
        staging_->upload(in->dev, host_input, in->bytes(), stream_);
    } else
        hip_check(hipMemcpyAsync(in->dev, host_input, in->bytes(), hipMemcpyHostToDevice, static_cast<hipStream_t>(stream_)),
                  "hipMemcpyAsync");
    uploaded_ = uploaded_ || (pageable && !staged);
    launch_layers(staged ? kStagedLayers : kLayers);
}

// A large host input goes to the device in shares of this many bytes or more, and the head follows each.
static constexpr size_t kShare = 8u << 20;

// The layers at the front that can run on some of the images: a stem that is one pass with its MaxPool over three channels, and the binary
// convolutions behind it that read nothing else.  Their results do not depend on how many images a launch has (the float
// layers' other kernels are chosen by that, and add in another order).
void Net::find_head() {
    auto stem = layers.empty() ? nullptr : std::dynamic_pointer_cast<FloatConv>(layers[0]);
    if (copy_input_ || blob(input_name_)->bytes() < 2 * kShare || !stem || !stem->fused_maxpool_out || stem->input_mat != stored_blob(input_name_) || stem->input_mat->c != 3) return;
    std::vector<const Mat *> rd, wr;
    std::set<const Mat *> made = {stem->input_mat.get()};
    for (size_t i = 0; i < layers.size(); ++i) {
        auto bc = std::dynamic_pointer_cast<BinConv>(layers[i]);
        if (bc && bc->inside_pass) {
            head_ = i + 1;
            continue;
        }
        if (i > 0 && (!bc || bc->method() != BinConv::DIRECT_CONV || bc->branch || bc->has_slices())) return;
        layer_io(layers[i], rd, wr);
        if (bc && bc->fused_sign_out) wr.push_back(bc->fused_sign_out.get());
        for (const Mat *m : rd)
            if (!made.count(m)) return;
        for (const auto *list : {&rd, &wr})
            for (const Mat *m : *list)
                if (m->n != batch_ || m->bytes() / batch_ % 16 != 0) return;  // (the kernels want aligned images)
        made.insert(wr.begin(), wr.end());
        head_ = i + 1;
    }
}

// The head's launches on images first .. first + count - 1: its blobs stand for those alone while they are made.
void Net::run_head(int first, int count) {
    std::vector<const Mat *> rd, wr;
    std::set<const Mat *> blobs;
    for (size_t i = 0; i < head_; ++i) {
        layer_io(layers[i], rd, wr);
        blobs.insert(rd.begin(), rd.end());
        blobs.insert(wr.begin(), wr.end());
        auto bc = std::dynamic_pointer_cast<BinConv>(layers[i]);
        if (bc && !bc->inside_pass && !bc->next_in_pass && bc->fused_sign_out) blobs.insert(bc->fused_sign_out.get());
    }
    struct View {
        Mat *m;
        void *dev;
        int n;
        View(Mat *m_, int first, int count) : m(m_), dev(m_->dev), n(m_->n) {
            m->dev = static_cast<unsigned char *>(dev) + m->bytes() / n * first;
            m->n = count;
        }
        ~View() { m->dev = dev, m->n = n; }
        View(const View &) = delete;
    };
    std::vector<std::unique_ptr<View>> views;
    for (const Mat *m : blobs)
        if (m->dev) views.push_back(std::make_unique<View>(const_cast<Mat *>(m), first, count));
    for (size_t i = 0; i < head_; ++i) layers[i]->forward();
}

// Behind each share the head's launches on the images that are whole by then, so that only the last share's are left when the input is
// there.  A share's event holds up what follows it on its stream by about 20 us, so the next share takes the other stream.  bireal18
// from pageable memory, us, before, in shares of 4 MB and of 8: 16 images 494 / 469 / 519, 40 867 / 831 / 802, 64 1268 / 1235 / 1159,
// 100 1908 / 1766 / 1755, 256 4196 / 3794 / 3643; all shares on one stream: 40 811, 100 1814, 256 3830.  From pinned memory: 40 722 ->
// 673, 100 1613 -> 1484.
void Net::upload_and_run_head(const void *host_input, bool pageable) {
    auto in = blob(input_name_);
    const size_t image = in->bytes() / batch_;
    hipStream_t s = static_cast<hipStream_t>(stream_);
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");  // (a run that failed may have left kernels that read the input)
    void *up = nullptr;
    {
        std::lock_guard<std::mutex> lock(capture_mutex());
        up = shares_->begin(in->bytes() / kShare + 1);  // (all but the last are of kShare or more)
    }
    int done = 0;
    auto arriving = [&](size_t bytes) -> void * {
        const int there = (int)(bytes / image);
        if (there < batch_ && (size_t)(there - done) * image < kShare) return shares_->at_hand();
        void *next = shares_->pass(s);
        run_head(done, there - done);
        done = there;
        return next;
    };
    try {
        if (pageable) {
            {
                std::lock_guard<std::mutex> lock(capture_mutex());
                staging_->grow(in->bytes());
            }
            staging_->upload(in->dev, host_input, in->bytes(), up, arriving);
        } else {
            for (size_t at = 0; at < in->bytes();) {
                const size_t n = std::min(kShare + image, in->bytes() - at);  // (with kShare of whole images)
                hip_check(hipMemcpyAsync(static_cast<unsigned char *>(in->dev) + at, static_cast<const unsigned char *>(host_input) + at, n,
                                         hipMemcpyHostToDevice, static_cast<hipStream_t>(up)),
                          "hipMemcpyAsync");
                at += n;
                up = arriving(at);
            }
        }
    } catch (...) {
        shares_->synchronize();
        (void)hipStreamSynchronize(s);
        throw;
    }
}

void Net::run_device(const void *device_input) {
    BNN_ASSERT(prepared_, "run before read");
    bind_input(device_input, kLayers);
    launch_layers(kLayers);
}

// Points the input blob at the memory this run reads: the caller's device buffer in place, or the blob's own
// allocation (host inputs, unaligned buffers, callers whose buffers keep changing), filled here from device_input.
void Net::bind_input(const void *device_input, Kind kind) {
    auto in = blob(input_name_);
    const bool in_place = device_input != nullptr && !copy_input_ && reinterpret_cast<uintptr_t>(device_input) % 256 == 0;
    void *want = in_place ? const_cast<void *>(device_input) : input_own_dev_;
    Graph &graph = graphs_[kind];
    if (graph.exec && graph.input != want) {
        // the graph's kernels hold the address they were captured with
        if (in_place && ++input_rebinds_ >= 3) {
            copy_input_ = true;
            want = input_own_dev_;
        }
        if (graph.input != want) {
            std::lock_guard<std::mutex> lock(capture_mutex());
            (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph.exec));
            graph.exec = nullptr;
        }
    }
    in->dev = want;
    if (device_input != nullptr && want == input_own_dev_ && device_input != input_own_dev_)
        hip_check(hipMemcpyAsync(in->dev, device_input, in->bytes(), hipMemcpyDeviceToDevice, static_cast<hipStream_t>(stream_)),
                  "hipMemcpyAsync");
}

void Net::enqueue_layers(Kind kind) {
    if (kind == kStagedLayers) {
        const auto in = blob(input_name_);
        dab_check(dab_copy_f32(static_cast<float *>(in->dev), reinterpret_cast<const float *>(staging_->memory()), (int64_t)in->total(), stream_));
    }
    for (const Mirror &m : mirrors_)
        if (m.writer) m.writer->copy_to = m.copied ? m.host : nullptr;
    for (size_t i = kind == kBehindHead ? head_ : 0; i < layers.size(); ++i) layers[i]->forward();
    for (const Mirror &m : mirrors_)
        if (m.copied && !m.writer) dab_check(dab_copy_f32(m.host, static_cast<const float *>(m.mat->dev), (int64_t)m.mat->total(), stream_));
}

void Net::launch_layers(Kind kind) {
    BNN_ASSERT(!(strict && !run_fconv), "fconv must be run in strict mode");
    hipStream_t s = static_cast<hipStream_t>(stream_);
    Graph &graph = graphs_[kind];
    int copies = 0;
    for (Mirror &m : mirrors_) {
        m.valid = false;
        m.copied = m.asked || runs_ < 2;
        copies += m.copied;
    }
    if (graph.exec && graph.copies != copies) {
        std::lock_guard<std::mutex> lock(capture_mutex());
        (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph.exec));
        graph.exec = nullptr;
    }
    if (profile || !use_graph || (kind == kBehindHead && head_ == layers.size())) {  // (no layer behind the head: nothing to capture)
        enqueue_layers(kind);
    } else if (graph.exec) {
        hip_check(hipGraphLaunch(static_cast<hipGraphExec_t>(graph.exec), s), "hipGraphLaunch");
    } else if (runs_ >= 2) {
        // capture the kernels of one forward pass; nothing in the layers allocates, synchronises or memsets
        std::lock_guard<std::mutex> lock(capture_mutex());
        hipGraph_t captured = nullptr;
        hip_check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        try {
            enqueue_layers(kind);
        } catch (...) {
            (void)hipStreamEndCapture(s, &captured);
            if (captured) (void)hipGraphDestroy(captured);
            throw;
        }
        hip_check(hipStreamEndCapture(s, &captured), "hipStreamEndCapture");
        hipGraphExec_t exec = nullptr;
        hip_check(hipGraphInstantiate(&exec, captured, nullptr, nullptr, 0), "hipGraphInstantiate");
        (void)hipGraphDestroy(captured);
        graph.exec = exec;
        graph.input = blob(input_name_)->dev;
        graph.copies = copies;
        hip_check(hipGraphLaunch(exec, s), "hipGraphLaunch");
    } else {
        enqueue_layers(kind);
    }
    for (const auto &kv : contiguous_) kv.first->gather_to(kv.second->dev, s);
    for (const auto &l : alone_) l->forward_alone();
    for (const auto &bc : columns_) bc->fill_columns();
    ++runs_;
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
    for (const auto &kv : contiguous_) kv.second->mark_device_written();
    for (const auto &kv : mat_map_) kv.second->mark_device_written();  // host mirrors show the previous run
    for (Mirror &m : mirrors_) m.valid = m.copied;
}

std::vector<std::string> Net::layer_descriptions() const {
    std::vector<std::string> out;
    for (const auto &l : layers) out.push_back(l->to_str());
    return out;
}

std::string Net::time_report() const {
    std::stringstream ss;
    double total = 0;
    for (const auto &kv : layer_time_) total += kv.second;
    for (const auto &kv : layer_time_) ss << kv.first << ": " << kv.second << "ms\n";
    ss << "total: " << total << "ms\n";
    return ss.str();
}

}  // namespace bnn
