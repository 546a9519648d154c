#include "mat.h"

#include <hip/hip_runtime_api.h>

#include <cmath>
#include <fstream>
#include <ostream>
#include <stdexcept>

#include "staging.h"

namespace bnn {

static void hip_check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

Mat::Mat(int n_, int h_, int w_, int c_, DataType type, const std::string &name_)
    : n(n_), h(h_), w(w_), data_type(type), name(name_) {
    if (type == DataType::Bit) {
        if (c_ % 64 != 0) throw std::runtime_error("Bit Mat needs a channel count that is a multiple of 64, got " + std::to_string(c_));
        elem_c = c_;
        c = c_ / 64;
        elemsize = 8;
    } else {
        elem_c = c = c_;
        elemsize = 4;
    }
    if (bytes() > 0) hip_check(hipMalloc(&dev, bytes()), "hipMalloc");
}

Mat::Mat(size_t len, DataType type, const std::string &name_) : n(1), h(1), w(1), data_type(type), name(name_) {
    c = (int)len;
    elem_c = type == DataType::Bit ? (int)len * 64 : (int)len;
    elemsize = type == DataType::Bit ? 8 : 4;
    data_num_ = len;
    if (bytes() > 0) hip_check(hipMalloc(&dev, bytes()), "hipMalloc");
}

Mat::Mat(int n_, int h_, int w_, int c_, void *device_data, DataType type, size_t data_num)
    : n(n_), h(h_), w(w_), data_type(type), dev(device_data), external_memory(true), data_num_(data_num) {
    if (type == DataType::Bit) {
        elem_c = c_;
        c = c_ / 64;
        elemsize = 8;
    } else {
        elem_c = c = c_;
        elemsize = 4;
    }
}

Mat::~Mat() {
    if (dev && !external_memory) (void)hipFree(dev);
}

// Copies between host and device go over the current device's copy stream and wait for it.
static hipStream_t copy_stream() {
    int device = 0;
    hip_check(hipGetDevice(&device), "hipGetDevice");
    return static_cast<hipStream_t>(copy_stream(device));
}

std::shared_ptr<Mat> Mat::planned(int n, int h, int w, int c, DataType type, const std::string &name) {
    if (type == DataType::Bit && c % 64 != 0)
        throw std::runtime_error("Bit Mat needs a channel count that is a multiple of 64, got " + std::to_string(c));
    auto m = std::make_shared<Mat>(n, h, w, c, nullptr, type);
    m->external_memory = false;
    m->name = name;
    return m;
}

std::shared_ptr<Mat> Mat::planned(size_t len, DataType type, const std::string &name) {
    auto m = std::make_shared<Mat>((size_t)0, type, name);
    m->c = (int)len, m->elem_c = type == DataType::Bit ? (int)len * 64 : (int)len;
    m->data_num_ = len;
    return m;
}

void Mat::allocate() {
    if (!dev && !external_memory && bytes() > 0) hip_check(hipMalloc(&dev, bytes()), "hipMalloc");
}

void Mat::become_slice(std::shared_ptr<Mat> whole, int first) {
    whole->allocate();
    if (dev && !external_memory) hip_check(hipFree(dev), "hipFree");
    dev = static_cast<unsigned char *>(whole->dev) + (size_t)first * elemsize;
    ld = whole->c;
    external_memory = true;
    storage = std::move(whole);
    host_valid_ = false;
}

void Mat::gather_to(void *dst, void *stream) const {
    const size_t row = (size_t)c * elemsize, pitch = ld ? (size_t)ld * elemsize : row;
    hip_check(hipMemcpy2DAsync(dst, row, dev, pitch, row, total() / c, hipMemcpyDeviceToDevice, static_cast<hipStream_t>(stream)),
              "hipMemcpy2DAsync");
}

void Mat::upload(const void *host, size_t nbytes) {
    if (ld) throw std::runtime_error("Mat::upload: the tensor is a slice of another one");
    if (nbytes > bytes()) throw std::runtime_error("Mat::upload: source larger than the tensor");
    hip_check(hipMemcpyAsync(dev, host, nbytes, hipMemcpyHostToDevice, copy_stream()), "hipMemcpyAsync H2D");
    hip_check(hipStreamSynchronize(copy_stream()), "hipStreamSynchronize");
    host_valid_ = false;
}

void Mat::download(void *host, size_t nbytes, Staging *via) const {
    if (nbytes > bytes()) throw std::runtime_error("Mat::download: destination larger than the tensor");
    if (via && !ld) {
        via->download(host, dev, nbytes);
        return;
    }
    if (ld) {
        // whole pixels, and what is left of nbytes from the pixel behind them
        const size_t row = (size_t)c * elemsize, pitch = (size_t)ld * elemsize, rows = nbytes / row, rest = nbytes - rows * row;
        if (rows)
            hip_check(hipMemcpy2DAsync(host, row, dev, pitch, row, rows, hipMemcpyDeviceToHost, copy_stream()), "hipMemcpy2DAsync D2H");
        if (rest)
            hip_check(hipMemcpyAsync(static_cast<unsigned char *>(host) + rows * row, static_cast<const unsigned char *>(dev) + rows * pitch, rest,
                                     hipMemcpyDeviceToHost, copy_stream()),
                      "hipMemcpyAsync D2H");
        hip_check(hipStreamSynchronize(copy_stream()), "hipStreamSynchronize");
        return;
    }
    hip_check(hipMemcpyAsync(host, dev, nbytes, hipMemcpyDeviceToHost, copy_stream()), "hipMemcpyAsync D2H");
    hip_check(hipStreamSynchronize(copy_stream()), "hipStreamSynchronize");
}

std::vector<float> Mat::to_host_float() const {
    if (data_type != DataType::Float) throw std::runtime_error("to_host_float on a Bit Mat");
    std::vector<float> out(total());
    if (!out.empty()) download(out.data(), bytes());
    return out;
}

std::vector<uint64_t> Mat::to_host_bits() const {
    if (data_type != DataType::Bit) throw std::runtime_error("to_host_bits on a Float Mat");
    std::vector<uint64_t> out(total());
    if (!out.empty()) download(out.data(), bytes());
    return out;
}

void Mat::sync_to_host(Staging *via) const {
    if (host_valid_) return;
    if (host_.size() != bytes()) {
        host_.resize(bytes());
        data = host_.empty() ? nullptr : host_.data();
    }
    // the copy does not wait for work queued on other streams; a Net synchronises its own stream at the end of run()
    if (!host_.empty()) download(host_.data(), host_.size(), via);
    host_valid_ = true;
}

bool Mat::operator==(const Mat &m) const {
    if (this == &m || (dev != nullptr && dev == m.dev && c == m.c && ld == m.ld)) return true;
    if (!(elemsize == m.elemsize && n == m.n && w == m.w && h == m.h && c == m.c && data_type == m.data_type &&
          total() == m.total()))
        return false;
    sync_to_host();
    m.sync_to_host();
    if (data_type == DataType::Float) {
        const float *a = static_cast<const float *>(data), *b = static_cast<const float *>(m.data);
        for (size_t i = 0; i < total(); ++i) {
            if (std::isnan(a[i]) != std::isnan(b[i])) return false;
            if (std::abs(a[i] - b[i]) > 1e-5) return false;
        }
    } else {
        const uint64_t *a = static_cast<const uint64_t *>(data), *b = static_cast<const uint64_t *>(m.data);
        for (size_t i = 0; i < total(); ++i)
            if (a[i] != b[i]) return false;
    }
    return true;
}

void Mat::dump(const std::string &filename) const {
    if (data_type != DataType::Float) throw std::runtime_error("dump writes float Mats");
    std::ofstream ofs(filename);
    for (size_t i = 0; i < total(); ++i) ofs << (*this)[(int)i] << std::endl;
}

std::ostream &operator<<(std::ostream &os, const Mat &mat) {
    os << "n: " << mat.n << ", width: " << mat.w << ", height: " << mat.h << ", channels: " << mat.c << std::endl;
    mat.sync_to_host();
    const size_t shown = mat.total() < 10 ? mat.total() : 10;
    for (size_t i = 0; i < shown; ++i) {
        if (mat.data_type == DataType::Float)
            os << static_cast<const float *>(mat.data)[i] << ", ";
        else
            os << std::hex << static_cast<const uint64_t *>(mat.data)[i] << std::dec << ", ";
    }
    return os;
}

}  // namespace bnn
