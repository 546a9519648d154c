// The layers Net::prepare of the reference builds (dabnn/layers/{BinConv,FloatConv,
// Affine,Add,AvePool,MaxPool,Relu,PRelu,Concat,Split,Shuffle}.{h,cpp}); constructor
// signatures follow the reference.
#pragma once

#include "layer.h"

namespace bnn {

using css = const std::string &;

class FloatConv;

class BNN_API BinConv : public Layer {
   public:
    MatP input_mat;
    MatP binarized_mat;  // packed input of the direct method
    MatP col_mat;        // column matrix of the bgemm method; no memory while nobody needs it
    MatP weight_mat;
    MatP transposed_weight_mat;
    MatP output_mat;
    const int pad_h, pad_w, stride_h, stride_w;

    enum Method { DIRECT_CONV = 0, BGEMM = 1 };

    // Set by Net::prepare when the layers that follow are Affine (and Add) on this layer's output and the direct
    // kernel applies: the three run as one pass with identical results.
    MatP fused_a, fused_b, fused_shortcut;
    // Also set by Net::prepare: the fused pass of this layer writes the sign-packed copy of its result that the next
    // direct BinConv on that blob needs (fused_sign_out = that layer's binarized_mat), and a layer whose packed input
    // is made that way skips its own pack_mat (input_prepacked).
    MatP fused_sign_out;
    bool input_prepacked = false;
    // The packed input, the output or the packed output is a slice of a wider tensor (Mat::ld): dab_bconv runs, which
    // takes the distance between pixels, whatever the method.
    bool has_slices() const;

    // Also set by Net::prepare: this layer and the next one, `next_in_pass`, run as one pass (dab_bconv3x3_pair), which writes
    // neither this layer's output nor its packed copy; the next layer's own forward() has nothing left to do (inside_pass).
    std::shared_ptr<BinConv> next_in_pass;
    bool inside_pass = false;
    // Of the second layer of such a pass, where its result is only wanted pooled 2x2 (by `branch` of its reader) and as sign bits
    // (dab_bconv3x3_pair_pool): the pooled blob.  output_mat is then only made for who asks for it.
    MatP pooled_in_pass;
    const BinConv *first_in_pass = nullptr;
    void forward_pass(bool pooled) const;  // of the first layer: both layers
    // The layer by itself, for who asks for those blobs (which must have memory) after a run.
    void forward_alone() const override;

    // Also set by Net::prepare: the 1x1 convolution of this layer's shortcut branch runs in this layer's pass
    // (dab_bconv3x3_down), which does not write the branch's blob.
    std::shared_ptr<FloatConv> branch;
    MatP branch_pooled;  // the branch's pooled input, where input_mat is not written
    void forward_with_branch(float *branch_out) const;  // branch_out: where the branch's blob is wanted, or null

    BinConv(NetCP net, css name, css input, css weight, css output, int pad_h, int pad_w, int stride_h, int stride_w);
    void forward_impl() const override;
    std::string to_str() const override;
    Method method() const;
    bool reads_packed() const;  // works on the packed input (a producer may write it), not on the fp32 blob
    // The column matrix of the last forward(), from the packed input it left: for a layer that reads_packed() and that
    // somebody wants the matrix of.  col_mat must have memory.
    void fill_columns() const;

   private:
    int kernel_h() const { return weight_mat->h; }
    int kernel_w() const { return weight_mat->w; }
    bool direct_conv_compatible() const;
};

class BNN_API FloatConv : public Layer {
   public:
    MatP input_mat, weight_mat, bias_mat, output_mat;
    // Affine (and Relu) layers that follow on the output blob, applied in the convolution's epilogue when set
    MatP fused_a, fused_b;
    bool fused_relu = false;
    // A PRelu that follows instead of the Relu, and the packed copy of the result for the BinConvs that read it: the
    // convolution's epilogue makes both, and its output may be a slice of a wider tensor.
    MatP fused_slope, fused_sign_out;
    // Set by Net::prepare for a 1x1 convolution that reads the output of an AvePool 2x2 stride 2: the pool's input.
    // The layer then pools it itself and convolves the result; the pooled blob (input_mat) is written as a side product
    // when it has device memory, and is a shape without memory when the net dropped the blob.
    MatP fused_pool_input;
    // The same for a global AvePool (one window over the whole image) at small batch: fused_pool_input is its input.
    bool fused_pool_global = false;
    // The same for a MaxPool 2x2 stride 2 before large problems, with a Relu or a PRelu and slices: the pooled blob is only
    // made for who asks for it (MaxPool::inside_conv).
    bool fused_pool_max = false;
    // Set by Net::prepare when a MaxPool 3x3 stride 2 pad 1 is the only reader of the output: the pool's output blob,
    // the packed copy of it a direct BinConv wants (or null) and the workspace of the one-pass kernel.  output_mat is
    // null then: the convolution's result is never written.
    MatP fused_maxpool_out, fused_maxpool_sign, fused_maxpool_carry;
    // Set by Net::prepare: the binary convolution that adds this layer's result runs both (BinConv::branch); the layer by itself
    // makes output_mat, which must have memory, for who asks for it after a run.
    const BinConv *inside_block = nullptr;
    void forward_alone() const override;
    // Whether forward() can write the result a second time, and where to; set by the net for the launches it enqueues.
    bool can_copy() const { return output_mat && !output_mat->ld && !fused_pool_max && !fused_slope && !inside_block && (!fused_pool_input || fused_pool_global); }
    float *copy_to = nullptr;
    const int pad_h, pad_w, stride_h, stride_w, dilation;
    FloatConv(NetCP net, css name, css input, css weight, css bias, css output, int pad_h, int pad_w, int stride_h,
              int stride_w, int dilation);
    FloatConv(NetCP net, css name, css input, css weight, css output, int pad_h, int pad_w, int stride_h, int stride_w,
              int dilation);
    void forward_impl() const override;
    std::string to_str() const override;

   private:
    void check_operands() const;
};

class BNN_API Affine : public Layer {
   public:
    MatP data_mat, a_mat, b_mat;
    Affine(NetCP net, css name, css data, css a, css b);
    void forward_impl() const override;
};

class BNN_API Add : public Layer {
   public:
    MatP input1_mat, input2_mat;
    Add(NetCP net, css name, css input1, css input2);
    void forward_impl() const override;
};

class BNN_API Relu : public Layer {
   public:
    MatP data_mat;
    Relu(NetCP net, css name, css data);
    void forward_impl() const override;
};

class BNN_API PRelu : public Layer {
   public:
    MatP data_mat, slope_mat;
    bool inside_conv = false;  // set by Net::prepare: the float convolution before it applies it
    PRelu(NetCP net, css name, css data, css slope);
    void forward_impl() const override;
    std::string to_str() const override;
};

class BNN_API Concat : public Layer {
   public:
    MatP input1_mat, input2_mat, output_mat;
    bool in_place = false;  // set by Net::prepare: both inputs are slices of the output, written there by their producers
    Concat(NetCP net, css name, css input1, css input2, css output);
    void forward_impl() const override;
    std::string to_str() const override;
};

// dabnn/layers/Split.{h,cpp}: a Bit blob's words per pixel cut in two halves (first half -> output 1).
class BNN_API Split : public Layer {
   public:
    MatP input_mat, output_mat1, output_mat2;
    Split(NetCP net, css name, css input, css output1, css output2);
    void forward_impl() const override;
};

// dabnn/layers/Shuffle.{h,cpp}: the channel shuffle of a two-group network on packed words, in place.
class BNN_API Shuffle : public Layer {
   public:
    MatP data_mat;
    Shuffle(NetCP net, css name, css data);
    void forward_impl() const override;
};

class BNN_API AvePool : public Layer {
   public:
    MatP input_mat, output_mat;
    const int kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w;
    AvePool(NetCP net, css name, css input, css output, int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h,
            int stride_w);
    void forward_impl() const override;
};

class BNN_API MaxPool : public Layer {
   public:
    MatP input_mat, output_mat;
    // Set by Net::prepare when a direct BinConv reads the pooled blob: its packed input, written in the same pass.
    MatP fused_sign_out;
    bool inside_conv = false;  // set by Net::prepare: the 1x1 convolution behind it pools for itself
    const int kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w;
    MaxPool(NetCP net, css name, css input, css output, int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h,
            int stride_w);
    void forward_impl() const override;
    void forward_alone() const override;
    std::string to_str() const override;
};

}  // namespace bnn
