// The operators of the CNN forward hot path, under the reference's class names so that an unmodified
// topology resolves to them through the registry: operation_convolution (on operation_general_conv),
// operation_convolutiondepthwise, operation_pooling, operation_eltwise, operation_binaryop, operation_relu,
// operation_innerproduct, operation_split. Each overrides the forward_gpu_* virtuals and calls the exhip C ABI.
#pragma once
#include <cfloat>
#include <map>

#include "operation.hpp"

namespace glasssix {
namespace excalibur {

// Convolution hyper-parameters as parsed by the reference (src/Excalibur/operation_general_conv.cpp:9-124),
// member names kept.
template <typename Dtype>
class operation_general_conv : public operation<Dtype> {
public:
    explicit operation_general_conv(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }

    int output_channel_ = 0;
    int kernel_size_w_ = 0, kernel_size_h_ = 0;
    int dilation_w_ = 1, dilation_h_ = 1;
    int stride_w_ = 1, stride_h_ = 1;
    int group_ = 1;
    int pad_left_ = 0, pad_right_ = 0, pad_top_ = 0, pad_bottom_ = 0;
    bool int8_scale_term_ = false;
    bool bias_term_ = false;
    int weight_data_size_ = 0;
    int activation_type_ = 0;
    int impl_type_ = 0;
    int output_pad_right_ = 0, output_pad_bottom_ = 0, output_dim_h_ = 0, output_dim_w_ = 0;
    int input_channels() const { return weight_data_size_ * group_ / output_channel_ / kernel_size_h_ / kernel_size_w_; }
};

template <typename Dtype>
class operation_convolutiondepthwise;
template <typename Dtype>
class operation_input;
template <typename Dtype>
class operation_reshape;

template <typename Dtype>
class operation_convolution : public operation_general_conv<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_convolution(const operation_param& param);
    ~operation_convolution() override;
    int init_weights() override;
    int init_weights(FILE* fp) override;

    // Dequantization scale per output channel, fabs(ws) <= 1e-6 ? 0 : 1.0f / (ws * fs), computed on the
    // host in float exactly as src/Excalibur/operation_convolution.cpp:400-403.
    std::vector<float> dequantize_scales() const;
    float featmap_scale() const;
    // device copies (created on first use)
    const float* bias_gpu();
    const float* scale_gpu();
    // weights packed for the MFMA kernel for one input geometry; cached per (dtype, n, h, w, c_stride)
    const void* packed_weights(int dtype, const exhip_conv_desc& d);
    // A holder that keeps the pointer across forwards (a fused plan) pins the copy: pinned copies are never evicted.
    const void* pin_packed_weights(int dtype, const exhip_conv_desc& d);
    void unpin_packed_weights(const void* ptr);
    exhip_conv_desc describe(int n, int h, int w, int c_stride, int k_stride) const;
    // The activation layer behind this one, applied in the kernel's epilogue by the next forward calls: post_op 0 = none,
    // else 1 + EXHIP_UNARY_* with its two parameters; relu = a ReLU layer. False, and nothing set, where this layer's
    // kernel cannot apply it (the definition-order kernel of grouped layers, the sigmoid's double-precision exp).
    virtual bool set_post_activation(int post_op, float alpha, float beta, bool relu);
    // the same for a PReLU layer: its device-resident slopes, one per output channel or one for all
    virtual bool set_post_prelu(const float* slopes, bool shared);
    void clear_post() {
        post_op_ = 0; post_alpha_ = post_beta_ = 0.f; post_relu_ = false;
        post_slope_ = nullptr; post_slope_shared_ = false;
        post_sum_.reset(); post_sum_used_ = false; post_sum_last_ = false;
    }
    // fp16 layers: the other operand of the two-input sum layer behind this one, or (behind_activation) behind the
    // activation layer set with set_post_activation / set_post_prelu. The next forward adds it in the kernel's epilogue
    // if it can (NHWC result, an NHWC operand of the result's shape) and says so in post_sum_used().
    void set_post_sum(const std::shared_ptr<memory::tensor<unsigned short>>& other, bool behind_activation = false) {
        post_sum_ = other; post_sum_used_ = false; post_sum_last_ = behind_activation;
    }
    bool post_sum_used() const { return post_sum_used_; }
    // fp16: this layer, a pointwise one, with the 3x3 depthwise layer that it alone reads in front of it in one kernel, each with
    // the layers set behind it; `bottoms` are the depthwise layer's. False, with nothing done, where the pair runs as two layers.
    bool forward_behind_depthwise(operation_convolutiondepthwise<Dtype>& dw, const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops);
    // the same with the pointwise layer `first` that the depthwise layer alone reads: a mobile network's block; `bottoms` are that layer's
    bool forward_block(operation_convolution<Dtype>& first, operation_convolutiondepthwise<Dtype>& dw, const tensor_list<unsigned short>& bottoms,
                       tensor_list<unsigned short>& tops);
    // fp16: this layer and `next`, pointwise ones of which neither reads the other, in one launch where their forms allow it. False, with nothing done, where a layer's
    // tensors are not for it.
    bool forward_beside(operation_convolution<Dtype>& next, const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops,
                        const tensor_list<unsigned short>& next_bottoms, tensor_list<unsigned short>& next_tops);
    bool beside_form(const tensor_list<unsigned short>& bottoms, exhip_conv_desc* d) const;
    // fp16: this layer, of at most four input channels, straight on its NCHW input, with the Input layer that it alone reads in front of it
    // (or NULL) and the layers set behind it; `bottoms` are the first one's. False, with nothing done, where the layers run by themselves.
    bool forward_stem(operation_input<Dtype>* input, const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops);
    // fp16: this layer, a pointwise one, with the Reshape of its channels into groups and the Transpose of the last two axes behind it (a detection
    // head) as one launch; `tops` are the Transpose layer's. False, with nothing done, where the three run by themselves.
    bool forward_head(const operation_reshape<Dtype>& reshape, const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops);
    // Whether that launch is for these layers and pixels; the layers by themselves then make the NCHW result from NHWC rows, so that they run the
    // kernel, and add in the order, of the one launch. (Others do not: 128 -> 255 3x3 at 16 x 80 x 80 takes 80 us straight to NCHW, 123 through rows.)
    bool head_form(const operation_reshape<Dtype>& reshape, const tensor_list<unsigned short>& bottoms, exhip_conv_desc* d, std::vector<int>* to) const;
    void set_through_rows(bool on) { through_rows_ = on; }
    // int8 layers on the MFMA kernel. The next forward calls also write the int8 NHWC form of the output that a reader
    // quantizing with `fs` into `stride` channels per pixel would make of it (attached to the top blob as its
    // `quantized` copy), and with `only` leave the float data unwritten; fs = 0 switches it off. False where this
    // layer cannot (not int8, another kernel).
    virtual bool set_quantized_output(float fs, int stride, bool only);
    // what this layer's quantizer produces from its input: the scale and the channel stride (0, 0 if it has none)
    virtual void quantized_input(float* fs, int* stride) const;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_i8(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
    bool mfma_path_ok() const;
    bool through_rows_ = false;
    const unsigned short* sum_operand(const tensor_list<unsigned short>& tops, exhip_conv_desc* d);
    int post_op_ = 0;
    float post_alpha_ = 0.f, post_beta_ = 0.f;
    bool post_relu_ = false;
    const float* post_slope_ = nullptr;
    bool post_slope_shared_ = false;
    std::shared_ptr<memory::tensor<unsigned short>> post_sum_;
    bool post_sum_used_ = false, post_sum_last_ = false;
    float q_out_fs_ = 0.f;
    int q_out_stride_ = 0;
    bool q_out_only_ = false;

private:
    struct packed_entry { void* ptr; size_t bytes; unsigned long long last_use; int pins = 0; };
    unsigned long long packed_clock_ = 0;
    std::map<std::vector<int>, packed_entry> packed_;
    std::shared_ptr<memory::tensor<float>> scale_dev_;
};

template <typename Dtype>
class operation_convolutiondepthwise : public operation_convolution<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_convolutiondepthwise(const operation_param& param) : operation_convolution<Dtype>(param) {}
    bool set_post_activation(int, float, float, bool) override { return false; }
    bool set_post_prelu(const float* slopes, bool shared) override;  // the 3x3 kernels apply it; other shapes do not pair
    bool set_quantized_output(float, int, bool) override { return false; }
    void quantized_input(float* fs, int* stride) const override { *fs = 0.f; *stride = 0; }

protected:
    friend class operation_convolution<Dtype>;
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_i8(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
    bool fast3x3() const;
};

template <typename Dtype>
class operation_pooling : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_pooling(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }

    int kernel_size_w_ = 0, kernel_size_h_ = 0, stride_w_ = 1, stride_h_ = 1;
    int pad_left_ = 0, pad_right_ = 0, pad_top_ = 0, pad_bottom_ = 0;
    int type_ = 0;  // 0 MAX, 1 AVE
    bool global_pooling_ = false;
    int pad_mode_ = 1;  // 0 ceil, 1 floor
    int avgpool_count_include_pad_ = 0;
    // effective window for an input of h x w (global pooling overrides kernel, stride and padding)
    void geometry(int h, int w, int* kh, int* kw, int* sh, int* sw, int* pt, int* pb, int* pl, int* pr, int* oh, int* ow) const;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

template <typename Dtype>
class operation_eltwise : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_eltwise(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    enum eltwise_type { PROD = 0, SUM = 1, MAX = 2 };
    int type_ = SUM;
    std::vector<float> coeffs_;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
    void eltwise_general_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops);
};

template <typename Dtype>
class operation_binaryop : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_binaryop(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int op_type_ = 0;  // 0 ADD, 1 SUB, 2 MUL, 3 DIV
    int with_scalar_ = 0;
    float coef_ = 0.f;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

template <typename Dtype>
class operation_relu : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_relu(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    float slope_ = 0.f;  // parsed and ignored, as in the reference (src/Excalibur/operation_relu.cpp:14-17)

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

template <typename Dtype>
class operation_split : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_split(const operation_param& param) : operation<Dtype>(param) {}
    const char* type() const override { return this->params_.type_.c_str(); }

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

template <typename Dtype>
class operation_innerproduct : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_innerproduct(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int init_weights() override;
    int init_weights(FILE* fp) override;
    int num_output_ = 0;
    bool bias_term_ = false;
    int weight_data_size_ = 0;
    bool int8_scale_term_ = false;
    int activation_type_ = 0;  // parsed, never applied (as in the reference)

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
    // The reference reads the int8 blob (one weight scale, one feature-map scale) but has no forward for it
    // (include/Excalibur/operation.hpp:353-357). Here the layer is the int8 1x1 convolution of the flattened input, with
    // the int8 convolution's arithmetic: q8(x * fs), int32 sum, fmaf(acc, 1 / (ws * fs), bias).
    void forward_gpu_i8(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    std::shared_ptr<memory::tensor<float>> scale_dev_;
};

// ---- activation / glue layers of the shipped topologies (float32 kernels; fp16 pipelines take the base class's
// convert-and-call wrapper) ----

// HardSwish, LeakyRelu, Sigmoid, HardSigmoid: one elementwise kernel with two parameters.
// src/Excalibur/operation_hardswish.cpp:10-63, operation_leakyrelu.cpp:12-58, operation_sigmoid.cpp:10-33,
// operation_hardsigmoid.cpp:10-46 (keys 0 = alpha, 1 = beta).
template <typename Dtype>
class operation_unary : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    operation_unary(const operation_param& param, int op, float alpha, float beta, int n_keys);
    const char* type() const override { return this->params_.type_.c_str(); }
    int op_;
    float alpha_, beta_;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};
template <typename Dtype>
struct operation_hardswish : operation_unary<Dtype> {
    explicit operation_hardswish(const operation_param& p) : operation_unary<Dtype>(p, EXHIP_UNARY_HARDSWISH, 0.f, 0.f, 2) {}
};
template <typename Dtype>
struct operation_leakyrelu : operation_unary<Dtype> {
    explicit operation_leakyrelu(const operation_param& p) : operation_unary<Dtype>(p, EXHIP_UNARY_LEAKYRELU, 0.f, 0.f, 1) {}
};
template <typename Dtype>
struct operation_sigmoid : operation_unary<Dtype> {
    explicit operation_sigmoid(const operation_param& p) : operation_unary<Dtype>(p, EXHIP_UNARY_SIGMOID, 0.f, 0.f, 0) {}
};
template <typename Dtype>
struct operation_hardsigmoid : operation_unary<Dtype> {
    explicit operation_hardsigmoid(const operation_param& p) : operation_unary<Dtype>(p, EXHIP_UNARY_HARDSIGMOID, 0.2f, 0.5f, 2) {}
};

// src/Excalibur/operation_clip.cpp:11-58: keys 0 = lower bound, 1 = upper bound.
template <typename Dtype>
struct operation_clip : operation_unary<Dtype> {
    explicit operation_clip(const operation_param& p) : operation_unary<Dtype>(p, EXHIP_UNARY_CLIP, -FLT_MAX, FLT_MAX, 2) {}
};

// src/Excalibur/operation_prelu.cpp:9-124: key 0 = number of slopes (1 = shared), blob = the slopes.
template <typename Dtype>
class operation_prelu : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_prelu(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int init_weights() override;
    int init_weights(FILE* fp) override;
    int num_slope_ = 0;
    bool share_channel_ = false;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_batchnorm.cpp:10-156: keys 0 = channels, 1 = eps; blob = slope, mean, var, bias;
// a = bias - slope*mean/sqrt(var + eps), b = slope/sqrt(var + eps) at load time, y = b*x + a.
template <typename Dtype>
class operation_batchnorm : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_batchnorm(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int init_weights() override;
    int init_weights(FILE* fp) override;
    int channels_ = 0;
    float eps_ = 0.f;
    std::shared_ptr<memory::tensor<float>> a_, b_;
    // fp16 pipeline: the activation layer on the next line (an EXHIP_UNARY_* operation other than the sigmoid) runs in this
    // layer's kernel when the blob is NHWC; post_used() says whether it did.
    void set_post_unary(int op, float alpha, float beta) { post_unary_ = op; post_alpha_ = alpha; post_beta_ = beta; post_used_ = false; }
    void clear_post() { post_unary_ = -1; post_used_ = false; }
    bool post_used() const { return post_used_; }

protected:
    int post_unary_ = -1;
    float post_alpha_ = 0.f, post_beta_ = 0.f;
    bool post_used_ = false;
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
    void fold();
};

// src/Excalibur/operation_input.cpp:10-151: keys 0/1/2 = w/h/c, 3 = means, 4 = scales; (x - mean[c]) * scale[c].
template <typename Dtype>
class operation_input : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_input(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int w_ = 0, h_ = 0, c_ = 0;
    std::vector<float> means_, vars_;
    std::shared_ptr<memory::tensor<float>> means_dev_, vars_dev_;
    void upload_tables(int ch);

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_concat.cpp:10-103: key 0 = axis - 2 (the files carry -1 for the channel axis).
template <typename Dtype>
class operation_concat : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_concat(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int axis_ = 0;
    // fp16 pipeline: the BatchNorm layer on the next line (its device-resident a / b; null = none) and the activation layer
    // behind that (-1 = none) run in this layer's kernel when every blob is NHWC; post_used() says whether they did.
    void set_post(const float* bn_a, const float* bn_b, int unary_op, float alpha, float beta) {
        post_bn_a_ = bn_a; post_bn_b_ = bn_b; post_unary_ = unary_op; post_alpha_ = alpha; post_beta_ = beta; post_set_ = true; post_used_ = false;
    }
    void clear_post() { post_set_ = false; post_used_ = false; post_bn_a_ = post_bn_b_ = nullptr; post_unary_ = -1; }
    bool post_used() const { return post_used_; }
    // fp16: this layer and the max pools with windows 5, 9 and 13 of x in front of it, whose results stand behind x in it, as one launch. False, with nothing done,
    // where the four run by themselves.
    bool forward_pyramid(const std::shared_ptr<memory::tensor<unsigned short>>& x, tensor_list<unsigned short>& tops);

protected:
    const float *post_bn_a_ = nullptr, *post_bn_b_ = nullptr;
    int post_unary_ = -1;
    float post_alpha_ = 0.f, post_beta_ = 0.f;
    bool post_set_ = false, post_used_ = false;
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_interp.cpp:185-268: keys 0 = type (1 nearest), 1 -> width scale, 2 -> height scale,
// 3 / 4 = output width / height, 6 = align corners. Nearest without align-corners is the form on the path.
template <typename Dtype>
class operation_interp : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_interp(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int resize_type_ = 0, output_width_ = 0, output_height_ = 0, align_corner_ = 0;
    float width_scale_ = 1.f, height_scale_ = 1.f;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_yolov5focus.cpp:12-50.
template <typename Dtype>
class operation_yolov5focus : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_yolov5focus(const operation_param& param) : operation<Dtype>(param) {}
    const char* type() const override { return this->params_.type_.c_str(); }

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_reshape.cpp:8-131: keys 0 / 1 / 2 = new width / height / channels (-233 when absent: that
// dimension is then derived from the element count, in the order channels, height, width), 3 = permute (unused). The
// bottom tensor's shape is changed in place and the top is the same tensor.
template <typename Dtype>
class operation_reshape : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_reshape(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int n_ = 0, c_ = -233, h_ = -233, w_ = -233, permute_ = 0;
    // the shape the layer gives a tensor of `old_shape` with `count` elements
    std::vector<int> new_shape(const std::vector<int>& old_shape, int count) const;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_flatten.cpp:11-113: key 0 = axis (default 1); a copy with shape [n][1][h'][w'].
template <typename Dtype>
class operation_flatten : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_flatten(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int axis_ = 1;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
};

// src/Excalibur/operation_softmax.cpp:10-96: key 0 = axis (read, not used: the sum always runs over the channels).
template <typename Dtype>
class operation_softmax : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_softmax(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    int axis_ = 0;

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
};

// src/Excalibur/operation_transpose.cpp:9-70: key 0 = order of (h, w, c) as "a,b,c". (0,1,2) passes the tensor on,
// (1,0,2) swaps rows and columns of every plane; the reference's other orders index past their planes and are refused.
template <typename Dtype>
class operation_transpose : public operation<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_transpose(const operation_param& param);
    const char* type() const override { return this->params_.type_.c_str(); }
    std::vector<int> perms_{0, 1, 2};

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;
    void forward_gpu_f16(const tensor_list<unsigned short>& bottoms, tensor_list<unsigned short>& tops) override;
};

// src/Excalibur/operation_deconvolution.cpp:11-171: the convolution's keys; float32 weights [C][K][kh][kw]; group 1.
template <typename Dtype>
class operation_deconvolution : public operation_general_conv<Dtype> {
public:
    template <typename T>
    using tensor_list = typename operation<Dtype>::template tensor_list<T>;
    explicit operation_deconvolution(const operation_param& param) : operation_general_conv<Dtype>(param) {}
    ~operation_deconvolution() override;
    int init_weights() override;
    int init_weights(FILE* fp) override;
    // A 2x2 stride-2 layer without padding gives every output pixel one input pixel and one tap: four 1x1 convolutions whose
    // results interleave (EXHIP_PLACE_SHUFFLED). Their packed weights and their bias, made once.
    bool four_pointwise() const;
    int deconv_input_channels() const { return this->weight_data_size_ / (this->output_channel_ * this->kernel_size_h_ * this->kernel_size_w_); }
    const void* pointwise_weights(const exhip_conv_desc& d);
    const float* pointwise_bias();

protected:
    void forward_gpu_f32(const tensor_list<float>& bottoms, tensor_list<float>& tops) override;

private:
    void* pointwise_ = nullptr;
    size_t pointwise_bytes_ = 0;
    std::shared_ptr<memory::tensor<float>> pointwise_bias_;
};

}  // namespace excalibur
}  // namespace glasssix
