// unet.hpp — internal interface of the denoiser: kernel launchers
// (unet_conv.hip, unet_grad.hip, unet_kernels.hip) and the U-Net that strings
// them together (unet.hip).
#pragma once

#include "internal.hpp"

namespace aur {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16;

__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((uint32_t)h << 16); }
// round to nearest even (gfx950's v_cvt_pk_bf16_f32; NaN stays NaN)
__device__ __forceinline__ u16 f2bf(float f) { return __builtin_bit_cast(u16, (__bf16)f); }

// Convolution input: full-resolution A (Ca channels) concatenated with a
// half-resolution B (Cb channels) read through nearest upsampling.
struct ConvIn {
    const uint16_t* a;
    const uint16_t* b;
    int ca, cb;
};

// bias + ReLU; pool: also the 2x2 average of the output (where conv_pools says so)
Status conv_relu(const ConvIn& in, const uint16_t* w, const float* bias, uint16_t* out, uint16_t* pool, int N, int H,
                 int W, int cout, hipStream_t s);
// the size from which conv_relu can pool
bool conv_pools(int N, int H, int W);
// the output layer: 3 floats per pixel, the residual, or (noisy given) the image
// max(expm1(noisy + residual), 0)
Status conv_residual(const ConvIn& in, const uint16_t* w, const float* bias, const float* noisy, float* out, int N,
                     int H, int W, hipStream_t s);
// data gradient of a gradient g of cg channels: BF16 masked by act > 0, or FP32
Status conv_data_grad(const uint16_t* g, int cg, const uint16_t* w, const uint16_t* act, uint16_t* out, int N, int H,
                      int W, int cout, hipStream_t s);
Status conv_data_grad_f32(const uint16_t* g, int cg, const uint16_t* w, float* out, int N, int H, int W, int cout,
                          hipStream_t s);

// Weight gradient of one layer with respect to one part of its input.
struct DwPart {
    const uint16_t *x, *g;  // the part (cx channels; half: at half resolution), the layer's output gradient
    int cx, cout, cin, ci0; // channels; ci0: the part's first channel in the layer's input of cin
    bool half;
    int N, H, W;
    float *dw, *db;         // [cout][9][cin]; db null: not this part's
};
constexpr uint32_t kDwBlocks = 128;  // most blocks, and partial sums, of a part
size_t dw_partial_floats(const DwPart& p);
// all parts; scratch holds the sum of their dw_partial_floats
Status weight_grads(const DwPart* parts, int n, float* scratch, hipStream_t s);
Status avgpool2(const uint16_t* in, int N, int H, int W, int C, uint16_t* out, hipStream_t s);
Status upsample_grad(const float* d, const uint16_t* act, int N, int H, int W, int C, uint16_t* g, hipStream_t s);
Status skip_grad(const float* skip, const float* pool, const uint16_t* act, int N, int H, int W, int C, uint16_t* g,
                 hipStream_t s);
Status prep_input(const float* rgb, const float* alb, const float* nrm, size_t npix, float inv_spp, uint16_t* x,
                  float* noisy_log, hipStream_t s);
Status loss_grad(const float* res, const float* noisy_log, const float* target, size_t npix, int kind, uint16_t* g,
                 float* loss_partial, hipStream_t s);
Status adam_step(float* w, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2, float eps,
                 int t, hipStream_t s);
Status pack_weights(const float* w, int cout, int cin, int kpad, int kpad_t, uint16_t* wk, uint16_t* wt,
                    hipStream_t s);
Status mfma_selftest(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s);

// 4-level U-Net (channels 32/48/64/64), 15 3x3 convolutions.
class Unet {
   public:
    struct Layer {
        int a, b;          // activation slots of the A / B inputs (b < 0: none)
        int out;           // activation slot written
        int ca, cb, cout;  // channels
        int level;         // resolution level 0..3
        bool relu;
        int kpad, kpad_t;
        size_t w_off, b_off;
        DevBuf wk, wt;     // BF16 forward / data-gradient weight copies
    };
    explicit Unet(hipStream_t s) : s_(s) {}
    Status init(uint32_t seed);
    size_t param_count() const { return n_params_; }
    Status get_params(float* host);
    Status set_params(const float* host);
    // forward on N images of H x W (H, W multiples of 8): the denoised image
    // into img, or (img null) the residual, kept for backward
    Status forward(const float* rgb, const float* alb, const float* nrm, float inv_spp, int N, int H, int W,
                   float* img);
    // loss against targets (mean radiance) and gradients into grads_
    Status backward(const float* target, float* loss);
    Status adam(float lr);
    void set_loss(int kind) { loss_kind_ = kind; }  // 0 log-space L2, 1 relative L2
    Status grads_to_host(float* host);
    void release();

   private:
    Status alloc(int N, int H, int W);
    Status repack();
    hipStream_t s_;
    std::vector<Layer> layers_;
    size_t n_params_ = 0;
    DevBuf params_, grads_, m_, v_;
    int N_ = 0, H_ = 0, W_ = 0;
    int t_ = 0;
    int loss_kind_ = 0;
    static constexpr int kSlots = 19;  // x, 14 hidden, 3 pools, out
    DevBuf act_[kSlots];               // BF16 activations (slot 18: the FP32 residual, 3 per pixel)
    DevBuf grad_[kSlots];              // BF16 gradients of the layers' outputs, masked by their ReLU
    // FP32 gradients that are summed with another one: of the skip connections'
    // and the pooled slots, and of a decoder's upsampled input (full resolution)
    DevBuf fgrad_[kSlots], dup_;
    DevBuf noisy_log_, scratch_, loss_part_;
    int slot_c_[kSlots] = {0};
    int slot_lv_[kSlots] = {0};
};

}  // namespace aur
