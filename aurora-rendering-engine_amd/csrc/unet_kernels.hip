// unet_kernels.hip — the denoiser's elementwise kernels on gfx950: input
// preparation, average pooling, Adam, the BF16 operand copies of the weights,
// and the MFMA lane-layout self-test.  The convolutions are in unet_conv.hip,
// the gradients in unet_grad.hip.
//
// No reference counterpart: the reference has no learned component.
#include "unet.hpp"

#include <algorithm>

namespace aur {
namespace {

union Pack8 {
    uint4 u;
    bf16x8 v;
    u16 h[8];
};

// ------------------------------------------------------- elementwise ---
// 2x2 average of BF16 activations, eight channels (one 16-byte load of
// each of the four pixels) per thread; C is a multiple of 8
__global__ void k_avgpool(const u16* __restrict__ in, int N, int H, int W, int C, u16* __restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // group of 8 output channels
    const int h2 = H / 2, w2 = W / 2, cg = C / 8;
    const size_t total = (size_t)N * h2 * w2 * cg;
    if (i >= total) return;
    const int g = (int)(i % cg);
    size_t q = i / cg;
    const int x = (int)(q % w2);
    q /= w2;
    const int y = (int)(q % h2);
    const int n = (int)(q / h2);
    auto at = [&](int yy, int xx) {
        Pack8 p;
        p.u = *reinterpret_cast<const uint4*>(in + (((size_t)n * H + yy) * W + xx) * C + 8 * g);
        return p;
    };
    const Pack8 a = at(2 * y, 2 * x), b = at(2 * y, 2 * x + 1), c = at(2 * y + 1, 2 * x), d = at(2 * y + 1, 2 * x + 1);
    Pack8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float s = (bf2f(a.h[k]) + bf2f(b.h[k])) + (bf2f(c.h[k]) + bf2f(d.h[k]));
        o.h[k] = f2bf(0.25f * s);
    }
    *reinterpret_cast<uint4*>(out + (((size_t)n * h2 + y) * w2 + x) * C + 8 * g) = o.u;
}

// network input: 16 channels = log(1 + radiance mean), albedo mean, normal
// mean, zeros; also keeps log(1 + radiance) for the residual output
__global__ void k_prep(const float* __restrict__ rgb, const float* __restrict__ alb, const float* __restrict__ nrm,
                       size_t npix, float inv_spp, u16* __restrict__ x, float* __restrict__ noisy_log) {
    const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= npix) return;
    Pack8 lo, hi;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float l = log1pf(fmaxf(rgb[3 * p + c] * inv_spp, 0.0f));
        noisy_log[3 * p + c] = l;
        lo.h[c] = f2bf(l);
        lo.h[3 + c] = f2bf(alb ? alb[3 * p + c] * inv_spp : 0.0f);
    }
    lo.h[6] = f2bf(nrm ? nrm[3 * p] * inv_spp : 0.0f);
    lo.h[7] = f2bf(nrm ? nrm[3 * p + 1] * inv_spp : 0.0f);
    hi.u = make_uint4(0, 0, 0, 0);
    hi.h[0] = f2bf(nrm ? nrm[3 * p + 2] * inv_spp : 0.0f);
    reinterpret_cast<uint4*>(x + 16 * p)[0] = lo.u;
    reinterpret_cast<uint4*>(x + 16 * p)[1] = hi.u;
}

// Adam on the FP32 master parameters
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       size_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// BF16 operand copies of one layer: forward [Cout][Kpad] (k = tap*Cin+ci)
// and data-gradient [Cin][Kpad'] (k' = tap'*Cout+co, tap' = 8 - tap)
__global__ void k_pack_weights(const float* __restrict__ w, int cout, int cin, int kpad, int kpad_t,
                               u16* __restrict__ wk, u16* __restrict__ wt) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int nf = cout * kpad, nt = cin * kpad_t;
    if (i < nf) {
        const int co = i / kpad, k = i % kpad;
        wk[i] = k < 9 * cin ? f2bf(w[(size_t)co * 9 * cin + k]) : (u16)0;
    } else if (i < nf + nt) {
        const int j = i - nf;
        const int ci = j / kpad_t, k = j % kpad_t;
        u16 v = 0;
        if (k < 9 * cout) {
            const int tap = k / cout, co = k % cout;
            v = f2bf(w[((size_t)co * 9 + (8 - tap)) * cin + ci]);
        }
        wt[j] = v;
    }
}

// 16x16x32 MFMA on one tile: the lane layout self-test
__global__ void k_mfma_selftest(const u16* A, const u16* B, float* D) {
    const int l = threadIdx.x;
    Pack8 a, b;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        a.h[j] = A[(l % 16) * 32 + 8 * (l / 16) + j];  // A is 16 x 32 row-major
        b.h[j] = B[(8 * (l / 16) + j) * 16 + l % 16];  // B is 32 x 16 row-major
    }
    floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) D[(4 * (l / 16) + r) * 16 + l % 16] = acc[r];
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// ---------------------------------------------------------------- host ---
Status avgpool2(const uint16_t* in, int N, int H, int W, int C, uint16_t* out, hipStream_t s) {
    if (C % 8) return Status{AURORA_ERR_INVALID, "avgpool: channel count must be a multiple of 8"};
    k_avgpool<<<nblocks((size_t)N * (H / 2) * (W / 2) * (C / 8)), 256, 0, s>>>(in, N, H, W, C, out);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status prep_input(const float* rgb, const float* alb, const float* nrm, size_t npix, float inv_spp, uint16_t* x,
                  float* noisy_log, hipStream_t s) {
    k_prep<<<nblocks(npix), 256, 0, s>>>(rgb, alb, nrm, npix, inv_spp, x, noisy_log);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status adam_step(float* w, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2, float eps,
                 int t, hipStream_t s) {
    const float c1 = 1.0f / (1.0f - powf(b1, (float)t)), c2 = 1.0f / (1.0f - powf(b2, (float)t));
    k_adam<<<nblocks(n), 256, 0, s>>>(w, g, m, v, n, lr, b1, b2, eps, c1, c2);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status pack_weights(const float* w, int cout, int cin, int kpad, int kpad_t, uint16_t* wk, uint16_t* wt,
                    hipStream_t s) {
    k_pack_weights<<<nblocks((size_t)cout * kpad + (size_t)cin * kpad_t), 256, 0, s>>>(w, cout, cin, kpad, kpad_t,
                                                                                       wk, wt);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status mfma_selftest(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s) {
    k_mfma_selftest<<<1, 64, 0, s>>>(A, B, D);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

}  // namespace aur
