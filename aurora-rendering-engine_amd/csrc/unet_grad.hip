// unet_grad.hip — the denoiser's weight and bias gradients on MFMA, their
// reduction, and the elementwise steps between the data-gradient convolutions
// of the backward pass.
//
// No reference counterpart: the reference has no learned component.
#include "unet.hpp"

#include <algorithm>

namespace aur {
namespace {

union Frag {
    uint4 u;
    uint32_t w[4];
    bf16x8 v;
};

// ---------------------------------------------------- weight gradient ---
// dW[co][tap][ci] = sum_p g[p][co] * X[p + tap][ci]: MFMA with M = 16 output
// channels, N = 16 input channels, K = 32 pixels of a row, and both operands
// need consecutive pixels of one channel.  A block stages tiles of 2 rows x 64
// pixels of g, and of X with its halo, in shared memory transposed to [channel]
// [pixel] (16-byte loads of 8 channels, 4 pixels per thread, regrouped by byte
// permutes), so an operand fragment is one 16-byte read, and the three column
// shifts of a row are taken from a 12-pixel window in registers.  A wave owns
// one input-channel tile with every output-channel tile and all 9 taps (for 16
// and 32 input channels the waves split the pixels instead, and are summed at
// the end).  Gathering each operand value by itself cost 79 VALU instructions
// per MFMA.  The bias gradient is one more MFMA against ones.
//
// A launch takes all layers of one shape as jobs: the coarse levels have few
// tiles, and one launch per layer left most of the chip idle.  Loss and
// gradients of an 8 x 128^2 batch 1296 -> 793 us: the weight gradients 302 -> 190
// us in 9 launches instead of 15, the sums of their partials 121 -> 35 in one
// instead of 15, the bias gradients (147 us, 30 launches) in them, and the masks,
// fills and adds of FP32 gradients (190 us, 40 launches) in the convolutions'
// epilogues.
constexpr int kRows = 2, kPix = 64, kPixStride = 72;  // 144 bytes: 16 channels start in distinct banks
constexpr int kMaxJobs = 6;
struct DwJob {
    const u16 *x, *g;
    float* part;           // nblk x ((9 * NCO * NCI) * 256 + 16 * NCO) floats
    int N, H, W, half;     // half: X is read at half resolution through nearest upsampling
    uint32_t nblk, first;  // blocks of the job, first block in the launch
};
struct DwArgs {
    DwJob job[kMaxJobs];
    int n;
};

// 4 pixels x 8 channels to 8 channels x 4 pixels
__device__ __forceinline__ void store_transposed(u16* dst, const uint4 p[4]) {
    const uint32_t a[4][4] = {{p[0].x, p[0].y, p[0].z, p[0].w},
                              {p[1].x, p[1].y, p[1].z, p[1].w},
                              {p[2].x, p[2].y, p[2].z, p[2].w},
                              {p[3].x, p[3].y, p[3].z, p[3].w}};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint2 even = make_uint2(__builtin_amdgcn_perm(a[1][d], a[0][d], 0x05040100u),
                                      __builtin_amdgcn_perm(a[3][d], a[2][d], 0x05040100u));
        const uint2 odd = make_uint2(__builtin_amdgcn_perm(a[1][d], a[0][d], 0x07060302u),
                                     __builtin_amdgcn_perm(a[3][d], a[2][d], 0x07060302u));
        *reinterpret_cast<uint2*>(dst + (2 * d) * kPixStride) = even;
        *reinterpret_cast<uint2*>(dst + (2 * d + 1) * kPixStride) = odd;
    }
}

constexpr int dw_split(int nci) { return nci == 1 ? 4 : nci == 2 ? 2 : 1; }
constexpr int dw_lds(int nci, int nco) {
    const int stage = ((kRows + 2) * nci * 16 + kRows * nco * 16) * kPixStride * 2;
    const int sum = dw_split(nci) > 1 ? (9 * nco * nci * 256 + nco * 256) * 4 : 0;
    return stage > sum ? stage : sum;
}

template <int NCI, int NCO>
__global__ __launch_bounds__(256) void k_dw(DwArgs args) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int C = 16 * NCI, CO = 16 * NCO, SPLIT = dw_split(NCI);
    u16* const xt = reinterpret_cast<u16*>(smem);  // [row][channel][pixel x0-2 ..]
    u16* const gt = xt + (kRows + 2) * C * kPixStride;
    int jn = 0;
    while (jn + 1 < args.n && blockIdx.x >= args.job[jn + 1].first) ++jn;
    const DwJob& J = args.job[jn];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int ci = SPLIT == 4 ? 0 : SPLIT == 2 ? (wave & 1) : wave;
    const int part_of = SPLIT == 4 ? wave : SPLIT == 2 ? (wave >> 1) : 0;
    const int H = J.H, W = J.W;
    const uint32_t segs = (W + kPix - 1) / kPix, bands = (H + kRows - 1) / kRows;
    const uint32_t tiles = (uint32_t)J.N * bands * segs, blk = blockIdx.x - J.first;
    const uint32_t t0 = (uint32_t)((uint64_t)tiles * blk / J.nblk), t1 = (uint32_t)((uint64_t)tiles * (blk + 1) / J.nblk);
    floatx4 acc[NCO][9], accb[NCO];
#pragma unroll
    for (int t = 0; t < NCO; ++t) {
        accb[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 9; ++k) acc[t][k] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    Frag ones;
    ones.u = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    for (uint32_t tl = t0; tl < t1; ++tl) {
        const int x0 = (int)(tl % segs) * kPix, y0 = (int)((tl / segs) % bands) * kRows, n = (int)(tl / (segs * bands));
        // X: rows y0-1 .., pixels x0-2 .. x0+65 in groups of 4 (x0 - 2 is even: a
        // half-resolution pair shares its pixel)
        constexpr int XU = (kRows + 2) * 17 * (C / 8), XJ = (XU + 255) / 256;
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const int u = tid + 256 * j;
            if (u < XU) {
                const int pg = u % 17, q = u / 17, r = q % (kRows + 2), g8 = q / (kRows + 2);
                const int y = y0 - 1 + r, x = x0 - 2 + 4 * pg;
                uint4 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = make_uint4(0, 0, 0, 0);
                    if (J.half && (i & 1)) {
                        if ((unsigned)(x + i) < (unsigned)W) v[i] = v[i - 1];
                    } else if ((unsigned)y < (unsigned)H && (unsigned)(x + i) < (unsigned)W) {
                        const size_t px = J.half ? ((size_t)n * (H >> 1) + (y >> 1)) * (W >> 1) + ((x + i) >> 1)
                                                 : ((size_t)n * H + y) * W + x + i;
                        v[i] = *reinterpret_cast<const uint4*>(J.x + px * C + 8 * g8);
                    }
                }
                store_transposed(xt + (r * C + 8 * g8) * kPixStride + 4 * pg, v);
            }
        }
        constexpr int GU = kRows * 16 * (CO / 8), GJ = (GU + 255) / 256;
#pragma unroll
        for (int j = 0; j < GJ; ++j) {
            const int u = tid + 256 * j;
            if (u < GU) {
                const int pg = u % 16, q = u / 16, r = q % kRows, g8 = q / kRows;
                const int y = y0 + r, x = x0 + 4 * pg;
                uint4 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = make_uint4(0, 0, 0, 0);
                    if (y < H && x + i < W)
                        v[i] = *reinterpret_cast<const uint4*>(J.g + (((size_t)n * H + y) * W + x + i) * CO + 8 * g8);
                }
                store_transposed(gt + (r * CO + 8 * g8) * kPixStride + 4 * pg, v);
            }
        }
        __syncthreads();
        if (ci < NCI) {
#pragma unroll
            for (int ch = 0; ch < kRows * 2; ++ch) {
                const int r = ch >> 1, c = ch & 1;
                if (ch % SPLIT != part_of || y0 + r >= H || x0 + 32 * c >= W) continue;  // wave-uniform
                Frag a[NCO];
#pragma unroll
                for (int t = 0; t < NCO; ++t)
                    a[t].u = *reinterpret_cast<const uint4*>(gt + (r * CO + 16 * t + m) * kPixStride + 32 * c + 8 * kg);
#pragma unroll
                for (int dy = 0; dy < 3; ++dy) {
                    // pixels x - 2 .. x + 9 of this lane's first pixel x, two per word
                    const u16* src = xt + ((r + dy) * C + 16 * ci + m) * kPixStride + 32 * c + 8 * kg;
                    const uint4 lo = *reinterpret_cast<const uint4*>(src);
                    const uint2 up = *reinterpret_cast<const uint2*>(src + 8);
                    const uint32_t d[6] = {lo.x, lo.y, lo.z, lo.w, up.x, up.y};
                    uint32_t s[5];  // pixels (x - 1, x), (x + 1, x + 2), ...
#pragma unroll
                    for (int k = 0; k < 5; ++k) s[k] = __builtin_amdgcn_alignbit(d[k + 1], d[k], 16);
                    Frag b[3];
                    b[0].u = make_uint4(s[0], s[1], s[2], s[3]);
                    b[1].u = make_uint4(d[1], d[2], d[3], d[4]);
                    b[2].u = make_uint4(s[1], s[2], s[3], s[4]);
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int t = 0; t < NCO; ++t)
                            acc[t][3 * dy + dx] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t].v, b[dx].v, acc[t][3 * dy + dx], 0, 0, 0);
                }
                if (ci == 0) {
#pragma unroll
                    for (int t = 0; t < NCO; ++t)
                        accb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t].v, ones.v, accb[t], 0, 0, 0);
                }
            }
        }
        __syncthreads();  // the tiles are staged anew
    }
    // D[4*kg + r][m]: row = co offset, column = ci offset
    if constexpr (SPLIT > 1) {
        // waves that split the pixels, summed in order through shared memory
        float* const sum = reinterpret_cast<float*>(smem);
        for (int k = SPLIT - 1; k > 0; --k) {
            if (part_of == k) {
#pragma unroll
                for (int t = 0; t < NCO; ++t) {
#pragma unroll
                    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            sum[((tap * NCO + t) * NCI + ci) * 256 + (4 * kg + r) * 16 + m] = acc[t][tap][r];
                    if (ci == 0) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            sum[(9 * NCO * NCI + t) * 256 + (4 * kg + r) * 16 + m] = accb[t][r];
                    }
                }
            }
            __syncthreads();
            if (part_of == k - 1) {
#pragma unroll
                for (int t = 0; t < NCO; ++t) {
#pragma unroll
                    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[t][tap][r] += sum[((tap * NCO + t) * NCI + ci) * 256 + (4 * kg + r) * 16 + m];
                    if (ci == 0) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            accb[t][r] += sum[(9 * NCO * NCI + t) * 256 + (4 * kg + r) * 16 + m];
                    }
                }
            }
            __syncthreads();
        }
    }
    if (ci < NCI && part_of == 0) {
        float* part = J.part + (size_t)blk * (9 * NCO * NCI * 256 + CO);
#pragma unroll
        for (int t = 0; t < NCO; ++t) {
#pragma unroll
            for (int tap = 0; tap < 9; ++tap)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    part[((tap * NCO + t) * NCI + ci) * 256 + (4 * kg + r) * 16 + m] = acc[t][tap][r];
            if (ci == 0 && m == 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) part[9 * NCO * NCI * 256 + 16 * t + 4 * kg + r] = accb[t][r];
            }
        }
    }
}

// Sums of the blocks' partials of every job, in a fixed order: eight
// interleaved sums keep eight loads in flight.
constexpr int kMaxReduce = 24;
struct ReduceJob {
    const float* part;
    float *dw, *db;             // db null: not the layer's first input part
    int nblk, nci, nco, cin, ci0;  // ci0: first input channel of the part in the layer
    uint32_t first;             // first block in the launch
};
struct ReduceArgs {
    ReduceJob job[kMaxReduce];
    int n;
};
__global__ __launch_bounds__(256) void k_dw_reduce(ReduceArgs args) {
    int jn = 0;
    while (jn + 1 < args.n && blockIdx.x >= args.job[jn + 1].first) ++jn;
    const ReduceJob& J = args.job[jn];
    const int nw = 9 * J.nci * J.nco * 256, stride = nw + 16 * J.nco;
    const int e = (int)(blockIdx.x - J.first) * 256 + threadIdx.x;
    if (e >= stride) return;
    const float* p = J.part + e;
    float q[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    int b = 0;
    for (; b + 8 <= J.nblk; b += 8) {
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] += p[(size_t)(b + k) * stride];
    }
    for (int k = 0; b < J.nblk; ++b, ++k) q[k] += p[(size_t)b * stride];
    const float s = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
    if (e >= nw) {
        if (J.db) J.db[e - nw] = s;
        return;
    }
    const int tile = e / 256, in = e % 256;
    const int ci = tile % J.nci, t = (tile / J.nci) % J.nco, tap = tile / (J.nci * J.nco);
    J.dw[((size_t)(16 * t + in / 16) * 9 + tap) * J.cin + J.ci0 + 16 * ci + in % 16] = s;
}

// ------------------------------------------------------- elementwise ---
// kind 0: loss = mean over pixels and channels of (z - log(1 + target))^2,
//   z = log(1 + noisy) + res, the prediction in log space;
// kind 1: loss = mean of (D - T)^2 / (D^2 + 0.01), D = expm1(z), with the
//   denominator held constant in the gradient: the relative MSE of the
//   error metric, unbiased under noisy targets (Lehtinen et al. 2018,
//   Noise2Noise); dD/dz = D + 1.
// g = dloss/dres as the 16 BF16 channels of the output layer's gradient (3 and
// zeros), per-block partial loss
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ res, const float* __restrict__ noisy_log,
                                              const float* __restrict__ target, size_t npix, int kind,
                                              u16* __restrict__ g, float* __restrict__ loss_partial) {
    __shared__ float red[256];
    const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
    float l = 0.0f;
    if (p < npix) {
        const float scale = 2.0f / (float)(3 * npix);
        u16 h[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float z = noisy_log[3 * p + c] + res[3 * p + c];
            const float t = fmaxf(target[3 * p + c], 0.0f);
            float gv;
            if (kind == 0) {
                const float d = z - log1pf(t);
                l += d * d;
                gv = scale * d;
            } else {
                const float D = expm1f(z);
                const float e = D - t;
                const float inv = 1.0f / (D * D + 0.01f);
                l += e * e * inv;
                gv = scale * e * inv * (D + 1.0f);
            }
            h[c] = f2bf(gv);
        }
        uint4* o = reinterpret_cast<uint4*>(g + 16 * p);
        o[0] = make_uint4((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2], 0u, 0u);
        o[1] = make_uint4(0u, 0u, 0u, 0u);
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_partial[blockIdx.x] = red[0];
}

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ uint2 masked(float4 v, const u16* act) {
    const uint2 a = *reinterpret_cast<const uint2*>(act);
    const float x = bf2f((u16)a.x) > 0.0f ? v.x : 0.0f, y = bf2f((u16)(a.x >> 16)) > 0.0f ? v.y : 0.0f;
    const float z = bf2f((u16)a.y) > 0.0f ? v.z : 0.0f, w = bf2f((u16)(a.y >> 16)) > 0.0f ? v.w : 0.0f;
    return make_uint2((uint32_t)f2bf(x) | ((uint32_t)f2bf(y) << 16), (uint32_t)f2bf(z) | ((uint32_t)f2bf(w) << 16));
}

// the gradient of an upsampled tensor: the 2x2 sums of d (full resolution),
// masked by the activation, 4 channels per thread
__global__ __launch_bounds__(256) void k_upsample_grad(const float* __restrict__ d, const u16* __restrict__ act, int N,
                                                       int H, int W, int C, u16* __restrict__ g) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int cg = C / 4, h2 = H / 2, w2 = W / 2;
    if (i >= (size_t)N * h2 * w2 * cg) return;
    const int c = 4 * (int)(i % cg);
    const size_t q = i / cg;  // half-resolution pixel
    const int x = (int)(q % w2), y = (int)(q / w2 % h2);
    const size_t n = q / ((size_t)w2 * h2);
    const float* p = d + ((n * H + 2 * y) * W + 2 * x) * C + c;
    const float4 a = ld4(p), b = ld4(p + C), e = ld4(p + (size_t)W * C), f = ld4(p + (size_t)W * C + C);
    const float4 s = make_float4((a.x + b.x) + (e.x + f.x), (a.y + b.y) + (e.y + f.y), (a.z + b.z) + (e.z + f.z),
                                 (a.w + b.w) + (e.w + f.w));
    *reinterpret_cast<uint2*>(g + q * C + c) = masked(s, act + q * C + c);
}

// the gradient of a tensor with a skip connection and a pooled copy: the skip's
// plus a quarter of the pooled pixel's, masked, 4 channels per thread
__global__ __launch_bounds__(256) void k_skip_grad(const float* __restrict__ skip, const float* __restrict__ pool,
                                                   const u16* __restrict__ act, int N, int H, int W, int C,
                                                   u16* __restrict__ g) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int cg = C / 4;
    if (i >= (size_t)N * H * W * cg) return;
    const int c = 4 * (int)(i % cg);
    const size_t q = i / cg;
    const int x = (int)(q % W), y = (int)(q / W % H);
    const size_t n = q / ((size_t)W * H);
    const float4 a = ld4(skip + q * C + c);
    const float4 b = ld4(pool + ((n * (H / 2) + y / 2) * (W / 2) + x / 2) * C + c);
    const float4 s = make_float4(a.x + 0.25f * b.x, a.y + 0.25f * b.y, a.z + 0.25f * b.z, a.w + 0.25f * b.w);
    *reinterpret_cast<uint2*>(g + q * C + c) = masked(s, act + q * C + c);
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + 255) / 256); }

// blocks of a job: at most kDwBlocks, so that the partials stay small against the
// activations (full resolution of an 8 x 128^2 batch: eight tiles each)
uint32_t job_blocks(const DwPart& p) {
    const uint32_t tiles = (uint32_t)p.N * ((p.H + kRows - 1) / kRows) * ((p.W + kPix - 1) / kPix);
    return std::max(1u, std::min(tiles, kDwBlocks));
}

}  // namespace

size_t dw_partial_floats(const DwPart& p) {
    return (size_t)job_blocks(p) * (9 * (p.cx / 16) * (p.cout / 16) * 256 + p.cout);
}

Status weight_grads(const DwPart* parts, int n, float* scratch, hipStream_t s) {
    ReduceArgs red{};
    if (n > kMaxReduce) return Status{AURORA_ERR_INVALID, "denoiser: too many gradient parts"};
    std::vector<float*> at((size_t)n);
    uint32_t rb = 0;
    for (int i = 0; i < n; ++i) {
        const DwPart& p = parts[i];
        at[(size_t)i] = scratch;
        ReduceJob& r = red.job[i];
        r = ReduceJob{scratch, p.dw, p.db, (int)job_blocks(p), p.cx / 16, p.cout / 16, p.cin, p.ci0, rb};
        rb += nblocks((size_t)9 * (p.cx / 16) * (p.cout / 16) * 256 + p.cout);
        scratch += dw_partial_floats(p);
    }
    red.n = n;
    for (int nci = 1; nci <= 4; ++nci)
        for (int nco = 1; nco <= 4; ++nco) {
            int i = 0;
            while (i < n) {
                DwArgs a{};
                uint32_t blocks = 0;
                for (; i < n && a.n < kMaxJobs; ++i) {
                    const DwPart& p = parts[i];
                    if (p.cx != 16 * nci || p.cout != 16 * nco) continue;
                    const uint32_t nb = job_blocks(p);
                    a.job[a.n++] = DwJob{p.x, p.g, at[(size_t)i], p.N, p.H, p.W, p.half ? 1 : 0, nb, blocks};
                    blocks += nb;
                }
                if (!a.n) break;
                const int lds = dw_lds(nci, nco);
#define AUR_DW(I, O) \
    case 4 * (I) + (O): k_dw<I, O><<<blocks, 256, lds, s>>>(a); break;
                switch (4 * nci + nco) {
                    AUR_DW(1, 2)
                    AUR_DW(2, 1) AUR_DW(2, 2) AUR_DW(2, 3)
                    AUR_DW(3, 2) AUR_DW(3, 3) AUR_DW(3, 4)
                    AUR_DW(4, 3) AUR_DW(4, 4)
                    default: return Status{AURORA_ERR_INVALID, "denoiser: no weight gradient for these channel counts"};
                }
#undef AUR_DW
                AUR_HIP(hipGetLastError());
            }
        }
    k_dw_reduce<<<rb, 256, 0, s>>>(red);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

Status loss_grad(const float* res, const float* noisy_log, const float* target, size_t npix, int kind, uint16_t* g,
                 float* loss_partial, hipStream_t s) {
    if (kind != 0 && kind != 1) return Status{AURORA_ERR_INVALID, "unknown loss kind"};
    k_loss<<<nblocks(npix), 256, 0, s>>>(res, noisy_log, target, npix, kind, g, loss_partial);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status upsample_grad(const float* d, const uint16_t* act, int N, int H, int W, int C, uint16_t* g, hipStream_t s) {
    k_upsample_grad<<<nblocks((size_t)N * (H / 2) * (W / 2) * (C / 4)), 256, 0, s>>>(d, act, N, H, W, C, g);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}
Status skip_grad(const float* skip, const float* pool, const uint16_t* act, int N, int H, int W, int C, uint16_t* g,
                 hipStream_t s) {
    k_skip_grad<<<nblocks((size_t)N * H * W * (C / 4)), 256, 0, s>>>(skip, pool, act, N, H, W, C, g);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

}  // namespace aur
