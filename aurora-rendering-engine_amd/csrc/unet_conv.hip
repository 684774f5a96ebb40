// unet_conv.hip — the denoiser's 3x3 convolutions for gfx950: implicit GEMM on
// MFMA (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32 accumulation), forward
// and data gradient, with the network's elementwise steps in their epilogues
// (bias and ReLU, the 2x2 pooling, the output image, the ReLU mask of a
// gradient).
//
// Tensors are NHWC, BF16.  A convolution input is the concatenation of a
// full-resolution tensor A (CA channels) and a half-resolution tensor B (CB
// channels) read through nearest upsampling, so the decoder's upsample + skip
// concat is never materialised.  Weights of a layer are [Cout][9][Cin] (k =
// tap*Cin + c, tap = 3*(dy+1) + (dx+1)), padded to ceil(9*Cin/32)*32.
//
// MFMA operand layout (16x16x32, wave64): lane l holds A[l%16][8*(l/16)+j]
// and B[8*(l/16)+j][l%16] for j = 0..7 and returns D[4*(l/16)+r][l%16] for
// r = 0..3 (checked on the device by aurora_selftest_mfma).
//
// No reference counterpart: the reference has no learned component.
#include "unet.hpp"

#include <algorithm>

namespace aur {
namespace {

__device__ __forceinline__ uint32_t pack2(float a, float b) { return (uint32_t)f2bf(a) | ((uint32_t)f2bf(b) << 16); }

union Frag {
    uint4 u;
    bf16x8 v;
};

struct ConvArgs {
    const u16 *a, *b;      // input
    const u16* w;          // weights, padded rows
    const float* bias;     // forward
    void* out;
    u16* pool;             // EPI_RELU_POOL: the 2x2 average of the output
    const float* noisy;    // EPI_IMAGE: log(1 + noisy radiance), 3 per pixel
    const u16* act;        // EPI_MASK: activation whose sign masks the output
    int N, H, W;
    int ostride;           // channels of an output pixel
};

// What the epilogue writes.
enum { EPI_RELU, EPI_RELU_POOL, EPI_IMAGE, EPI_RES3, EPI_MASK, EPI_PLAIN };

// A pixel's channels sit in shared memory at a stride of 2*C + 16 bytes: 16
// consecutive pixels then start in distinct banks, so a fragment (16 pixels x 8
// channels per k group) reads without conflicts.
constexpr int pix_stride(int c) { return 2 * c + 16; }
constexpr int tile_bytes(int ca, int cb, int rpw) {
    return (4 * rpw + 2) * 66 * pix_stride(ca) + (cb ? (2 * rpw + 2) * 34 * pix_stride(cb) : 0);
}

// A block of 4 waves computes 4*RPW rows x 64 pixels x 16*NT channels, each
// wave RPW rows: it stages the input rows (halo of one pixel included; the
// half-resolution part at its own resolution) in shared memory once, then runs
// K = 9*(CA+CB) in chunks of 32.  Channel counts are template arguments: the K
// loop is unrolled, and a chunk's shared-memory addresses are a lane base plus
// constants, where runtime counts cost 14.7 VALU instructions per MFMA
// (tap, column and channel of each lane's k group, address products) and
// bound the kernel together with staging loads that took a lane per pixel
// (64 cache lines per load; now consecutive lanes read consecutive bytes).
// K order and every rounding are those of the runtime-count kernel.
//
// One 1024x1024 inference 590 -> 495 us (316 -> 376 TFLOP/s), the 14 hidden
// layers of an 8 x 128^2 training batch 10-20% faster each.  The full-resolution
// 32 -> 32 layer takes 44 us (47 before) where a copy of its tensors takes 20:
// its waves wait 61% of their time, on the staging loads first (a block stages,
// waits, multiplies, stores); MFMA busy 17%.
//
// The MFMAs compute each tile transposed (weights as the A operand); row r of
// tile t is channel (r/4)*4*NT + 4*t + r%4, so a lane ends with 4*NT
// consecutive channels of a pixel: 8*NT bytes per store.
template <int CA, int CB, int NT, int RPW, int EPI>
__global__ __launch_bounds__(256) void k_conv(ConvArgs p) {
    extern __shared__ __align__(16) unsigned char tile[];
    constexpr int C = CA + CB, PA = pix_stride(CA), PB = pix_stride(CB);
    constexpr int ROWS = 4 * RPW + 2, HROWS = 2 * RPW + 2;
    constexpr int KP = (9 * C + 31) / 32 * 32, CHUNKS = KP / 32, HALVES = 9 * C / 16;
    constexpr int TB = ROWS * 66 * PA;  // the half-resolution part
    const int H = p.H, W = p.W;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int segs = (W + 63) / 64, bands = (H + 4 * RPW - 1) / (4 * RPW);
    // neighbouring tiles on one XCD (blocks are dealt to the 8 XCDs in turn):
    // they share halo rows in its L2
    unsigned bid = blockIdx.x;
    if ((gridDim.x & 7u) == 0) bid = (bid & 7u) * (gridDim.x >> 3) + (bid >> 3);
    const int x0 = (int)(bid % segs) * 64;
    const int y0 = (int)((bid / segs) % bands) * 4 * RPW;
    const int n = (int)(bid / (segs * bands));
    const int co_base = blockIdx.y * 16 * NT;

    {
        constexpr int G = CA / 8, TOTAL = ROWS * 66 * G, J = (TOTAL + 255) / 256;
        // rows y0-1 .., pixels x0-1 .. x0+64: a row's pieces are consecutive
        const u16* src = p.a + ((int64_t)((int64_t)n * H + y0 - 1) * W + x0 - 1) * CA;
        uint4 v[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int idx = tid + 256 * j, r = idx / (66 * G), rem = idx - r * (66 * G), px = rem / G;
            const bool in = idx < TOTAL && (unsigned)(y0 - 1 + r) < (unsigned)H && (unsigned)(x0 - 1 + px) < (unsigned)W;
            v[j] = make_uint4(0, 0, 0, 0);
            if (in) v[j] = *reinterpret_cast<const uint4*>(src + r * (W * CA) + rem * 8);
        }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int idx = tid + 256 * j, q = idx / G;  // pixel of the tile, row-major
            if (idx < TOTAL) *reinterpret_cast<uint4*>(tile + q * PA + 16 * (idx - q * G)) = v[j];
        }
    }
    if constexpr (CB > 0) {
        constexpr int G = CB / 8, TOTAL = HROWS * 34 * G, J = (TOTAL + 255) / 256;
        const int h2 = H >> 1, w2 = W >> 1, hy0 = y0 / 2 - 1, hx0 = x0 / 2 - 1;
        const u16* src = p.b + ((int64_t)((int64_t)n * h2 + hy0) * w2 + hx0) * CB;
        uint4 v[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int idx = tid + 256 * j, r = idx / (34 * G), rem = idx - r * (34 * G), px = rem / G;
            const bool in = idx < TOTAL && (unsigned)(hy0 + r) < (unsigned)h2 && (unsigned)(hx0 + px) < (unsigned)w2;
            v[j] = make_uint4(0, 0, 0, 0);
            if (in) v[j] = *reinterpret_cast<const uint4*>(src + r * (w2 * CB) + rem * 8);
        }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int idx = tid + 256 * j, q = idx / G;
            if (idx < TOTAL) *reinterpret_cast<uint4*>(tile + TB + q * PB + 16 * (idx - q * G)) = v[j];
        }
    }
    __syncthreads();
    if (y0 + wave * RPW >= H) return;  // no barrier follows

    const int m = lane & 15, kg = lane >> 4;  // pixel of a fragment, k group of 8
    const bool hi = kg >= 2;                  // the chunk's second 16 channels
    const int abase = (wave * RPW * 66 + m) * PA + (kg & 1) * 16, abase2 = abase + (hi ? 32 : 0);
    int bcol[3] = {0, 0, 0}, brow[RPW + 2] = {};
    if constexpr (CB > 0) {
#pragma unroll
        for (int tx = 0; tx < 3; ++tx) bcol[tx] = TB + (((m + tx - 1) >> 1) + 1) * PB + (kg & 1) * 16;
#pragma unroll
        for (int q = 0; q < RPW + 2; ++q) brow[q] = (((wave * RPW + q - 1) >> 1) + 1) * 34 * PB;
    }
    const u16* wrow[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        wrow[t] = p.w + (size_t)(co_base + (m >> 2) * 4 * NT + 4 * t + (m & 3)) * KP + 8 * kg;

    floatx4 acc[RPW][4][NT];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[r][mt][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // address of the 16 channels `h` (tap h / (C/16)) for row r
    auto at = [&](int h, int r) {
        const int tap = h / (C / 16), cb = h % (C / 16), ty = tap / 3, tx = tap % 3;
        return cb < CA / 16 ? abase + ((r + ty) * 66 + tx) * PA + cb * 32
                            : bcol[tx] + brow[r + ty] + (cb - CA / 16) * 32;
    };
    auto in_a = [&](int h) { return h % (C / 16) < CA / 16; };
    auto load = [&](int q, Frag (&fa)[RPW][4], Frag (&fb)[NT]) {
        const int h0 = 2 * q, h1 = 2 * q + 1;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            if (h1 >= HALVES) {  // the last chunk's second half lies past the last tap
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    fa[r][mt].u = make_uint4(0, 0, 0, 0);
                    if (!hi)
                        fa[r][mt].u = *reinterpret_cast<const uint4*>(tile + at(h0, r) + mt * (in_a(h0) ? 16 * PA : 8 * PB));
                }
            } else if (in_a(h0) && in_a(h1) && h0 / (C / 16) == h1 / (C / 16)) {
                const unsigned char* s = tile + abase2 + (at(h0, r) - abase);
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) fa[r][mt].u = *reinterpret_cast<const uint4*>(s + mt * 16 * PA);
            } else {
                const unsigned char* s = tile + (hi ? at(h1, r) : at(h0, r));
                const int s0 = in_a(h0) ? 16 * PA : 8 * PB, s1 = in_a(h1) ? 16 * PA : 8 * PB;
#pragma unroll
                for (int mt = 0; mt < 4; ++mt)
                    fa[r][mt].u = *reinterpret_cast<const uint4*>(s + mt * (s0 == s1 ? s0 : hi ? s1 : s0));
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) fb[t].u = *reinterpret_cast<const uint4*>(wrow[t] + 32 * q);
    };
    auto mma = [&](Frag (&fa)[RPW][4], Frag (&fb)[NT]) {
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[r][mt][t] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[t].v, fa[r][mt].v, acc[r][mt][t], 0, 0, 0);
    };
    Frag a0[RPW][4], b0[NT], a1[RPW][4], b1[NT];
    load(0, a0, b0);
#pragma unroll
    for (int q = 0; q < CHUNKS; q += 2) {
        if (q + 1 < CHUNKS) load(q + 1, a1, b1);
        mma(a0, b0);
        if (q + 1 < CHUNKS) {
            if (q + 2 < CHUNKS) load(q + 2, a0, b0);
            mma(a1, b1);
        }
    }

    // this lane: channels co .. co + 4*NT - 1 of pixels x0 + 16*mt + m
    const int co = co_base + kg * 4 * NT;
    constexpr bool kForward = EPI == EPI_RELU || EPI == EPI_RELU_POOL || EPI == EPI_IMAGE || EPI == EPI_RES3;
    float bv[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) bv[t][k] = kForward ? p.bias[co + 4 * t + k] : 0.0f;
    uint32_t keep[RPW][4][2 * NT];  // EPI_RELU_POOL: the stored channels
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int y = y0 + wave * RPW + r;
        if (y >= H) continue;
        const size_t row = ((size_t)n * H + y) * W;
        if constexpr (EPI == EPI_IMAGE || EPI == EPI_RES3) {
            // the three channels sit in the 16 lanes of k group 0, for four
            // pixels each: spread them to one pixel per lane, so that the wave
            // evaluates expm1f once per channel and its accesses are contiguous
            const int x = x0 + lane;
            float v[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[c] = 0.0f;
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    const float u = __shfl(acc[r][mt][0][c] + bv[0][c], m);
                    v[c] = kg == mt ? u : v[c];
                }
            }
            if (x < W) {
                float* o = static_cast<float*>(p.out) + 3 * (row + x);
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    o[c] = EPI == EPI_RES3 ? v[c] : fmaxf(expm1f(p.noisy[3 * (row + x) + c] + v[c]), 0.0f);
            }
            continue;
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const int x = x0 + 16 * mt + m;
            float v[NT][4];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v[t][k] = acc[r][mt][t][k];
                    if (kForward) v[t][k] += bv[t][k];
                    if (EPI == EPI_RELU || EPI == EPI_RELU_POOL) v[t][k] = fmaxf(v[t][k], 0.0f);
                }
            if constexpr (EPI == EPI_PLAIN) {
                if (x < W) {
                    float* o = static_cast<float*>(p.out) + (row + x) * p.ostride + co;
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        reinterpret_cast<float4*>(o)[t] = make_float4(v[t][0], v[t][1], v[t][2], v[t][3]);
                }
            } else {
                if constexpr (EPI == EPI_MASK) {
                    if (x < W) {
                        const u16* ap = p.act + (row + x) * p.ostride + co;
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const uint2 av = reinterpret_cast<const uint2*>(ap)[t];
                            const u16 ah[4] = {(u16)av.x, (u16)(av.x >> 16), (u16)av.y, (u16)(av.y >> 16)};
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                if (!(bf2f(ah[k]) > 0.0f)) v[t][k] = 0.0f;
                        }
                    }
                }
                uint32_t h[2 * NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    h[2 * t] = pack2(v[t][0], v[t][1]);
                    h[2 * t + 1] = pack2(v[t][2], v[t][3]);
                }
                if (x < W) {
                    u16* o = static_cast<u16*>(p.out) + (row + x) * p.ostride + co;
                    if constexpr (NT % 2 == 0) {
#pragma unroll
                        for (int t = 0; t < NT / 2; ++t)
                            reinterpret_cast<uint4*>(o)[t] = make_uint4(h[4 * t], h[4 * t + 1], h[4 * t + 2], h[4 * t + 3]);
                    } else {
#pragma unroll
                        for (int t = 0; t < NT; ++t) reinterpret_cast<uint2*>(o)[t] = make_uint2(h[2 * t], h[2 * t + 1]);
                    }
                }
                if constexpr (EPI == EPI_RELU_POOL) {
#pragma unroll
                    for (int k = 0; k < 2 * NT; ++k) keep[r][mt][k] = h[k];
                }
            }
        }
    }
    if constexpr (EPI == EPI_RELU_POOL) {
        static_assert(RPW == 2, "a wave holds both rows of a pooled pixel");
        // H and W are even: both rows and both pixels of a pair are inside or
        // neither is; the odd lanes hand their pixel to the even ones
        const int y = y0 + wave * 2;
        const size_t prow = ((size_t)n * (H >> 1) + (y >> 1)) * (W >> 1);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const int x = x0 + 16 * mt + m;
            uint32_t h[2 * NT];
#pragma unroll
            for (int k = 0; k < 2 * NT; ++k) {
                const uint32_t a = keep[0][mt][k], c = keep[1][mt][k];
                const uint32_t b = (uint32_t)__builtin_amdgcn_mov_dpp((int)a, 0xB1, 0xf, 0xf, true);
                const uint32_t d = (uint32_t)__builtin_amdgcn_mov_dpp((int)c, 0xB1, 0xf, 0xf, true);
                const float lo = (bf2f((u16)a) + bf2f((u16)b)) + (bf2f((u16)c) + bf2f((u16)d));
                const float up = (bf2f((u16)(a >> 16)) + bf2f((u16)(b >> 16))) +
                                 (bf2f((u16)(c >> 16)) + bf2f((u16)(d >> 16)));
                h[k] = pack2(0.25f * lo, 0.25f * up);
            }
            if (x < W && (m & 1) == 0) {
                u16* o = p.pool + (prow + (x >> 1)) * p.ostride + co;
#pragma unroll
                for (int t = 0; t < NT; ++t) reinterpret_cast<uint2*>(o)[t] = make_uint2(h[2 * t], h[2 * t + 1]);
            }
        }
    }
}

template <int CA, int CB, int NT, int RPW, int EPI>
Status launch(const ConvArgs& p, int groups, hipStream_t s) {
    const size_t blocks = (size_t)p.N * ((p.H + 4 * RPW - 1) / (4 * RPW)) * ((p.W + 63) / 64);
    if (blocks > 0x7fffffffull) return Status{AURORA_ERR_INVALID, "denoiser: image too large"};
    k_conv<CA, CB, NT, RPW, EPI>
        <<<dim3((unsigned)blocks, (unsigned)groups), 256, tile_bytes(CA, CB, RPW), s>>>(p);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

// Two rows per wave read a 1.29x halo instead of 1.55x and use every weight
// fragment eight times; from 512 blocks (two per CU) on: inference 517 us, 519
// from 256, 542 from 1024, 536 never; a training batch, whose layers have at most
// 256 such blocks, 790 us, and 830 with the limit at 256.  The tiles of the layers
// without a pooled output must also leave room for two blocks per CU.  With one,
// 64 channels take 95 KB, one block per CU, which still beats a pooling kernel of
// its own: 2048x2048 1616 us against 1627, 4096x4096 6003 against 6065.
// Pixel blocks of the one-row-per-wave form below which a layer splits its
// output channels over the grid (one 16-channel tile per wave), and of the
// two-row form from which that one is taken.
constexpr size_t kSplitBlocks = 128, kTwoRowBlocks = 512;

template <int CA, int CB, int NT, int EPI>
Status dispatch(const ConvArgs& p, hipStream_t s) {
    const size_t cols = (size_t)p.N * ((p.W + 63) / 64);
    const size_t one = cols * ((p.H + 3) / 4), two = cols * ((p.H + 7) / 8);
    if constexpr (EPI == EPI_RELU_POOL) return launch<CA, CB, NT, 2, EPI>(p, 1, s);
    if constexpr (EPI != EPI_RELU_POOL) {
        if constexpr (NT > 1) {
            if (one < kSplitBlocks) return launch<CA, CB, 1, 1, EPI>(p, NT, s);
        }
        if constexpr (tile_bytes(CA, CB, 2) <= 81920) {
            if (two >= kTwoRowBlocks) return launch<CA, CB, NT, 2, EPI>(p, 1, s);
        }
        return launch<CA, CB, NT, 1, EPI>(p, 1, s);
    }
}

inline int shape(int ca, int cb, int cout) { return (ca << 16) | (cb << 8) | cout; }
Status unknown() { return Status{AURORA_ERR_INVALID, "denoiser: no convolution for these channel counts"}; }

}  // namespace

bool conv_pools(int N, int H, int W) {
    return (size_t)N * ((W + 63) / 64) * ((H + 7) / 8) >= kTwoRowBlocks;
}

Status conv_relu(const ConvIn& in, const uint16_t* w, const float* bias, uint16_t* out, uint16_t* pool, int N, int H,
                 int W, int cout, hipStream_t s) {
    ConvArgs p{};
    p.a = in.a;
    p.b = in.b;
    p.w = w;
    p.bias = bias;
    p.out = out;
    p.pool = pool;
    p.N = N;
    p.H = H;
    p.W = W;
    p.ostride = cout;
    const int sh = shape(in.ca, in.cb, cout);
    if (pool) {
        switch (sh) {
            case (32 << 16) | 32: return dispatch<32, 0, 2, EPI_RELU_POOL>(p, s);
            case (48 << 16) | 48: return dispatch<48, 0, 3, EPI_RELU_POOL>(p, s);
            case (64 << 16) | 64: return dispatch<64, 0, 4, EPI_RELU_POOL>(p, s);
        }
        return unknown();
    }
    switch (sh) {
        case (16 << 16) | 32: return dispatch<16, 0, 2, EPI_RELU>(p, s);
        case (32 << 16) | 32: return dispatch<32, 0, 2, EPI_RELU>(p, s);
        case (32 << 16) | 48: return dispatch<32, 0, 3, EPI_RELU>(p, s);
        case (48 << 16) | 48: return dispatch<48, 0, 3, EPI_RELU>(p, s);
        case (48 << 16) | 64: return dispatch<48, 0, 4, EPI_RELU>(p, s);
        case (64 << 16) | 64: return dispatch<64, 0, 4, EPI_RELU>(p, s);
        case (64 << 16) | (64 << 8) | 64: return dispatch<64, 64, 4, EPI_RELU>(p, s);
        case (48 << 16) | (64 << 8) | 48: return dispatch<48, 64, 3, EPI_RELU>(p, s);
        case (32 << 16) | (48 << 8) | 32: return dispatch<32, 48, 2, EPI_RELU>(p, s);
    }
    return unknown();
}

Status conv_residual(const ConvIn& in, const uint16_t* w, const float* bias, const float* noisy, float* out, int N,
                     int H, int W, hipStream_t s) {
    if (in.ca != 32 || in.cb != 0) return unknown();
    ConvArgs p{};
    p.a = in.a;
    p.w = w;
    p.bias = bias;
    p.out = out;
    p.noisy = noisy;
    p.N = N;
    p.H = H;
    p.W = W;
    return noisy ? dispatch<32, 0, 1, EPI_IMAGE>(p, s) : dispatch<32, 0, 1, EPI_RES3>(p, s);
}

Status conv_data_grad(const uint16_t* g, int cg, const uint16_t* w, const uint16_t* act, uint16_t* out, int N, int H,
                      int W, int cout, hipStream_t s) {
    ConvArgs p{};
    p.a = g;
    p.w = w;
    p.act = act;
    p.out = out;
    p.N = N;
    p.H = H;
    p.W = W;
    p.ostride = cout;
    switch (shape(cg, 0, cout)) {
        case (16 << 16) | 32: return dispatch<16, 0, 2, EPI_MASK>(p, s);
        case (32 << 16) | 32: return dispatch<32, 0, 2, EPI_MASK>(p, s);
        case (48 << 16) | 48: return dispatch<48, 0, 3, EPI_MASK>(p, s);
        case (64 << 16) | 64: return dispatch<64, 0, 4, EPI_MASK>(p, s);
    }
    return unknown();
}

Status conv_data_grad_f32(const uint16_t* g, int cg, const uint16_t* w, float* out, int N, int H, int W, int cout,
                          hipStream_t s) {
    ConvArgs p{};
    p.a = g;
    p.w = w;
    p.out = out;
    p.N = N;
    p.H = H;
    p.W = W;
    p.ostride = cout;
    switch (shape(cg, 0, cout)) {
        case (32 << 16) | 32: return dispatch<32, 0, 2, EPI_PLAIN>(p, s);
        case (32 << 16) | 48: return dispatch<32, 0, 3, EPI_PLAIN>(p, s);
        case (48 << 16) | 32: return dispatch<48, 0, 2, EPI_PLAIN>(p, s);
        case (48 << 16) | 48: return dispatch<48, 0, 3, EPI_PLAIN>(p, s);
        case (48 << 16) | 64: return dispatch<48, 0, 4, EPI_PLAIN>(p, s);
        case (64 << 16) | 48: return dispatch<64, 0, 3, EPI_PLAIN>(p, s);
        case (64 << 16) | 64: return dispatch<64, 0, 4, EPI_PLAIN>(p, s);
    }
    return unknown();
}

}  // namespace aur
