// denoise.hip — learned denoiser for path-traced frames (no reference counterpart: the
// reference renders one primary sample per pixel and has no denoiser).
//
// Network: a 5-level convolutional U-Net over 10 per-pixel features (log radiance, albedo,
// normal, log distance; padded to 16 channels).  Encoder level l: two 3x3 convolutions with
// ReLU (widths E[l]) then 2x2 average pooling; level 4 is the bottleneck.  Decoder level l:
// nearest 2x upsampling, concatenation with the encoder's level-l output, two 3x3
// convolutions with ReLU (widths D[l]); a final 3x3 convolution gives linear RGB radiance.
//
// Numerics: activations, weights and activation gradients in BF16 (round to nearest even);
// every convolution is an implicit GEMM on v_mfma_f32_16x16x32_bf16 with FP32 accumulation;
// biases, the loss, weight gradients (split-K partial sums reduced in a fixed order, so runs
// are deterministic) and Adam state are FP32.
//
// Kernels:
//   forward conv (+bias, ReLU) and backward-data conv: dX = conv(dY, W') with W'[ci][8-tap][co] =
//                    W[co][tap][ci]; its epilogue multiplies by the ReLU mask of the layer that
//                    produced X (X > 0).  A fragments are 8 channels of one pixel at one tap, read
//                    from an LDS tile of the NHWC input with its halo, B fragments 8 channels of a
//                    [co][tap][ci] weight row.  Weights are the first MFMA operand, so a lane's
//                    outputs are 4 consecutive channels of one pixel.
//   k_conv3x3_res    persistent workgroups, each wave with the weights of 16 output channels in registers,
//                    16 x 8 (or 16 x 16) pixel tiles double-buffered in LDS: inputs of up to 96
//                    channels (64 for 80 and 96 outputs) where every CU has two tiles.
//   k_conv3x3_split  16 x 8 pixel tiles with the output channels split over workgroups, weights from L2
//                    into registers several K steps ahead: everything else.
//                    Both can pool their output (2x2 mean) in the epilogue, read the decoder's
//                    upsampled channels from the lower level in their staging, and sum the gradient
//                    of an upsampling in their epilogue.
//   k_conv3x3_wgrad  dW[co][tap][ci] = sum_p dY[p][co] X[p+tap][ci] of all layers, over chunks of pixel
//                    tiles, all nine taps of a block of input channels in registers, the operands
//                    transposed on the way out of LDS; dbias in the same pass.
//   k_wgrad_reduce   the chunks' sums added up; in training with the Adam step and the BF16 weights.
//   pooling (backward), feature, loss and weight-layout kernels are element-wise.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "vt_internal.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kInCh = 16;       // input feature channels (10 used)
constexpr int kOutCh = 3;
constexpr int kLayers = 19;
constexpr int kMaxWidth = 96;   // widest layer (six groups of 16 output channels)
constexpr float kAlbedoEps = 0.01f;  // demodulation: irradiance = radiance / (albedo + eps)
constexpr float kLogMax = 16.0f;     // clamp of the predicted log irradiance

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint32_t b) { return __uint_as_float((b & 0xFFFFu) << 16); }
// two floats to packed BF16 (lo in bits 0-15), round to nearest even: f2bf's result for finite
// values, in one v_cvt_pk_bf16_f32
__device__ __forceinline__ uint32_t pk2bf(float lo, float hi) {
    typedef float f32x2v __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{lo, hi}), bf16x2v));
}
__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u}); }
__device__ __forceinline__ uint32_t half16(const u32x4& v, int t) { return (v[t >> 1] >> (16 * (t & 1))) & 0xFFFFu; }

// ---- convolution (forward and backward-data) ------------------------------------------
struct ConvArgs {
    const uint16_t* in;      // N x H x W x in_stride, channels [0, Cin)
    const uint16_t* w;       // [Cout][9 * Cin]
    const float* bias;       // [Cout] or null
    void* out;               // N x H x W x out_stride, channels [out_off, out_off + Cout)
    const uint16_t* mask;    // MASK: N x H x W x mask_stride; out = 0 where mask <= 0
    uint16_t* pool;          // optional: 2x2 mean pool of the BF16 output, N x H/2 x W/2 x Cout
    const uint16_t* up;      // input channels [0, up_C) read from this N x H/2 x W/2 x up_C tensor at
                             // (y/2, x/2) (nearest upsampling), the rest from `in`; up_C = 0: `in`
    uint32_t up_C;
    // MASK: the mask of channels [0, low_C) is `low_mask`'s (N x H/2 x W/2 x low_C) at (y/2, x/2), and those
    // channels of the output are summed over 2x2 pixels into `low_sum` (N x H/2 x W/2 x low_C): the gradient
    // of the level whose upsampling they are.  H and W even; low_C = 0: none
    const uint16_t* low_mask;
    uint16_t* low_sum;
    uint32_t low_C;
    uint32_t in_stride, out_stride, out_off, mask_stride;
    uint32_t N, H, W, Cin, Cout;
};

// Sums over 2x2 pixels, times `scale`, rounded to BF16: o0, o1 are this lane's outputs (4 channels) at pixels
// (x, y0) and (x, y0 + 1), y0 even, and lanes r, r ^ 1 an even/odd column pair, so the sum comes from
// this lane and its neighbour, in row-major order.  Every lane reaches the shuffles; the even ones store to
// dst, N x H/2 x W/2 x C.
__device__ __forceinline__ void put_quad(const ConvArgs& a, uint16_t* dst, uint32_t C, float scale, const uint2& o0,
                                         const uint2& o1, uint32_t co0, uint32_t n, int x, int y0, uint32_t r, bool in) {
    const uint32_t own[2][2] = {{o0.x, o0.y}, {o1.x, o1.y}};
    uint32_t nb[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) nb[m][t] = (uint32_t)__shfl_xor((int)own[m][t], 1, 64);
    if ((r & 1u) != 0u || !in) return;
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = i >> 1, sh = 16 * (i & 1);
        const float s = ((bf2f(own[0][t] >> sh) + bf2f(nb[0][t] >> sh)) + bf2f(own[1][t] >> sh)) + bf2f(nb[1][t] >> sh);
        o[i] = scale * s;
    }
    const size_t q = ((size_t)n * (a.H / 2u) + (size_t)(y0 >> 1)) * (a.W / 2u) + (size_t)(x >> 1);
    *reinterpret_cast<uint2*>(dst + q * C + co0) = make_uint2(pk2bf(o[0], o[1]), pk2bf(o[2], o[3]));
}

// Epilogue of the convolutions for a wave's ROWS rows of 16 pixels from (tx0, y0), y0 even: a lane holds
// output channels co0 .. co0 + 3 of pixel r of each row (weights are the first MFMA operand).  BF16
// outputs (widths and strides are multiples of 8) go out as one 8-byte store, the mask read the
// same way; FP32 ones channel by channel.  A row's address is wave-uniform and a lane's place in it
// the same for every tile, so no vector instruction goes into addresses.
template <int ROWS, bool RELU, bool OUTF, bool MASK>
__device__ __forceinline__ void put_rows(const ConvArgs& a, const f32x4 (&acc)[ROWS], const float (&bias)[4], uint32_t co0,
                                         uint32_t n, int tx0, int y0, uint32_t r) {
    const bool in_x = tx0 + (int)r < (int)a.W && co0 < a.Cout;
    // (a wave's 16 channels lie below low_C or at and above it: widths are multiples of 16)
    const bool low = MASK && (uint32_t)__builtin_amdgcn_readfirstlane(co0) < a.low_C;
    const uint32_t at = r * a.out_stride + co0, at_mask = low ? (r >> 1) * a.low_C + co0 : r * a.mask_stride + co0;
    uint2 o[2] = {make_uint2(0u, 0u), make_uint2(0u, 0u)};
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
        const int y = y0 + m;
        if (y >= (int)a.H) break;   // (uniform)
        const size_t p = ((size_t)n * a.H + (size_t)y) * a.W + (size_t)tx0;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = acc[m][i] + bias[i];
            if (RELU) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
        }
        if constexpr (OUTF) {
            float* const row = reinterpret_cast<float*>(a.out) + p * a.out_stride + a.out_off;
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                if (in_x && co0 + i < a.Cout) row[at + i] = v[i];
        } else {
            if (MASK && in_x) {
                const size_t pl = ((size_t)n * (a.H / 2u) + (size_t)(y >> 1)) * (a.W / 2u) + (size_t)(tx0 >> 1);
                const uint2 mk = *reinterpret_cast<const uint2*>((low ? a.low_mask + pl * a.low_C : a.mask + p * a.mask_stride) + at_mask);
                if (!(bf2f(mk.x) > 0.0f)) v[0] = 0.0f;
                if (!(bf2f(mk.x >> 16) > 0.0f)) v[1] = 0.0f;
                if (!(bf2f(mk.y) > 0.0f)) v[2] = 0.0f;
                if (!(bf2f(mk.y >> 16) > 0.0f)) v[3] = 0.0f;
            }
            o[m & 1] = make_uint2(pk2bf(v[0], v[1]), pk2bf(v[2], v[3]));
            if (in_x && !low) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + p * a.out_stride + a.out_off + at) = o[m & 1];
            if constexpr (MASK) {
                if ((m & 1) && low) put_quad(a, a.low_sum, a.low_C, 1.0f, o[0], o[1], co0, n, tx0 + (int)r, y - 1, r, in_x);
            } else {
                if ((m & 1) && a.pool) put_quad(a, a.pool, a.Cout, 0.25f, o[0], o[1], co0, n, tx0 + (int)r, y - 1, r, in_x);
            }
        }
    }
}

// 16 bytes of a tile's halo: channels c .. c + 7 of pixel (y, x) of image n, zeros outside the image.  The
// load is unconditional (a clamped address): conditional ones make a branch each, and a wait
// for every outstanding load where the branches join.  in: whether to keep the value (the
// caller selects, where it stores).
__device__ __forceinline__ u32x4 halo_chunk(const ConvArgs& a, uint32_t n, int y, int x, uint32_t c, bool& in) {
    in = in && y >= 0 && y < (int)a.H && x >= 0 && x < (int)a.W;
    const uint32_t yc = (uint32_t)min(max(y, 0), (int)a.H - 1), xc = (uint32_t)min(max(x, 0), (int)a.W - 1);
    const uint16_t* const p = a.in + ((size_t)(n * a.H + yc) * a.W + xc) * a.in_stride + c;
    const uint16_t* const q = a.up + ((size_t)(n * (a.H >> 1) + (yc >> 1)) * (a.W >> 1) + (xc >> 1)) * a.up_C + c;
    return *reinterpret_cast<const u32x4*>(c < a.up_C ? q : p);
}

// Convolution over kTileX x kTileY pixel tiles with the output channels split over workgroups (4
// waves, grid: tiles x groups of 16 channels), for the layers that do not fill the GPU otherwise: the
// lower levels of the network, training batches, small frames.  The input tile with a one-pixel
// halo is staged in LDS once (zeros outside the image), so the nine taps of each pixel read LDS.  Each wave
// owns two rows of 16 pixels.  Weight fragments come straight from the [co][tap][ci] rows in L2, kDepth
// K steps ahead in registers, the first ones before the tile is staged: the K loop has no barrier
// and waits for no load it has just issued.
// Bound by latency: a launch of 8 images of 8 x 8 to 64 x 64 pixels is a few microseconds of dependent
// steps (the tile, 9 Cin / 32 K steps) on workgroups that used to be too few (8 for the lowest level, each
// with all output channels and a barrier per K step): 27 such launches of a fine-tuning step 431 -> 224
// us, the lower levels of a 720p inference 170 -> 122 us.  Two groups of channels per wave were no
// faster anywhere (218 and 126 us).
constexpr int kTileX = 16, kTileY = 8;
constexpr uint32_t kDepth = 9;

inline size_t conv_split_lds(uint32_t cin) { return (size_t)(kTileY + 2) * (kTileX + 2) * (cin + 8u) * 2u; }

template <bool RELU, bool OUTF, bool MASK>
__global__ __launch_bounds__(256) void k_conv3x3_split(ConvArgs a, uint32_t ntx, uint32_t nty) {
    constexpr int MT = 2;   // rows of pixels of a wave
    extern __shared__ __align__(16) uint16_t tile[];  // (kTileY + 2) x (kTileX + 2) pixels x cs
    const uint32_t cs = a.Cin + 8u;                   // LDS pixel stride (16 B of padding)
    const uint32_t tx = blockIdx.x % ntx, rest = blockIdx.x / ntx, n = rest / nty;
    const int tx0 = (int)tx * kTileX, ty0 = (int)(rest % nty) * kTileY;
    const uint32_t cobase = blockIdx.y * 16u;
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t g = lane >> 4, r = lane & 15u;
    const uint32_t K = 9u * a.Cin;
    const uint32_t S = (K + 32u * kDepth - 1u) / (32u * kDepth) * kDepth;   // K steps, whole rings
    // this lane's weight row (past Cout the last again: outputs nobody stores)
    const uint16_t* const wrow = a.w + (size_t)min(cobase + r, a.Cout - 1u) * K;
    u32x4 B[kDepth];
    // (past 9 Cin a clamped address; the zeros are selected where the fragment is used)
    auto fetch = [&](uint32_t ks, u32x4& dst) {
        dst = *reinterpret_cast<const u32x4*>(wrow + min(32u * ks + 8u * g, K - 8u));
    };
    // cpp + 1 chunks of 16 B per pixel: its channels, then its padding, set to zeros (K past
    // the end reads the padding, so no select is needed)
    const uint32_t cpp = a.Cin / 8u + 1u;
    const uint32_t total = (uint32_t)((kTileY + 2) * (kTileX + 2)) * cpp;
    // i / cpp as (i * inv) >> 20: exact while i < 2^20 / cpp (cpp <= 25, i < 6600); i * inv
    // stays below 2^32 since cpp >= 2
    const uint32_t inv = ((1u << 20) + cpp - 1u) / cpp;
    // staging in batches: all loads of a batch are issued before its LDS stores, so a thread
    // waits for one round trip per batch instead of one per 16-byte chunk
    constexpr uint32_t kBatch = 8;
    auto stage = [&](uint32_t i0, bool first) {
        u32x4 v[kBatch];
        bool ok[kBatch];
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b) {
            const uint32_t i = min(i0 + threadIdx.x + 256u * b, total - 1u);
            const uint32_t pix = (i * inv) >> 20, c8 = i - pix * cpp;
            ok[b] = c8 + 1u < cpp;
            v[b] = halo_chunk(a, n, ty0 + (int)(pix / (uint32_t)(kTileX + 2)) - 1, tx0 + (int)(pix % (uint32_t)(kTileX + 2)) - 1,
                              8u * min(c8, cpp - 2u), ok[b]);
        }
        if (first) {   // after the tile's loads, which complete first
#pragma unroll
            for (uint32_t d = 0; d < kDepth; ++d) fetch(d, B[d]);
        }
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b) {
            const uint32_t i = i0 + threadIdx.x + 256u * b;
            const uint32_t pix = (i * inv) >> 20, c8 = i - pix * cpp;
            if (i < total) *reinterpret_cast<u32x4*>(tile + (size_t)pix * cs + 8u * c8) = ok[b] ? v[b] : u32x4{0u, 0u, 0u, 0u};
        }
    };
    stage(0u, true);
    for (uint32_t i0 = 256u * kBatch; i0 < total; i0 += 256u * kBatch) stage(i0, false);
    __syncthreads();
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // k = 32 s + 8 g as (tap, channel): tap = (k * invc) >> 20, exact while k < 2^20 / Cin
    // (k < 9 Cin + 32 kDepth <= 2016)
    const uint32_t invc = ((1u << 20) + a.Cin - 1u) / a.Cin;
    const uint32_t rowbase = (uint32_t)MT * wave;
    const uint16_t* const abase = tile + (size_t)((rowbase + 1u) * (kTileX + 2) + r + 1u) * cs;
    const uint32_t rstep = (uint32_t)(kTileX + 2) * cs;
    auto load_a = [&](uint32_t ks, bf16x8 (&A)[MT]) {
        const uint32_t k = 32u * ks + 8u * g;
        const uint32_t tap = (k * invc) >> 20;
        const bool kv = tap < 9u;
        const int tp = kv ? (int)tap : 4, cc = kv ? (int)(k - tap * a.Cin) : (int)a.Cin;   // past K: the zero padding
        const int ty = (tp >= 3 ? 1 : 0) + (tp >= 6 ? 1 : 0);
        const uint16_t* const p = abase + ((ty - 1) * (kTileX + 2) + tp - 3 * ty - 1) * (int)cs + cc;
#pragma unroll
        for (int m = 0; m < MT; ++m) A[m] = ld8(p + (size_t)m * rstep);
    };
    bf16x8 A[2][MT];
    load_a(0u, A[0]);
    // two rings per iteration, so that ring and operand buffers have fixed indexes
    auto ring = [&](uint32_t s0, uint32_t par) {
#pragma unroll
        for (uint32_t d = 0; d < kDepth; ++d) {
            const uint32_t ks = s0 + d, cur = (par + d) & 1u;
            load_a(ks + 1u, A[cur ^ 1u]);
            const bool kv = 32u * ks + 8u * g < K;
            const bf16x8 w = __builtin_bit_cast(bf16x8, kv ? B[d] : u32x4{0u, 0u, 0u, 0u});
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, A[cur][m], acc[m], 0, 0, 0);
            fetch(ks + kDepth, B[d]);
        }
    };
    for (uint32_t s0 = 0;;) {
        ring(s0, 0u);
        if ((s0 += kDepth) >= S) break;
        ring(s0, kDepth & 1u);
        if ((s0 += kDepth) >= S) break;
    }
    const uint32_t co0 = cobase + 4u * g;
    float bias[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) bias[i] = (a.bias && co0 + i < a.Cout) ? a.bias[co0 + i] : 0.0f;
    put_rows<MT, RELU, OUTF, MASK>(a, acc, bias, co0, n, tx0, ty0 + (int)rowbase, r);
}

// Resident-weight form for the layers with tiles enough for every CU: persistent workgroups walk the
// kTileX x res_y pixel tiles, each wave with the weights of 16 output channels in registers and ROWS
// rows of 16 pixels, so the only operand it reads from LDS is the input.  Tiles with their halo are
// double-buffered in LDS, the next one fetched into registers while the current one is computed: one
// barrier a tile.
// K is walked in steps of 32 as in the split form: k = tap CI + channel, 9 CI rounded up to whole steps
// (CI: the input channels; a multiple of 16), so every output is the same sum in the same order there and here.
// 8 channels (the output layer's gradient) are padded to 32: a step holds one tap where the split form's holds
// four.  An MFMA adds its four groups of 8 products one after another, so the zeros between the taps change
// nothing and the bits are the same all the same (test_gpu_conv_forms.py, with taps that cancel).
// A pixel's neighbours in x follow it in LDS, so the 32 values
// of a step that lies within one row of taps are at one offset for all of a row's pixels (CI an odd
// multiple of 16: the second half of a step may lie in the next pixel, beyond its padding), and a
// fragment read once feeds the steps of up to three output rows: ROWS + 2 reads for 3 ROWS MFMAs where
// CI is a multiple of 32.  Otherwise steps of the middle row of taps start half a step off (reads of
// their own), one step holds the end of the first row of taps and the start of the second, and
// the last one ends in the padding.
// Bound by the LDS reads and MFMAs where there are many channels (64 -> 64 at 1088 x 1920: 154 GFLOP and 535
// MB in 141 us, 1.1 PFLOP/s and 3.8 TB/s; 80 -> 64: 223 us), by HBM where there are few (32 -> 32: 38 GFLOP and
// 268 MB in 50 us).  The form before kept the weights in LDS and read (2 + Cout / 16) operands for
// every 2 Cout / 16 MFMAs, more LDS time than MFMA time: 241, 291 and 112 us, and 64 -> 3 122 us (now 74).
// Rows of a tile: 8, so that two workgroups or more share a CU and one's epilogue runs beside
// another's MFMAs (64 -> 64 channels at 1088 x 1920 161 -> 148 us against 16 rows); 16 for 80 and 96 output
// channels, whose five or six waves would leave SIMDs uneven (64 -> 80 channels of 8 images of 128 x
// 128 27 -> 38 us with 8 rows).
constexpr int res_y(int nt) { return nt <= 4 ? 8 : 16; }
constexpr uint32_t res_pix(int nt) { return (uint32_t)(res_y(nt) + 2) * (kTileX + 2); }
constexpr uint32_t res_waves(int nt) { return nt <= 2 ? 4u : nt == 3 ? 6u : nt == 4 ? 4u : 2u * (uint32_t)nt; }
// waves per SIMD the registers are cut for, and the workgroups per CU they allow
constexpr uint32_t res_simd(int nt, int ci) { return ci <= 32 ? 4u : (nt == 3 && ci <= 64) || nt >= 5 ? 3u : 2u; }
constexpr uint32_t res_per_cu(int nt, int ci) { return 4u * res_simd(nt, ci) / res_waves(nt); }
constexpr size_t res_lds(int nt, int ci) { return 2u * res_pix(nt) * ((uint32_t)ci + 8u) * 2u; }

template <int NT, int CI, bool RELU, bool OUTF, bool MASK>
__global__ __launch_bounds__(64 * res_waves(NT)) __attribute__((amdgpu_waves_per_eu(res_simd(NT, CI)))) void k_conv3x3_res(
    ConvArgs a, uint32_t ntx, uint32_t nty, uint32_t ntiles) {
    constexpr uint32_t kWaves = res_waves(NT), kThreads = 64u * kWaves, kResPix = res_pix(NT);
    constexpr int kResY = res_y(NT), ROWS = kResY * NT / (int)kWaves;
    constexpr int cs = CI + 8;                             // LDS pixel stride (16 B of padding, zeros)
    constexpr uint32_t kCh = (kResPix * (CI / 8u) + kThreads - 1u) / kThreads;
    constexpr int kRow = 3 * CI, KS = (9 * CI + 31) / 32;   // K values of a row of taps, K steps
    extern __shared__ __align__(16) uint16_t lds[];        // 2 x kResPix pixels x cs
    const uint32_t tid = threadIdx.x, lane = tid & 63u, g = lane >> 4, r = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t co16 = 16u * (wave % NT), rowbase = ROWS * (wave / NT);
    for (uint32_t i = tid; i < 2u * kResPix * (cs / 8u); i += kThreads)
        *reinterpret_cast<u32x4*>(lds + 8u * i) = u32x4{0u, 0u, 0u, 0u};
    // input tiles: cpp chunks of 16 B per pixel; chunk i -> pixel (i * inv) >> 20, exact for i < 2^20 / 12
    const uint32_t cpp = a.Cin / 8u, total = kResPix * cpp;
    const uint32_t inv = ((1u << 20) + cpp - 1u) / cpp;
    u32x4 pre[kCh];
    uint32_t keep = 0;   // bit b: pre[b] lies in the image (else zeros)
    // this thread's chunks: byte offsets from the tile's first halo pixel, in the tensor they come from
    // (where registers are left for them: 64 -> 64 channels at 1088 x 1920 148 -> 138 us, 80 -> 64 223 -> 243)
    constexpr bool kOff = CI <= 64 && NT <= 4;
    uint32_t voff[kCh], from_up = 0;
#pragma unroll
    for (uint32_t b = 0; b < kCh && kOff; ++b) {
        const uint32_t i = min(tid + kThreads * b, total - 1u), pix = (i * inv) >> 20, c = 8u * (i - pix * cpp);
        const uint32_t ly = pix / (uint32_t)(kTileX + 2), lx = pix % (uint32_t)(kTileX + 2);
        const bool up = c < a.up_C;
        voff[b] = 2u * (up ? (((ly + 1u) >> 1) * (a.W >> 1) + ((lx + 1u) >> 1)) * a.up_C + c : (ly * a.W + lx) * a.in_stride + c);
        from_up |= up ? 1u << b : 0u;
    }
    auto origin = [&](uint32_t t, uint32_t& n, int& tx0, int& ty0) {
        const uint32_t tx = t % ntx, rest = t / ntx;
        tx0 = (int)(tx * (uint32_t)kTileX);
        ty0 = (int)((rest % nty) * (uint32_t)kResY);
        n = rest / nty;
    };
    auto fetch_tile = [&](uint32_t t) {
        uint32_t n;
        int tx0, ty0;
        origin(t, n, tx0, ty0);
        if (kOff && tx0 > 0 && ty0 > 0 && tx0 + kTileX < (int)a.W && ty0 + kResY < (int)a.H) {   // the halo lies inside
            const char* const pi = reinterpret_cast<const char*>(
                a.in + (((size_t)n * a.H + (size_t)(ty0 - 1)) * a.W + (size_t)(tx0 - 1)) * a.in_stride);
            const char* const pu = reinterpret_cast<const char*>(
                a.up + (((size_t)n * (a.H >> 1) + (size_t)(ty0 / 2 - 1)) * (a.W >> 1) + (size_t)(tx0 / 2 - 1)) * a.up_C);
            keep = ~0u;
            if (a.up_C == 0u) {
#pragma unroll
                for (uint32_t b = 0; b < kCh; ++b) pre[b] = *reinterpret_cast<const u32x4*>(pi + voff[b]);
            } else {
#pragma unroll
                for (uint32_t b = 0; b < kCh; ++b)
                    pre[b] = *reinterpret_cast<const u32x4*>(((from_up >> b & 1u) ? pu : pi) + voff[b]);
            }
            return;
        }
        keep = 0u;
#pragma unroll
        for (uint32_t b = 0; b < kCh; ++b) {
            const uint32_t i = min(tid + kThreads * b, total - 1u);
            const uint32_t pix = (i * inv) >> 20;
            bool ok = true;
            pre[b] = halo_chunk(a, n, ty0 + (int)(pix / (uint32_t)(kTileX + 2)) - 1, tx0 + (int)(pix % (uint32_t)(kTileX + 2)) - 1,
                                8u * (i - pix * cpp), ok);
            keep |= ok ? 1u << b : 0u;
        }
    };
    auto store_tile = [&](uint16_t* tile) {
#pragma unroll
        for (uint32_t b = 0; b < kCh; ++b) {
            const uint32_t i = tid + kThreads * b;
            const uint32_t pix = (i * inv) >> 20, c8 = i - pix * cpp;
            if (i < total)
                *reinterpret_cast<u32x4*>(tile + pix * cs + 8u * c8) = (keep >> b & 1u) ? pre[b] : u32x4{0u, 0u, 0u, 0u};
        }
    };
    uint32_t t = blockIdx.x;
    if (t < ntiles) fetch_tile(t);
    // this lane's weights (past Cout the last row again: outputs nobody stores) and biases
    bf16x8 w[KS];
    const uint16_t* const wrow = a.w + (size_t)min(co16 + r, a.Cout - 1u) * (9u * a.Cin);
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)KS; ++k) {
        const uint32_t kk = 32u * k + 8u * g, tap = kk / (uint32_t)CI, ci = kk % (uint32_t)CI;
        const u32x4 v = *reinterpret_cast<const u32x4*>(wrow + min(tap, 8u) * a.Cin + min(ci, a.Cin - 8u));
        w[k] = __builtin_bit_cast(bf16x8, tap < 9u && ci < a.Cin ? v : u32x4{0u, 0u, 0u, 0u});
    }
    const uint32_t co0 = co16 + 4u * g;
    float bias[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) bias[i] = (a.bias && co0 + i < a.Cout) ? a.bias[co0 + i] : 0.0f;
    __syncthreads();   // the zeros
    uint32_t buf = 0;
    if (t < ntiles) store_tile(lds);
    __syncthreads();
    for (; t < ntiles; t += gridDim.x, buf ^= 1u) {
        const bool more = t + gridDim.x < ntiles;
        if (more) fetch_tile(t + gridDim.x);
        const uint16_t* const base = lds + buf * (kResPix * cs) + (rowbase * (kTileX + 2) + r) * cs + 8u * g;
        // of a step whose second half lies in the next pixel, of the one whose second half lies in the next
        // row of taps (its first half is the end of this one), and of the one whose second half is padding
        const bool up = g >= 2u;
        const uint16_t* const cross = base + (up ? 8 : 0);
        const uint16_t* const mixed = base + (up ? (kTileX + 2) * cs - 16 : 2 * cs + CI - 16);
        const uint16_t* const last = base + 2 * cs + CI - 16 + (up ? 16 - 8 * (int)g : 0);
        f32x4 acc[ROWS];
#pragma unroll
        for (int m = 0; m < ROWS; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (CI == 64 && res_simd(NT, CI) == 2) {
            // the next row's fragments are read while this row's MFMAs run (64 -> 64 channels at 1088 x 1920 149 ->
            // 141 us; fewer channels gain nothing, more have no registers for it)
            bf16x8 A[2][kRow / 32];
            auto read_row = [&](int i, bf16x8 (&dst)[kRow / 32]) {
#pragma unroll
                for (int k = 0; k < kRow / 32; ++k) dst[k] = ld8(base + (i * (kTileX + 2) + 32 * k / CI) * cs + 32 * k % CI);
            };
            read_row(0, A[0]);
#pragma unroll
            for (int i = 0; i < ROWS + 2; ++i) {   // a row of the halo: dy of output row i - dy
                if (i < ROWS + 1) read_row(i + 1, A[(i + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < kRow / 32; ++k)
#pragma unroll
                    for (int dy = 0; dy < 3; ++dy)
                        if (i - dy >= 0 && i - dy < ROWS)
                            acc[i - dy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[dy * (kRow / 32) + k], A[i & 1][k],
                                                                                 acc[i - dy], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < ROWS + 2; ++i) {   // a row of the halo: dy of output row i - dy
                if (CI % 32 != 0 && i >= 1 && i - 1 < ROWS)
                    acc[i - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kRow / 32], ld8(mixed + (i - 1) * (kTileX + 2) * cs),
                                                                         acc[i - 1], 0, 0, 0);
#pragma unroll
                for (int rel = 0; rel + 32 <= kRow; rel += 16) {   // a step's start within its row of taps
                    const bool first = rel % 32 == 0;              // dy 0 and 2 (and 1 where CI is a multiple of 32)
                    if (!first && CI % 32 == 0) continue;
                    const uint16_t* const at = rel / CI != (rel + 31) / CI ? cross : base;
                    const bf16x8 A = ld8(at + (i * (kTileX + 2) + rel / CI) * cs + rel % CI);
#pragma unroll
                    for (int dy = 0; dy < 3; ++dy) {
                        if ((dy * kRow + rel) % 32 != 0 || i - dy < 0 || i - dy >= ROWS) continue;
                        acc[i - dy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[(dy * kRow + rel) / 32], A, acc[i - dy], 0, 0, 0);
                    }
                }
                if (CI % 32 != 0 && i >= 2)
                    acc[i - 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[KS - 1], ld8(last + i * (kTileX + 2) * cs), acc[i - 2], 0,
                                                                         0, 0);
            }
        }
        if (more) store_tile(lds + (buf ^ 1u) * (kResPix * cs));
        uint32_t n;
        int tx0, ty0;
        origin(t, n, tx0, ty0);
        put_rows<ROWS, RELU, OUTF, MASK>(a, acc, bias, co0, n, tx0, ty0 + (int)rowbase, r);
        __syncthreads();   // this tile is no longer read, the next one is written
    }
}

// ---- weight gradient ----------------------------------------------------------------------
struct WGradArgs {
    const uint16_t* in;   // forward input, N x H x W x in_stride, channels [up_C, Cin)
    const uint16_t* up;   // its channels [0, up_C), N x H/2 x W/2 x up_C at (y/2, x/2)
    uint32_t up_C;
    const uint16_t* g;    // gradient of the pre-activation output, N x H x W x g_stride (g_stride % 8 == 0)
    float* part;          // [chunks][Cout * 9 * Cin weights, then Cout biases]
    uint32_t in_stride, g_stride;
    uint32_t N, H, W, Cin, Cout;
    uint32_t ntx, nty, tiles;   // kWgX x kWgY pixel tiles: per row, per column, of the batch
    uint32_t tiles_chunk;       // consecutive tiles of one workgroup
    uint32_t nco, nci;          // 16-channel groups of a workgroup's outputs and inputs
    uint32_t cob, cib;          // workgroups that share a chunk: per outputs and per inputs
    uint32_t first;             // its first workgroup in the launch
};
struct WGradTable {
    WGradArgs l[kLayers];
};

// dW[co][tap][ci] = sum_p dY[p][co] X[p + tap][ci] as a GEMM over pixels: rows co, columns ci, one
// accumulator tile per tap.  A workgroup takes a chunk of kWgX x kWgY pixel tiles, 16 NCI of the
// input channels and 16 NCO of the outputs and holds all nine taps' sums in registers: wave w
// the taps of row dy = w - 1 (three shifts in x share every dY fragment).  A tile of dY and of X with
// a one-pixel halo is staged in LDS as it lies in memory (pixel by pixel); ds_read_b64_tr_b16
// transposes on the way to the registers (16 lanes read 4 pixels x 16 channels, lane i gets channel i
// of the 4 pixels), so a tap is an offset of whole LDS pixels and both tensors are read from memory
// once for all taps.  The next tile is fetched into registers while the current one is multiplied.
// A K step is 2 rows of 16 pixels: k = 8 g + 4 h + j is the pixel 4 (g & 1) + 8 h + j of row g >> 1,
// the same for both operands.  LDS pixels lie an odd multiple of 32 B apart, so the 8 pixels that
// half a wave reads are in different banks.
// Bound by the matrix pipe and the staging together.
constexpr uint32_t kWgX = 16, kWgY = 4, kWgThreads = 192;
constexpr uint32_t wg_pitch(uint32_t n16) { return 16u * (n16 | 1u); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
// 16 channels x 8 pixels of an MFMA operand: pixels at p and p + 8 (LDS pixels of `pitch` elements)
__device__ __forceinline__ bf16x8 ld_tr(const uint16_t* p, uint32_t pitch) {
    typedef __attribute__((address_space(3))) s16x4 LdsS16x4;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4*)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4*)(p + 8u * pitch));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

constexpr uint32_t kWgMaxCo = 3, kWgMaxCi = 2;   // more accumulators leave two waves per SIMD
constexpr uint32_t kWgLds = kWgX * kWgY * wg_pitch(kWgMaxCo) + (kWgX + 2u) * (kWgY + 2u) * wg_pitch(kWgMaxCi);

template <int NCO, int NCI>
__device__ __forceinline__ void wgrad_block(const WGradArgs& a, uint32_t chunk, uint32_t cib, uint32_t cob, uint16_t* lds) {
    constexpr uint32_t GP = wg_pitch(NCO), XP = wg_pitch(NCI), XW = kWgX + 2u, XH = kWgY + 2u;
    constexpr uint32_t GCH = kWgX * kWgY * 2u * NCO, XCH = XW * XH * 2u * NCI;   // 16-byte chunks of a tile
    constexpr uint32_t GB = (GCH + kWgThreads - 1u) / kWgThreads, XB = (XCH + kWgThreads - 1u) / kWgThreads;
    uint16_t* const gt = lds;
    uint16_t* const xt = lds + kWgX * kWgY * GP;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // tap row: dy = wave - 1
    const uint32_t ci0 = cib * 16u * NCI, co0 = cob * 16u * NCO;
    const uint32_t cout8 = (a.Cout + 7u) & ~7u;
    const uint32_t t1 = min(a.tiles, (chunk + 1u) * a.tiles_chunk);
    // This thread's chunks: byte offsets from the tile's first pixel (gradient), from the halo's first pixel (input),
    // and their place in the tile.  Chunks outside the image or the channels read the tile's first pixel and are
    // zeros in LDS: every load is unconditional, with a wave-uniform base and a few instructions for its
    // bounds (addresses made anew for each chunk: 92 us a step, or 125 with the upsampled channels read from
    // below; this 76).
    u32x4 gpre[GB], xpre[XB];
    uint32_t goff[GB], xoff[XB], gpos[GB], xpos[XB], from_up = 0, keep = 0;
    const uint32_t gsafe = 2u * co0, xsafe = 2u * ((a.W + 1u) * a.in_stride);
#pragma unroll
    for (uint32_t b = 0; b < GB; ++b) {
        const uint32_t i = tid + kWgThreads * b, pix = i / (2u * NCO), c = co0 + 8u * (i % (2u * NCO));
        const bool ok = i < GCH && c < cout8;
        gpos[b] = ok ? pix % kWgX | (pix / kWgX) << 16 : 0xFFFFFFFFu;   // (no such pixel)
        goff[b] = ok ? 2u * ((pix / kWgX * a.W + pix % kWgX) * a.g_stride + c) : gsafe;
    }
#pragma unroll
    for (uint32_t b = 0; b < XB; ++b) {
        const uint32_t i = tid + kWgThreads * b, pix = i / (2u * NCI), c = ci0 + 8u * (i % (2u * NCI));
        const uint32_t lx = pix % XW, ly = pix / XW;
        const bool ok = i < XCH && c < a.Cin, up = ok && c < a.up_C;
        xpos[b] = ok ? lx | ly << 16 : 0xFFFFFFFFu;
        xoff[b] = up ? 2u * ((((ly + 1u) >> 1) * (a.W >> 1) + ((lx + 1u) >> 1)) * a.up_C + c) : 2u * ((ly * a.W + lx) * a.in_stride + c);
        from_up |= up ? 1u << b : 0u;
    }
    auto fetch = [&](uint32_t t) {
        const uint32_t tx = t % a.ntx, rest = t / a.ntx, ty = rest % a.nty, n = rest / a.nty;
        const uint32_t x0 = tx * kWgX, y0 = ty * kWgY;
        const size_t p0 = ((size_t)n * a.H + y0) * a.W + x0;
        const char* const pg = reinterpret_cast<const char*>(a.g + p0 * a.g_stride);
        const char* const px = reinterpret_cast<const char*>(a.in + p0 * a.in_stride) - xsafe;
        keep = 0u;
#pragma unroll
        for (uint32_t b = 0; b < GB; ++b) {
            const bool ok = x0 + (gpos[b] & 0xFFFFu) < a.W && y0 + (gpos[b] >> 16) < a.H;
            gpre[b] = *reinterpret_cast<const u32x4*>(pg + (ok ? goff[b] : gsafe));
            keep |= ok ? 1u << b : 0u;
        }
        bool ok[XB];
#pragma unroll
        for (uint32_t b = 0; b < XB; ++b) {   // (the halo's first pixel is (x0 - 1, y0 - 1): unsigned, so outside is large)
            ok[b] = x0 + (xpos[b] & 0xFFFFu) - 1u < a.W && y0 + (xpos[b] >> 16) - 1u < a.H;
            keep |= ok[b] ? 1u << (GB + b) : 0u;
        }
        if (a.up_C == 0u) {
#pragma unroll
            for (uint32_t b = 0; b < XB; ++b) xpre[b] = *reinterpret_cast<const u32x4*>(px + (ok[b] ? xoff[b] : xsafe));
        } else {
            const size_t q0 = ((size_t)n * (a.H >> 1) + y0 / 2u) * (a.W >> 1) + x0 / 2u;
            const char* const pu = reinterpret_cast<const char*>(a.up + q0 * a.up_C) - 2u * ((a.W >> 1) + 1u) * a.up_C;
#pragma unroll
            for (uint32_t b = 0; b < XB; ++b)
                xpre[b] = *reinterpret_cast<const u32x4*>(ok[b] ? ((from_up >> b & 1u) ? pu : px) + xoff[b] : px + xsafe);
        }
    };
    // this lane's pixel and channels of a transposed read
    const uint32_t g = lane >> 4, r = lane & 15u;
    const uint32_t col = 4u * (g & 1u) + (r >> 2), row = g >> 1;
    const uint16_t* const gbase = gt + (row * kWgX + col) * GP + 4u * (r & 3u);
    const uint16_t* const xbase = xt + ((row + wave) * XW + col) * XP + 4u * (r & 3u);
    const bool do_bias = wave == 1u && cib == 0u;
    const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    f32x4 acc[3][NCI][NCO], bacc[NCO];
#pragma unroll
    for (int j = 0; j < NCO; ++j) {
        bacc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 3 * NCI; ++k) acc[k / NCI][k % NCI][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    uint32_t t = chunk * a.tiles_chunk;
    if (t < t1) fetch(t);
    for (; t < t1; ++t) {
        __syncthreads();   // the previous tile is no longer read
#pragma unroll
        for (uint32_t b = 0; b < GB; ++b) {
            const uint32_t i = tid + kWgThreads * b;
            if (i < GCH) *reinterpret_cast<u32x4*>(gt + i / (2u * NCO) * GP + 8u * (i % (2u * NCO))) = (keep >> b & 1u) ? gpre[b] : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (uint32_t b = 0; b < XB; ++b) {
            const uint32_t i = tid + kWgThreads * b;
            if (i < XCH) *reinterpret_cast<u32x4*>(xt + i / (2u * NCI) * XP + 8u * (i % (2u * NCI))) =
                    (keep >> (GB + b) & 1u) ? xpre[b] : u32x4{0u, 0u, 0u, 0u};
        }
        __syncthreads();
        if (t + 1u < t1) fetch(t + 1u);
#pragma unroll
        for (uint32_t ks = 0; ks < kWgY / 2u; ++ks) {
            bf16x8 A[NCO];
#pragma unroll
            for (int j = 0; j < NCO; ++j) A[j] = ld_tr(gbase + 2u * ks * kWgX * GP + 16u * j, GP);
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                for (int c = 0; c < NCI; ++c) {
                    const bf16x8 B = ld_tr(xbase + (2u * ks * XW + dx) * XP + 16u * c, XP);
#pragma unroll
                    for (int j = 0; j < NCO; ++j)
                        acc[dx][c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], B, acc[dx][c][j], 0, 0, 0);
                }
            if (do_bias)
#pragma unroll
                for (int j = 0; j < NCO; ++j)
                    bacc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], ones, bacc[j], 0, 0, 0);
        }
    }
    // D layout: lane holds output channels co0 + 16 j + 4 g + i (rows) at input channel r (column)
    const uint32_t K = 9u * a.Cin;
    float* const part = a.part + (size_t)chunk * (a.Cout * K + a.Cout);
#pragma unroll
    for (int j = 0; j < NCO; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t co = co0 + 16u * j + 4u * g + (uint32_t)i;
            if (co >= a.Cout) continue;
#pragma unroll
            for (int c = 0; c < NCI; ++c) {
                const uint32_t ci = ci0 + 16u * c + r;
                if (ci >= a.Cin) continue;
#pragma unroll
                for (uint32_t dx = 0; dx < 3; ++dx) part[(size_t)co * K + (3u * wave + dx) * a.Cin + ci] = acc[dx][c][j][i];
            }
            if (do_bias && r == 0u) part[a.Cout * K + co] = bacc[j][i];
        }
}

// Every layer's weight gradient in one launch at the end of the backward pass: a layer alone has
// too little work to fill the GPU and to hide its start (19 launches: 175 us a step of 8 crops of 128 x
// 128, this one 76; 99 with the workgroups of a chunk on different XCDs and addresses made for each load).
__global__ __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_conv3x3_wgrad(WGradTable T) {
    __shared__ __align__(16) uint16_t lds[kWgLds];
    uint32_t l = 0;
    while (l + 1u < (uint32_t)kLayers && blockIdx.x >= T.l[l + 1].first) ++l;
    const WGradArgs& a = T.l[l];
    // workgroups are dealt to the 8 XCDs in turn: the ones that share a chunk are 8 apart, on one L2
    const uint32_t b = blockIdx.x - a.first, per = a.cib * a.cob, sub = b / 8u % per;
    const uint32_t chunk = b / (8u * per) * 8u + b % 8u, cib = sub % a.cib, cob = sub / a.cib;
    if (chunk * a.tiles_chunk >= a.tiles) return;   // (uniform: chunks come in eights)
    switch (a.nco * 4u + a.nci) {
        case 5: wgrad_block<1, 1>(a, chunk, cib, cob, lds); break;
        case 6: wgrad_block<1, 2>(a, chunk, cib, cob, lds); break;
        case 9: wgrad_block<2, 1>(a, chunk, cib, cob, lds); break;
        case 10: wgrad_block<2, 2>(a, chunk, cib, cob, lds); break;
        case 13: wgrad_block<3, 1>(a, chunk, cib, cob, lds); break;
        default: wgrad_block<3, 2>(a, chunk, cib, cob, lds); break;
    }
}

struct LayerDev {
    uint32_t cin, cout, cout8;
    uint32_t w_off, b_off;     // in the FP32 parameter vector
    uint32_t wb_off, wt_off;   // BF16 forward weights [co][tap][ci], transposed [ci][8-tap][cout8]
    uint32_t nw;               // cout * 9 * cin
};
// weight i of a layer into its BF16 forward and transposed (tap-flipped) copies
__device__ __forceinline__ void put_weight(const LayerDev& d, uint32_t i, float w, uint16_t* __restrict__ wb,
                                           uint16_t* __restrict__ wt) {
    const uint32_t co = i / (9u * d.cin), rem = i - co * 9u * d.cin;
    const uint32_t tap = rem / d.cin, ci = rem - tap * d.cin;
    const uint16_t b = f2bf(w);
    wb[d.wb_off + i] = b;
    wt[d.wt_off + (ci * 9u + (8u - tap)) * d.cout8 + co] = b;
}

// The chunks' partial sums of every layer, added up in chunk order (deterministic): parameter i of
// layer l is part[off + c * n + i - first] over its chunks c.  One launch for the whole network:
// a layer alone is too few threads to fill the GPU.  ADAM: the step (Kingma & Ba 2015) on the
// FP32 master parameters and their BF16 copies in the same pass, else the gradient into `grads`.
struct PartTable {
    struct {
        uint64_t off;
        uint32_t chunks, n, first;   // n: the layer's weights and biases, from parameter `first`
    } l[kLayers];
};
struct AdamArgs {
    float *w, *m, *v;
    const LayerDev* layers;
    uint16_t *wb, *wt;
    float lr, b1, b2, eps, bc1, bc2;
};
template <bool ADAM>
__global__ __launch_bounds__(256) void k_wgrad_reduce(const float* __restrict__ part, PartTable T, uint32_t nparam,
                                                      float* __restrict__ grads, AdamArgs o) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= nparam) return;
    uint32_t l = 0;
    while (l + 1u < (uint32_t)kLayers && i >= T.l[l + 1].first) ++l;
    const uint32_t n = T.l[l].n, chunks = T.l[l].chunks, k = i - T.l[l].first;
    const float* p = part + T.l[l].off + k;
    float s = 0.0f;
#pragma unroll 8
    for (uint32_t c = 0; c < chunks; ++c) s += p[(size_t)c * n];
    if (!ADAM) {
        grads[i] = s;
        return;
    }
    const float mi = o.b1 * o.m[i] + (1.0f - o.b1) * s;
    const float vi = o.b2 * o.v[i] + (1.0f - o.b2) * s * s;
    o.m[i] = mi;
    o.v[i] = vi;
    const float w = o.w[i] - o.lr * (mi / o.bc1) / (sqrtf(vi / o.bc2) + o.eps);
    o.w[i] = w;
    if (k < o.layers[l].nw) put_weight(o.layers[l], k, w, o.wb, o.wt);
}

// ---- element-wise kernels (8 channels per thread) ----------------------------------------
// g (N x H x W x C) = (gpool[parent] / 4 + gcat[p, off..]) * (act[p, off..] > 0)
__global__ void k_pool_bwd(const uint16_t* __restrict__ gpool, const uint16_t* __restrict__ gcat,
                           const uint16_t* __restrict__ act, uint32_t stride, uint32_t off, uint16_t* __restrict__ g,
                           uint32_t N, uint32_t H, uint32_t W, uint32_t C) {
    const uint32_t c8n = C / 8u;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * H * W * c8n) return;
    const uint32_t c8 = i % c8n, p = i / c8n;
    const uint32_t x = p % W, y = (p / W) % H, n = p / (W * H);
    const uint32_t parent = (n * (H / 2u) + y / 2u) * (W / 2u) + x / 2u;
    const u32x4 vp = *reinterpret_cast<const u32x4*>(gpool + (size_t)parent * C + c8 * 8u);
    const u32x4 vc = *reinterpret_cast<const u32x4*>(gcat + (size_t)p * stride + off + c8 * 8u);
    const u32x4 va = *reinterpret_cast<const u32x4*>(act + (size_t)p * stride + off + c8 * 8u);
    u32x4 o;
    for (int t = 0; t < 4; ++t) {
        uint32_t h2[2];
        for (int e = 0; e < 2; ++e) {
            const int k = 2 * t + e;
            const float v = 0.25f * bf2f(half16(vp, k)) + bf2f(half16(vc, k));
            h2[e] = bf2f(half16(va, k)) > 0.0f ? f2bf(v) : 0u;
        }
        o[t] = h2[0] | (h2[1] << 16);
    }
    *reinterpret_cast<u32x4*>(g + (size_t)p * C + c8 * 8u) = o;
}

// features of an h x w frame into an hp x wp tensor (edge-replicated padding), 16 channels:
// log(1 + max(rad, 0) / (albedo + 0.01)) x3 (demodulated irradiance), albedo x3, normal x3,
// log(1 + distance) / 8, log2(spp) / 8, zeros x5
__global__ void k_features(const float4* __restrict__ rad, const float4* __restrict__ gbuf, uint32_t h, uint32_t w,
                           uint32_t hp, uint32_t wp, float spp_feature, uint16_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hp * wp) return;
    const uint32_t x = min(i % wp, w - 1u), y = min(i / wp, h - 1u);
    const uint32_t s = y * w + x;
    const float4 L = rad[s], A = gbuf[2 * s], Nn = gbuf[2 * s + 1];
    // the albedo the network sees (and remodulates with) is the BF16-rounded one
    const float ar = bf2f(f2bf(A.x)) + kAlbedoEps, ag = bf2f(f2bf(A.y)) + kAlbedoEps, ab = bf2f(f2bf(A.z)) + kAlbedoEps;
    float f[16] = {log1pf(fmaxf(L.x, 0.0f) / ar), log1pf(fmaxf(L.y, 0.0f) / ag), log1pf(fmaxf(L.z, 0.0f) / ab),
                   A.x, A.y, A.z, Nn.x, Nn.y, Nn.z, log1pf(fmaxf(A.w, 0.0f)) * 0.125f, spp_feature,
                   0, 0, 0, 0, 0};
    u32x4 o0, o1;
    for (int t = 0; t < 4; ++t) {
        o0[t] = (uint32_t)f2bf(f[2 * t]) | ((uint32_t)f2bf(f[2 * t + 1]) << 16);
        o1[t] = (uint32_t)f2bf(f[8 + 2 * t]) | ((uint32_t)f2bf(f[9 + 2 * t]) << 16);
    }
    *reinterpret_cast<u32x4*>(out + (size_t)i * 16u) = o0;
    *reinterpret_cast<u32x4*>(out + (size_t)i * 16u + 8u) = o1;
}

__global__ void k_f32_to_bf16(const float* __restrict__ in, uint16_t* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f2bf(in[i]);
}

// crop of an h x w frame's RGB target rows (RGBA32F) into N x c x c x 3 at (y0, x0)
struct CropDesc {
    uint32_t frame, y0, x0, pad;
};
struct FrameDesc {
    const uint16_t* feat;   // h x w x 16
    const float* target;    // h x w x 3
    uint32_t h, w;
};
__global__ void k_gather_crops(const FrameDesc* __restrict__ frames, const CropDesc* __restrict__ crops, uint32_t N,
                               uint32_t c, uint16_t* __restrict__ x0, float* __restrict__ tgt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * c * c) return;
    const uint32_t x = i % c, y = (i / c) % c, n = i / (c * c);
    const CropDesc cd = crops[n];
    const FrameDesc fd = frames[cd.frame];
    const size_t s = (size_t)(cd.y0 + y) * fd.w + cd.x0 + x;
    const u32x4* f = reinterpret_cast<const u32x4*>(fd.feat + s * 16u);
    u32x4* o = reinterpret_cast<u32x4*>(x0 + (size_t)i * 16u);
    o[0] = f[0];
    o[1] = f[1];
    for (int k = 0; k < 3; ++k) tgt[(size_t)i * 3u + k] = fd.target[s * 3u + k];
}

__global__ void k_rgba_to_rgb(const float4* __restrict__ in, float* __restrict__ out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = in[i];
    out[3 * i] = v.x;
    out[3 * i + 1] = v.y;
    out[3 * i + 2] = v.z;
}

// The network predicts a correction y to the input's log irradiance b (feature channels 0..2
// of x): irradiance E = exp(min(b + y, kLogMax)) - 1, radiance a * E with a = albedo + eps
// (feature channels 3..5).  relMSE loss mean((a E - t)^2 / (t^2 + 0.01)) over P pixels x 3
// channels; gy = dLoss/dy (BF16, stride 8, channels 3..7 zero); per-block partial sums.
__device__ __forceinline__ float irradiance(float b, float y, float* dE) {
    const float z = b + y;
    if (z > kLogMax) {
        *dE = 0.0f;
        return expm1f(kLogMax);
    }
    *dE = expf(z);
    return expm1f(z);
}

__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ y, const float* __restrict__ t,
                                              const uint16_t* __restrict__ x, uint32_t P, float scale,
                                              uint16_t* __restrict__ gy, float* __restrict__ part) {
    __shared__ float red[256];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (i < P) {
        u32x4 o = {0u, 0u, 0u, 0u};
        uint32_t h[3];
        for (int c = 0; c < 3; ++c) {
            const float b = bf2f(x[(size_t)i * 16u + (uint32_t)c]);
            const float a = bf2f(x[(size_t)i * 16u + 3u + (uint32_t)c]) + kAlbedoEps;
            float dE;
            const float E = irradiance(b, y[3 * i + c], &dE);
            const float d = a * E - t[3 * i + c];
            const float den = t[3 * i + c] * t[3 * i + c] + 0.01f;
            l += d * d / den;
            h[c] = f2bf(2.0f * d / den * a * dE * scale);
        }
        o[0] = h[0] | (h[1] << 16);
        o[1] = h[2];
        *reinterpret_cast<u32x4*>(gy + (size_t)i * 8u) = o;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_loss_sum(const float* __restrict__ part, uint32_t n, float scale,
                                                  float* __restrict__ out) {
    __shared__ float red[256];
    float s = 0.0f;
    for (uint32_t i = threadIdx.x; i < n; i += 256u) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0] * scale;
}

// FP32 master -> BF16 forward and transposed (tap-flipped) weights of every layer
__global__ void k_prep_weights(const float* __restrict__ params, const LayerDev* __restrict__ L, uint32_t nl,
                               uint16_t* __restrict__ wb, uint16_t* __restrict__ wt, uint32_t total) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    uint32_t l = 0;
    while (l + 1 < nl && i >= L[l].nw) {
        i -= L[l].nw;
        ++l;
    }
    put_weight(L[l], i, params[L[l].w_off + i], wb, wt);
}

// network output (hp x wp x 3 log-irradiance corrections, FP32) -> h x w RGBA32F radiance
// (irradiance remodulated with the albedo of the features x, clamped at 0); alpha < 1 blends
// with the input radiance: alpha * denoised + (1 - alpha) * input
__global__ void k_output(const float* __restrict__ y, const uint16_t* __restrict__ x, uint32_t h, uint32_t w,
                         uint32_t wp, const float4* __restrict__ rad, float alpha, float4* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= h * w) return;
    const uint32_t xx = i % w, yy = i / w;
    const size_t q = (size_t)yy * wp + xx;
    const float* v = y + q * 3u;
    const uint16_t* f = x + q * 16u;
    float r[3];
    for (int c = 0; c < 3; ++c) {
        float dE;
        r[c] = fmaxf((bf2f(f[3 + c]) + kAlbedoEps) * irradiance(bf2f(f[c]), v[c], &dE), 0.0f);
    }
    if (alpha < 1.0f) {
        const float4 in = rad[i];
        const float b = 1.0f - alpha;
        r[0] = alpha * r[0] + b * in.x;
        r[1] = alpha * r[1] + b * in.y;
        r[2] = alpha * r[2] + b * in.z;
    }
    out[i] = make_float4(r[0], r[1], r[2], 1.0f);
}

// ---- host side ---------------------------------------------------------------------------
inline uint32_t blocks(size_t n, uint32_t b = 256) { return (uint32_t)((n + b - 1) / b); }
inline uint32_t up8(uint32_t c) { return (c + 7u) & ~7u; }

struct Layer {
    uint32_t cin, cout;
    bool relu;
    LayerDev d;
};

struct Tensor {
    uint16_t* p = nullptr;
    uint32_t C = 0;   // channels (row stride)
};

struct Net {
    bool on = false;
    uint32_t E[5] = {}, D[4] = {}, U[4] = {};
    Layer L[kLayers];
    size_t nparam = 0, nwb = 0, nwt = 0;
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    uint16_t *wb = nullptr, *wt = nullptr;
    LayerDev* ldev = nullptr;
    uint64_t adam_t = 0;
    bool weights_dirty = true;
    // activations (capacity in level-0 pixels)
    size_t cap = 0;
    void* act_mem = nullptr;
    Tensor x0, a[4], cat[4], pool[4], b1, b2, d1[4], d2[4];
    float* y = nullptr;
    // gradients
    size_t gcap = 0;
    void* grad_mem = nullptr;
    Tensor gy, gd2[4], gd1[4], gcat[4], gb2, gb1, gpool[4], gskip[4], ga[4];
    float* target = nullptr;
    float* lpart = nullptr;
    float* part = nullptr;
    size_t part_cap = 0;
    WGradTable wg{};           // the weight gradients' launch and where its partial sums lie
    PartTable parts{};         // (plan_wgrad)
    uint32_t wg_blocks = 0;
    float* losses = nullptr;   // device, one per training iteration
    size_t losses_cap = 0;
    // training frames
    std::vector<void*> frame_mem;
    std::vector<FrameDesc> frames;
    FrameDesc* frames_dev = nullptr;
    size_t frames_dev_cap = 0;
    CropDesc* crops_dev = nullptr;
    size_t crops_cap = 0;
    // staging for host <-> device frames
    void* io = nullptr;
    size_t io_cap = 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // output blend weights for spp = 2^k, k < nblend (none: the network output alone)
    float blend[32] = {};
    uint32_t nblend = 0;
};

Net net;

// blend weight for spp samples: linear in log2(spp) between the table's entries, clamped to
// its ends; 1 without a table
float blend_alpha(uint32_t spp) {
    if (net.nblend == 0) return 1.0f;
    const float t = log2f((float)(spp ? spp : 1u));
    if (t <= 0.0f) return net.blend[0];
    if (t >= (float)(net.nblend - 1)) return net.blend[net.nblend - 1];
    const uint32_t k = (uint32_t)t;
    const float f = t - (float)k;
    return net.blend[k] + f * (net.blend[k + 1] - net.blend[k]);
}

void set_layer(int i, uint32_t cin, uint32_t cout, bool relu) {
    net.L[i].cin = cin;
    net.L[i].cout = cout;
    net.L[i].relu = relu;
}

void free_act() {
    hipFree(net.act_mem);
    net.act_mem = nullptr;
    net.cap = 0;
}
void free_grad() {
    hipFree(net.grad_mem);
    net.grad_mem = nullptr;
    net.gcap = 0;
}

void free_all() {
    free_act();
    free_grad();
    for (void* p : net.frame_mem) hipFree(p);
    hipFree(net.params); hipFree(net.grads); hipFree(net.adam_m); hipFree(net.adam_v);
    hipFree(net.wb); hipFree(net.wt); hipFree(net.ldev); hipFree(net.part); hipFree(net.losses);
    hipFree(net.frames_dev); hipFree(net.crops_dev); hipFree(net.io);
    if (net.e0) hipEventDestroy(net.e0);
    if (net.e1) hipEventDestroy(net.e1);
    net = Net{};
}

// Bump allocation of tensors out of one device block (256-byte aligned).
struct Bump {
    char* base;
    size_t off = 0;
    bool count_only;
    void* take(size_t bytes) {
        void* p = count_only ? nullptr : base + off;
        off += (bytes + 255) & ~(size_t)255;
        return p;
    }
    Tensor t(size_t px, uint32_t C) {
        Tensor x;
        x.p = static_cast<uint16_t*>(take(px * C * 2));
        x.C = C;
        return x;
    }
};

size_t layout_act(Bump& b, size_t P0) {
    net.x0 = b.t(P0, kInCh);
    for (int l = 0; l < 4; ++l) {
        const size_t P = P0 >> (2 * l);
        net.a[l] = b.t(P, net.E[l]);
        net.cat[l] = b.t(P, net.U[l] + net.E[l]);
        net.pool[l] = b.t(P >> 2, net.E[l]);
        net.d1[l] = b.t(P, net.D[l]);
        net.d2[l] = b.t(P, net.D[l]);
    }
    net.b1 = b.t(P0 >> 8, net.E[4]);
    net.b2 = b.t(P0 >> 8, net.E[4]);
    net.y = static_cast<float*>(b.take(P0 * 3 * 4));
    return b.off;
}

size_t layout_grad(Bump& b, size_t P0) {
    net.gy = b.t(P0, 8);
    for (int l = 0; l < 4; ++l) {
        const size_t P = P0 >> (2 * l);
        net.gd2[l] = b.t(P, net.D[l]);
        net.gd1[l] = b.t(P, net.D[l]);
        net.gcat[l] = b.t(P, net.U[l] + net.E[l]);
        net.gpool[l] = b.t(P >> 2, net.E[l]);
        net.gskip[l] = b.t(P, net.E[l]);
        net.ga[l] = b.t(P, net.E[l]);
    }
    net.gb1 = b.t(P0 >> 8, net.E[4]);
    net.gb2 = b.t(P0 >> 8, net.E[4]);
    net.target = static_cast<float*>(b.take(P0 * 3 * 4));
    net.lpart = static_cast<float*>(b.take((P0 / 256 + 1) * 4));
    return b.off;
}

int ensure_act(size_t P0) {
    if (P0 <= net.cap && net.act_mem) {
        Bump b{static_cast<char*>(net.act_mem), 0, false};
        layout_act(b, P0);
        return 0;
    }
    free_act();
    Bump c{nullptr, 0, true};
    const size_t bytes = layout_act(c, P0);
    if (hipMalloc(&net.act_mem, bytes) != hipSuccess) {
        net.act_mem = nullptr;
        return -1;
    }
    net.cap = P0;
    Bump b{static_cast<char*>(net.act_mem), 0, false};
    layout_act(b, P0);
    return 0;
}

int ensure_grad(size_t P0) {
    if (!(P0 <= net.gcap && net.grad_mem)) {
        free_grad();
        Bump c{nullptr, 0, true};
        const size_t bytes = layout_grad(c, P0);
        if (hipMalloc(&net.grad_mem, bytes) != hipSuccess) {
            net.grad_mem = nullptr;
            return -1;
        }
        net.gcap = P0;
    }
    Bump b{static_cast<char*>(net.grad_mem), 0, false};
    layout_grad(b, P0);
    return 0;
}

// ---- launches ----------------------------------------------------------------------------
// compute units of the current device (queried once)
uint32_t device_cus() {
    static int n = 0;
    if (n == 0 && (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, vt_rt_device()) != hipSuccess || n <= 0))
        n = 256;
    return (uint32_t)n;
}

// resident-weight launch when there are two tiles for every CU; returns 1 when not applicable.  Fewer
// workgroups than the CUs hold where those would get less than two tiles each: the weights are read
// once a workgroup.
template <int NT, int CI, bool RELU, bool OUTF, bool MASK>
int launch_res(const ConvArgs& a, hipStream_t s) {
    const uint32_t ntx = (a.W + kTileX - 1u) / kTileX, nty = (a.H + (uint32_t)res_y(NT) - 1u) / (uint32_t)res_y(NT);
    const size_t ntiles = (size_t)ntx * nty * a.N;
    size_t grid = (size_t)device_cus() * res_per_cu(NT, CI);
    if (ntiles < 2u * device_cus() || ntiles > 0xFFFFFFFFu) return 1;
    if (ntiles < 2u * grid) grid = std::max<size_t>(device_cus(), ntiles / 2u);
    static bool allowed = false;
    if (!allowed) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv3x3_res<NT, CI, RELU, OUTF, MASK>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)res_lds(NT, CI)) != hipSuccess)
            return -1;
        allowed = true;
    }
    hipLaunchKernelGGL((k_conv3x3_res<NT, CI, RELU, OUTF, MASK>), dim3((uint32_t)grid), dim3(64u * res_waves(NT)), res_lds(NT, CI),
                       s, a, ntx, nty, (uint32_t)ntiles);
    return 0;
}
template <int NT, bool RELU, bool OUTF, bool MASK>
int launch_res(const ConvArgs& a, hipStream_t s) {
    switch (a.Cin) {
        case 16: return launch_res<NT, 16, RELU, OUTF, MASK>(a, s);
        case 8: case 32: return launch_res<NT, 32, RELU, OUTF, MASK>(a, s);
        case 48: return launch_res<NT, 48, RELU, OUTF, MASK>(a, s);
        case 64: return launch_res<NT, 64, RELU, OUTF, MASK>(a, s);
        default: break;
    }
    if constexpr (NT <= 4) {   // (more waves have no registers for the weights of 80 and 96 channels)
        if (a.Cin == 80u) return launch_res<NT, 80, RELU, OUTF, MASK>(a, s);
        if (a.Cin == 96u) return launch_res<NT, 96, RELU, OUTF, MASK>(a, s);
    }
    return 1;
}

// LDS above 64 KiB is allowed first (once per instantiation and size)
template <bool RELU, bool OUTF, bool MASK>
int launch_split(const ConvArgs& a, uint32_t groups, hipStream_t s) {
    const uint32_t ntx = (a.W + kTileX - 1u) / kTileX, nty = (a.H + kTileY - 1u) / kTileY;
    const size_t lds = conv_split_lds(a.Cin);
    static size_t allowed = 65536;
    if (lds > allowed) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv3x3_split<RELU, OUTF, MASK>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return -1;
        allowed = lds;
    }
    hipLaunchKernelGGL((k_conv3x3_split<RELU, OUTF, MASK>), dim3(ntx * nty * a.N, groups), dim3(256), lds, s, a, ntx,
                       nty);
    return 0;
}

// nt: 16-channel groups of the output
template <bool RELU, bool OUTF, bool MASK>
int launch_conv_nt(uint32_t nt, const ConvArgs& a, hipStream_t s) {
    // resident weights where there are tiles enough, else split output channels
    int rc = 1;
    switch (nt) {
        case 1: rc = launch_res<1, RELU, OUTF, MASK>(a, s); break;
        case 2: rc = launch_res<2, RELU, OUTF, MASK>(a, s); break;
        case 3: rc = launch_res<3, RELU, OUTF, MASK>(a, s); break;
        case 4: rc = launch_res<4, RELU, OUTF, MASK>(a, s); break;
        case 5: rc = launch_res<5, RELU, OUTF, MASK>(a, s); break;
        case 6: rc = launch_res<6, RELU, OUTF, MASK>(a, s); break;
        default: break;
    }
    if (rc <= 0) return rc;
    return launch_split<RELU, OUTF, MASK>(a, nt, s);
}

// forward conv of layer li: in (Cin channels, stride in.C) -> out (stride out_stride, offset out_off)
// pool (optional, BF16 outputs only, H and W even): also writes the 2x2 mean pool of the output
// (N x H/2 x W/2 x Cout), fused into the epilogue
// up (optional, H and W even): input channels [0, up.C) are the nearest 2x upsampling of `up`
// (N x H/2 x W/2), read by the kernels' staging
int conv_fwd(int li, const Tensor& in, void* out, uint32_t out_stride, uint32_t out_off, uint32_t N, uint32_t H,
             uint32_t W, bool outf, hipStream_t s, uint16_t* pool = nullptr, const Tensor* up = nullptr) {
    const Layer& L = net.L[li];
    ConvArgs a{};
    a.in = in.p;
    a.in_stride = in.C;
    a.w = net.wb + L.d.wb_off;
    a.bias = net.params + L.d.b_off;
    a.out = out;
    a.out_stride = out_stride;
    a.out_off = out_off;
    a.N = N; a.H = H; a.W = W;
    a.Cin = L.cin;
    a.Cout = L.cout;
    a.pool = pool;
    a.up = up ? up->p : in.p;
    a.up_C = up ? up->C : 0u;
    const uint32_t nt = (L.cout + 15u) / 16u;
    if (outf) return launch_conv_nt<false, true, false>(nt, a, s);
    return L.relu ? launch_conv_nt<true, false, false>(nt, a, s) : launch_conv_nt<false, false, false>(nt, a, s);
}

// backward-data of layer li: g (Cout channels, stride g.C, g.C % 8 == 0) -> dX (Cin channels),
// masked by the forward input X (> 0) when mask is given
// low, low_g (optional, H and W even): X's channels [0, low.C) are the upsampling of `low`, whose gradient (masked
// by it) goes to low_g instead of dX
int conv_bwd_data(int li, const Tensor& g, const Tensor& dx, const Tensor* mask, uint32_t N, uint32_t H, uint32_t W,
                  hipStream_t s, const Tensor* low = nullptr, const Tensor* low_g = nullptr) {
    const Layer& L = net.L[li];
    ConvArgs a{};
    a.in = a.up = g.p;
    a.in_stride = g.C;
    a.w = net.wt + L.d.wt_off;
    a.bias = nullptr;
    a.out = dx.p;
    a.out_stride = dx.C;
    a.out_off = 0;
    a.mask = mask ? mask->p : nullptr;
    a.mask_stride = mask ? mask->C : 0;
    if (low) {
        a.low_mask = low->p;
        a.low_sum = low_g->p;
        a.low_C = low->C;
    }
    a.N = N; a.H = H; a.W = W;
    a.Cin = L.d.cout8;
    a.Cout = L.cin;
    const uint32_t nt = (L.cin + 15u) / 16u;
    return mask ? launch_conv_nt<false, false, true>(nt, a, s) : launch_conv_nt<false, false, false>(nt, a, s);
}

// level of a layer's pixels: 0 at full size, each next one half the width and height
uint32_t layer_level(int li) { return li < 10 ? (uint32_t)li / 2u : li < 18 ? 3u - (uint32_t)(li - 10) / 2u : 0u; }

// How the weight gradients of a batch of N x H x W are split over one launch's workgroups, and where
// their partial sums lie: about kWgPerCu workgroups per CU in all, as many as are resident (more write and
// read more partial sums; 8 fine-tuning steps 4.92 ms with 4, 4.94 with 3, 5.15 with 8, with 64 output channels
// a workgroup and 2 per CU 5.18, with 32 and 5 5.10), each of about the same work: a tile costs its staging,
// about as much as 4 blocks of 16 x 16 channels, and its blocks.
constexpr uint32_t kWgPerCu = 4;
int plan_wgrad(uint32_t N, uint32_t H, uint32_t W) {
    uint64_t work = 0;
    auto cost = [](const WGradArgs& a) { return 4u + a.nco * a.nci; };
    for (int i = 0; i < kLayers; ++i) {
        const Layer& L = net.L[i];
        WGradArgs& a = net.wg.l[i];
        const uint32_t lvl = layer_level(i), co = (L.cout + 15u) / 16u, ci = (L.cin + 15u) / 16u;
        a.N = N; a.H = H >> lvl; a.W = W >> lvl;
        a.Cin = L.cin;
        a.Cout = L.cout;
        a.cob = (co + kWgMaxCo - 1u) / kWgMaxCo;
        a.nco = (co + a.cob - 1u) / a.cob;
        a.nci = std::min(ci, kWgMaxCi);
        a.cib = (ci + a.nci - 1u) / a.nci;
        a.ntx = (a.W + kWgX - 1u) / kWgX;
        a.nty = (a.H + kWgY - 1u) / kWgY;
        a.tiles = N * a.ntx * a.nty;
        work += (uint64_t)a.tiles * a.cob * a.cib * cost(a);
    }
    const uint64_t share = work / (kWgPerCu * device_cus()) + 1u;   // of one workgroup
    uint64_t off = 0;
    uint32_t first = 0;
    for (int i = 0; i < kLayers; ++i) {
        const Layer& L = net.L[i];
        WGradArgs& a = net.wg.l[i];
        a.tiles_chunk = (uint32_t)std::max<uint64_t>(1u, std::min<uint64_t>(a.tiles, (share + cost(a) - 1u) / cost(a)));
        const uint32_t chunks = (a.tiles + a.tiles_chunk - 1u) / a.tiles_chunk;
        a.first = first;
        first += (chunks + 7u) / 8u * 8u * a.cob * a.cib;
        net.parts.l[i].off = off;
        net.parts.l[i].chunks = chunks;
        net.parts.l[i].n = L.d.nw + L.cout;
        net.parts.l[i].first = L.d.w_off;
        off += (uint64_t)chunks * (L.d.nw + L.cout);
    }
    net.wg_blocks = first;
    if (off > net.part_cap || !net.part) {
        hipFree(net.part);
        net.part = nullptr;
        net.part_cap = 0;
        if (hipMalloc(&net.part, off * 4) != hipSuccess) {
            net.part = nullptr;
            return -1;
        }
        net.part_cap = off;
    }
    for (int i = 0; i < kLayers; ++i) net.wg.l[i].part = net.part + net.parts.l[i].off;
    return 0;
}

// the operands of layer li's weight gradient: its input x (channels [0, up.C) the upsampling of up) and its
// output's gradient g
void wgrad_of(int li, const Tensor& x, const Tensor& g, const Tensor* up = nullptr) {
    WGradArgs& a = net.wg.l[li];
    a.up = up ? up->p : x.p;
    a.up_C = up ? up->C : 0u;
    a.in = x.p;
    a.in_stride = x.C;
    a.g = g.p;
    a.g_stride = g.C;
}

int prep_weights(hipStream_t s) {
    if (!net.weights_dirty) return 0;
    uint32_t total = 0;
    for (auto& L : net.L) total += L.d.nw;
    hipLaunchKernelGGL(k_prep_weights, dim3(blocks(total)), dim3(256), 0, s, net.params, net.ldev, (uint32_t)kLayers,
                       net.wb, net.wt, total);
    if (hipGetLastError() != hipSuccess) return -1;
    net.weights_dirty = false;
    return 0;
}

// forward pass on net.x0 (N x H x W, H and W multiples of 16) -> net.y
// The decoder's upsampled channels are read straight from the lower level wherever they are needed; cat[l]
// holds the skip, in its channels of the concatenation, or (dense: inference) by itself, pixel by
// pixel: half of each 160 B row of the level-0 concatenation lies in lines that the other half shares.
int forward(uint32_t N, uint32_t H, uint32_t W, hipStream_t s, bool dense = false) {
    if (prep_weights(s) != 0) return -1;
    int rc = 0;
    Tensor in = net.x0;
    for (int l = 0; l < 4 && rc == 0; ++l) {
        const uint32_t h = H >> l, w = W >> l;
        rc |= conv_fwd(2 * l, in, net.a[l].p, net.a[l].C, 0, N, h, w, false, s);
        rc |= conv_fwd(2 * l + 1, net.a[l], net.cat[l].p, dense ? net.E[l] : net.cat[l].C, dense ? 0u : net.U[l], N, h,
                       w, false, s, net.pool[l].p);
        in = net.pool[l];
    }
    const uint32_t h4 = H >> 4, w4 = W >> 4;
    rc |= conv_fwd(8, in, net.b1.p, net.b1.C, 0, N, h4, w4, false, s);
    rc |= conv_fwd(9, net.b1, net.b2.p, net.b2.C, 0, N, h4, w4, false, s);
    Tensor prev = net.b2;
    for (int l = 3; l >= 0 && rc == 0; --l) {
        const uint32_t h = H >> l, w = W >> l;
        const int li = 10 + 2 * (3 - l);
        // (dense: channel U of a pixel is the skip's first; those below are never read from here)
        const Tensor skip = dense ? Tensor{net.cat[l].p - net.U[l], net.E[l]} : net.cat[l];
        rc |= conv_fwd(li, skip, net.d1[l].p, net.d1[l].C, 0, N, h, w, false, s, nullptr, &prev);
        rc |= conv_fwd(li + 1, net.d1[l], net.d2[l].p, net.d2[l].C, 0, N, h, w, false, s);
        prev = net.d2[l];
    }
    rc |= conv_fwd(18, net.d2[0], net.y, 3, 0, N, H, W, true, s);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

// loss of net.y against net.target and the backward pass; loss into *loss_dev.  lr null: gradient
// -> net.grads, else an Adam step at that rate (parameters and their BF16 copies)
int backward(uint32_t N, uint32_t H, uint32_t W, float* loss_dev, const float* lr, hipStream_t s) {
    const size_t P0 = (size_t)N * H * W;
    const float scale = 1.0f / (float)(3 * P0);
    const uint32_t lb = blocks(P0);
    if (plan_wgrad(N, H, W) != 0) return -1;
    hipLaunchKernelGGL(k_loss, dim3(lb), dim3(256), 0, s, net.y, net.target, net.x0.p, (uint32_t)P0, scale,
                       net.gy.p, net.lpart);
    hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(256), 0, s, net.lpart, lb, scale, loss_dev);
    int rc = 0;
    // output layer
    wgrad_of(18, net.d2[0], net.gy);
    rc |= conv_bwd_data(18, net.gy, net.gd2[0], &net.d2[0], N, H, W, s);
    // decoder, level 0 up to 3
    for (int l = 0; l < 4 && rc == 0; ++l) {
        const uint32_t h = H >> l, w = W >> l;
        const int li = 10 + 2 * (3 - l);
        wgrad_of(li + 1, net.d1[l], net.gd2[l]);
        rc |= conv_bwd_data(li + 1, net.gd2[l], net.gd1[l], &net.d1[l], N, h, w, s);
        // the up part of the concatenation: the coarser level's output and its gradient
        const Tensor &prev = l < 3 ? net.d2[l + 1] : net.b2, &gprev = l < 3 ? net.gd2[l + 1] : net.gb2;
        wgrad_of(li, net.cat[l], net.gd1[l], &prev);
        rc |= conv_bwd_data(li, net.gd1[l], net.gcat[l], &net.cat[l], N, h, w, s, &prev, &gprev);
    }
    // bottleneck
    const uint32_t h4 = H >> 4, w4 = W >> 4;
    wgrad_of(9, net.b1, net.gb2);
    rc |= conv_bwd_data(9, net.gb2, net.gb1, &net.b1, N, h4, w4, s);
    wgrad_of(8, net.pool[3], net.gb1);
    rc |= conv_bwd_data(8, net.gb1, net.gpool[3], nullptr, N, h4, w4, s);
    // encoder, level 3 down to 0
    for (int l = 3; l >= 0 && rc == 0; --l) {
        const uint32_t h = H >> l, w = W >> l;
        const size_t n8 = (size_t)N * h * w * (net.E[l] / 8);
        hipLaunchKernelGGL(k_pool_bwd, dim3(blocks(n8)), dim3(256), 0, s, net.gpool[l].p, net.gcat[l].p,
                           net.cat[l].p, net.cat[l].C, net.U[l], net.gskip[l].p, N, h, w, net.E[l]);
        // enc conv 2: input a[l], output (skip) in cat[l]
        Tensor skip_in = net.a[l];
        wgrad_of(2 * l + 1, skip_in, net.gskip[l]);
        rc |= conv_bwd_data(2 * l + 1, net.gskip[l], net.ga[l], &net.a[l], N, h, w, s);
        // enc conv 1: input pool[l-1] (or x0)
        const Tensor& in = l > 0 ? net.pool[l - 1] : net.x0;
        wgrad_of(2 * l, in, net.ga[l]);
        if (l > 0) rc |= conv_bwd_data(2 * l, net.ga[l], net.gpool[l - 1], nullptr, N, h, w, s);
    }
    if (rc != 0) return -1;
    hipLaunchKernelGGL(k_conv3x3_wgrad, dim3(net.wg_blocks), dim3(kWgThreads), 0, s, net.wg);
    // no step on gradients that are not there: where a launch above failed, the partial sums are an earlier pass's
    if (hipGetLastError() != hipSuccess) return -1;
    AdamArgs o{};
    if (lr) {
        net.adam_t += 1;
        const float b1 = 0.9f, b2 = 0.999f;
        o = AdamArgs{net.params, net.adam_m, net.adam_v, net.ldev, net.wb, net.wt, *lr, b1, b2, 1e-8f,
                     1.0f - powf(b1, (float)net.adam_t), 1.0f - powf(b2, (float)net.adam_t)};
        hipLaunchKernelGGL(k_wgrad_reduce<true>, dim3(blocks(net.nparam)), dim3(256), 0, s, net.part, net.parts,
                           (uint32_t)net.nparam, net.grads, o);
    } else {
        hipLaunchKernelGGL(k_wgrad_reduce<false>, dim3(blocks(net.nparam)), dim3(256), 0, s, net.part, net.parts,
                           (uint32_t)net.nparam, net.grads, o);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int ensure_io(size_t bytes) {
    if (bytes <= net.io_cap && net.io) return 0;
    hipFree(net.io);
    net.io = nullptr;
    net.io_cap = 0;
    if (hipMalloc(&net.io, bytes) != hipSuccess) return -1;
    net.io_cap = bytes;
    return 0;
}

uint32_t pcg(uint32_t v) {
    const uint32_t state = v * 747796405u + 2891336453u;
    const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}

// denoise an h x w frame whose radiance and G-buffer are in device memory; out_dev RGBA32F
float spp_feature(uint32_t spp) { return log2f((float)(spp ? spp : 1u)) * 0.125f; }

int denoise_device(const float4* rad, const float4* gbuf, uint32_t h, uint32_t w, uint32_t spp, float4* out_dev,
                   float* ms, hipStream_t s) {
    const uint32_t hp = (h + 15u) & ~15u, wp = (w + 15u) & ~15u;
    if (ensure_act((size_t)hp * wp) != 0) return -1;
    hipEventRecord(net.e0, s);
    hipLaunchKernelGGL(k_features, dim3(blocks((size_t)hp * wp)), dim3(256), 0, s, rad, gbuf, h, w, hp, wp,
                       spp_feature(spp), net.x0.p);
    if (forward(1, hp, wp, s, true) != 0) return -1;
    hipLaunchKernelGGL(k_output, dim3(blocks((size_t)h * w)), dim3(256), 0, s, net.y, net.x0.p, h, w, wp, rad,
                       blend_alpha(spp), out_dev);
    hipEventRecord(net.e1, s);
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    if (ms) hipEventElapsedTime(ms, net.e0, net.e1);
    return 0;
}

}  // namespace

extern "C" {

int32_t vt_dn_init(const vt_dn_config* cfg) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!vt_rt_inited() || !cfg) return -1;
    hipSetDevice(vt_rt_device());
    if (net.on) free_all();
    for (int l = 0; l < 5; ++l)
        if (cfg->enc[l] == 0 || cfg->enc[l] % 16 || cfg->enc[l] > (uint32_t)kMaxWidth) {
            vt_rt_set_error("vt_dn_init: widths must be multiples of 16, at most 96");
            return -1;
        }
    for (int l = 0; l < 4; ++l)
        if (cfg->dec[l] == 0 || cfg->dec[l] % 16 || cfg->dec[l] > (uint32_t)kMaxWidth) {
            vt_rt_set_error("vt_dn_init: widths must be multiples of 16, at most 96");
            return -1;
        }
    for (int l = 0; l < 5; ++l) net.E[l] = cfg->enc[l];
    for (int l = 0; l < 4; ++l) net.D[l] = cfg->dec[l];
    net.U[3] = net.E[4];
    for (int l = 2; l >= 0; --l) net.U[l] = net.D[l + 1];
    set_layer(0, kInCh, net.E[0], true);
    set_layer(1, net.E[0], net.E[0], true);
    for (int l = 1; l < 4; ++l) {
        set_layer(2 * l, net.E[l - 1], net.E[l], true);
        set_layer(2 * l + 1, net.E[l], net.E[l], true);
    }
    set_layer(8, net.E[3], net.E[4], true);
    set_layer(9, net.E[4], net.E[4], true);
    for (int l = 3; l >= 0; --l) {
        const int li = 10 + 2 * (3 - l);
        set_layer(li, net.U[l] + net.E[l], net.D[l], true);
        set_layer(li + 1, net.D[l], net.D[l], true);
    }
    set_layer(18, net.D[0], kOutCh, false);
    size_t off = 0, wb = 0, wt = 0;
    LayerDev ld[kLayers];
    for (int i = 0; i < kLayers; ++i) {
        Layer& L = net.L[i];
        L.d.cin = L.cin;
        L.d.cout = L.cout;
        L.d.cout8 = up8(L.cout);
        L.d.nw = L.cout * 9u * L.cin;
        L.d.w_off = (uint32_t)off;
        off += L.d.nw;
        L.d.b_off = (uint32_t)off;
        off += L.cout;
        L.d.wb_off = (uint32_t)wb;
        wb += L.d.nw;
        L.d.wt_off = (uint32_t)wt;
        wt += (size_t)L.cin * 9u * L.d.cout8;
        wb = (wb + 127) & ~(size_t)127;  // keep every layer's rows 16-byte aligned
        wt = (wt + 127) & ~(size_t)127;
        ld[i] = L.d;
    }
    net.nparam = off;
    net.nwb = wb;
    net.nwt = wt;
    hipStream_t s = vt_rt_stream();
    if (hipMalloc(&net.params, off * 4) != hipSuccess || hipMalloc(&net.grads, off * 4) != hipSuccess ||
        hipMalloc(&net.adam_m, off * 4) != hipSuccess || hipMalloc(&net.adam_v, off * 4) != hipSuccess ||
        hipMalloc(&net.wb, wb * 2) != hipSuccess || hipMalloc(&net.wt, wt * 2) != hipSuccess ||
        hipMalloc(&net.ldev, sizeof(ld)) != hipSuccess || hipMalloc(&net.losses, 1024 * 4) != hipSuccess ||
        hipEventCreate(&net.e0) != hipSuccess ||
        hipEventCreate(&net.e1) != hipSuccess) {
        vt_rt_set_error("vt_dn_init: allocation failed");
        free_all();
        return -1;
    }
    hipMemsetAsync(net.params, 0, off * 4, s);
    hipMemsetAsync(net.grads, 0, off * 4, s);
    hipMemsetAsync(net.adam_m, 0, off * 4, s);
    hipMemsetAsync(net.adam_v, 0, off * 4, s);
    hipMemsetAsync(net.wb, 0, wb * 2, s);
    hipMemsetAsync(net.wt, 0, wt * 2, s);  // padding columns (co >= Cout) stay zero
    hipMemcpyAsync(net.ldev, ld, sizeof(ld), hipMemcpyHostToDevice, s);
    if (hipStreamSynchronize(s) != hipSuccess) {
        free_all();
        return -1;
    }
    net.losses_cap = 1024;
    net.on = true;
    net.weights_dirty = true;
    return 0;
}

int32_t vt_dn_layers(uint32_t* out4, uint32_t max_layers) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on) return -1;
    for (uint32_t i = 0; i < (uint32_t)kLayers && i < max_layers && out4; ++i) {
        out4[4 * i] = net.L[i].cin;
        out4[4 * i + 1] = net.L[i].cout;
        out4[4 * i + 2] = net.L[i].d.w_off;
        out4[4 * i + 3] = net.L[i].d.b_off;
    }
    return kLayers;
}

uint64_t vt_dn_param_count(void) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    return net.on ? net.nparam : 0;
}

int32_t vt_dn_set_params(const float* params, uint64_t n) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !params || n != net.nparam) return -1;
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const hipError_t e = vt_copy_in(net.params, params, n * 4, s);
    hipMemsetAsync(net.adam_m, 0, n * 4, s);
    hipMemsetAsync(net.adam_v, 0, n * 4, s);
    net.adam_t = 0;
    net.weights_dirty = true;
    return hipStreamSynchronize(s) == hipSuccess && e == hipSuccess ? 0 : -1;
}

int32_t vt_dn_get_params(float* params, uint64_t n) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !params || n != net.nparam) return -1;
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const hipError_t e = vt_copy_out(params, net.params, n * 4, s);
    return hipStreamSynchronize(s) == hipSuccess && e == hipSuccess ? 0 : -1;
}

int32_t vt_dn_grad(const float* x, const float* target, uint32_t n, uint32_t h, uint32_t w, float* y, float* grad,
                   float* loss) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !x || !target || n == 0 || h == 0 || w == 0 || h % 16 || w % 16) {
        vt_rt_set_error("vt_dn_grad: bad arguments (h and w must be multiples of 16)");
        return -1;
    }
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t P0 = (size_t)n * h * w;
    if (ensure_act(P0) != 0 || ensure_grad(P0) != 0 || ensure_io(P0 * kInCh * 4) != 0) {
        vt_rt_set_error("vt_dn_grad: allocation failed");
        return -1;
    }
    hipMemcpyAsync(net.io, x, P0 * kInCh * 4, hipMemcpyHostToDevice, s);
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(blocks(P0 * kInCh)), dim3(256), 0, s, static_cast<const float*>(net.io),
                       net.x0.p, P0 * kInCh);
    hipMemcpyAsync(net.target, target, P0 * 3 * 4, hipMemcpyHostToDevice, s);
    if (forward(n, h, w, s) != 0 || backward(n, h, w, net.losses, nullptr, s) != 0) {
        vt_rt_set_error("vt_dn_grad: launch failed");
        return -1;
    }
    if (y) hipMemcpyAsync(y, net.y, P0 * 3 * 4, hipMemcpyDeviceToHost, s);
    if (grad) hipMemcpyAsync(grad, net.grads, net.nparam * 4, hipMemcpyDeviceToHost, s);
    if (loss) hipMemcpyAsync(loss, net.losses, 4, hipMemcpyDeviceToHost, s);
    return hipStreamSynchronize(s) == hipSuccess ? 0 : -1;
}

int32_t vt_dn_features(const float* rad_rgba, const float* gbuf8, uint32_t h, uint32_t w, uint32_t spp, float* out16) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !rad_rgba || !gbuf8 || !out16 || h == 0 || w == 0) return -1;
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t npx = (size_t)h * w;
    if (ensure_io(npx * (16 + 32 + 32 + 64)) != 0) return -1;
    char* io = static_cast<char*>(net.io);
    float4* rad = reinterpret_cast<float4*>(io);
    float4* gb = reinterpret_cast<float4*>(io + npx * 16);
    uint16_t* f = reinterpret_cast<uint16_t*>(io + npx * 48);
    hipMemcpyAsync(rad, rad_rgba, npx * 16, hipMemcpyHostToDevice, s);
    hipMemcpyAsync(gb, gbuf8, npx * 32, hipMemcpyHostToDevice, s);
    hipLaunchKernelGGL(k_features, dim3(blocks(npx)), dim3(256), 0, s, rad, gb, h, w, h, w, spp_feature(spp), f);
    std::vector<uint16_t> hb(npx * 16);
    hipMemcpyAsync(hb.data(), f, npx * 32, hipMemcpyDeviceToHost, s);
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    for (size_t i = 0; i < hb.size(); ++i) {
        const uint32_t u = (uint32_t)hb[i] << 16;
        std::memcpy(&out16[i], &u, 4);
    }
    return 0;
}

int32_t vt_dn_add_frame(const float* rad_rgba, const float* gbuf8, const float* target_rgba, uint32_t h, uint32_t w,
                        uint32_t spp) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !rad_rgba || !gbuf8 || !target_rgba || h < 16 || w < 16) return -1;
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t npx = (size_t)h * w;
    if (ensure_io(npx * 64) != 0) return -1;
    void* mem = nullptr;
    const size_t fbytes = (npx * 32 + 255) & ~(size_t)255;
    if (hipMalloc(&mem, fbytes + npx * 12) != hipSuccess) {
        vt_rt_set_error("vt_dn_add_frame: allocation failed");
        return -1;
    }
    char* io = static_cast<char*>(net.io);
    float4* rad = reinterpret_cast<float4*>(io);
    float4* gb = reinterpret_cast<float4*>(io + npx * 16);
    FrameDesc fd;
    fd.feat = static_cast<const uint16_t*>(mem);
    fd.target = reinterpret_cast<const float*>(static_cast<char*>(mem) + fbytes);
    fd.h = h;
    fd.w = w;
    hipError_t e = vt_copy_in(rad, rad_rgba, npx * 16, s);
    if (e == hipSuccess) e = vt_copy_in(gb, gbuf8, npx * 32, s);
    hipLaunchKernelGGL(k_features, dim3(blocks(npx)), dim3(256), 0, s, rad, gb, h, w, h, w, spp_feature(spp),
                       static_cast<uint16_t*>(mem));
    if (e == hipSuccess) e = vt_copy_in(rad, target_rgba, npx * 16, s);
    hipLaunchKernelGGL(k_rgba_to_rgb, dim3(blocks(npx)), dim3(256), 0, s, rad, const_cast<float*>(fd.target),
                       (uint32_t)npx);
    if (hipStreamSynchronize(s) != hipSuccess || e != hipSuccess) {
        hipFree(mem);
        return -1;
    }
    net.frame_mem.push_back(mem);
    net.frames.push_back(fd);
    return (int32_t)net.frames.size() - 1;
}

int32_t vt_dn_clear_frames(void) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on) return -1;
    hipSetDevice(vt_rt_device());
    hipStreamSynchronize(vt_rt_stream());
    for (void* p : net.frame_mem) hipFree(p);
    net.frame_mem.clear();
    net.frames.clear();
    return 0;
}

int32_t vt_dn_train(uint32_t iters, uint32_t batch, uint32_t crop, float lr, uint32_t seed, float* losses) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || net.frames.empty() || iters == 0 || batch == 0 || crop < 16 || crop % 16) {
        vt_rt_set_error("vt_dn_train: no frames or bad arguments (crop must be a multiple of 16)");
        return -1;
    }
    for (auto& f : net.frames)
        if (f.h < crop || f.w < crop) {
            vt_rt_set_error("vt_dn_train: a frame is smaller than the crop");
            return -1;
        }
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t P0 = (size_t)batch * crop * crop;
    if (ensure_act(P0) != 0 || ensure_grad(P0) != 0) {
        vt_rt_set_error("vt_dn_train: allocation failed");
        return -1;
    }
    if (net.losses_cap < iters) {
        hipFree(net.losses);
        net.losses = nullptr;
        net.losses_cap = 0;
        if (hipMalloc(&net.losses, (size_t)iters * 4) != hipSuccess) return -1;
        net.losses_cap = iters;
    }
    if (net.frames_dev_cap < net.frames.size()) {
        hipFree(net.frames_dev);
        net.frames_dev = nullptr;
        if (hipMalloc(&net.frames_dev, net.frames.size() * sizeof(FrameDesc)) != hipSuccess) return -1;
        net.frames_dev_cap = net.frames.size();
    }
    hipMemcpyAsync(net.frames_dev, net.frames.data(), net.frames.size() * sizeof(FrameDesc), hipMemcpyHostToDevice, s);
    const size_t ncrop = (size_t)iters * batch;
    if (net.crops_cap < ncrop) {
        hipFree(net.crops_dev);
        net.crops_dev = nullptr;
        if (hipMalloc(&net.crops_dev, ncrop * sizeof(CropDesc)) != hipSuccess) return -1;
        net.crops_cap = ncrop;
    }
    // crop positions: a seeded PCG stream, uniform over frames and positions
    std::vector<CropDesc> crops(ncrop);
    uint32_t st = pcg(seed ^ 0x9E3779B9u);
    for (auto& c : crops) {
        st = pcg(st);
        c.frame = st % (uint32_t)net.frames.size();
        const FrameDesc& f = net.frames[c.frame];
        st = pcg(st);
        c.y0 = st % (f.h - crop + 1u);
        st = pcg(st);
        c.x0 = st % (f.w - crop + 1u);
        c.pad = 0;
    }
    hipMemcpyAsync(net.crops_dev, crops.data(), ncrop * sizeof(CropDesc), hipMemcpyHostToDevice, s);
    if (hipStreamSynchronize(s) != hipSuccess) return -1;  // the host vector must outlive the copy
    const uint32_t warm = std::min<uint32_t>(100u, iters / 10u + 1u);
    for (uint32_t it = 0; it < iters; ++it) {
        hipLaunchKernelGGL(k_gather_crops, dim3(blocks(P0)), dim3(256), 0, s, net.frames_dev,
                           net.crops_dev + (size_t)it * batch, batch, crop, net.x0.p, net.target);
        // linear warm-up, then cosine decay to 5% of lr
        const float t = (float)it / (float)iters;
        float lr_t = lr * (0.05f + 0.95f * 0.5f * (1.0f + cosf(3.14159265f * t)));
        if (it < warm) lr_t *= (float)(it + 1) / (float)warm;
        if (forward(batch, crop, crop, s) != 0 || backward(batch, crop, crop, net.losses + it, &lr_t, s) != 0) {
            vt_rt_set_error("vt_dn_train: launch failed");
            return -1;
        }
    }
    if (losses) hipMemcpyAsync(losses, net.losses, (size_t)iters * 4, hipMemcpyDeviceToHost, s);
    return hipStreamSynchronize(s) == hipSuccess ? 0 : -1;
}

int32_t vt_dn_denoise(const float* rad_rgba, const float* gbuf8, uint32_t h, uint32_t w, uint32_t spp,
                      float* out_rgba, float* gpu_ms) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || !rad_rgba || !gbuf8 || !out_rgba || h == 0 || w == 0) return -1;
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t npx = (size_t)h * w;
    if (ensure_io(npx * 64) != 0) return -1;
    char* io = static_cast<char*>(net.io);
    float4* rad = reinterpret_cast<float4*>(io);
    float4* gb = reinterpret_cast<float4*>(io + npx * 16);
    float4* out = reinterpret_cast<float4*>(io + npx * 48);
    if (vt_copy_in(rad, rad_rgba, npx * 16, s) != hipSuccess || vt_copy_in(gb, gbuf8, npx * 32, s) != hipSuccess ||
        denoise_device(rad, gb, h, w, spp, out, gpu_ms, s) != 0) {
        vt_rt_set_error("vt_dn_denoise: failed");
        return -1;
    }
    const hipError_t e = vt_copy_out(out_rgba, out, npx * 16, s);
    return hipStreamSynchronize(s) == hipSuccess && e == hipSuccess ? 0 : -1;
}

int32_t vt_dn_denoise_frame(float* out_rgba, float* gpu_ms) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    const float4 *rad = nullptr, *gb = nullptr;
    uint32_t w = 0, h = 0, spp = 1;
    if (!net.on || !out_rgba || !vt_rt_frame(&rad, &gb, &w, &h, &spp)) {
        vt_rt_set_error("vt_dn_denoise_frame: no network or no frame with a G-buffer");
        return -1;
    }
    hipSetDevice(vt_rt_device());
    hipStream_t s = vt_rt_stream();
    const size_t npx = (size_t)h * w;
    if (ensure_io(npx * 16) != 0) return -1;
    float4* out = static_cast<float4*>(net.io);
    if (denoise_device(rad, gb, h, w, spp, out, gpu_ms, s) != 0) {
        vt_rt_set_error("vt_dn_denoise_frame: failed");
        return -1;
    }
    const hipError_t e = vt_copy_out(out_rgba, out, npx * 16, s);
    return hipStreamSynchronize(s) == hipSuccess && e == hipSuccess ? 0 : -1;
}

int32_t vt_dn_set_blend(const float* alpha, uint32_t n) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    if (!net.on || n > 32 || (n && !alpha)) return -1;
    for (uint32_t k = 0; k < n; ++k)
        if (!(alpha[k] >= 0.0f && alpha[k] <= 1.0f)) return -1;
    for (uint32_t k = 0; k < n; ++k) net.blend[k] = alpha[k];
    net.nblend = n;
    return 0;
}

void vt_dn_shutdown(void) {
    std::lock_guard<std::mutex> lk(vt_rt_lock());
    vt_dn_release();
}

}  // extern "C"

// Frees the denoiser; the caller holds the runtime lock (cleanup() calls it too).
void vt_dn_release() {
    if (!net.on && !net.params) return;
    hipSetDevice(vt_rt_device());
    hipStreamSynchronize(vt_rt_stream());
    free_all();
}
