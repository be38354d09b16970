// nrc.hip -- neural radiance cache: MLP inference, training (forward + backward) and Adam,
// hand-written for gfx950 bf16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation.
//
// Network: 96 input features (12-frequency sin/cos of the position, direction, normal,
// albedo, roughness, a constant 1, zero padding) -> 5 hidden layers of 64 (ReLU) -> 32
// outputs of which 0..2 are RGB radiance.  No biases (the constant feature biases the
// first layer).  Weights: FP32 master copy updated by Adam, and two bf16 copies in the
// order the matrix instructions read them (fwd_pos, bwd_pos).
//
// MFMA operand mapping (v_mfma_f32_16x16x32_bf16: one 16x16 output tile, 32-deep reduction;
// r = lane % 16, g = lane / 16):
//   A: lane supplies row r, eight reduction elements j = 0 .. 7 of its group g
//   B: lane supplies column r, the same reduction elements
//   D: lane holds rows 4g .. 4g + 3 of column r
// Reduction element (g, j) of 32-deep chunk c is feature 32 c + 8 g + j in every product.  (Another
// assignment would give sums that differ in their FP32 roundings and, through the rounding to
// bf16, predictions that differ by 2e-4.)  Every product is formed transposed: A = weights
// (rows = output features), B = activations (columns = samples), and row 4 g + i of row tile
// 2 c + h is output feature 32 c + 8 g + 4 h + i (feature_of).  The result then has a sample per
// lane, and two result tiles together are, converted to bf16, the B operand of chunk c of the
// next layer.  Activations never leave the registers; the weights are stored in that order
// instead, so a fragment is one 16-byte load per lane.
//
// A product with the identity turns a tile with a sample per lane into one with a feature per
// lane (exact: one term per sum), the operand form of dW = X^T G.
#include <hip/hip_runtime.h>
#include <math.h>
#include "crt_internal.h"
#include "nrc.h"

namespace crt {

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short  s16x4 __attribute__((ext_vector_type(4)));
typedef float  f32x4 __attribute__((ext_vector_type(4)));

constexpr int kFrag = 512;   // elements of one weight fragment: 64 lanes x 8

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// 16-deep product: lane supplies reduction elements 4g .. 4g + 3
__device__ __forceinline__ f32x4 mma16(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}

// A value the compiler takes for new at each call: the weight addresses of a tile go through
// it, or every fragment would be loaded before the loop over tiles and spilled.
__device__ __forceinline__ int fresh(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}

__device__ __forceinline__ bf16 to_bf16(float x) { return (bf16)x; }   // round to nearest even
__device__ __forceinline__ bf16x8 ld8(const bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }

__host__ __device__ constexpr int layer_k(int l) { return l == 0 ? kNrcIn : kNrcHid; }
__host__ __device__ constexpr int layer_n(int l) { return l == kNrcLayers - 1 ? kNrcOut : kNrcHid; }
// first forward fragment of layer l: (row tile, 32-deep chunk) fragments, 12 + 4 x 8 + 4 = 48
__host__ __device__ constexpr int fwd_frag(int l) { return l == 0 ? 0 : 12 + 8 * (l - 1); }
// first backward fragment of layer l >= 1: 4 x 8 + 4 = 36
__host__ __device__ constexpr int bwd_frag(int l) { return 8 * (l - 1); }

// feature of row (or column) r of the 16-wide tile t of a layer's outputs
__device__ __forceinline__ int feature_of(int t, int r) { return 32 * (t >> 1) + 8 * (r >> 2) + 4 * (t & 1) + (r & 3); }
// and back: feature f is row tile_row(f) of tile tile_of(f)
__device__ __forceinline__ int tile_of(int f) { return 2 * (f >> 5) + ((f >> 2) & 1); }
__device__ __forceinline__ int tile_row(int f) { return 4 * ((f >> 3) & 3) + (f & 3); }
// element of a fragment: row r, reduction feature k
__device__ __forceinline__ int frag_elem(int r, int k) { return (((k >> 3) & 3) * 16 + r) * 8 + (k & 7); }

// position of weight (k, c) of layer l among the forward fragments
__device__ __forceinline__ int fwd_pos(int l, int k, int c)
{
    return (fwd_frag(l) + tile_of(c) * (layer_k(l) / 32) + (k >> 5)) * kFrag + frag_elem(tile_row(c), k);
}

// position of weight (k, c) of layer l >= 1 among the backward fragments (rows = input
// features, reduction over the output features)
__device__ __forceinline__ int bwd_pos(int l, int k, int c)
{
    return (bwd_frag(l) + tile_of(k) * (layer_n(l) / 32) + (c >> 5)) * kFrag + frag_elem(tile_row(k), c);
}

// two features in one register
__device__ __forceinline__ uint32_t pack2(float lo, float hi)
{
    typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{to_bf16(lo), to_bf16(hi)});
}

// sin and cos of x times the FP32 number 2^freq pi.  sincosf on that product: the features are FP32
// sines and cosines before they become bf16 ones, for any x (the hardware's v_sin and v_cos take
// revolutions, and one known to 2^-25 leaves few correct bits near a zero crossing and none
// far outside the unit box).  kNear: the product is below 2^17 in magnitude, where sincosf needs
// no table for its reduction; told so, the compiler leaves that part out, 100 of 150 instructions.
template <bool kNear>
__device__ __forceinline__ uint32_t sincos_pair(float x, int freq)
{
    const float a = x * __uint_as_float(0x40490FDBu + ((uint32_t)freq << 23));
    if (kNear) __builtin_assume(__builtin_fabsf(a) < 131072.0f);
    float s, c;
    sincosf(a, &s, &c);
    return pack2(s, c);
}

// The lane's 24 input features of its sample (three B operands).  q: the sample's query (any
// query of the batch for the lanes beyond it, whose results are not used).  Features 2 p and
// 2 p + 1 are the pair of component p / 12 and frequency p % 12: pairs 16 c + 4 g .. in chunks
// c = 0 and 1, whose four belong to one component; the pairs 32 .. 35 of chunk 2 are all lane
// group 0's, so every group computes one of them and group 0 gathers them.
__device__ __forceinline__ void encode(const float *q, int g, bf16x8 (&f)[3])
{
    typedef float    f4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const float x0 = q[g < 3 ? 0 : 1], x1 = q[g < 2 ? 1 : 2], x2 = q[2];
    // direction, normal, albedo and roughness: features 72 .. 79 are group 1's, 80 and 81 group 2's
    const f4  ea = *reinterpret_cast<const f4 *>(q + (g == 1 ? 3 : 9));
    const f4  eb = *reinterpret_cast<const f4 *>(q + (g == 1 ? 7 : 9));
    const int f0 = g < 3 ? 4 * g : 0, f1 = g < 2 ? 4 + 4 * g : 4 * g - 8;
    uint32_t  v[9];
    // 16 * 2^11 pi < 2^17; a NaN is not near
    if (__all(fabsf(x0) <= 16.0f && fabsf(x1) <= 16.0f && fabsf(x2) <= 16.0f)) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            v[m]     = sincos_pair<true>(x0, f0 + m);
            v[4 + m] = sincos_pair<true>(x1, f1 + m);
        }
        v[8] = sincos_pair<true>(x2, 8 + g);
    } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) v[k] = 0u;
#pragma unroll 1
        for (int m = 0; m < 9; ++m) {
            const uint32_t p = sincos_pair<false>(m < 4 ? x0 : m < 8 ? x1 : x2, m < 4 ? f0 + m : m < 8 ? f1 + m - 4 : 8 + g);
#pragma unroll
            for (int k = 0; k < 9; ++k) v[k] = k == m ? p : v[k];
        }
    }
    const int   r    = __lane_id() & 15;
    const u32x4 mid  = {pack2(ea[0], ea[1]), pack2(ea[2], ea[3]), pack2(eb[0], eb[1]), pack2(eb[2], eb[3])};
    const u32x4 last = {pack2(ea[2], ea[3]), pack2(1.0f, 0.0f), 0u, 0u};
    u32x4 c2;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const uint32_t p = (uint32_t)__shfl((int)v[8], 16 * m + r);
        c2[m] = g == 0 ? p : g == 1 ? mid[m] : g == 2 ? last[m] : 0u;
    }
    f[0] = __builtin_bit_cast(bf16x8, u32x4{v[0], v[1], v[2], v[3]});
    f[1] = __builtin_bit_cast(bf16x8, u32x4{v[4], v[5], v[6], v[7]});
    f[2] = __builtin_bit_cast(bf16x8, c2);
}

// max(x, 0), 0 for NaN, in one instruction where fmaxf takes two (it first quiets its operand).
// The upper bound changes nothing: the largest float, like infinity, becomes infinity in bf16.
__device__ __forceinline__ float relu(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 3.402823466e+38f); }

// D tiles 2c, 2c + 1 as the B operand of the next product; relu: clamp below at 0.
template <bool kRelu>
__device__ __forceinline__ bf16x8 pack(f32x4 lo, f32x4 hi)
{
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[i]     = to_bf16(kRelu ? relu(lo[i]) : lo[i]);
        r[4 + i] = to_bf16(kRelu ? relu(hi[i]) : hi[i]);
    }
    return r;
}

// acc[rt][ct] = rows 16 rt .. of (weights x activations) for CT tiles of 16 samples.
template <int NK, int NR, int CT, class Load>
__device__ __forceinline__ void product(Load frag, const bf16x8 (&b)[3][CT], f32x4 (&acc)[4][CT])
{
#pragma unroll
    for (int rt = 0; rt < NR; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kc = 0; kc < NK; ++kc)
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
            const bf16x8 a = frag(rt * NK + kc);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = mma(a, b[kc][ct], acc[rt][ct]);
        }
}

template <int CT>
__device__ __forceinline__ void activate(const f32x4 (&acc)[4][CT], bf16x8 (&b)[3][CT])
{
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) b[c][ct] = pack<true>(acc[2 * c][ct], acc[2 * c + 1][ct]);
}

// Inference.  Bound by vector instructions (conversion, ReLU and, the larger part, the 36 sines
// and cosines of a sample: about 1550 per 64 samples, 81 us for 2.07M samples) beside the matrix
// pipe (184 products of 16 cycles, 39 us) and the query bytes (133 MB).  A block of four waves
// keeps the 46 used weight fragments in LDS (46 KB: three blocks, 12 waves per CU, which 160
// registers a lane also allow) and loops over tiles of 256 samples; a wave owns 64 samples, so
// a fragment read from LDS serves four products.  2,073,600 queries: 409 us with activations
// passed through LDS, weights re-read from L2 by every wave and the sines with their reduction
// for any argument inline; 147 us like this, with the same predictions bit for bit.
constexpr int kInferWaves = 4, kInferBlocks = 768;
constexpr int kInferFrags = 46;   // 44 of the hidden layers, row tile 0 of the output

// n_dev (when set) is a device-side count, clamped to the buffers' capacity n_host.
__global__ __launch_bounds__(64 * kInferWaves, 3) void k_nrc_infer(const float *__restrict__ q, float *__restrict__ out,
                                                                   uint32_t n_host, const uint32_t *__restrict__ n_dev,
                                                                   const bf16 *__restrict__ WF)
{
    __shared__ bf16x8 ws[kInferFrags * 64];
    const uint32_t n = n_dev ? min(*n_dev, n_host) : n_host;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint32_t wv = threadIdx.x >> 6;
    constexpr uint32_t kTile = 64 * kInferWaves;
    const uint32_t ntiles = (uint32_t)(((uint64_t)n + kTile - 1) / kTile);
    if (blockIdx.x >= ntiles) return;
    for (int i = threadIdx.x; i < kInferFrags * 64; i += 64 * kInferWaves) ws[i] = ld8(WF + (size_t)i * 8);
    __syncthreads();
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint32_t s0 = tile * kTile + wv * 64;
        bf16x8 b[3][4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
            const uint32_t s = s0 + ct * 16 + r;
            bf16x8 f[3];
            encode(q + (size_t)min(s, n - 1u) * kNrcQuery, g, f);
#pragma unroll
            for (int c = 0; c < 3; ++c) b[c][ct] = f[c];
        }
        f32x4 acc[4][4];
#define FWD(L, NK, NR)                                                                        \
    {                                                                                         \
        const bf16x8 *w = ws + fwd_frag(L) * 64 + fresh(lane);                                \
        product<NK, NR, 4>([&](int f) { return w[f * 64]; }, b, acc);                         \
    }
        FWD(0, 3, 4)
        activate<4>(acc, b);
        FWD(1, 2, 4)
        activate<4>(acc, b);
        FWD(2, 2, 4)
        activate<4>(acc, b);
        FWD(3, 2, 4)
        activate<4>(acc, b);
        FWD(4, 2, 4)
        activate<4>(acc, b);
        FWD(5, 2, 1)
#undef FWD
        if (g == 0) {
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                const uint32_t s = s0 + ct * 16 + r;
                if (s < n)
                    for (int i = 0; i < 3; ++i) out[(size_t)s * 3 + i] = acc[0][ct][i];
            }
        }
    }
}

// Training.  A block of four waves owns tiles of 64 samples, 16 per wave.  Forward and the
// backward data products stay in each wave's registers (no barrier); for dW the waves exchange
// the layer's activations and output gradients, a feature per lane, through LDS, and wave w
// forms the column tile w of the layer's dW over all 64 samples.  The dW tiles accumulate in
// registers over all the block's tiles (92 registers a lane), so a batch writes one gradient
// partial per block, at most kNrcMaxParts of them, instead of one per 64 samples.  Two exchange
// buffers alternate, so a layer costs one barrier.  40 KB of LDS fit in beside three
// traversal blocks on a CU, that is once one of the four has ended.  Bound by the chain of 12 products of one tile (a few microseconds)
// for batches below 16,384; for larger ones by the weight fragments from L2 (82 KB per wave and
// tile).  16,384 samples: 28 us with the activations saved to HBM and gathered from there by 2
// bytes, 23 us like this; with the partials' sum (60 -> 5 us) and one pinned copy of gradient and
// loss a gradient call went from 131 to 50 us.
constexpr int kXt = 6 * 4 * 64, kGt = 4 * 4 * 64;   // exchanged fragments of 4 elements

__global__ __launch_bounds__(256, 1) void k_nrc_train(const float *__restrict__ q, const float *__restrict__ target,
                                                      uint32_t n, float inv_count, const bf16 *__restrict__ WF,
                                                      const bf16 *__restrict__ WB, float *__restrict__ partial,
                                                      float *__restrict__ partial_loss)
{
    __shared__ bf16x4 xs[2][kXt], gs[2][kGt];
    __shared__ float  wloss[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const uint32_t ntiles = (n + 63u) / 64u;
    // column r of ident[h] selects reduction element (r / 4, 4 h + r % 4)
    bf16x8 ident[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) ident[h][j] = to_bf16(g == (r >> 2) && j == 4 * h + (r & 3) ? 1.0f : 0.0f);
    const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto turn = [&](bf16x8 f, int h) {   // feature tile h of a chunk, samples in the registers
        const f32x4 d = mma(f, ident[h], zero);
        return bf16x4{to_bf16(d[0]), to_bf16(d[1]), to_bf16(d[2]), to_bf16(d[3])};
    };
    f32x4 dw0[6], dwh[4][4], dw5 = zero;   // dW tiles of column tile wv (layer 5: row tile wv)
#pragma unroll
    for (int k = 0; k < 6; ++k) dw0[k] = zero;
#pragma unroll
    for (int l = 0; l < 4; ++l)
#pragma unroll
        for (int k = 0; k < 4; ++k) dwh[l][k] = zero;
    float lsum = 0.0f;
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint32_t s = tile * 64u + wv * 16 + r;
        bf16x8 b[3][1];
        bf16x4 xt[6];            // input features, turned
        bf16x4 ht[5][4];         // hidden activations, turned
        uint32_t live[5];        // bit 8 c + j: hidden activation (c, j) of this lane is positive
        {
            bf16x8 f[3];
            encode(q + (size_t)min(s, n - 1u) * kNrcQuery, g, f);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                b[c][0] = f[c];
                xt[2 * c]     = turn(f[c], 0);
                xt[2 * c + 1] = turn(f[c], 1);
            }
        }
        f32x4 acc[4][1];
#define FWD(L, NK, NR)                                                                  \
    {                                                                                   \
        const bf16 *w = WF + fwd_frag(L) * kFrag + fresh(lane * 8);                     \
        product<NK, NR, 1>([&](int f) { return ld8(w + f * kFrag); }, b, acc);          \
    }
#define HIDDEN(L, NK)                                                                   \
    FWD(L, NK, 4)                                                                       \
    activate<1>(acc, b);                                                                \
    live[L] = 0u;                                                                       \
    _Pragma("unroll") for (int c = 0; c < 2; ++c)                                       \
    {                                                                                   \
        ht[L][2 * c]     = turn(b[c][0], 0);                                            \
        ht[L][2 * c + 1] = turn(b[c][0], 1);                                            \
        _Pragma("unroll") for (int j = 0; j < 8; ++j)                                   \
            live[L] |= (float)b[c][0][j] > 0.0f ? 1u << (8 * c + j) : 0u;               \
    }
        HIDDEN(0, 3)
        HIDDEN(1, 2)
        HIDDEN(2, 2)
        HIDDEN(3, 2)
        HIDDEN(4, 2)
#undef HIDDEN
        FWD(5, 2, 1)
#undef FWD
        // loss and dL/dy: the lanes of group 0 hold the three outputs of their sample
        bf16x8 gy;
#pragma unroll
        for (int j = 0; j < 8; ++j) gy[j] = to_bf16(0.0f);
        if (g == 0 && s < n) {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const float y = acc[0][0][i], e = y - target[(size_t)s * 3 + i], den = y * y + kNrcEpsRel;
                lsum += e * e / den * inv_count;
                gy[i] = to_bf16(2.0f * e / den * inv_count);
            }
        }
        // Layer L: share its input X (NX feature tiles) and output gradient G (NG tiles), then
        // accumulate dW.  The barrier also keeps this layer's stores behind the reads of the
        // layer before last, which used the same buffer.
        auto share = [&](const auto &x, const auto &gt, int buf) {
#pragma unroll
            for (int k = 0; k < (int)(sizeof x / sizeof x[0]); ++k) xs[buf][(k * 4 + wv) * 64 + lane] = x[k];
#pragma unroll
            for (int k = 0; k < (int)(sizeof gt / sizeof gt[0]); ++k) gs[buf][(k * 4 + wv) * 64 + lane] = gt[k];
            __syncthreads();
        };
        b[0][0] = gy;
        {
            const bf16x4 gt[1] = {turn(gy, 0)};
            share(ht[4], gt, 0);
#pragma unroll
            for (int p = 0; p < 4; ++p) dw5 = mma16(xs[0][(wv * 4 + p) * 64 + lane], gs[0][p * 64 + lane], dw5);
        }
        // gradient of layer L's input from b, masked by relu' of that input (hidden layer L - 1)
#define DX(L, NC)                                                                                              \
    {                                                                                                          \
        const bf16 *w = WB + bwd_frag(L) * kFrag + fresh(lane * 8);                                            \
        product<NC, 4, 1>([&](int f) { return ld8(w + f * kFrag); }, b, acc);                                  \
    }                                                                                                          \
    _Pragma("unroll") for (int t = 0; t < 4; ++t) _Pragma("unroll") for (int i = 0; i < 4; ++i)                \
        acc[t][0][i] = live[L - 1] >> (8 * (t >> 1) + 4 * (t & 1) + i) & 1u ? acc[t][0][i] : 0.0f;             \
    _Pragma("unroll") for (int c = 0; c < 2; ++c) b[c][0] = pack<false>(acc[2 * c][0], acc[2 * c + 1][0]);
#define DW(L, X, NX, D, BUF)                                                                                   \
    {                                                                                                          \
        const bf16x4 gt[4] = {turn(b[0][0], 0), turn(b[0][0], 1), turn(b[1][0], 0), turn(b[1][0], 1)};         \
        share(X, gt, BUF);                                                                                     \
        _Pragma("unroll") for (int p = 0; p < 4; ++p)                                                          \
        {                                                                                                      \
            const bf16x4 gg = gs[BUF][(wv * 4 + p) * 64 + lane];                                               \
            _Pragma("unroll") for (int k = 0; k < NX; ++k)                                                     \
                D[k] = mma16(xs[BUF][(k * 4 + p) * 64 + lane], gg, D[k]);                                      \
        }                                                                                                      \
    }
        DX(5, 1)
        DW(4, ht[3], 4, dwh[3], 1)
        DX(4, 2)
        DW(3, ht[2], 4, dwh[2], 0)
        DX(3, 2)
        DW(2, ht[1], 4, dwh[1], 1)
        DX(2, 2)
        DW(1, ht[0], 4, dwh[0], 0)
        DX(1, 2)
        DW(0, xt, 6, dw0, 1)
#undef DX
#undef DW
        // buffer 1 was read last and buffer 0 before a barrier: the next tile may start with 0
    }
    // the block's partial, in parameter order (columns 16 .. 31 of the output layer are zero)
    float *P = partial + (size_t)blockIdx.x * kNrcParams;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int k = 0; k < 6; ++k) P[feature_of(k, 4 * g + i) * kNrcHid + feature_of(wv, r)] = dw0[k][i];
#pragma unroll
        for (int l = 0; l < 4; ++l)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                P[nrc_w_off(l + 1) + feature_of(k, 4 * g + i) * kNrcHid + feature_of(wv, r)] = dwh[l][k][i];
        float *p5 = P + nrc_w_off(5) + feature_of(wv, 4 * g + i) * kNrcOut + r;
        p5[0]  = dw5[i];
        p5[16] = 0.0f;
    }
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
    if (lane == 0) wloss[wv] = lsum;
    __syncthreads();
    if (threadIdx.x == 0) partial_loss[blockIdx.x] = wloss[0] + wloss[1] + wloss[2] + wloss[3];
}

// Sum of the partials of 256 parameters per block: 16 waves take the rows in turn, a lane four
// consecutive parameters (16 bytes), and the waves' sums meet in LDS.  Thread t < 256 returns
// the sum of parameter 256 blockIdx + t.  With one thread per parameter walking all the rows,
// 256 rows (25 MB) took 60 us.
constexpr int kSumWaves = 16;

__device__ __forceinline__ float sum_rows(const float *__restrict__ partial, uint32_t nrows)
{
    __shared__ float4 part[kSumWaves][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float *src = partial + blockIdx.x * 256 + lane * 4;
#pragma unroll 4
    for (uint32_t t = wv; t < nrows; t += kSumWaves) {
        const float4 v = *reinterpret_cast<const float4 *>(src + (size_t)t * kNrcParams);
        a.x += v.x;
        a.y += v.y;
        a.z += v.z;
        a.w += v.w;
    }
    part[wv][lane] = a;
    __syncthreads();
    float s = 0.0f;
    if (threadIdx.x < 256)
        for (int w = 0; w < kSumWaves; ++w) s += reinterpret_cast<const float *>(part[w])[threadIdx.x];
    return s;
}

// Adam on the FP32 master weights from the summed partials; refreshes the bf16 copies.
// Padded outputs (columns >= 3 of the last layer) and padded input features (rows >= 83 of
// the first layer) stay zero.
__global__ __launch_bounds__(64 * kSumWaves) void k_nrc_adam(const float *__restrict__ partial, uint32_t nrows,
                                                             float *params, float *m, float *v, bf16 *WF, bf16 *WB,
                                                             float lr, float b1, float b2, float eps, float bc1,
                                                             float bc2, int update)
{
    const float gsum = update ? sum_rows(partial, nrows) : 0.0f;
    if (threadIdx.x >= 256) return;
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    int l = 0;
    while (l + 1 < kNrcLayers && p >= (uint32_t)nrc_w_off(l + 1)) ++l;
    const uint32_t N = layer_n(l);
    const uint32_t local = p - nrc_w_off(l), k = local / N, c = local % N;
    const bool frozen = (l == kNrcLayers - 1 && c >= 3) || (l == 0 && k >= 83);
    float w = params[p];
    if (update && !frozen) {
        const float mm = b1 * m[p] + (1.0f - b1) * gsum;
        const float vv = b2 * v[p] + (1.0f - b2) * gsum * gsum;
        m[p] = mm;
        v[p] = vv;
        w -= lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
        params[p] = w;
    }
    if (frozen) {
        w = 0.0f;
        params[p] = 0.0f;
    }
    WF[fwd_pos(l, (int)k, (int)c)] = to_bf16(w);
    if (l > 0) WB[bwd_pos(l, (int)k, (int)c)] = to_bf16(w);
}

// out[0 .. kNrcParams) = the summed gradient, out[kNrcParams] = the loss (summed in FP64 by a
// wave that has no parameter to finish), so the caller fetches both with one copy.
__global__ __launch_bounds__(64 * kSumWaves) void k_nrc_sum_partials(const float *__restrict__ partial,
                                                                     const float *__restrict__ partial_loss,
                                                                     uint32_t nrows, float *out)
{
    const float s = sum_rows(partial, nrows);
    if (threadIdx.x < 256) out[blockIdx.x * 256 + threadIdx.x] = s;
    if (blockIdx.x == 0 && threadIdx.x >= 256 && threadIdx.x < 320) {
        double d = 0.0;
        for (uint32_t t = threadIdx.x - 256; t < nrows; t += 64) d += partial_loss[t];
        for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o);
        if (threadIdx.x == 256) out[kNrcParams] = (float)d;
    }
}

static_assert(kNrcParams % 256 == 0, "sum_rows takes whole groups of 256 parameters");

hipError_t launch_infer(const float *q, float *out, uint32_t n, const uint32_t *n_dev, const __bf16 *WF, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    const uint32_t tiles = (uint32_t)(((uint64_t)n + 64 * kInferWaves - 1) / (64 * kInferWaves));
    // three blocks per CU are resident; each loads the weights once
    k_nrc_infer<<<std::min<uint32_t>(tiles, kInferBlocks), 64 * kInferWaves, 0, s>>>(q, out, n, n_dev, WF);
    return hipGetLastError();
}

}  // namespace

hipError_t nrc_launch_infer(const float *q, float *out, uint32_t n, const __bf16 *WF, hipStream_t s)
{
    return launch_infer(q, out, n, nullptr, WF, s);
}

hipError_t nrc_launch_infer_dev(const float *q, float *out, const uint32_t *n_dev, uint32_t n_max, const __bf16 *WF,
                                hipStream_t s)
{
    return launch_infer(q, out, n_max, n_dev, WF, s);
}

hipError_t nrc_launch_train(const float *q, const float *target, uint32_t n, const __bf16 *WF, const __bf16 *WB,
                            float *partial, float *partial_loss, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    k_nrc_train<<<nrc_partial_rows(n), 256, 0, s>>>(q, target, n, 1.0f / (3.0f * (float)n), WF, WB, partial, partial_loss);
    return hipGetLastError();
}

hipError_t nrc_launch_adam(const float *partial, uint32_t nrows, float *params, float *m, float *v, __bf16 *WF,
                           __bf16 *WB, float lr, float b1, float b2, float eps, uint64_t step, int update,
                           hipStream_t s)
{
    const float bc1 = 1.0f - powf(b1, (float)step), bc2 = 1.0f - powf(b2, (float)step);
    k_nrc_adam<<<kNrcParams / 256, 64 * kSumWaves, 0, s>>>(partial, nrows, params, m, v, WF, WB, lr, b1, b2, eps,
                                                           update ? bc1 : 1.0f, update ? bc2 : 1.0f, update);
    return hipGetLastError();
}

hipError_t nrc_launch_sum_partials(const float *partial, const float *partial_loss, uint32_t nrows, float *out,
                                   hipStream_t s)
{
    k_nrc_sum_partials<<<kNrcParams / 256, 64 * kSumWaves, 0, s>>>(partial, partial_loss, nrows, out);
    return hipGetLastError();
}

}  // namespace crt
