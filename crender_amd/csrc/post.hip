// post.hip -- GPU post-processing and denoising of the renderer's images.
//
// Post-processing restates cr::post_processor (CRender src/render/post/post_processor.cpp:
// 110-312 with assets/app/shaders/post_process.comp and blur.comp):
//   bloom  brightness pass (luma 0.2126/0.7152/0.0722 below `threshold` -> black, alpha 1),
//          then 10 separable blur passes alternating horizontal / vertical (15 taps, the
//          weights of blur.comp, texels outside the image read as 0), added to the colour
//          times `strength`;
//   gray   0.2126 r + 0.7162 g + 0.0722 b (post_process.comp's weights);
//   tonemapping  linear / Reinhard / Hejl-Burgess-Dawson ("Jim and Richard") / Uncharted 2,
//          with exposure and 1/gamma (not applied by Hejl-Burgess-Dawson).
// The reference dispatches floor(W/8) x floor(H/8) groups of 8x8, so pixels right of
// 8*floor(W/8) or below 8*floor(H/8) keep the cleared value 0; full_coverage = 0 keeps that
// behaviour, 1 processes every pixel.  Products and sums are evaluated in the shaders'
// order without contraction, so the CPU restatement in the oracle matches bit for bit
// except where pow() rounds differently.
//
// Denoising: the reference calls Intel Open Image Denoise (src/util/denoise.h:10-42), a
// pretrained network that is not part of this build.  Its inputs (colour, normal and albedo
// images) feed here an edge-avoiding a-trous wavelet filter (Dammertz et al. 2010,
// "Edge-Avoiding A-Trous Wavelet Transform for fast Global Illumination Filtering"):
// 5 levels of a 5x5 B3-spline kernel with hole spacing 2^level, each tap weighted by
// exp(-|dc|^2/sc^2) exp(-|dn|^2/sn^2) exp(-|da|^2/sa^2).
#include <hip/hip_runtime.h>
#include <float.h>
#include <math.h>

#include "crt_internal.h"

#pragma clang fp contract(off)

namespace crt {

namespace {

__constant__ float kBlurW[8] = {0.19744746769063704f, 0.1746973469158936f,  0.12099884565428047f,
                                0.06560233156931679f, 0.027839605612666265f, 0.009246250740395456f,
                                0.002403157286908872f, 0.00048872837522002f};

__device__ __forceinline__ bool covered(uint32_t x, uint32_t y, const PostDev &p)
{
    return x < p.cover_w && y < p.cover_h;
}

__device__ __forceinline__ float uncharted_map(float x)
{
    const float A = 0.15f, B = 0.50f, C = 0.10f, D = 0.20f, E = 0.02f, F = 0.30f;
    return ((x * (A * x + C * B) + D * E) / (x * (A * x + B) + D * F)) - E / F;
}

// post_process.comp after the bloom was added: gray, exposure and tone map.
__device__ __forceinline__ float4 graded(float r, float g0, float b0, const PostDev &p)
{
    float c[3] = {r, g0, b0};
    if (p.gray) {
        const float g = 0.2126f * c[0] + 0.7162f * c[1] + 0.0722f * c[2];
        c[0] = c[1] = c[2] = g;
    }
    if (p.tonemap) {
        const float ig = 1.0f / p.gamma;
        for (int k = 0; k < 3; ++k) c[k] = c[k] * p.exposure;
        if (p.tonemap_type == 0) {
            for (int k = 0; k < 3; ++k) c[k] = powf(c[k], ig);
        } else if (p.tonemap_type == 1) {
            for (int k = 0; k < 3; ++k) c[k] = powf(c[k] / (c[k] + 1.0f), ig);
        } else if (p.tonemap_type == 2) {
            for (int k = 0; k < 3; ++k) {
                const float v = fmaxf(0.0f, c[k] - 0.004f);
                c[k] = (v * (6.2f * v + 0.5f)) / (v * (6.2f * v + 1.7f) + 0.06f);
            }
        } else if (p.tonemap_type == 3) {
            const float ws = 1.0f / uncharted_map(11.2f);
            for (int k = 0; k < 3; ++k) c[k] = powf(uncharted_map(2.0f * c[k]) * ws, ig);
        }
    }
    return make_float4(c[0], c[1], c[2], 1.0f);
}

__global__ __launch_bounds__(256) void k_composite(const float4 *src, float4 *out, PostDev p)
{
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= p.w || y >= p.h) return;
    const size_t i = (size_t)y * p.w + x;
    const float4 s = src[i];
    out[i] = covered(x, y, p) ? graded(s.x, s.y, s.z, p) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// One horizontal and one vertical blur pass of a tile of 64 x 32 pixels.  The passes apart read
// and wrote the image once each (24 us at 1080p, 2.7 TB/s); together the horizontal result
// stays in LDS, at the price of reading the tile's border of 7 pixels again (1.75 times the
// tile, mostly from L2).  A thread computes runs of eight pixels, so a run of a row or column
// takes 22 LDS reads per channel instead of 120.  Row pitches of 79 words put the 8 runs of 8
// neighbouring rows on 64 different banks.  kFirst: the source is the image itself and its
// pixels pass the brightness threshold as they are loaded (k_bright).  kLast: the result is
// added to the image and graded instead of stored.  1080p, the whole of post-processing with
// bloom and tone map (Uncharted 2): brightness 13 + 10 blurs x 24 + composite 30 us before, now
// 33 + 3 x 31 + 60 us.  Bound by vector instructions: the sums keep blur.comp's order, so a tap
// is a product and a sum, and the border costs the horizontal pass 1.4 times the tile.
constexpr int kBlurR = 7, kBlurW_ = 64, kBlurH = 32, kRun = 8;
constexpr int kBlurIn = kBlurW_ + 2 * kBlurR, kBlurRows = kBlurH + 2 * kBlurR, kBlurPitch = kBlurIn + 1;

// eight neighbouring sums of the 15 taps in v[0 .. 21], each in blur.comp's order
__device__ __forceinline__ void blur_run(const float (&v)[kRun + 2 * kBlurR], float (&o)[kRun])
{
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
        float s = v[j + kBlurR] * kBlurW[0];
#pragma unroll
        for (int k = 1; k <= kBlurR; ++k) {
            s = s + v[j + kBlurR + k] * kBlurW[k];
            s = s + v[j + kBlurR - k] * kBlurW[k];
        }
        o[j] = s;
    }
}

template <bool kFirst, bool kLast>
__global__ __launch_bounds__(256) void k_blur2(const float4 *src, const float4 *image, float4 *dst, PostDev p)
{
    __shared__ float a[3][kBlurRows * kBlurPitch];   // source tile and border
    __shared__ float h[3][kBlurRows * kBlurW_];      // horizontal result
    const int x0 = blockIdx.x * kBlurW_, y0 = blockIdx.y * kBlurH, t = threadIdx.x;
    for (int i = t; i < kBlurRows * kBlurIn; i += 256) {
        const int r = i / kBlurIn, c = i - r * kBlurIn, x = x0 + c - kBlurR, y = y0 + r - kBlurR;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (x >= 0 && y >= 0 && x < (int)p.w && y < (int)p.h) {
            v = src[(size_t)y * p.w + x];
            // glm::dot(at, vec3(0.2126, 0.7152, 0.0722)) (post_processor.cpp:305)
            if (kFirst && v.x * 0.2126f + v.y * 0.7152f + v.z * 0.0722f < p.threshold) v = make_float4(0, 0, 0, 0);
        }
        a[0][r * kBlurPitch + c] = v.x;
        a[1][r * kBlurPitch + c] = v.y;
        a[2][r * kBlurPitch + c] = v.z;
    }
    __syncthreads();
    for (int i = t; i < kBlurRows * (kBlurW_ / kRun); i += 256) {
        const int r = i / (kBlurW_ / kRun), c = i % (kBlurW_ / kRun) * kRun, y = y0 + r - kBlurR;
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            float v[kRun + 2 * kBlurR], o[kRun];
#pragma unroll
            for (int k = 0; k < kRun + 2 * kBlurR; ++k) v[k] = a[ch][r * kBlurPitch + c + k];
            blur_run(v, o);
#pragma unroll
            for (int k = 0; k < kRun; ++k)   // glClearTexImage: 0 beyond the dispatch
                h[ch][r * kBlurW_ + c + k] = y >= 0 && covered(x0 + c + k, y, p) ? o[k] : 0.0f;
        }
    }
    __syncthreads();
    const int c = t % kBlurW_, r0 = t / kBlurW_ * kRun;   // 64 columns x 4 runs
    float o[3][kRun];
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
        float v[kRun + 2 * kBlurR];
#pragma unroll
        for (int k = 0; k < kRun + 2 * kBlurR; ++k) v[k] = h[ch][(r0 + k) * kBlurW_ + c];
        blur_run(v, o[ch]);
    }
    const uint32_t x = x0 + c;
    if (x >= p.w) return;
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
        const uint32_t y = y0 + r0 + k;
        if (y >= p.h) break;
        const size_t i  = (size_t)y * p.w + x;
        float4       px = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (covered(x, y, p)) {
            px = make_float4(o[0][k], o[1][k], o[2][k], 1.0f);
            if (kLast) {
                const float4 s = image[i];
                px = graded(s.x + px.x * p.strength, s.y + px.y * p.strength, s.z + px.z * p.strength, p);
            }
        }
        dst[i] = px;
    }
}

// One a-trous level: out = sum_k w_k * in_k / sum_k w_k over a 5x5 footprint with holes.
// A thread computes kRows pixels of a column that are `step` rows apart, so that they share
// taps: 5 (kRows + 4) taps for kRows pixels instead of 25 per pixel.  The weight is one
// exponential, 2^(log2 k - |dc|^2 ic - |dn|^2 in - |da|^2 ia) with log2 e in ic, in and ia.
constexpr int kRows = 4;

struct AtrousArgs {
    const float4 *in, *nrm, *alb;
    int           w, h, step;
    float         ic, in_, ia;
};
struct Tap {
    float3 c, n, a;   // colour, normal, albedo
};

// Sums of the thread's pixels (x, y0 + k step).  tap(ry, dx) is the tap `ry` steps below y0 and
// dx steps to the right; kInside: every tap lies in the image, otherwise those outside have
// weight 0 (their values are those of some pixel).
template <bool kInside, class Load>
__device__ __forceinline__ void atrous_rows(const AtrousArgs &g, int x, int y0, Load tap, float4 (&o)[kRows])
{
    // log2 of the 5x5 kernel (3/8, 1/4, 1/16 per axis)
    constexpr float kLog[3] = {-1.4150374992788437f, -2.0f, -4.0f};
    Tap   t0[kRows];
    float sr[kRows], sg[kRows], sb[kRows], sw[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        t0[k] = tap(k, 0);
        sr[k] = sg[k] = sb[k] = sw[k] = 0.0f;
    }
    // not unrolled: the compiler would load all 40 taps first and spill them
#pragma unroll 1
    for (int dx = -2; dx <= 2; ++dx) {
        const float lx  = dx == 0 ? kLog[0] : (dx == -1 || dx == 1 ? kLog[1] : kLog[2]);
        const int   xx  = x + dx * g.step;
        const bool  inx = kInside || (xx >= 0 && xx < g.w);
#pragma unroll
        for (int ry = -2; ry < kRows + 2; ++ry) {
            const int  yy = y0 + ry * g.step;
            const bool ok = kInside || (inx && yy >= 0 && yy < g.h);
            Tap t = tap(ry, dx);
            if (!kInside && !ok) t.c = make_float3(0.0f, 0.0f, 0.0f);   // 0 x weight 0, also for infinities
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                const int dy = ry - k;
                if (dy < -2 || dy > 2) continue;
                const float cx = t.c.x - t0[k].c.x, cy = t.c.y - t0[k].c.y, cz = t.c.z - t0[k].c.z;
                const float nx = t.n.x - t0[k].n.x, ny = t.n.y - t0[k].n.y, nz = t.n.z - t0[k].n.z;
                const float ax = t.a.x - t0[k].a.x, ay = t.a.y - t0[k].a.y, az = t.a.z - t0[k].a.z;
                const float dc = fmaf(cx, cx, fmaf(cy, cy, cz * cz));
                const float dn = fmaf(nx, nx, fmaf(ny, ny, nz * nz));
                const float da = fmaf(ax, ax, fmaf(ay, ay, az * az));
                const float lk = lx + kLog[dy < 0 ? -dy : dy];
                float wt = __builtin_amdgcn_exp2f(fmaf(-dc, g.ic, fmaf(-dn, g.in_, fmaf(-da, g.ia, lk))));
                if (!kInside && !ok) wt = 0.0f;
                sr[k] = fmaf(wt, t.c.x, sr[k]);
                sg[k] = fmaf(wt, t.c.y, sg[k]);
                sb[k] = fmaf(wt, t.c.z, sb[k]);
                sw[k] = sw[k] + wt;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kRows; ++k) o[k] = make_float4(sr[k] / sw[k], sg[k] / sw[k], sb[k] / sw[k], 1.0f);
}

__device__ __forceinline__ void atrous_store(const AtrousArgs &g, float4 *out, int x, int y0, const float4 (&o)[kRows])
{
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        const int y = y0 + k * g.step;
        if (y < g.h) out[(size_t)y * g.w + x] = o[k];
    }
}

// Whether the footprints of pixels x .. x + nx - 1 of kRows * ng rows from y0 lie in the image.
__device__ __forceinline__ bool atrous_inside(const AtrousArgs &g, int x, int nx, int y0, int ng)
{
    const int m = 2 * g.step;
    return x >= m && x + nx - 1 + m < g.w && y0 >= m && y0 + (kRows * ng - 1) * g.step + m < g.h;
}

// Any step: taps from global memory.  A wave is 64 pixels of a row group.  Levels with holes
// wider than kTileStep rows only; closer ones re-read lines from beyond L2 this way (155 us a
// level at 1080p, whether a thread computes one pixel or four).
__global__ __launch_bounds__(256, 4) void k_atrous(AtrousArgs g, float4 *out)
{
    const int xb = (int)(blockIdx.x * 64), x = xb + (int)threadIdx.x;
    const int q  = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * 4 + threadIdx.y));
    // rows y0 + k step of the group: residue class q % step, kRows rows of the class
    const int y0 = q / g.step * (kRows * g.step) + q % g.step;
    if (x >= g.w || y0 >= g.h) return;
    auto tap = [&](int ry, int dx) {
        const size_t j = (size_t)min(max(y0 + ry * g.step, 0), g.h - 1) * g.w + min(max(x + dx * g.step, 0), g.w - 1);
        const float4 c = g.in[j], n = g.nrm[j], a = g.alb[j];
        return Tap{make_float3(c.x, c.y, c.z), make_float3(n.x, n.y, n.z), make_float3(a.x, a.y, a.z)};
    };
    float4 o[kRows];
    if (atrous_inside(g, xb, 64, y0, 1)) atrous_rows<true>(g, x, y0, tap, o);
    else atrous_rows<false>(g, x, y0, tap, o);
    atrous_store(g, out, x, y0, o);
}

// Steps up to kTileStep: a block stages the taps of a tile -- TW pixels of 16 rows that are
// `step` apart, and two steps on every side -- in LDS, 36 bytes a tap, so every line comes from
// L2 about 1.3 (step 1) to 1.9 times (step 16) instead of ten.  Tiles are 64 wide while two
// blocks fit on a CU (step 8: 69 KB), 128 wide at step 16, where one block of eight waves
// (138 KB) hides more than one of four (92 KB).  A level at 1080p, by step 1, 2, 4, 8, 16: 51,
// 50, 56, 63, 79 us, near the 47 us of its vector instructions; 123 us at step 16 with tiles 64 wide.
constexpr int kTileGroups = 4, kTileRows = kRows * kTileGroups + 4, kTileStep = 16;
constexpr int    tile_width(int step) { return step <= 8 ? 64 : 128; }
constexpr size_t tile_bytes(int step) { return (size_t)kTileRows * (tile_width(step) + 4 * step) * 36; }

template <int TW>
__global__ __launch_bounds__(TW * kTileGroups, 2) void k_atrous_tile(AtrousArgs g, float4 *out)
{
    extern __shared__ float4 tile[];
    const int wpx = TW + 4 * g.step, npx = kTileRows * wpx;
    float4 *ta = tile, *tb = tile + npx;                 // colour, normal.x | normal.yz, albedo.xy
    float  *tc = reinterpret_cast<float *>(tile + 2 * npx);   // albedo.z
    const int q  = (int)blockIdx.y;                      // rows of residue class q % step
    const int yb = q / g.step * (kRows * kTileGroups * g.step) + q % g.step;
    const int xb = (int)blockIdx.x * TW, tid = (int)(threadIdx.y * TW + threadIdx.x);
    if (yb >= g.h) return;
    for (int i = tid; i < npx; i += TW * kTileGroups) {
        const int r = i / wpx, c = i - r * wpx;
        const int y = min(max(yb + (r - 2) * g.step, 0), g.h - 1), x = min(max(xb + c - 2 * g.step, 0), g.w - 1);
        const size_t j = (size_t)y * g.w + x;
        const float4 pc = g.in[j], pn = g.nrm[j], pa = g.alb[j];
        ta[i] = make_float4(pc.x, pc.y, pc.z, pn.x);
        tb[i] = make_float4(pn.y, pn.z, pa.x, pa.y);
        tc[i] = pa.z;
    }
    __syncthreads();
    const int x = xb + (int)threadIdx.x, y0 = yb + (int)threadIdx.y * kRows * g.step;
    if (x >= g.w || y0 >= g.h) return;
    const int base = (int)(threadIdx.y * kRows + 2) * wpx + (int)threadIdx.x + 2 * g.step;
    auto tap = [&](int ry, int dx) {
        const int    i = base + ry * wpx + dx * g.step;
        const float4 a = ta[i], b = tb[i];
        return Tap{make_float3(a.x, a.y, a.z), make_float3(a.w, b.x, b.y), make_float3(b.z, b.w, tc[i])};
    };
    float4 o[kRows];
    if (atrous_inside(g, xb, TW, yb, kTileGroups)) atrous_rows<true>(g, x, y0, tap, o);
    else atrous_rows<false>(g, x, y0, tap, o);
    atrous_store(g, out, x, y0, o);
}

}  // namespace

hipError_t launch_post(const PostDev &p, const float4 *in, float4 *out, float4 *t0, float4 *t1, hipStream_t s)
{
    if (!p.bloom) {
        k_composite<<<dim3((p.w + 63) / 64, (p.h + 3) / 4), dim3(64, 4), 0, s>>>(in, out, p);
        return hipGetLastError();
    }
    // blur.comp ping-pong (post_processor.cpp:270-300): ten passes, horizontal first
    const dim3 g((p.w + kBlurW_ - 1) / kBlurW_, (p.h + kBlurH - 1) / kBlurH);
    k_blur2<true, false><<<g, 256, 0, s>>>(in, nullptr, t0, p);
    k_blur2<false, false><<<g, 256, 0, s>>>(t0, nullptr, t1, p);
    k_blur2<false, false><<<g, 256, 0, s>>>(t1, nullptr, t0, p);
    k_blur2<false, false><<<g, 256, 0, s>>>(t0, nullptr, t1, p);
    k_blur2<false, true><<<g, 256, 0, s>>>(t1, in, out, p);
    return hipGetLastError();
}

hipError_t launch_atrous(const float4 *colour, const float4 *normal, const float4 *albedo, float4 *out, float4 *t0,
                         float4 *t1, uint32_t w, uint32_t h, int levels, float sc, float sn, float sa, hipStream_t s)
{
    // tiles of more LDS than a launch may use by default
    auto allow = [](const void *kernel, size_t bytes) {
        return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    };
    hipError_t e = allow(reinterpret_cast<const void *>(k_atrous_tile<64>), tile_bytes(8));
    if (e == hipSuccess) e = allow(reinterpret_cast<const void *>(k_atrous_tile<128>), tile_bytes(kTileStep));
    if (e != hipSuccess) return e;
    const float4 *src = colour;
    for (int l = 0; l < levels; ++l) {
        float4 *dst = l == levels - 1 ? out : (l % 2 == 0 ? t0 : t1);
        // the colour tolerance halves per level (finer detail survives at coarse scales)
        const float scl = sc * exp2f(-(float)l);
        const int     step = 1 << l;
        // log2 e / sigma^2; finite where 1 / sigma^2 is, so that taps of equal values keep their weight
        auto coeff = [](float sigma) {
            const float v = 1.4426950408889634f / (sigma * sigma);
            return 1.0f / (sigma * sigma) <= FLT_MAX ? fminf(v, FLT_MAX) : v;
        };
        const AtrousArgs a = {src, normal, albedo, (int)w, (int)h, step, coeff(scl), coeff(sn), coeff(sa)};
        // groups of rows that are `step` apart, in every residue class
        auto groups = [&](uint32_t rows) { return step * ((h + rows * step - 1) / (rows * step)); };
        auto tiles = [&](auto *kernel, uint32_t tw) {
            kernel<<<dim3((w + tw - 1) / tw, groups(kRows * kTileGroups)), dim3(tw, kTileGroups), tile_bytes(step), s>>>(a, dst);
        };
        if (step <= kTileStep) tile_width(step) == 64 ? tiles(k_atrous_tile<64>, 64) : tiles(k_atrous_tile<128>, 128);
        else
            k_atrous<<<dim3((w + 63) / 64, (groups(kRows) + 3) / 4), dim3(64, 4), 0, s>>>(a, dst);
        src = dst;
    }
    return hipGetLastError();
}

}  // namespace crt
