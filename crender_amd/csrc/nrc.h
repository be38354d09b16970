// nrc.h -- layout constants and launchers of the neural radiance cache (nrc.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace crt {

constexpr int   kNrcQuery  = 13;   // p[3] (scene-normalised), d[3], n[3], albedo[3], roughness
constexpr int   kNrcIn     = 96;   // encoded features (82 used + constant 1 + padding)
constexpr int   kNrcHid    = 64;
constexpr int   kNrcOut    = 32;   // outputs 0..2 = RGB
constexpr int   kNrcLayers = 6;    // 96->64, 4 x 64->64, 64->32
constexpr int   kNrcParams = kNrcIn * kNrcHid + 4 * kNrcHid * kNrcHid + kNrcHid * kNrcOut;   // 24576
constexpr uint32_t kNrcMaxParts = 256;   // gradient partials (training blocks) per step: one per CU
constexpr float kNrcEpsRel = 0.01f;

__host__ __device__ constexpr int nrc_w_off(int l)
{
    return l == 0 ? 0 : kNrcIn * kNrcHid + (l - 1) * kNrcHid * kNrcHid;
}

// Gradient partial rows and loss partials written by nrc_launch_train for n samples: one per
// block, which owns every kNrcMaxParts-th tile of 64 samples.
__host__ __device__ constexpr uint32_t nrc_partial_rows(uint32_t n)
{
    return (n + 63u) / 64u < kNrcMaxParts ? (n + 63u) / 64u : kNrcMaxParts;
}

// WF, WB: bf16 weights as the forward and backward products read them, kNrcParams elements
// each, written by nrc_launch_adam (update 0: from the parameters as they are).
hipError_t nrc_launch_infer(const float *q, float *out, uint32_t n, const __bf16 *WF, hipStream_t s);
hipError_t nrc_launch_train(const float *q, const float *target, uint32_t n, const __bf16 *WF, const __bf16 *WB,
                            float *partial, float *partial_loss, hipStream_t s);
hipError_t nrc_launch_adam(const float *partial, uint32_t nrows, float *params, float *m, float *v, __bf16 *WF,
                           __bf16 *WB, float lr, float b1, float b2, float eps, uint64_t step, int update,
                           hipStream_t s);
// out: kNrcParams gradient values, then the loss
hipError_t nrc_launch_sum_partials(const float *partial, const float *partial_loss, uint32_t nrows, float *out,
                                   hipStream_t s);

}  // namespace crt
