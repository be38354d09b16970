// material.h -- texture and material colour lookups of a scene on the device.
#pragma once
#include <hip/hip_runtime.h>
#include "crt_internal.h"

namespace crt {

// image.h:104-109: nearest texel, static_cast<uint64_t>(u * width) % width.  The cast of a
// negative product is undefined in C++; this follows what x86-64 code without AVX-512 does
// (the signed truncation reinterpreted as uint64), so u * width in (-1, 0] maps to column 0
// and -1.5 to (2^64 - 1) % width.  For power-of-two sizes that is the positive modulo.
__device__ __forceinline__ uint64_t texel_index(float u, uint32_t size)
{
    return (uint64_t)(int64_t)(u * (float)size) % (uint64_t)size;
}

__device__ __forceinline__ float4 tex_uv(const SceneDev &sc, int32_t t, float u, float v)
{
    const TextureDev td = sc.texs[t];
    const uint64_t   x = texel_index(u, td.w), y = texel_index(v, td.h);
    return sc.texels[td.offset + x + y * (uint64_t)td.w];
}

__device__ __forceinline__ float4 mat_colour(const SceneDev &sc, const MaterialDev &m, float u, float v)
{
    if (m.tex >= 0 && (uint32_t)m.tex < sc.ntex) return tex_uv(sc, m.tex, u, v);
    return make_float4(m.colour[0], m.colour[1], m.colour[2], m.colour[3]);
}

}  // namespace crt
