// scene_hash.hip -- the checkpoint's scene hash (FNV-1a, 64 bits) of device arrays (gfx950).
//
// h = (h ^ byte) * p for every byte is one chain of 64-bit multiplications: 1.1 ns a byte on a
// host core, 15 of the 25 ms in which a 400,000-triangle model was loaded.  The chain splits because the XOR
// touches the low byte only: with l = h mod 256, h ^ b = h + ((l ^ b) - l), so
//   * the low bytes form a chain of their own, l' = ((l ^ b) * 0xB3) mod 256, a map of 256 states
//     per chunk of the data that composes with its neighbours';
//   * given the low byte l at its start, a chunk of L bytes takes any h with that low byte to
//     h p^L + (f - l p^L), f being the chunk's own chain started from l.
// So: the state maps of all chunks (a wave per chunk, four states a lane), their composition
// (the start state of every chunk), the chunks' own chains (a lane per chunk), and the sum of
// their contributions.  Same value as the byte by byte chain, beside the BVH build on the second stream.
#include "crt_internal.h"

namespace crt {

namespace {

constexpr uint64_t kPrime = 1099511628211ull;   // 2^40 + 0x1B3
constexpr uint32_t kChunkBytes = 1024, kChunkWords = kChunkBytes / 4;
constexpr uint32_t kSpan = 128;                 // chunks composed by one block
constexpr uint32_t kPieceChunks = 65536;        // chunks per round (64 MB of data)

__host__ __device__ constexpr uint64_t prime_pow(uint32_t n)
{
    uint64_t r = 1, b = kPrime;
    for (; n; n >>= 1, b *= b)
        if (n & 1u) r *= b;
    return r;
}

// map[chunk][state] = low byte after the chunk's bytes, started from each state.  A lane holds
// states 4 lane .. 4 lane + 3 in the halves of two registers; 0xB3 times a byte fits in 16 bits.
__global__ __launch_bounds__(256) void k_fnv_maps(const uint32_t *__restrict__ words, uint32_t nwords, uint32_t *map)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t chunk = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
    const uint32_t w0 = chunk * kChunkWords;
    if (w0 >= nwords) return;
    const uint32_t w1 = min(w0 + kChunkWords, nwords);
    uint32_t e = (4u * lane) | (4u * lane + 2u) << 16, o = (4u * lane + 1u) | (4u * lane + 3u) << 16;
    for (uint32_t w = w0; w < w1; ++w) {
        const uint32_t v = words[w];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t b = (v >> (8 * k)) & 0xFFu, bb = b | b << 16;
            e = __umul24(e ^ bb, 0xB3u) & 0x00FF00FFu;
            o = __umul24(o ^ bb, 0xB3u) & 0x00FF00FFu;
        }
    }
    map[(size_t)chunk * 64u + lane] = e | o << 8;
}

// The composed map of the block's kSpan chunks; thread = start state.
__global__ __launch_bounds__(256) void k_fnv_compose(const uint32_t *__restrict__ map, uint32_t nchunks, uint8_t *super)
{
    __shared__ uint32_t m[kSpan * 64];
    const uint32_t c0 = blockIdx.x * kSpan, n = min(kSpan, nchunks - c0);
    for (uint32_t i = threadIdx.x; i < n * 64u; i += 256) m[i] = map[(size_t)c0 * 64u + i];
    __syncthreads();
    const uint8_t *bytes = reinterpret_cast<const uint8_t *>(m);
    uint32_t s = threadIdx.x;
    for (uint32_t c = 0; c < n; ++c) s = bytes[c * 256u + s];
    super[blockIdx.x * 256u + threadIdx.x] = (uint8_t)s;
}

// The low byte at the start of every span: one chain over the spans, kSpan maps in LDS at a time.
__global__ __launch_bounds__(256) void k_fnv_span_starts(const uint8_t *__restrict__ super, uint32_t nspans,
                                                         const uint64_t *h, uint8_t *start)
{
    __shared__ uint32_t m[kSpan * 64];
    uint32_t s = (uint32_t)(*h & 0xFFu);
    for (uint32_t p0 = 0; p0 < nspans; p0 += kSpan) {
        const uint32_t n = min(kSpan, nspans - p0);
        for (uint32_t i = threadIdx.x; i < n * 64u; i += 256)
            m[i] = reinterpret_cast<const uint32_t *>(super)[(size_t)p0 * 64u + i];
        __syncthreads();
        if (threadIdx.x == 0)
            for (uint32_t c = 0; c < n; ++c) {
                start[p0 + c] = (uint8_t)s;
                s = reinterpret_cast<const uint8_t *>(m)[c * 256u + s];
            }
        __syncthreads();
    }
}

// term[c] = f - l p^L of every chunk: the low bytes at the span's chunks first, then a chunk's
// own chain per thread.
__global__ __launch_bounds__(kSpan) void k_fnv_terms(const uint32_t *__restrict__ words, uint32_t nwords,
                                                     const uint32_t *__restrict__ map, uint32_t nchunks,
                                                     const uint8_t *__restrict__ span_start, uint64_t *term)
{
    __shared__ uint32_t m[kSpan * 64];
    __shared__ uint8_t  st[kSpan];
    const uint32_t c0 = blockIdx.x * kSpan, n = min(kSpan, nchunks - c0);
    for (uint32_t i = threadIdx.x; i < n * 64u; i += kSpan) m[i] = map[(size_t)c0 * 64u + i];
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = span_start[blockIdx.x];
        for (uint32_t c = 0; c < n; ++c) {
            st[c] = (uint8_t)s;
            s = reinterpret_cast<const uint8_t *>(m)[c * 256u + s];
        }
    }
    __syncthreads();
    if (threadIdx.x >= n) return;
    const uint32_t c = c0 + threadIdx.x, w0 = c * kChunkWords, w1 = min(w0 + kChunkWords, nwords);
    const uint64_t l = st[threadIdx.x];
    uint64_t f = l;
    for (uint32_t w = w0; w < w1; ++w) {
        const uint32_t v = words[w];
#pragma unroll
        for (int k = 0; k < 4; ++k) f = (f ^ ((v >> (8 * k)) & 0xFFu)) * kPrime;
    }
    term[c] = f - l * (w1 - w0 == kChunkWords ? prime_pow(kChunkBytes) : prime_pow(4u * (w1 - w0)));
}

// h = h p^bytes + the terms, each times p^(bytes after its chunk): a Horner chain per thread
// over neighbouring chunks, then one over the threads; the last chunk may be shorter.
__global__ __launch_bounds__(256) void k_fnv_fold(const uint64_t *__restrict__ term, uint32_t nwords, uint32_t nchunks,
                                                  uint64_t *h)
{
    __shared__ uint64_t sum[256], mul[256];
    constexpr uint64_t  kP = prime_pow(kChunkBytes);
    const uint32_t full = nwords / kChunkWords, per = (full + 255u) / 256u;   // whole chunks
    const uint32_t c0 = min(threadIdx.x * per, full), c1 = min(c0 + per, full);
    uint64_t s = 0, q = 1;
    for (uint32_t c = c0; c < c1; ++c) {
        s = s * kP + term[c];
        q *= kP;
    }
    sum[threadIdx.x] = s;
    mul[threadIdx.x] = q;
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint64_t r = *h;
    for (int i = 0; i < 256; ++i) r = r * mul[i] + sum[i];
    if (full < nchunks) r = r * prime_pow(4u * (nwords - full * kChunkWords)) + term[full];
    *h = r;
}

__global__ void k_hash_set(uint64_t *h, uint64_t v) { *h = v; }

}  // namespace

// whole spans for the chunks of a round over at most max_words
static uint32_t round_chunks(size_t max_words)
{
    const size_t c = std::min<size_t>((max_words + kChunkWords - 1) / kChunkWords, kPieceChunks);
    return (uint32_t)((c + kSpan - 1) / kSpan * kSpan);
}

size_t hash_scratch_bytes(size_t max_words)
{
    const size_t chunks = round_chunks(max_words), spans = chunks / kSpan;
    return chunks * (8 + 256) + spans * (256 + 1);
}

hipError_t launch_hash_init(uint64_t *h, hipStream_t s)
{
    k_hash_set<<<1, 1, 0, s>>>(h, 1469598103934665603ull);
    return hipGetLastError();
}

hipError_t launch_hash(const void *words, size_t nwords, uint64_t *h, void *scratch, hipStream_t s)
{
    const uint32_t chunks = round_chunks(nwords);
    uint64_t *term  = static_cast<uint64_t *>(scratch);
    uint32_t *map   = reinterpret_cast<uint32_t *>(term + chunks);
    uint8_t  *super = reinterpret_cast<uint8_t *>(map + (size_t)chunks * 64);
    uint8_t  *start = super + (size_t)(chunks / kSpan) * 256;
    constexpr size_t piece = (size_t)kPieceChunks * kChunkWords;
    for (size_t w0 = 0; w0 < nwords; w0 += piece) {
        const uint32_t *p = static_cast<const uint32_t *>(words) + w0;
        const uint32_t  n = (uint32_t)std::min(piece, nwords - w0), nc = (n + kChunkWords - 1) / kChunkWords,
                        spans = (nc + kSpan - 1) / kSpan;
        k_fnv_maps<<<(nc + 3) / 4, 256, 0, s>>>(p, n, map);
        k_fnv_compose<<<spans, 256, 0, s>>>(map, nc, super);
        k_fnv_span_starts<<<1, 256, 0, s>>>(super, spans, h, start);
        k_fnv_terms<<<spans, kSpan, 0, s>>>(p, n, map, nc, start, term);
        k_fnv_fold<<<1, 256, 0, s>>>(term, n, nc, h);
    }
    return hipGetLastError();
}

}  // namespace crt
