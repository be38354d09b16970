// traverse.hip -- wide-BVH ray traversal for the crt path tracer (gfx950).
//
// Replaces rtcIntersect1 (CRender src/objects/model.cpp:27): closest hit in (tnear, tfar]
// with equal t resolved to the smaller primID; plus an any-hit variant for shadow rays.
//
// Execution model (wave64):
//   * persistent grid: a fixed number of 256-thread blocks per CU; every wave loops
//     fetching rays until the queue is drained, so the launch shape never depends on the
//     ray count (which lives in device memory and is produced by the previous kernel).
//   * XCD-aware fetch: the ray range is cut into 8 contiguous slices, one per XCD
//     (blocks are dispatched round-robin over XCDs), so neighbouring rays share an L2;
//     an XCD that drains its slice takes from the others.  A wave owns 64 rays from the
//     start and takes further ones in chunks (RaySupply).
//   * refill: when 16 or more lanes of a wave are idle, they take rays of the wave's chunk
//     by ballot rank.
//   * per-lane short stack in LDS (entry-major (ref, distance) pairs; 8, 16 or 32 entries, growing
//     downwards), spilled a full stack at a time to a per-lane global region when full.  Entries carry
//     the child's entry distance so popped nodes beyond the current hit are skipped.
//   * children are ordered by entry distance with a sorting network; the nearest is
//     visited next and the others are written behind it, nearest on top.
//   * leaf parking: a lane that reaches a leaf keeps it aside (up to two) and continues
//     down the tree until most lanes of the wave hold their leaves (fewer than 16 can still
//     park one), so the triangle phase runs with more lanes busy (Aila and Laine 2009,
//     "speculative traversal").
#include <hip/hip_runtime.h>
#include "crt_internal.h"
#include "material.h"

namespace crt {

namespace {

constexpr float kInf = __builtin_huge_valf();
constexpr uint32_t kEmpty = kInvalidRef;
constexpr uint32_t kMissKey = 0x7FE00000u;   // behind every distance
// The defaults of the three thresholds, at 1080p: soup of 1M triangles 8 passes / 20 passes, terrain
// of 1M triangles 8 passes, ms; 9.40 / 22.13 / 9.92 with all of them.
// Idle lanes that trigger a refill: 8 -> 9.34 / 22.08 / 9.89, 24 -> 9.37 / 22.40 / 9.91, 32 -> 9.68 /
// 22.68 / 9.89.
constexpr uint32_t kRefillIdle = 16;
// A wave leaves the inner-node phase for its parked leaves once fewer lanes than this can still
// park one: 4 -> 9.79 / 23.12 / 9.97, 8 -> 9.49 / 22.42 / 9.88, 32 -> 9.64 / 22.71 / 10.25.
constexpr uint32_t kParkMin    = 16;
// After so many leaf-loop rounds, once every parked leaf is tested, a wave resumes the inner-node
// phase (lanes still at a leaf park it there) instead of following chains of popped leaves with
// few lanes busy: 1 -> 9.71 / 22.90 / 10.26, 2 -> 9.65 / 22.74 / 10.13, 4 -> 9.51 / 22.39 / 10.00,
// unlimited 9.66 / 22.73 / 10.09.
constexpr uint32_t kLeafRounds = 3;
constexpr uint32_t kInstExit   = 0xFFFFFFFEu;   // stack marker: leave the current instance
// Ize, "Robust BVH Ray Traversal" (JCGT 2013): scaling the far slab distance by
// 1 + 2*gamma(3) keeps FP32 box tests conservative.
constexpr float kFarScale = 1.0000003576278687f;
// 4-wide nodes: entry distances are compared with a hit's, when a child is tested and when it
// is popped, this much nearer than they are.  The hit distance of a triangle in a box face rounds
// apart from the face's, the more so the flatter the ray: of 18.6M random hits of triangles in an
// axis-aligned plane, 28 % lie before their own box, 0.03 % by more than 2^-20 of the distance, 20
// by more than 2^-12.  A coincident or coplanar triangle in another leaf would be lost.  (8-wide
// boxes are rounded outwards to their grid and by the bound in NodeOps<8>.)
constexpr float kNearScale = 1.0f - 1.0f / 4096.0f;

struct RayState {
    f3     o, d, inv;
    float  tn, tmax;
    wt_ray wt;
    uint32_t best_tri, best_prim;
    float  bu, bv;
};

// Child of a node to be sorted: entry distance bits above, ref below, read as one FP64 number.
// Distances are non-negative floats and kMissKey is below the bits of an FP64 infinity, so the
// order of the numbers is that of the distances (of the refs among equal ones) and none is a NaN.
typedef double Child;

__device__ __forceinline__ Child make_child(uint32_t key, uint32_t ref)
{
    return __builtin_bit_cast(double, make_uint2(ref, key));
}
__device__ __forceinline__ uint32_t child_key(Child c) { return __builtin_bit_cast(uint2, c).y; }
__device__ __forceinline__ uint32_t child_ref(Child c) { return __builtin_bit_cast(uint2, c).x; }

// compare-exchange: FP64 min and max move all 64 bits of the smaller and the larger one
// (FP64 denormals are kept, and a distance of 0 gives one) at FP32 rate on gfx950: 2
// instructions a comparator instead of a compare and four selects, 38 of the 95 for eight children.
// With the pair pushed as it is and rows a constant apart a node step takes about 230 VALU
// instructions instead of 300; the step is bound by these and by the latency of the node's
// load.  1080p, before -> after: soup 8 passes 11.0 -> 10.2 ms, terrain 8 passes 12.5 -> 10.5 ms,
// camera rays 694 -> 634 us.
__device__ __forceinline__ void cswap(Child &a, Child &b)
{
    Child lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

template <int W>
__device__ __forceinline__ void sort_children(Child (&c)[W])
{
#define CS(i, j) cswap(c[i], c[j])
    if constexpr (W == 4) {
        CS(0, 1); CS(2, 3);
        CS(0, 2); CS(1, 3);
        CS(1, 2);
    } else {
        // optimal 19-comparator network for 8 inputs
        CS(0, 2); CS(1, 3); CS(4, 6); CS(5, 7);
        CS(0, 4); CS(1, 5); CS(2, 6); CS(3, 7);
        CS(0, 1); CS(2, 3); CS(4, 5); CS(6, 7);
        CS(2, 4); CS(3, 5);
        CS(1, 4); CS(3, 6);
        CS(1, 2); CS(3, 4); CS(5, 6);
    }
#undef CS
}

// key = entry distance (non-negative float bits, low 3 bits cleared) | child slot
__device__ __forceinline__ uint32_t make_key(float t, int j)
{
    return (__float_as_uint(t) & ~7u) | (uint32_t)j;
}

// Finite reciprocal: a zero direction component gives +-1e30 instead of inf, so an
// axis-parallel ray whose origin lies on a slab plane yields [0, big] rather than the
// NaN of 0 * inf, and the box test stays conservative.
__device__ __forceinline__ float safe_rcp(float d)
{
    return fabsf(d) < 1e-30f ? copysignf(1e30f, d) : 1.0f / d;
}

__device__ __forceinline__ bool slab(float lx, float hx, float ly, float hy, float lz, float hz, const RayState &r,
                                     float &tentry)
{
    float t0x = (lx - r.o.x) * r.inv.x, t1x = (hx - r.o.x) * r.inv.x;
    float t0y = (ly - r.o.y) * r.inv.y, t1y = (hy - r.o.y) * r.inv.y;
    float t0z = (lz - r.o.z) * r.inv.z, t1z = (hz - r.o.z) * r.inv.z;
    const float tnx = fminf(t0x, t1x), tfx = fmaxf(t0x, t1x);
    const float tny = fminf(t0y, t1y), tfy = fmaxf(t0y, t1y);
    const float tnz = fminf(t0z, t1z), tfz = fmaxf(t0z, t1z);
    const float tmin = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, fmaxf(r.tn, 0.0f)));
    const float tmax = fminf(fminf(tfx, tfy), tfz) * kFarScale;
    tentry = tmin * kNearScale;
    return tmin <= tmax && tentry <= r.tmax;
}

// Keeps a load where it is written (the compiler would sink one that only some lanes need below
// the branch, behind the tests, and wait for memory a second time).  The child refs of a node:
// soup 8 passes 10.2 -> 9.8 ms, terrain 10.5 -> 10.2 ms, camera rays 615 -> 596 us.
__device__ __forceinline__ void keep_load(uint4 &v)
{
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
}

template <int W>
struct NodeOps;

template <>
struct NodeOps<4> {
    static __device__ __forceinline__ int expand(const void *nodes, uint32_t idx, const RayState &r, Child (&c)[4])
    {
        const float4 *p = reinterpret_cast<const float4 *>(static_cast<const Node4 *>(nodes) + idx);
        const float4  lx = p[0], hx = p[1], ly = p[2], hy = p[3], lz = p[4], hz = p[5];
        const uint4   ch = reinterpret_cast<const uint4 *>(p)[6];
        const uint32_t nc = reinterpret_cast<const uint4 *>(p)[7].x;
        const uint32_t ref[4] = {ch.x, ch.y, ch.z, ch.w};
        const float LX[4] = {lx.x, lx.y, lx.z, lx.w}, HX[4] = {hx.x, hx.y, hx.z, hx.w};
        const float LY[4] = {ly.x, ly.y, ly.z, ly.w}, HY[4] = {hy.x, hy.y, hy.z, hy.w};
        const float LZ[4] = {lz.x, lz.y, lz.z, lz.w}, HZ[4] = {hz.x, hz.y, hz.z, hz.w};
        int nh = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float t;
            const bool h = (uint32_t)j < nc && slab(LX[j], HX[j], LY[j], HY[j], LZ[j], HZ[j], r, t);
            c[j] = make_child(h ? __float_as_uint(t) : kMissKey, ref[j]);
            nh += h ? 1 : 0;
        }
        return nh;
    }
};

template <>
struct NodeOps<8> {
    // Plane distances in FMA form: t = q * (2^e * inv) + (origin - o) * inv, one rounding per
    // plane instead of decoding the plane first.  The rounding of the per-node base and of
    // the FMA is bounded by delta = 2^-20 * (|base| + 255 |2^e inv|) per axis; subtracting
    // it from the base of the entry plane and adding it to the base of the exit plane keeps
    // every child interval a superset of the exact one, at no per-child cost.
    // The entry plane of an axis is the low one for a positive direction and the high one for
    // a negative direction, so the byte words are picked once per node (lo <= hi holds for
    // every child slot below the child count) and a child costs no min/max per axis.
    static __device__ __forceinline__ int expand(const void *nodes, uint32_t idx, const RayState &r, Child (&c)[8])
    {
        const uint4 *p  = reinterpret_cast<const uint4 *>(static_cast<const Node8Q *>(nodes) + idx);
        const uint4  h  = p[0];
        uint4        c0 = p[1], c1 = p[2];
        const uint4  qx = p[3], qy = p[4], qz = p[5];
        keep_load(c0);
        keep_load(c1);
        const uint32_t ref[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const float sx = __uint_as_float((h.w & 0xFFu) << 23) * r.inv.x;
        const float sy = __uint_as_float(((h.w >> 8) & 0xFFu) << 23) * r.inv.y;
        const float sz = __uint_as_float(((h.w >> 16) & 0xFFu) << 23) * r.inv.z;
        const float bx = (__uint_as_float(h.x) - r.o.x) * r.inv.x;
        const float by = (__uint_as_float(h.y) - r.o.y) * r.inv.y;
        const float bz = (__uint_as_float(h.z) - r.o.z) * r.inv.z;
        const float dx = 9.5367431640625e-07f * (fabsf(bx) + 255.0f * fabsf(sx));
        const float dy = 9.5367431640625e-07f * (fabsf(by) + 255.0f * fabsf(sy));
        const float dz = 9.5367431640625e-07f * (fabsf(bz) + 255.0f * fabsf(sz));
        const float bnx = bx - dx, bfx = bx + dx, bny = by - dy, bfy = by + dy, bnz = bz - dz, bfz = bz + dz;
        // words [0..1] hold the low bytes of children 0-3 / 4-7, words [2..3] the high bytes
        const bool px = r.inv.x >= 0.0f, py = r.inv.y >= 0.0f, pz = r.inv.z >= 0.0f;
        const uint32_t nx0 = px ? qx.x : qx.z, nx1 = px ? qx.y : qx.w, fx0 = px ? qx.z : qx.x, fx1 = px ? qx.w : qx.y;
        const uint32_t ny0 = py ? qy.x : qy.z, ny1 = py ? qy.y : qy.w, fy0 = py ? qy.z : qy.x, fy1 = py ? qy.w : qy.y;
        const uint32_t nz0 = pz ? qz.x : qz.z, nz1 = pz ? qz.y : qz.w, fz0 = pz ? qz.z : qz.x, fz1 = pz ? qz.w : qz.y;
        const float tn0 = fmaxf(r.tn, 0.0f);
        const uint32_t nc = h.w >> 24;
        int nh = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int sh = 8 * (j & 3);
            const float tnx = fmaf((float)(((j < 4 ? nx0 : nx1) >> sh) & 0xFFu), sx, bnx);
            const float tfx = fmaf((float)(((j < 4 ? fx0 : fx1) >> sh) & 0xFFu), sx, bfx);
            const float tny = fmaf((float)(((j < 4 ? ny0 : ny1) >> sh) & 0xFFu), sy, bny);
            const float tfy = fmaf((float)(((j < 4 ? fy0 : fy1) >> sh) & 0xFFu), sy, bfy);
            const float tnz = fmaf((float)(((j < 4 ? nz0 : nz1) >> sh) & 0xFFu), sz, bnz);
            const float tfz = fmaf((float)(((j < 4 ? fz0 : fz1) >> sh) & 0xFFu), sz, bfz);
            const float tmin = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tn0));
            const float tmax = fminf(fminf(tfx, tfy), fminf(tfz, r.tmax));
            const bool hit = (uint32_t)j < nc && tmin <= tmax;
            c[j] = make_child(hit ? __float_as_uint(tmin) : kMissKey, ref[j]);
            nh += hit ? 1 : 0;
        }
        return nh;
    }
};

template <uint32_t S>
struct Stack {
    uint2    *s;        // this lane's column of the LDS stack, [S][kTraceBlock] of (ref, entry distance
                        // bits), filled from row S - 1 downwards
    uint4    *g;        // this lane's global spill: `depth` (ref, distance) entries, contiguous, so
                        // that a spill of S entries writes S * 8 bytes of whole lines (uint4 = 2 entries)
    uint32_t  top, gsp, depth;   // row of the top entry (S: none in LDS), entries spilled

    uint32_t *err;

    __device__ __forceinline__ void clear()
    {
        top = S;
        gsp = 0;
    }
    __device__ __forceinline__ void push(uint2 e)
    {
        if (top == 0) {
            if (gsp + S > depth) {
                // cannot happen for trees admitted at commit; never write out of bounds
                *err = 1u;
                return;
            }
            for (uint32_t k = 0; k < S; k += 2) {
                const uint2 a = s[k * kTraceBlock], b = s[(k + 1) * kTraceBlock];
                g[(gsp + k) / 2] = make_uint4(a.x, a.y, b.x, b.y);
            }
            gsp += S;
            top = S;
        }
        --top;
        s[top * kTraceBlock] = e;
    }
    // Writes c[K .. W - 1] to the rows from p on, up to the last hit: rows a constant apart, one
    // compare per child, and no further ones once no lane has any left.
    template <int W, int K>
    static __device__ __forceinline__ void store_children(uint2 *p, const Child (&c)[W], int nh)
    {
        if constexpr (K < W) {
            if (K < nh) {
                p[(K - 1) * kTraceBlock] = __builtin_bit_cast(uint2, c[K]);
                store_children<W, K + 1>(p, c, nh);
            }
        }
    }
    // Pushes the hit children of a node, sorted ascending with the nh - 1 hits behind the nearest
    // in slots 1..nh-1, so that slot 1 ends on top.
    template <int W>
    __device__ __forceinline__ void push_children(const Child (&c)[W], int nh)
    {
        const uint32_t m = (uint32_t)nh - 1u;
        if (m <= top) {
            top -= m;
            store_children<W, 1>(s + top * kTraceBlock, c, nh);
        } else {
#pragma unroll
            for (int k = W - 1; k >= 1; --k) {
                if (k < nh) push(__builtin_bit_cast(uint2, c[k]));
            }
        }
    }
    // pops the next entry closer than tmax; kEmpty when the stack is exhausted
    __device__ __forceinline__ uint32_t pop(float tmax)
    {
        for (;;) {
            if (top == S) {
                if (gsp == 0) return kEmpty;
                gsp -= S;
                for (uint32_t k = 0; k < S; k += 2) {
                    const uint4 v = g[(gsp + k) / 2];
                    s[k * kTraceBlock]       = make_uint2(v.x, v.y);
                    s[(k + 1) * kTraceBlock] = make_uint2(v.z, v.w);
                }
                top = 0;
            }
            const uint2 v = s[top * kTraceBlock];
            ++top;
            if (__uint_as_float(v.y) <= tmax) return v.x;
        }
    }
};

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// kMulti: rays of many scenes in one launch (batched rendering); each lane takes its
// ray's scene (nodes, triangles, root) when it fetches the ray.
// kInst: two-level scene.  A leaf of the instance BVH (level 0) names instances; entering
// one transforms the lane's ray into the instance's object space (direction renormalised,
// distances scaled by |inv * d|, model.cpp:107-113) and pushes kInstExit, whose pop
// restores the world ray; closest-hit distances are compared in world units.
// The 8-entry stack variant is also the high-occupancy one: its 16 KB of LDS per block
// leaves room for 8 waves per SIMD, so the register budget is capped to match (64 VGPRs).
// kStats: the instrumented variant; counts each lane's inner-node tests, leaf visits and
// triangle tests, each wave's iterations of the node and leaf loops, and the lanes idle in
// node-loop iterations by cause (no ray, ray finished but for parked leaves, waiting at a
// leaf with both parking slots full), and adds them to q.tstats when the wave leaves.
// The launch's epilogue (TraceQueue::done): every block that took part reports when its
// waves are done with the work counters; the last one clears the next bounce's counters.  No
// fence is needed: every work-counter atomic returned (its value was used) before the block's
// barrier, the last block reads nothing other blocks wrote, and the end of the kernel
// publishes its stores to the next launch.  (A device-scope fence here would write back and
// invalidate the XCD's L2 under the blocks still traversing.)
__device__ __forceinline__ void trace_clear(const TraceQueue &q, uint32_t n)
{
    for (uint32_t x = 0; x < kXcds; ++x) q.counters[x * kCntLine] = 0u;
    if (q.clear0) *q.clear0 = 0u;
    if (q.clear1) *q.clear1 = 0u;
    if (q.stat) atomicAdd(q.stat, (unsigned long long)n);
    *q.done = 0u;
}

__device__ __forceinline__ void trace_epilogue(const TraceQueue &q, uint32_t n, uint32_t nblocks)
{
    if (!q.done) return;
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (atomicAdd(q.done, 1u) != nblocks - 1u) return;
    trace_clear(q, n);
}

// How a launch's rays reach its waves.  The queue is cut into kXcds contiguous slices, one per
// XCD; a slice's first kStatic rays per wave belong to that slice's waves by position, so a
// launch that has no more rays than that needs no atomic at all, and blocks without rays leave
// at once.  The rest of a slice is handed out in chunks by the slice's counter; a wave keeps
// its chunk and refills its lanes from it.  Chunks shrink as the slice drains (a quarter of an
// even share of what is left, within [kChunkMin, kChunkMax]), so that the waves end together.
// Why: an atomic on one cache line from the whole chip takes about 18 ns (55 million a second),
// and with one atomic per refill on eight counters in one line that rate, not the traversal,
// set a launch's time: 298 us for 96 rays (2048 waves each draining eight slices) and 0.5 ms
// per million rays.  A drained wave reads all the counters with one load per lane instead of
// trying the slices one by one.
constexpr uint32_t kStatic   = 64;
constexpr uint32_t kChunkMin = 32;
constexpr uint32_t kChunkMax = 256;

struct RaySupply {
    uint32_t n, slice, nw;      // rays, rays per slice, waves per slice
    uint32_t pbeg, pend;        // the wave's own rays
    uint32_t x, chunk, tried;   // slice drawn from, next chunk size, slices found empty
    bool     dynamic;           // some slice has rays beyond the static ones

    __device__ __forceinline__ uint32_t slice_beg(uint32_t k) const { return min(k * slice, n); }
    __device__ __forceinline__ uint32_t slice_len(uint32_t k) const { return min(slice, n - slice_beg(k)); }
    __device__ __forceinline__ uint32_t dyn_len(uint32_t k) const
    {
        const uint32_t len = slice_len(k), st = nw * kStatic;
        return len > st ? len - st : 0u;
    }
    __device__ __forceinline__ uint32_t guided(uint32_t left) const
    {
        return min(max(left / (4u * nw), kChunkMin), kChunkMax);
    }
    // wave: index of the wave among its slice's waves
    __device__ __forceinline__ void init(uint32_t count, uint32_t xcd, uint32_t wave, uint32_t waves)
    {
        n       = count;
        nw      = waves;
        slice   = (n + kXcds - 1u) / kXcds;
        dynamic = slice > nw * kStatic;
        x       = xcd;
        tried   = 0u;
        const uint32_t len = slice_len(x), b = min(wave * kStatic, len);
        pbeg  = slice_beg(x) + b;
        pend  = pbeg + min(kStatic, len - b);
        chunk = guided(dyn_len(x));
    }
    // Blocks that have rays: all of them when some are handed out dynamically.
    __device__ __forceinline__ uint32_t active_blocks(uint32_t nblocks, uint32_t block_waves) const
    {
        if (dynamic) return nblocks;
        uint32_t a = 0;
        for (uint32_t k = 0; k < kXcds; ++k) {
            const uint32_t per = block_waves * kStatic;
            a += (slice_len(k) + per - 1u) / per;
        }
        return a;
    }
    // Takes the wave's next chunk; false when no slice has rays left.  All lanes call it.
    // Ends after at most kXcds failed takes: a slice found empty is not tried again.
    __device__ __forceinline__ bool take(uint32_t *counters, uint32_t lane)
    {
        if (!dynamic) return false;
        for (;;) {
            if (!(tried >> x & 1u)) {
                const uint32_t len = dyn_len(x);
                uint32_t b = len;
                if (len) {
                    if (lane == 0) b = atomicAdd(counters + x * kCntLine, chunk);
                    b = __builtin_amdgcn_readfirstlane(b);
                }
                if (b < len) {
                    const uint32_t base = slice_beg(x) + nw * kStatic;
                    const uint32_t e    = min(b + chunk, len);
                    pbeg  = base + b;
                    pend  = base + e;
                    chunk = guided(len - e);
                    return true;
                }
                tried |= 1u << x;
            }
            bool some = false;
            if (lane < kXcds && !(tried >> lane & 1u)) {
                const uint32_t v = __hip_atomic_load(counters + lane * kCntLine, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
                some = v < dyn_len(lane);
            }
            const uint32_t m = (uint32_t)__ballot(some) & ((1u << kXcds) - 1u);
            if (m == 0u) return false;
            // the next slice after x, so that the helpers spread over the slices left
            const uint32_t hi = m & ~((2u << x) - 1u);
            x     = __builtin_ctz(hi ? hi : m);
            chunk = kChunkMin;
        }
    }
};

// ---- few rays ---------------------------------------------------------------------------
// Eight lanes per ray: lane j of a group tests child j of the group's node, so a node costs
// one box test per lane instead of eight, its children are ranked by seven comparisons instead of
// a 19-step network, and up to eight culled stack entries or leaf triangles go in one step.
// A launch too small to fill the chip is bound by the chain of its longest ray, which this
// makes about half as long; a full chip does more with a ray per lane (TraceQueue::group_rays).
// The tests are those of the other mode, so are the hits.
constexpr uint32_t kGroup     = 8;
constexpr uint32_t kGroupRays = kTraceBlock / kGroup;   // rays of a block at a time

// Value of lane (l ^ m) of the lane's group of eight, m = 1 .. 7: DPP quad permutations, and
// the mirror of the half row (lane ^ 7) for the other quad.
template <int m>
__device__ __forceinline__ uint32_t group_xor(uint32_t v)
{
    constexpr int x    = m < 4 ? m : 7 - m;
    constexpr int quad = (0 ^ x) | (1 ^ x) << 2 | (2 ^ x) << 4 | (3 ^ x) << 6;   // quad_perm of lane ^ x
    if constexpr (m >= 4) v = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xF, 0xF, false);
    if constexpr (x > 0) v = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, quad, 0xF, 0xF, false);
    return v;
}

// The group's eight bits of a ballot.
__device__ __forceinline__ uint32_t group_ballot(bool b, uint32_t lane)
{
    return (uint32_t)(__ballot(b) >> (lane & ~(kGroup - 1u))) & 0xFFu;
}

// Between stack accesses of different lanes of a group.  One wave's LDS accesses stay in order, so it
// costs no instruction; it keeps the compiler from moving them across each other.
__device__ __forceinline__ void group_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); }

// Keeps the lane's or its partner's candidate: the nearer hit, at equal distance the smaller
// primID.
template <int m>
__device__ __forceinline__ void group_nearest(float &t, uint32_t &prim, uint32_t &who)
{
    const float    ot = __uint_as_float(group_xor<m>(__float_as_uint(t)));
    const uint32_t op = group_xor<m>(prim), ow = group_xor<m>(who);
    if (ot < t || (ot == t && op < prim)) {
        t    = ot;
        prim = op;
        who  = ow;
    }
}

// Writes the result of ray rid (one lane per ray calls it).
template <bool kAny>
__device__ __forceinline__ void store_ray(const TraceQueue &q, uint8_t *occ, uint32_t rid, const RayState &r)
{
    const bool h = r.best_tri != kInvalidRef;
    if (!kAny) {
        q.hits.t[rid]   = h ? r.tmax : kInf;
        q.hits.tri[rid] = r.best_tri;
        if (q.hits.u) q.hits.u[rid] = r.bu;
        if (q.hits.v) q.hits.v[rid] = r.bv;
    } else if (!q.res_rad) {
        occ[rid] = h ? 1 : 0;
    } else if (!h) {
        const uint32_t p = q.res_path[rid];
        const float4   c = q.res_contrib[rid];
        float4         v = q.res_rad[p];
        v.x += c.x;
        v.y += c.y;
        v.z += c.z;
        q.res_rad[p] = v;
    }
}

// Loads ray rid; false: it is degenerate and hits nothing (ntri: triangles of its scene).
__device__ __forceinline__ bool load_ray(const TraceQueue &q, uint32_t rid, uint32_t ntri, RayState &r)
{
    r.o = mk3(q.rays.ox[rid], q.rays.oy[rid], q.rays.oz[rid]);
    r.d = mk3(q.rays.dx[rid], q.rays.dy[rid], q.rays.dz[rid]);
    if (q.unit_dir && (r.d.x != 0.0f || r.d.y != 0.0f || r.d.z != 0.0f)) r.d = normalize(r.d);
    r.tn   = q.rays.tn ? q.rays.tn[rid] : kRayNear;
    r.tmax = q.rays.tf ? q.rays.tf[rid] : kInf;
    r.inv  = mk3(safe_rcp(r.d.x), safe_rcp(r.d.y), safe_rcp(r.d.z));
    r.wt   = wt_setup(r.d);
    r.best_tri = r.best_prim = kInvalidRef;
    r.bu = r.bv = 0.0f;
    return ntri > 0 && r.tn <= r.tmax && r.tmax == r.tmax && r.tn == r.tn &&
           (r.d.x != 0.0f || r.d.y != 0.0f || r.d.z != 0.0f);
}

// Shadow rays of scenes with transparent texels (renderer.cpp:330-345): a ray that stops on one
// (colour.w == 0) goes on from the hit + 0.1 * direction, up to kAlphaSteps traces, and adds its
// contribution if it escapes.  The lane restarts the ray itself, in the same launch: with a
// launch per step, its material test, compaction and counters as kernels of their own and the host
// reading the count between the steps, 640x360 with cut-outs took 950 us where it now takes 511.
constexpr uint32_t kAlphaSteps = 64;

// True if ray rid, stopped at r's hit, passes; o2 = where it goes on.
template <bool kMulti>
__device__ __forceinline__ bool alpha_passes(const SceneDev &sc_one, const TraceQueue &q, uint32_t rid,
                                             const RayState &r, f3 &o2)
{
#pragma clang fp contract(off)
    const SceneDev &sc = kMulti ? q.jobs[q.path_job[q.ray_path[rid]]].sc : sc_one;
    float u = 0.0f, v = 0.0f;
    if (sc.uv) {
        const float2 w0 = sc.uv[3 * (size_t)r.best_prim + 0], w1 = sc.uv[3 * (size_t)r.best_prim + 1],
                     w2 = sc.uv[3 * (size_t)r.best_prim + 2];
        const float b0 = 1.0f - r.bu - r.bv;
        u = b0 * w0.x + r.bu * w1.x + r.bv * w2.x;
        v = b0 * w0.y + r.bu * w1.y + r.bv * w2.y;
    }
    o2 = r.o + r.d * r.tmax + mk3(q.rays.dx[rid], q.rays.dy[rid], q.rays.dz[rid]) * 0.1f;
    return mat_colour(sc, sc.mats[sc.mat_idx[r.best_prim]], u, v).w == 0.0f;
}

// The launch's n rays with a group per ray; lds: `depth` entries for each of the block's groups.
template <bool kAny, bool kMulti>
__device__ __forceinline__ void trace_groups(const SceneDev &sc, const TraceQueue &q, uint8_t *occ, uint32_t n,
                                             uint2 *lds, uint32_t depth)
{
    const uint32_t lane = lane_id(), j = lane & (kGroup - 1u), slot = threadIdx.x / kGroup;
    uint2 *stack = lds + slot;
    for (uint32_t rid = blockIdx.x * kGroupRays + slot; rid < n; rid += gridDim.x * kGroupRays) {
        const void   *nodes = sc.nodes;
        const float4 *tris  = sc.tri;
        uint32_t root = sc.root, ntri = sc.ntri;
        if constexpr (kMulti) {
            const TraceScene ts = q.scenes[q.path_job[q.ray_path[rid]]];
            nodes = ts.nodes;
            tris  = ts.tri;
            root  = ts.root;
            ntri  = ts.ntri;
        }
        RayState r;
        uint32_t cur = load_ray(q, rid, ntri, r) ? root : kEmpty, sp = 0;
        while (cur != kEmpty) {
            if (ref_is_leaf(cur)) {
                const uint32_t first = leaf_first(cur), cnt = leaf_count(cur);
                for (uint32_t k0 = 0; k0 < cnt; k0 += kGroup) {   // leaves hold up to 16 triangles
                    float    t = kInf, u = 0.0f, v = 0.0f;
                    uint32_t prim = kInvalidRef, who = j;
                    bool     hit = false;
                    const size_t ti = (size_t)(first + k0 + j);
                    if (k0 + j < cnt) {
                        const float4 a = tris[3 * ti + 0], b = tris[3 * ti + 1], c = tris[3 * ti + 2];
                        hit = wt_test(r.wt, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), mk3(c.x, c.y, c.z), r.o, r.tn, r.tmax,
                                      t, u, v);
                        if (hit) prim = __float_as_uint(a.w);
                        else t = kInf;
                    }
                    if (group_ballot(hit, lane) == 0u) continue;
                    group_nearest<1>(t, prim, who);
                    group_nearest<2>(t, prim, who);
                    group_nearest<7>(t, prim, who);
                    if (t < r.tmax || prim < r.best_prim) {
                        const int src = (int)((lane & ~(kGroup - 1u)) | who);
                        r.tmax      = t;
                        r.best_prim = prim;
                        r.best_tri  = first + k0 + who;
                        r.bu        = __shfl(u, src);
                        r.bv        = __shfl(v, src);
                    }
                    if (kAny) break;
                }
                if (kAny && r.best_tri != kInvalidRef) break;
            } else {
                // child j of the node: NodeOps<8>::expand for one child
                const Node8Q  &nd = static_cast<const Node8Q *>(nodes)[cur];
                const uint4    h  = *reinterpret_cast<const uint4 *>(&nd);
                const uint32_t ref = nd.child[j];
                const uint32_t qlx = nd.qlox[j], qhx = nd.qhix[j], qly = nd.qloy[j], qhy = nd.qhiy[j], qlz = nd.qloz[j],
                               qhz = nd.qhiz[j];
                const float sx = __uint_as_float((h.w & 0xFFu) << 23) * r.inv.x;
                const float sy = __uint_as_float(((h.w >> 8) & 0xFFu) << 23) * r.inv.y;
                const float sz = __uint_as_float(((h.w >> 16) & 0xFFu) << 23) * r.inv.z;
                const float bx = (__uint_as_float(h.x) - r.o.x) * r.inv.x;
                const float by = (__uint_as_float(h.y) - r.o.y) * r.inv.y;
                const float bz = (__uint_as_float(h.z) - r.o.z) * r.inv.z;
                const float dx = 9.5367431640625e-07f * (fabsf(bx) + 255.0f * fabsf(sx));
                const float dy = 9.5367431640625e-07f * (fabsf(by) + 255.0f * fabsf(sy));
                const float dz = 9.5367431640625e-07f * (fabsf(bz) + 255.0f * fabsf(sz));
                const bool  px = r.inv.x >= 0.0f, py = r.inv.y >= 0.0f, pz = r.inv.z >= 0.0f;
                const float tnx = fmaf((float)(px ? qlx : qhx), sx, bx - dx), tfx = fmaf((float)(px ? qhx : qlx), sx, bx + dx);
                const float tny = fmaf((float)(py ? qly : qhy), sy, by - dy), tfy = fmaf((float)(py ? qhy : qly), sy, by + dy);
                const float tnz = fmaf((float)(pz ? qlz : qhz), sz, bz - dz), tfz = fmaf((float)(pz ? qhz : qlz), sz, bz + dz);
                const float tmin = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, fmaxf(r.tn, 0.0f)));
                const float tmax = fminf(fminf(tfx, tfy), fminf(tfz, r.tmax));
                const bool  hit  = j < h.w >> 24 && tmin <= tmax;
                const uint32_t key = hit ? make_key(tmin, (int)j) : kMissKey;
                const uint32_t nh = (uint32_t)__popc(group_ballot(hit, lane));
                if (nh > 0u) {
                    // hits nearer than this one; misses compare equal among themselves only
                    const uint32_t rank = (group_xor<1>(key) < key) + (group_xor<2>(key) < key) + (group_xor<3>(key) < key) +
                                          (group_xor<4>(key) < key) + (group_xor<5>(key) < key) + (group_xor<6>(key) < key) +
                                          (group_xor<7>(key) < key);
                    if (sp + nh - 1u > depth) {   // cannot happen for the scenes admitted; never write beyond
                        *q.error = 1u;
                        break;
                    }
                    group_fence();   // behind the loads that emptied these entries
                    if (hit && rank > 0u) stack[(sp + nh - 1u - rank) * kGroupRays] = make_uint2(ref, key & ~7u);
                    sp += nh - 1u;
                    const uint32_t near = __builtin_ctz(group_ballot(hit && rank == 0u, lane));
                    cur = __shfl(ref, (int)((lane & ~(kGroup - 1u)) | near));
                    continue;
                }
            }
            // next entry closer than the hit, eight entries at a time
            group_fence();   // behind the stores of the other lanes
            cur = kEmpty;
            while (sp > 0u) {
                uint2 e = make_uint2(kEmpty, 0u);
                if (j < sp) e = stack[(sp - 1u - j) * kGroupRays];
                const uint32_t m = group_ballot(j < sp && __uint_as_float(e.y) <= r.tmax, lane);
                if (m) {
                    const uint32_t i = __builtin_ctz(m);
                    cur = __shfl(e.x, (int)((lane & ~(kGroup - 1u)) | i));
                    sp -= i + 1u;
                    break;
                }
                sp -= min(sp, kGroup);
            }
        }
        if (j == 0u) store_ray<kAny>(q, occ, rid, r);
    }
}

template <int W, bool kAny, bool kMulti, uint32_t S, bool kInst, bool kStats = false, bool kAlpha = false>
__global__ __launch_bounds__(kTraceBlock, S == 8 ? 8 : 1) void k_trace(SceneDev sc, TraceQueue q, uint8_t *occ,
                                                                      uint32_t *spill)
{
    uint32_t c_nodes = 0, c_leaves = 0, c_tris = 0, c_wnode = 0, c_wleaf = 0;
    uint32_t c_noray = 0, c_empty = 0, c_leafwait = 0;   // idle lanes of node-loop iterations, by cause
    __shared__ uint2 s_stack[S * kTraceBlock];
    const uint32_t n = q.count ? *q.count : q.n;
    if (n == 0) {
        if (q.done && blockIdx.x == 0 && threadIdx.x == 0) trace_clear(q, n);
        return;
    }
    if constexpr (W == 8 && !kInst && !kStats && !kAlpha) {
        constexpr uint32_t kDepth = S * kTraceBlock / kGroupRays;
        static_assert(group_stack_fits(kDepth, S) && !group_stack_fits(kDepth + 1u, S), "the host's rule is this depth");
        if (n <= q.group_rays) {
            if (blockIdx.x * kGroupRays >= n) return;
            trace_groups<kAny, kMulti>(sc, q, occ, n, s_stack, kDepth);
            trace_epilogue(q, n, min(gridDim.x, (n + kGroupRays - 1u) / kGroupRays));
            return;
        }
    }
    const uint32_t lane = lane_id();
    constexpr uint32_t kWaves = kTraceBlock / 64;
    // wave-uniform by construction; readfirstlane keeps the supply in scalar registers
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    RaySupply sup;
    sup.init(n, blockIdx.x % kXcds, blockIdx.x / kXcds * kWaves + wave, gridDim.x / kXcds * kWaves);
    // no rays for any wave of the block: it does not count in the epilogue either
    if (!sup.dynamic && blockIdx.x / kXcds * kWaves * kStatic >= sup.slice_len(blockIdx.x % kXcds)) return;

    Stack<S> st;
    st.s      = s_stack + threadIdx.x;
    st.g      = reinterpret_cast<uint4 *>(spill) + (size_t)(blockIdx.x * blockDim.x + threadIdx.x) * (q.spill_depth / 2);
    st.depth  = q.spill_depth;
    st.err    = q.error;
    st.clear();

    RayState r;
    const void   *nodes = sc.nodes;
    const float4 *tris  = sc.tri;
    uint32_t rid = 0, cur = kEmpty;
    uint32_t aroot = sc.root, steps = 0, passed = 0;   // kAlpha: the ray's root, traces of it, passes of the lane
    // instance state (kInst): world ray while inside an instance, scale, instance ids
    f3       wo = mk3(0, 0, 0), wd = mk3(0, 0, 0);
    float    wtmax = 0.0f, ilen = 1.0f;
    uint32_t level = 0, cur_inst = kInvalidRef, best_inst = kInvalidRef;
    bool     inst_hit = false;
    auto enter_instance = [&](uint32_t inst) {
        const InstDev &I = sc.inst[inst];
        wo    = r.o;
        wd    = r.d;
        wtmax = r.tmax;
        const f3 o2 = mk3(I.inv[0] * r.o.x + I.inv[1] * r.o.y + I.inv[2] * r.o.z + I.inv[3],
                          I.inv[4] * r.o.x + I.inv[5] * r.o.y + I.inv[6] * r.o.z + I.inv[7],
                          I.inv[8] * r.o.x + I.inv[9] * r.o.y + I.inv[10] * r.o.z + I.inv[11]);
        const f3 d2 = mk3(I.inv[0] * r.d.x + I.inv[1] * r.d.y + I.inv[2] * r.d.z,
                          I.inv[4] * r.d.x + I.inv[5] * r.d.y + I.inv[6] * r.d.z,
                          I.inv[8] * r.d.x + I.inv[9] * r.d.y + I.inv[10] * r.d.z);
        ilen     = sqrtf(dot(d2, d2));
        r.o      = o2;
        r.d      = d2 * (1.0f / ilen);
        r.inv    = mk3(safe_rcp(r.d.x), safe_rcp(r.d.y), safe_rcp(r.d.z));
        r.wt     = wt_setup(r.d);
        r.tmax   = wtmax * ilen;
        level    = 1;
        cur_inst = inst;
        inst_hit = false;
        st.push(make_uint2(kInstExit, __float_as_uint(-kInf)));
        return I.root;
    };
    auto exit_instance = [&]() {
        r.o    = wo;
        r.d    = wd;
        r.inv  = mk3(safe_rcp(r.d.x), safe_rcp(r.d.y), safe_rcp(r.d.z));
        r.wt   = wt_setup(r.d);
        r.tmax = inst_hit ? r.tmax / ilen : wtmax;
        level  = 0;
    };
    // next node to visit: pops, leaving instances as their exit markers come up
    auto next = [&]() -> uint32_t {
        for (;;) {
            const uint32_t c = st.pop(r.tmax);
            if (!kInst || c != kInstExit) return c;
            exit_instance();
        }
    };
    // leaves parked by the inner-node phase, pend first (not for two-level scenes, whose
    // instance leaves change the lane's ray)
    constexpr bool kSpec = !kInst;
    uint32_t pend = kEmpty, pend2 = kEmpty;
    bool     active = false, exhausted = false;

    for (;;) {
        // ---- refill idle lanes ----
        uint64_t idle = __ballot(!active);
        uint32_t nidle = __popcll(idle);
        while (!exhausted && nidle >= q.refill_idle) {
            if (sup.pbeg == sup.pend && !sup.take(q.counters, lane)) {
                exhausted = true;
                break;
            }
            const uint32_t base = sup.pbeg, got = min(nidle, sup.pend - sup.pbeg);
            sup.pbeg += got;
            const uint32_t rank = __popcll(idle & ((1ull << lane) - 1ull));
            if (!active && rank < got) {
                rid = base + rank;
                st.clear();
                pend      = kEmpty;
                pend2     = kEmpty;
                level     = 0;
                best_inst = kInvalidRef;
                uint32_t root = sc.root, ntri = sc.ntri;
                if constexpr (kMulti) {
                    const TraceScene ts = q.scenes[q.path_job[q.ray_path[rid]]];
                    nodes = ts.nodes;
                    tris  = ts.tri;
                    root  = ts.root;
                    ntri  = ts.ntri;
                }
                const bool valid = load_ray(q, rid, ntri, r);
                cur    = valid ? root : kEmpty;
                active = true;
                if constexpr (kAlpha) {
                    aroot = root;
                    steps = 1;
                }
            }
            idle  = __ballot(!active);
            nidle = __popcll(idle);
        }
        if (__ballot(active) == 0) {
            if (exhausted) break;
            continue;
        }
        // ---- inner-node phase: lanes expand nodes until every lane holds a leaf or is done.
        // kSpec: a lane whose next node is a leaf parks it (two slots) and keeps traversing
        // until its slots are full, so that the leaf phase runs with more lanes busy ----
        for (;;) {
            if (kSpec && active && pend2 == kEmpty && cur != kEmpty && ref_is_leaf(cur)) {
                if (pend == kEmpty) pend = cur;
                else pend2 = cur;
                cur = next();
            }
            const bool inner = active && cur != kEmpty && !ref_is_leaf(cur);
            const uint64_t srch = __ballot(inner && (!kSpec || pend2 == kEmpty));
            if (srch == 0) break;
            // fewer than park_min lanes still searching and some holding a leaf: run the leaf
            // phase now rather than keep most of the wave waiting
            if (kSpec && __popcll(srch) < q.park_min && __ballot(active && pend != kEmpty) != 0) break;
            if constexpr (kStats) {
                ++c_wnode;
                c_noray += !active;
                c_empty += active && cur == kEmpty;
                c_leafwait += active && cur != kEmpty && ref_is_leaf(cur);
            }
            if (inner) {
                Child c[W];
                const int nh = NodeOps<W>::expand(nodes, cur, r, c);
                if constexpr (kStats) ++c_nodes;
                if (nh == 0) {
                    cur = next();
                } else {
                    sort_children<W>(c);
                    cur = child_ref(c[0]);
                    st.template push_children<W>(c, nh);
                }
            }
        }
        // ---- leaf phase: the parked leaf first, then leaves popped after it ----
        for (uint32_t round = 0;; ++round) {
            const bool parked = kSpec && active && pend != kEmpty;
            const bool leaf   = active && (parked || (cur != kEmpty && ref_is_leaf(cur)));
            if (__ballot(leaf) == 0) break;
            // a lane left holding an unparked leaf parks it in the next inner-node phase
            if (kSpec && q.leaf_rounds && round >= q.leaf_rounds && __ballot(parked) == 0) break;
            if constexpr (kStats) ++c_wleaf;
            if (kInst && leaf && level == 0) {
                // instance leaf: enter the first instance, keep the rest for later
                const uint32_t first = leaf_first(cur), cnt = leaf_count(cur);
                if (cnt > 1) st.push(make_uint2(ref_leaf(first + 1, cnt - 1), __float_as_uint(-kInf)));
                cur = enter_instance(sc.tlas_inst[first]);
            } else if (leaf) {
                const uint32_t lf = parked ? pend : cur;
                const uint32_t first = leaf_first(lf), cnt = leaf_count(lf);
                bool any = false;
                if constexpr (kStats) ++c_leaves;
                for (uint32_t k = 0; k < cnt; ++k) {
                    if constexpr (kStats) ++c_tris;
                    const size_t  ti = (size_t)(first + k);
                    const float4  a  = tris[3 * ti + 0];
                    const float4  b  = tris[3 * ti + 1];
                    const float4  c  = tris[3 * ti + 2];
                    float t, u, v;
                    if (wt_test(r.wt, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), mk3(c.x, c.y, c.z), r.o, r.tn, r.tmax,
                                t, u, v)) {
                        const uint32_t prim = __float_as_uint(a.w);
                        if (t < r.tmax || prim < r.best_prim) {
                            r.tmax      = t;
                            r.best_tri  = (uint32_t)ti;
                            r.best_prim = prim;
                            r.bu        = u;
                            r.bv        = v;
                            if (kInst) {
                                best_inst = cur_inst;
                                inst_hit  = true;
                            }
                        }
                        if (kAny) {
                            any = true;
                            break;
                        }
                    }
                }
                if (parked) {
                    pend  = pend2;
                    pend2 = kEmpty;
                    if (kAny && any) {
                        cur  = kEmpty;
                        pend = kEmpty;
                    }
                } else {
                    cur = (kAny && any) ? kEmpty : next();
                }
            }
        }
        if constexpr (kAlpha) {
            f3 o2;
            if (active && cur == kEmpty && r.best_tri != kInvalidRef && alpha_passes<kMulti>(sc, q, rid, r, o2)) {
                ++passed;
                if (steps < kAlphaSteps) {
                    ++steps;
                    r.o    = o2;
                    r.tmax = kInf;
                    r.best_tri = r.best_prim = kInvalidRef;
                    st.clear();
                    cur = aroot;
                }
            }
        }
        if (active && cur == kEmpty) {
            store_ray<kAny || kAlpha>(q, occ, rid, r);
            if (kInst && !kAny && q.hits.inst) q.hits.inst[rid] = r.best_tri != kInvalidRef ? best_inst : kInvalidRef;
            active = false;
        }
    }
    if constexpr (kStats) {
        unsigned long long a = c_nodes, b = c_leaves, c = c_tris, d = c_noray, e = c_empty, f = c_leafwait;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_xor(a, o);
            b += __shfl_xor(b, o);
            c += __shfl_xor(c, o);
            d += __shfl_xor(d, o);
            e += __shfl_xor(e, o);
            f += __shfl_xor(f, o);
        }
        if (lane == 0 && q.tstats) {
            atomicAdd(q.tstats + 0, a);
            atomicAdd(q.tstats + 1, b);
            atomicAdd(q.tstats + 2, c);
            atomicAdd(q.tstats + 3, (unsigned long long)c_wnode);   // wave-uniform counts
            atomicAdd(q.tstats + 4, (unsigned long long)c_wleaf);
            atomicAdd(q.tstats + 5, d);
            atomicAdd(q.tstats + 6, e);
            atomicAdd(q.tstats + 7, f);
        }
    }
    if constexpr (kAlpha) {
        for (int o = 32; o > 0; o >>= 1) passed += __shfl_xor(passed, o);
        if (lane == 0 && passed != 0u) atomicAdd(q.alpha_stat, (unsigned long long)passed);
    }
    trace_epilogue(q, n, sup.active_blocks(gridDim.x, kWaves));
}

}  // namespace

uint32_t trace_grid(int device, uint32_t blocks_per_cu)
{
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) != hipSuccess) return 1024;
    if (blocks_per_cu == 0) blocks_per_cu = kTraceBlocksPerCu;
    uint32_t g = (uint32_t)p.multiProcessorCount * blocks_per_cu;
    // whole multiple of the XCD count so every XCD gets the same number of blocks
    g = (g + kXcds - 1) / kXcds * kXcds;
    return g;
}

uint64_t trace_spill_bytes(uint32_t grid, uint32_t spill_depth)
{
    return (uint64_t)grid * kTraceBlock * spill_depth * 2u * sizeof(uint32_t);
}

namespace {

// Instantiates k_trace for the BVH width and LDS stack depth of the launch.
template <bool kAny, bool kMulti, bool kInst, bool kAlpha = false>
hipError_t dispatch_trace(uint32_t width, const TraceConfig &tc, const SceneDev &sc, const TraceQueue &qin, uint8_t *occ,
                          uint32_t *spill, hipStream_t s)
{
    const dim3 g(tc.grid), b(kTraceBlock);
    TraceQueue q   = qin;
    q.refill_idle  = tc.refill ? std::min(tc.refill, 64u) : kRefillIdle;
    q.park_min     = tc.park_min ? std::min(tc.park_min, 64u) : kParkMin;
    q.spill_depth  = tc.spill_depth;
    q.group_rays   = group_stack_fits(tc.stack_need, tc.stack) ? tc.group_rays : 0u;
    q.leaf_rounds  = tc.leaf_rounds ? (tc.leaf_rounds > 64u ? 0u : tc.leaf_rounds) : kLeafRounds;
    if (!kMulti && !kAlpha && q.tstats) {
        // instrumented traversal: one stack depth (the counts do not depend on it)
        if (width == 4) k_trace<4, kAny, false, 32, kInst, true><<<g, b, 0, s>>>(sc, q, occ, spill);
        else k_trace<8, kAny, false, 32, kInst, true><<<g, b, 0, s>>>(sc, q, occ, spill);
        return hipGetLastError();
    }
#define CRT_TRACE(Wd, Sd) k_trace<Wd, kAny, kMulti, Sd, kInst, false, kAlpha><<<g, b, 0, s>>>(sc, q, occ, spill)
    if (width == 4) {
        if (tc.stack == 8) CRT_TRACE(4, 8);
        else if (tc.stack == 32) CRT_TRACE(4, 32);
        else CRT_TRACE(4, 16);
    } else {
        if (tc.stack == 8) CRT_TRACE(8, 8);
        else if (tc.stack == 32) CRT_TRACE(8, 32);
        else CRT_TRACE(8, 16);
    }
#undef CRT_TRACE
    return hipGetLastError();
}

}  // namespace

hipError_t launch_trace_closest(const SceneDev &sc, const TraceQueue &q, uint32_t *spill, const TraceConfig &tc,
                                hipStream_t s)
{
    if (sc.instanced) return dispatch_trace<false, false, true>(sc.width, tc, sc, q, nullptr, spill, s);
    return dispatch_trace<false, false, false>(sc.width, tc, sc, q, nullptr, spill, s);
}

hipError_t launch_trace_any(const SceneDev &sc, const TraceQueue &q, uint8_t *occ, uint32_t *spill,
                            const TraceConfig &tc, hipStream_t s)
{
    if (sc.instanced) return dispatch_trace<true, false, true>(sc.width, tc, sc, q, occ, spill, s);
    return dispatch_trace<true, false, false>(sc.width, tc, sc, q, occ, spill, s);
}

hipError_t launch_trace_alpha(const SceneDev &sc, const TraceQueue &q, uint32_t *spill, const TraceConfig &tc,
                              hipStream_t s)
{
    if (sc.instanced) return dispatch_trace<false, false, true, true>(sc.width, tc, sc, q, nullptr, spill, s);
    return dispatch_trace<false, false, false, true>(sc.width, tc, sc, q, nullptr, spill, s);
}

hipError_t launch_trace_closest_multi(uint32_t width, const TraceQueue &q, uint32_t *spill, const TraceConfig &tc,
                                      hipStream_t s)
{
    SceneDev none{};
    none.ntri = 1;   // per-ray scenes decide
    return dispatch_trace<false, true, false>(width, tc, none, q, nullptr, spill, s);
}

hipError_t launch_trace_alpha_multi(uint32_t width, const TraceQueue &q, uint32_t *spill, const TraceConfig &tc,
                                    hipStream_t s)
{
    SceneDev none{};
    none.ntri = 1;
    return dispatch_trace<false, true, false, true>(width, tc, none, q, nullptr, spill, s);
}

hipError_t launch_trace_any_multi(uint32_t width, const TraceQueue &q, uint8_t *occ, uint32_t *spill,
                                  const TraceConfig &tc, hipStream_t s)
{
    SceneDev none{};
    none.ntri = 1;
    return dispatch_trace<true, true, false>(width, tc, none, q, occ, spill, s);
}

}  // namespace crt
