// Wavefront path-tracing kernels for gfx950 (CDNA4, wave64).
//
// Replaces the reference's device programs: __raygen__ Primary/Secondary/Shadow with
// the OptiX traversal behind optixTrace (Optix/GPU/optix.cu:225-343), the shading
// kernel PathTracingKernel (CUDA/GPU/Shade/PathTracing.h:8-175, launched from
// CUDA/GPU/cuda.cu:22-84), InitCudaCountersKernel and FimalizeFrameKernel
// (CUDA/GPU/CudaUtilityKernels.h:6-44).
//
// Design:
//  * Extend / Shadow: persistent waves refill idle lanes from a queue of
//    structure-of-arrays ray records (one atomic per refill); each lane walks the BVH2
//    (speculative while-while loop, leaf triangles dealt out over the wave) with a
//    two-tier stack: a 16-entry LDS ring per lane (lane-interleaved) over a global spill
//    area.
//  * Shade: the shared integrator step (trt/integrator.h) per ray; extension and
//    shadow rays are appended with one atomic per wave (ballot + mbcnt prefix) rather
//    than one atomic per ray as in the reference (PathTracing.h:135-141, 168-173).
//  * Queues are segmented (device.h: kSegs segments, each with its own counters on
//    separate cache lines) so that fetch and append atomics spread over 32 lines.
//  * RayGen writes thread t's ray to a fixed slot (no atomics; the primary queue is
//    dense), the paths of each sample in 8x8 pixel tiles.
//  * No host synchronisation between bounces: queue sizes stay in device counters.
//  * Radiance is accumulated per path (one writer per path per kernel) and reduced
//    per pixel in a fixed sample order in Finalize, so images are deterministic. Shade
//    lists emission rather than adding it; the bounce's Shadow launch, on a stream of its
//    own, adds first the listed emission and then its rays' contributions, so every term is
//    added in vertex order while Shade runs beside the previous bounce's Shadow.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.h"
#include "trt/segments.h"
#include "trt/slab32.h"
#include "trt/tonemap.h"

namespace trt {

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / 64;

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t prefix_count(uint64_t mask) {
  // number of set bits of mask below this lane
  const uint32_t lo = static_cast<uint32_t>(mask), hi = static_cast<uint32_t>(mask >> 32);
  return __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
}

// This lane's bit of a (wave-uniform) lane mask: predicates combined as masks stay in scalar
// registers, where combined bools would become vector integers.
__device__ __forceinline__ bool lane_bit(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

__device__ __forceinline__ uint32_t mask_count(uint64_t m) {
  // two 32-bit counts: a 64-bit compare of the count would be a vector instruction
  return static_cast<uint32_t>(__builtin_popcount(static_cast<uint32_t>(m))) +
         static_cast<uint32_t>(__builtin_popcount(static_cast<uint32_t>(m >> 32)));
}

__device__ __forceinline__ void wave_add_stat(unsigned long long* dst, uint32_t v) {
  // sum over the wave, one atomic
  uint32_t s = v;
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane_id() == 0 && s) atomicAdd(dst, static_cast<unsigned long long>(s));
}

// Fetches the next batch of up to `want` (1..64) items of a segmented queue for the
// wave: one atomic on the fetch cursor of the first segment, from `home` on, not yet
// found exhausted. `n_seg` holds, in lane s < kSegs, the item count of segment s
// (constant during the kernel); `done` collects exhausted segments (cursors only grow,
// so they stay exhausted; callers start it with seg_empty(), which also closes the
// segments outside the wave's fetch window). Every wave makes at most kFetchWindow
// failed attempts (kSegs in grids of fewer than kSegs waves), so the loop always ends. The cursors are not pre-read: coherent
// reads of a hot line serialise like the atomics themselves (measured: a pre-read of all
// 32 cursors per batch cost as much as the whole Shade kernel's work).
__device__ __forceinline__ bool seg_fetch_k(const SegIn& in, uint32_t n_seg, uint32_t home, uint64_t& done,
                                            uint32_t want, uint32_t& slot0, uint32_t& n_got) {
  const uint32_t lane = lane_id();
  const uint64_t all = (1ull << kSegs) - 1ull;
  for (;;) {
    const uint64_t m = ~done & all;
    if (m == 0ull) return false;
    const uint64_t rot = ((m >> home) | (m << (kSegs - home))) & all;
    uint32_t sgm = home + static_cast<uint32_t>(__builtin_ctzll(rot));
    if (sgm >= kSegs) sgm -= kSegs;
    uint32_t b = 0;
    if (lane == 0) b = atomicAdd(&in.work[sgm * kLine], want);
    b = __shfl(b, 0);
    const uint32_t ns = __shfl(n_seg, static_cast<int>(sgm));
    if (b < ns) {
      slot0 = sgm * in.cap + b;
      n_got = ns - b < want ? ns - b : want;
      return true;
    }
    done |= 1ull << sgm;
  }
}

__device__ __forceinline__ bool seg_fetch(const SegIn& in, uint32_t n_seg, uint32_t home, uint64_t& done,
                                          uint32_t& slot0, uint32_t& n_valid) {
  return seg_fetch_k(in, n_seg, home, done, 64u, slot0, n_valid);
}

// Home segment of the calling wave.
__device__ __forceinline__ uint32_t wave_home() { return (blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) % kSegs; }

// Initial `done` mask of seg_fetch (uniform per wave): segments without items, and every
// segment outside the wave's window {home, home + 1}. A wave thus only ever touches two
// fetch cursors; once the queue runs dry each cursor line takes (waves / kSegs) x 2
// failed attempts instead of one from every wave (the tail of small launches was spent
// in those serialised atomics). Every segment lies in the window of the waves whose
// home it is, so when every segment is some wave's home (at least kSegs waves in the
// grid with a home per wave, kSegs blocks with a home per block: every_segment_homed)
// every item is fetched; otherwise all segments stay open.
constexpr uint32_t kFetchWindow = 2;
__device__ __forceinline__ uint64_t seg_empty(uint32_t n_seg, uint32_t home, bool every_segment_homed) {
  const uint64_t all = (1ull << kSegs) - 1ull;
  uint64_t closed = ~__ballot(n_seg > 0u);
  if (every_segment_homed) {
    const uint64_t w = (1ull << kFetchWindow) - 1ull;
    closed |= ~(((w << home) | (w >> (kSegs - home))) & all);
  }
  return closed & all;
}
// seg_empty for a home per wave (wave_home).
__device__ __forceinline__ uint64_t seg_empty(uint32_t n_seg) {
  return seg_empty(n_seg, wave_home(), gridDim.x * kWavesPerBlock >= kSegs);
}

// Home segment of a wave in the single-level traversal and in Shade: one per block, so
// that the four waves of a block fetch neighbouring batches of the same part of the
// queue (neighbouring rays, which share nodes, triangles and materials in the CU's L1),
// and Shade's waves of a block append their outputs next to each other: 4 % faster Extend
// and 3.5 % faster Shade on the 1M-triangle soup than a home per wave. (The two-level
// traversal keeps a home per wave: there the block home measured 1.5 % slower, and a
// home per XCD, segment (b % 8) x 4 + (b / 8) % 4 for block b, slower on both scenes.)
// Every segment is some block's home once the grid has kSegs blocks.
__device__ __forceinline__ uint32_t block_home() { return blockIdx.x % kSegs; }

// Per-lane item count of segment `lane` (lanes >= kSegs: 0).
__device__ __forceinline__ uint32_t seg_counts(const SegIn& in) {
  const uint32_t lane = lane_id();
  if (lane >= kSegs) return 0u;
  const uint32_t c = in.cnt[lane * kLine];
  return c < in.cap ? c : in.cap;
}


// Appends the lanes in `mask` to a segmented queue; returns this lane's slot (kNoHit
// for lanes not in the mask). Starts at segment `home` and moves on while segments are
// full; a partly full segment takes what fits. Total capacity (kSegs * cap) is at
// least the number of items ever appended per queue, so the loop places everything
// within kSegs attempts; otherwise bit 1 of *overflow is set.
__device__ __forceinline__ uint32_t seg_append(uint32_t* cnt, uint32_t cap, uint32_t home, uint64_t mask,
                                               uint32_t* overflow) {
  const uint32_t lane = lane_id();
  const uint32_t need = static_cast<uint32_t>(__popcll(mask));
  const uint32_t rank = prefix_count(mask);
  const bool mine = (mask >> lane) & 1ull;
  uint32_t slot = kNoHit, done = 0, sgm = home;
  for (uint32_t t = 0; t < kSegs && done < need; ++t) {
    uint32_t b = 0;
    if (lane == 0) b = atomicAdd(&cnt[sgm * kLine], need - done);
    b = __shfl(b, 0);
    const uint32_t fit = b < cap ? (need - done < cap - b ? need - done : cap - b) : 0u;
    if (mine && rank >= done && rank < done + fit) slot = sgm * cap + b + (rank - done);
    done += fit;
    sgm = sgm + 1 == kSegs ? 0u : sgm + 1;
  }
  if (done < need && lane == 0) atomicOr(overflow, 2u);
  return slot;
}

struct TraceOut {
  float t, b1, b2;
  uint32_t prim, inst;
  uint32_t nodes, tests, spills;  // statistics: node visits, triangle tests, stack entries spilled
};

// Counting kernels: marks item i of a touch bitmap (null: not collected).
__device__ __forceinline__ void touch(uint32_t* bits, uint32_t i) {
  if (bits) atomicOr(&bits[i >> 5], 1u << (i & 31u));
}

// Ray/box slab tests of the device traversals (after Ize 2013's conservative form), on
// boxes stored as centre c and half extent h per axis; one class per node layout. Both
// are conservative: the far distance is widened by kBoxSlack, which covers errors
// relative to the distances themselves, and the stored half extents carry margins for the
// rest, so no box the ray touches is culled and traversal equals a brute-force loop. The
// axes are combined with max / min that ignore NaN. A node is visited by its byte offset
// from the (wave-uniform) array base: one 32-bit add per visit.
struct NodeHits {
  float n0, f0, n1, f1;  // per child: entry and (widened) exit; the ray meets the box when n <= f
  int32_t c0, c1;        // child references
};

// max / min as the instructions have them: NaN operands are ignored without first being
// made quiet (two more instructions per visit; no value here is a signalling NaN's).
__device__ __forceinline__ float max3_ft(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float min3_ft(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max_ft(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float min_ft(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// 48-byte nodes: fp32 boxes. With x = c - o and s = sign(inv) (per ray, +-1), a slab's
// entry and exit are (x - s h) inv and (x + s h) inv, each within a few ulp of itself plus
// u |x inv|. inv = 1/d is the IEEE reciprocal: for a zero direction component it is +-inf
// and the products give the exact slab of a ray parallel to the axis.
struct Nodes48 {
  static constexpr uint32_t kBytes = kNodeBytes;
  struct Ray {
    V3 o;
    V3 inv;  // 1 / d, infinite for a zero component
    V3 sgn;  // +-1, the sign of inv
  };
  static __device__ __forceinline__ Ray setup(const NodeGrid&, V3 o, V3 d) {
    Ray b;
    b.o = o;
    b.inv = v3(1.f / d.x, 1.f / d.y, 1.f / d.z);
    b.sgn = v3(__builtin_copysignf(1.f, b.inv.x), __builtin_copysignf(1.f, b.inv.y), __builtin_copysignf(1.f, b.inv.z));
    return b;
  }
  static __device__ __forceinline__ void slab(float cx, float hx, float cy, float hy, float cz, float hz, const Ray& b,
                                              float tmin, float tmax, float& n, float& f) {
    const float xx = cx - b.o.x, sx = hx * b.sgn.x;
    const float xy = cy - b.o.y, sy = hy * b.sgn.y;
    const float xz = cz - b.o.z, sz = hz * b.sgn.z;
    n = max_ft(max3_ft((xx - sx) * b.inv.x, (xy - sy) * b.inv.y, (xz - sz) * b.inv.z), tmin);
    f = min_ft(min3_ft((xx + sx) * b.inv.x, (xy + sy) * b.inv.y, (xz + sz) * b.inv.z), tmax) * kBoxSlack;
  }
  // Child reference from the low bytes of one node row (v_perm_b32 gathers two bytes per
  // instruction).
  static __device__ __forceinline__ int32_t child_ref(float4 r) {
    const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(r.y), __float_as_uint(r.x), 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(__float_as_uint(r.w), __float_as_uint(r.z), 0x04000c0cu);
    return static_cast<int32_t>(lo | hi);
  }
  static __device__ __forceinline__ NodeHits visit(const void* __restrict__ nodes, int32_t at, const Ray& b, float tmin,
                                                   float tmax) {
    const float4* p = reinterpret_cast<const float4*>(static_cast<const char*>(nodes) + static_cast<uint32_t>(at));
    const float4 r0 = p[0], r1 = p[1], r2 = p[2];
    NodeHits v;
    slab(r0.x, r0.y, r0.z, r0.w, r2.x, r2.y, b, tmin, tmax, v.n0, v.f0);
    slab(r1.x, r1.y, r1.z, r1.w, r2.z, r2.w, b, tmin, tmax, v.n1, v.f1);
    v.c0 = child_ref(r0);
    v.c1 = child_ref(r1);
    return v;
  }
};

// 32-byte nodes: fp16 boxes on the tree's grid (NodeSpace: world = org + step * c). Two
// 16-byte loads a visit instead of three (the load path bounds the traversal), and nothing
// to decode: v_fma_mix_f32 takes an fp16 operand as it is, so per axis
//   ct = fma(c, step inv, (org - o) inv),  entry = ct - h |step inv|,  exit = ct + h |step inv|
// are three instructions (six, plus six to gather the child references, with Nodes48).
// The terms that cancel in ct have an error of up to 3u (|x| + R) |inv| (u = 2^-24, x the
// distance to the box's centre, R the tree's half side on the axis): the part in |x| is
// relative to the distances, and the half extents' margins (bvh_build.h) exceed the part in R.
// The per-ray terms, and what they do with tiny direction components and extreme rays:
// slab32_ray.
struct Nodes32 {
  static constexpr uint32_t kBytes = sizeof(DevNode32);
  struct Ray {
    V3 o;
    V3 si;  // step / d
    V3 oi;  // (org - o) / d
  };
  static __device__ __forceinline__ Ray setup(const NodeGrid& g, V3 o, V3 d) {
    Ray b;
    b.o = o;
    slab32_ray(g.org, g.step, o, d, [](float x) { return __builtin_amdgcn_rcpf(x); }, b.si, b.oi);
    return b;
  }
  // v: fp16 (c, h) pairs of the axes, then the child reference
  static __device__ __forceinline__ void slab(uint4 v, const Ray& b, float tmin, float tmax, float& n, float& f) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 x = __builtin_bit_cast(h2, v.x), y = __builtin_bit_cast(h2, v.y), z = __builtin_bit_cast(h2, v.z);
    const float cx = __builtin_fmaf(static_cast<float>(x[0]), b.si.x, b.oi.x);
    const float cy = __builtin_fmaf(static_cast<float>(y[0]), b.si.y, b.oi.y);
    const float cz = __builtin_fmaf(static_cast<float>(z[0]), b.si.z, b.oi.z);
    const float ax = __builtin_fabsf(b.si.x), ay = __builtin_fabsf(b.si.y), az = __builtin_fabsf(b.si.z);
    n = max_ft(max3_ft(__builtin_fmaf(-static_cast<float>(x[1]), ax, cx), __builtin_fmaf(-static_cast<float>(y[1]), ay, cy),
                       __builtin_fmaf(-static_cast<float>(z[1]), az, cz)),
               tmin);
    f = min_ft(min3_ft(__builtin_fmaf(static_cast<float>(x[1]), ax, cx), __builtin_fmaf(static_cast<float>(y[1]), ay, cy),
                       __builtin_fmaf(static_cast<float>(z[1]), az, cz)),
               tmax) *
        kBoxSlack;
  }
  static __device__ __forceinline__ NodeHits visit(const void* __restrict__ nodes, int32_t at, const Ray& b, float tmin,
                                                   float tmax) {
    const uint4* p = reinterpret_cast<const uint4*>(static_cast<const char*>(nodes) + static_cast<uint32_t>(at));
    const uint4 r0 = p[0], r1 = p[1];
    NodeHits v;
    slab(r0, b, tmin, tmax, v.n0, v.f0);
    slab(r1, b, tmin, tmax, v.n1, v.f1);
    v.c0 = static_cast<int32_t>(r0.w);
    v.c1 = static_cast<int32_t>(r1.w);
    return v;
  }
};

// Sentinel of an exhausted traversal (never a leaf code: leaf first indices are < 2^28).
constexpr int32_t kTravDone = static_cast<int32_t>(0x80000000u);

// The traversal's node loop ends once at most kSearchBreakSpread of the lanes still walking
// have no leaf parked, instead of none: the last few searching lanes would otherwise
// hold the wave for a long tail of iterations in which most lanes idle. They keep their
// state and go on walking in the next round. 16 measured best on the 1M-triangle soup
// (Extend of a frame 7.97 ms; at 8 8.11, at 24 8.40) and as good as 8 on the instances.
constexpr uint32_t kSearchBreakSpread = 16;

// Persistent single-level BVH2 traversal of a segmented ray queue, in rounds of the
// "speculative while-while" form of Aila & Laine (2009, "Understanding the efficiency of
// ray traversal on GPUs"): lanes walk inner nodes until (nearly) every lane of the wave
// holds a leaf (a lane that meets its first leaf parks it and keeps walking), then the
// wave intersects leaves together. Before each round lanes whose ray has finished take new
// rays from the queue ("dynamic fetch", same paper) once at least kRefill of them are
// idle, so a few long rays do not hold the whole wave (40 of 64: a frame's Extend 7.97 ms
// on the soup, at 32 8.04, at 24 8.12; a refill's queue atomic, loads and divisions cost
// more lanes than they fill. Claiming 64 rays at a time and keeping them set up in
// registers made refills cheap but scatters a CU's rays over more of the queue: 9.0 ms at
// 24). The result does not depend on the visiting order (closest hit under the
// (t, inst, prim) order, or any hit).
// load(slot, o, d, tmin, tmax) reads a ray;
// finish(slot, r, hit) consumes a result (hit: a hit was found).
constexpr uint32_t kRefill = 40;

// Traversal stack of the queue traversals: the top entries live in an LDS ring of
// kRingEntries slots (entry k in slot k % kRingEntries, lane-interleaved), older ones are
// moved to the lane's area of a global spill buffer when the ring fills up and brought
// back when it runs empty. Deep traversals are rare, so the ring keeps LDS small (4 KiB
// per wave, beside the 1.6 KiB leaf-task area) and occupancy bound by registers, not by
// the tree depth.
//
// Pushes and pops are free of branches: the two lowest entries are sentinels (popping one
// ends the traversal, the second keeps the stack from looking empty then), every step
// reads the top entry ahead and stores its far child above the top whether or not it is
// pushed (one ring slot stays free for that), and stack_step moves the top. Only a ring
// about to overflow or running empty takes a branch (stack_move).
constexpr int kRingEntries = 16;

// LDS word at a byte address (ds_read / ds_write with a 32-bit address formed by integer
// arithmetic, so that a ring slot's address is one and-or of the lane's ring base and
// the slot offset).
typedef __attribute__((address_space(3))) uint32_t lds_u32;

__device__ __forceinline__ uint32_t lds_address(uint32_t* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u32*)p));  // address-space cast
}
__device__ __forceinline__ uint32_t lds_load(uint32_t a) { return *reinterpret_cast<lds_u32*>(static_cast<uintptr_t>(a)); }
__device__ __forceinline__ void lds_store(uint32_t a, uint32_t v) {
  *reinterpret_cast<lds_u32*>(static_cast<uintptr_t>(a)) = v;
}

// Entry counts are kept in units of kSlotBytes (the ring's slot stride: 64 lanes x 4 bytes),
// so that entry k's ring slot is at ring | (k * kSlotBytes & kRingMask). The wave's ring is
// 4 KiB aligned in LDS (the traversal kernels have no static LDS: dynamic LDS starts at 0,
// checked at start-up by traversal_lds_check), so the slot bits never meet the lane's base.
constexpr uint32_t kSlotBytes = 64 * 4;
constexpr uint32_t kRingMask = (kRingEntries - 1) * kSlotBytes;
constexpr uint32_t kSentinels = 2;
constexpr uint32_t kSpillStep = 4;  // entries moved at a time

struct TwoTierStack {
  uint32_t ring;         // LDS byte address of the lane's first ring slot
  uint32_t* spill_wave;  // the wave's spill area; lane l's `cap` entries start at l * cap
  uint32_t cap;          // capacity of the spill area (entries)
  uint32_t sp;           // entries on the stack, sentinels included, x kSlotBytes
  uint32_t lo1;          // (lo + 1) x kSlotBytes: entries [0, lo) are in the spill area, the rest in the ring
};

__device__ __forceinline__ void stack_reset(TwoTierStack& s) {
  for (uint32_t k = 0; k < kSentinels; ++k) lds_store(s.ring | (k * kSlotBytes), static_cast<uint32_t>(kTravDone));
  s.sp = kSentinels * kSlotBytes;
  s.lo1 = kSlotBytes;
}

// The wave's spill area of the traversal grid (stack_cap entries per thread), taken
// wave-uniform so that it stays in scalar registers; a lane's own area is formed only
// on the rare ring overflow or underflow.
__device__ __forceinline__ uint32_t* wave_spill(uint32_t* spill, int cap) {
  const uint32_t wave_first = __builtin_amdgcn_readfirstlane(threadIdx.x) & ~63u;
  return spill + static_cast<size_t>(blockIdx.x * kBlock + wave_first) * static_cast<uint32_t>(cap);
}

__device__ __forceinline__ uint32_t* lane_spill(const TwoTierStack& s) { return s.spill_wave + lane_id() * s.cap; }

// Top entry (the stack always holds one) and the store of the entry above it.
__device__ __forceinline__ int32_t stack_top(const TwoTierStack& s) {
  return static_cast<int32_t>(lds_load(s.ring | ((s.sp - kSlotBytes) & kRingMask)));
}
__device__ __forceinline__ void stack_above(const TwoTierStack& s, int32_t v) {
  lds_store(s.ring | (s.sp & kRingMask), static_cast<uint32_t>(v));
}

// Brings the ring back between its limits after sp moved: 1 to kRingEntries - 1 entries
// (one slot stays free for stack_above). At the capacity (a tree deeper than the stack was
// sized for) the top entry is dropped, which keeps every access in bounds, and on_full()
// reports the inexact traversal.
template <bool STATS, class OnFull>
__device__ __forceinline__ void stack_move(TwoTierStack& s, TraceOut& stats, OnFull on_full) {
  uint32_t* sp = lane_spill(s);
  const uint32_t lo = s.lo1 / kSlotBytes - 1u;
  if (s.sp < s.lo1) {  // ring empty: bring spilled entries back (lo > 0: the sentinels are below)
    const uint32_t n = lo < kSpillStep ? lo : kSpillStep;
    for (uint32_t k = lo - n; k < lo; ++k) lds_store(s.ring | ((k * kSlotBytes) & kRingMask), sp[k]);
    s.lo1 -= n * kSlotBytes;
  } else if (lo + kSpillStep > s.cap) {
    on_full();
    s.sp -= kSlotBytes;
  } else {  // ring full: move its oldest entries out
    for (uint32_t k = lo; k < lo + kSpillStep; ++k) sp[k] = lds_load(s.ring | ((k * kSlotBytes) & kRingMask));
    s.lo1 += kSpillStep * kSlotBytes;
    if (STATS) stats.spills += kSpillStep;
  }
}

// One entry pushed (already stored by stack_above) or popped (already read by stack_top),
// by the lanes of the masks.
template <bool STATS, class OnFull>
__device__ __forceinline__ void stack_step(TwoTierStack& s, uint64_t push, uint64_t pop, TraceOut& stats,
                                           OnFull on_full) {
  uint32_t by = lane_bit(push) ? kSlotBytes : 0u;
  by = lane_bit(pop) ? 0u - kSlotBytes : by;
  s.sp += by;
  if (s.sp - s.lo1 > (kRingEntries - 3) * kSlotBytes)  // not 1 .. kRingEntries - 2 entries in the ring
    stack_move<STATS>(s, stats, on_full);
}

// A ray's set-up of the watertight test (ray_tri_setup): axes packed 2 bits each, shear.
struct RayShear {
  int32_t kxyz;
  V3 s;
};
__device__ __forceinline__ RayShear ray_shear(V3 d) {
  const RayTri t = ray_tri_setup(v3(0.f), d);
  return RayShear{t.kx | (t.ky << 2) | (t.kz << 4), v3(t.sx, t.sy, t.sz)};
}

// Leaf phase of the traversal loops, spread over the whole wave: every (ray, triangle)
// pair of the leaves the lanes hold is a task, and the wave deals the tasks out 64 at a
// time, each lane testing one with the owning lane's ray (read across lanes), instead of
// each lane looping over its own leaves while most lanes wait (a round's leaves hold
// ~64 triangles, which a per-lane loop tests at ~16 active lanes per iteration).
// A task finds its owner without a list: lanes that own tasks mark the place of their
// first one, and a running maximum over the marks gives each place its owner (writing the
// tasks out, up to 14 per lane, took a quarter of the phase's instructions).
// An owner's closest hit is the minimum of a (t, prim) key over its tasks (LDS atomic
// min; the lexicographic order of the closest-hit search), and the task that holds the
// minimum writes the barycentrics. Per wave, in LDS: 64 marks, and a key and barycentrics
// per lane. One window of kTaskWin tasks per round.
constexpr uint32_t kTaskWin = 128;
constexpr uint32_t kTaskWords = 64 + 64 * 2 + 64 * 2;

struct LeafTasks {
  uint32_t* mark;           // [64] 1 + owning lane at an owner's first task, else 0
  unsigned long long* key;  // [64] hit key per lane
  float2* bary;             // [64] barycentrics of the key's hit
};

__device__ __forceinline__ LeafTasks leaf_tasks(uint32_t* base) {
  LeafTasks t;
  t.mark = base;
  t.key = reinterpret_cast<unsigned long long*>(base + 64);
  t.bary = reinterpret_cast<float2*>(base + 64 + 128);
  return t;
}

// Running maximum over the wave's lanes (all active), lane 0 first.
__device__ __forceinline__ uint32_t wave_scan_max(uint32_t v) {
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xf, 0xf, false)));  // row_shr 1
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xf, 0xf, false)));  // row_shr 2
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xf, 0xf, false)));  // row_shr 4
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xf, 0xf, false)));  // row_shr 8
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xa, 0xf, false)));  // row_bcast 15
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xc, 0xf, false)));  // row_bcast 31
  return v;
}

// Order-preserving (t, prim) key: t's bits mapped so that unsigned order is float
// order (-0 taken as +0), prim below.
__device__ __forceinline__ unsigned long long hit_key(float t, uint32_t prim) {
  uint32_t u = __float_as_uint(t + 0.f);
  u ^= (u >> 31) ? 0xffffffffu : 0x80000000u;
  return (static_cast<unsigned long long>(u) << 32) | prim;
}

__device__ __forceinline__ float key_t(unsigned long long k) {
  uint32_t u = static_cast<uint32_t>(k >> 32);
  u ^= (u >> 31) ? 0x80000000u : 0xffffffffu;
  return __uint_as_float(u);
}

// One leaf phase: lane l contributes the tasks of ca triangles from fa and cb from fb,
// tested with its ray (object-space origin o, axes and shear of ray_shear, tmin, tmax). A task hit counts if it beats the lane's best (t = tmax, prim0, and for
// TWO, instance inst0, with the lane's current instance cur). Returns whether the
// lane's tasks were in this round's window (false: it keeps its leaves for the next
// round); `better`: a task hit counted, the smallest (t, prim) key of those is kf, and
// its barycentrics are in tk.bary[lane].
template <bool STATS, bool TWO>
__device__ __forceinline__ bool leaf_phase(const LeafTasks& tk, const float4* __restrict__ tris, uint32_t lane,
                                           uint32_t fa, uint32_t ca, uint32_t fb, uint32_t cb, V3 o, const RayShear& rs,
                                           float tmin, float tmax, uint32_t prim0, uint32_t inst0,
                                           uint32_t cur, bool& better, unsigned long long& kf, TraceOut& stats,
                                           uint32_t* touch_tris) {
  const uint32_t n_tasks = ca + cb;  // at most 14
  uint32_t off = 0, total = 0;       // exclusive prefix and sum of n_tasks over the wave
  for (uint32_t bit = 0; bit < 4; ++bit) {
    const uint64_t m = __ballot((n_tasks >> bit) & 1u);
    off += prefix_count(m) << bit;
    total += static_cast<uint32_t>(__popcll(m)) << bit;
  }
  better = false;
  kf = 0;
  if (total == 0) return true;
  // one window of kTaskWin tasks per round: lanes whose tasks do not fit keep their
  // leaves for the next round (the first lane with tasks always fits)
  const bool fits = off + n_tasks <= kTaskWin;
  const uint64_t late = __ballot(!fits);
  const uint32_t m = late != 0 ? __shfl(off, static_cast<int>(__builtin_ctzll(late))) : total;
  // TWO: every hit up to tmax is a candidate, the owner's order is checked per hit
  const unsigned long long key0 = hit_key(tmax, TWO ? kNoHit : prim0);
  tk.key[lane] = key0;
  // triangle of place j: j + ta below ea, j + tb from there on
  const uint32_t ea = off + ca, ta = fa - off, tb = fb - ea;
  const bool owns = fits && n_tasks != 0;
  uint32_t last = 0;  // owner mark of the last place dealt out
  for (uint32_t s0 = 0; s0 < m; s0 += 64) {
    tk.mark[lane] = lane == 0 ? last : 0u;
    if (owns && off - s0 < 64u) tk.mark[off - s0] = lane + 1u;
    asm volatile("" ::: "memory");  // another lane may have marked this place
    const uint32_t mark = wave_scan_max(tk.mark[lane]);
    last = __builtin_amdgcn_readlane(mark, 63);
    const int own = static_cast<int>(mark) - 1;
    const uint32_t j = s0 + lane;
    const bool act = j < m;
    const uint32_t oea = __shfl(ea, own), ota = __shfl(ta, own), otb = __shfl(tb, own);
    const uint32_t ti = j + (j < oea ? ota : otb);
    RayTri ort;
    ort.o = v3(__shfl(o.x, own), __shfl(o.y, own), __shfl(o.z, own));
    const int kk = __shfl(rs.kxyz, own);
    ort.kx = kk & 3;
    ort.ky = (kk >> 2) & 3;
    ort.kz = kk >> 4;
    ort.sx = __shfl(rs.s.x, own);
    ort.sy = __shfl(rs.s.y, own);
    ort.sz = __shfl(rs.s.z, own);
    const float otmin = __shfl(tmin, own), otmax = __shfl(tmax, own);
    uint32_t oprim = 0, oinst = 0, ocur = 0;
    if (TWO) {
      oprim = __shfl(prim0, own);
      oinst = __shfl(inst0, own);
      ocur = __shfl(cur, own);
    }
    if (act) {
      const float4* tp = tris + static_cast<size_t>(ti) * 3u;
      const float4 a = tp[0], b = tp[1], cc = tp[2];
      if (STATS) {
        stats.tests++;
        touch(touch_tris, ti);
      }
      TriHit th;
      const uint32_t prim = __float_as_uint(a.w);
      if (intersect_triangle(ort, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), v3(cc.x, cc.y, cc.z), otmin, otmax, th) &&
          (!TWO || th.t < otmax || ocur < oinst || (ocur == oinst && prim < oprim))) {
        const unsigned long long key = hit_key(th.t, prim);
        atomicMin(&tk.key[own], key);
        if (tk.key[own] == key) tk.bary[own] = make_float2(th.b1, th.b2);
      }
    }
  }
  if (fits && n_tasks != 0) {
    kf = tk.key[lane];
    better = kf < key0;
  }
  return fits;
}

template <class Nodes, bool ANY, bool STATS, class Load, class Finish>
__device__ __forceinline__ void trace_queue(const DevAccel& acc, const SegIn& in, uint32_t* stk, uint32_t* tsk,
                                            uint32_t* overflow, TraceOut& stats, Load load, Finish finish) {
  const uint32_t lane = lane_id();
  const uint32_t n_seg = seg_counts(in), home = block_home();
  const int cap = acc.stack_cap;
  const void* __restrict__ nodes = acc.nodes;
  const float4* __restrict__ tris = acc.tris;
  uint64_t seg_done = seg_empty(n_seg, home, gridDim.x >= kSegs);
  bool drained = false;
  uint32_t slot = kNoHit;
  typename Nodes::Ray rb{};
  float tmin = 0.f;
  RayShear rs{};
  TraceOut r;
  r.t = 0.f;
  r.b1 = r.b2 = 0.f;
  r.prim = kNoHit;
  r.inst = kNoInstance;
  TwoTierStack st;
  st.ring = lds_address(stk);
  st.spill_wave = wave_spill(acc.spill, cap);
  st.cap = static_cast<uint32_t>(cap);
  stack_reset(st);
  int32_t node = kTravDone, leaf = 0;
  const auto on_full = [&] { atomicOr(overflow, 1u); };
  const LeafTasks tk = leaf_tasks(tsk);
  for (;;) {
    const uint64_t idle = __ballot(slot == kNoHit);
    const uint32_t n_idle = mask_count(idle);
    if (!drained && n_idle >= kRefill) {
      uint32_t base = 0, got = 0;
      if (seg_fetch_k(in, n_seg, home, seg_done, n_idle, base, got)) {
        const uint32_t rank = prefix_count(idle);
        if (slot == kNoHit && rank < got) {
          slot = base + rank;
          V3 o, d;
          float tmax;
          load(slot, o, d, tmin, tmax);
          rs = ray_shear(d);
          rb = Nodes::setup(acc.space, o, d);
          r.t = tmax;
          r.prim = kNoHit;
          r.inst = kNoInstance;
          stack_reset(st);
          node = 0;
          leaf = 0;
        }
      } else {
        drained = true;
      }
    }
    if (!__any(slot != kNoHit)) break;  // drained and every lane idle
    // Inner nodes: a wave-uniform loop in which lanes without an inner node idle, and one
    // straight line of predicated steps instead of a branch per outcome (both children,
    // one, none, a leaf to park), each of which some lane takes on almost every iteration:
    // the loop is bound by the instructions it issues. A popped leaf is parked by the next
    // iteration (whose box test that lane wastes on the root) rather than by a second pop.
    for (uint64_t walk = __ballot(node >= 0);;) {
      if (lane_bit(walk)) {
        const uint64_t inner = __ballot(node >= 0);  // the others hold a popped leaf
        const int32_t top = stack_top(st);
        const NodeHits v = Nodes::visit(nodes, max(node, 0), rb, tmin, r.t);
        if (STATS && node >= 0) {
          stats.nodes++;
          touch(acc.touch_nodes, static_cast<uint32_t>(node) / Nodes::kBytes);
        }
        const uint64_t h0 = __ballot(v.n0 <= v.f0) | ~inner, h1 = __ballot(v.n1 <= v.f1) & inner;
        const int32_t c0 = lane_bit(inner) ? v.c0 : node;
        const uint64_t both = h0 & h1, first1 = (both & __ballot(v.n1 < v.n0)) | ~h0;
        const int32_t nearc = lane_bit(first1) ? v.c1 : c0, farc = lane_bit(first1) ? c0 : v.c1;
        const uint64_t park = (h0 | h1) & __ballot(nearc < 0) & __ballot(leaf == 0);
        stack_above(st, farc);
        leaf = lane_bit(park) ? nearc : leaf;
        const uint64_t pop = ~(h0 | h1) | (park & ~both);
        node = lane_bit(park) ? farc : nearc;
        node = lane_bit(pop) ? top : node;
        stack_step<STATS>(st, both & ~park, pop, stats, on_full);
      }
      // the loop ends (for the whole wave) once no lane walks, or at most
      // kSearchBreakSpread of those that walked hold no parked leaf
      const uint64_t no_leaf = __ballot(leaf == 0), searching = walk & no_leaf;
      walk = __ballot(node >= 0) | (no_leaf & __ballot(node != kTravDone));
      if (walk == 0 || mask_count(searching) <= kSearchBreakSpread) break;
    }
    // leaves (the parked one, and `node` when it is a leaf), spread over the wave
    bool hit = false;
    const bool node_leaf = node < 0 && node != kTravDone;
    const uint32_t ca = leaf != 0 ? (~static_cast<uint32_t>(leaf) & 7u) : 0u;
    const uint32_t cb = node_leaf ? (~static_cast<uint32_t>(node) & 7u) : 0u;
    bool better;
    unsigned long long kf;
    if (leaf_phase<STATS, false>(tk, tris, lane, ~static_cast<uint32_t>(leaf) >> 3, ca, ~static_cast<uint32_t>(node) >> 3,
                                 cb, rb.o, rs, tmin, r.t, r.prim, kNoInstance, kNoInstance, better, kf,
                                 stats, acc.touch_tris) &&
        (leaf != 0 || node_leaf)) {  // not ca + cb != 0: an empty child's leaf holds no triangle
      if (better) {  // the barycentrics stay in tk.bary[lane] until the ray finishes
        r.t = key_t(kf);
        r.prim = static_cast<uint32_t>(kf);
        hit = ANY;
      }
      leaf = 0;
      if (node_leaf) {
        node = stack_top(st);
        stack_step<STATS>(st, 0ull, ~0ull, stats, on_full);
      }
    }
    if (slot != kNoHit && (hit || (node == kTravDone && leaf == 0))) {
      r.b1 = r.b2 = 0.f;
      if (r.prim != kNoHit) {
        const float2 bb = tk.bary[lane];
        r.b1 = bb.x;
        r.b2 = bb.y;
      }
      finish(slot, r, hit || r.prim != kNoHit);
      slot = kNoHit;
      node = kTravDone;
      leaf = 0;
    }
  }
}

// Two-level counterpart of trace_queue (instanced scenes): the same loop with lane refill,
// two-tier stack and wave-wide leaf phase, walking the top-level tree over instance boxes
// and, inside an instance, its mesh's tree with the ray in object space (leaf tasks use the
// owner's object-space ray). A third phase of each round changes spaces: a lane that meets a
// top-level leaf, or the marker pushed on entering an instance, waits for the round's end,
// and all of those then leave and enter instances together (a transform and a ray set-up of
// some 150 instructions, which inside the node loop ran for a lane or two at almost every
// iteration). A lane with a parked leaf never leaves its instance: the leaf is tested in
// that instance's space, before this phase.
constexpr int32_t kTravExit = static_cast<int32_t>(0x80000001u);  // leave the instance (stack marker); below every leaf code

template <class Nodes, bool ANY, bool STATS, class Load, class Finish>
__device__ __forceinline__ void trace_queue2(const DevAccel& acc, const SegIn& in, uint32_t* stk, uint32_t* tsk,
                                             uint32_t* overflow, TraceOut& stats, Load load, Finish finish) {
  const uint32_t lane = lane_id();
  const uint32_t n_seg = seg_counts(in), home = wave_home();
  const int cap = acc.stack_cap;
  const void* __restrict__ blas = acc.nodes;
  const void* __restrict__ tlas = acc.tlas;
  const float4* __restrict__ tris = acc.tris;
  uint64_t seg_done = seg_empty(n_seg);
  bool drained = false;
  uint32_t slot = kNoHit;
  V3 ow = v3(0.f), dw = v3(0.f);
  typename Nodes::Ray rb{};  // in the current space (world outside instances)
  RayShear rs{};  // in the current instance
  float tmin = 0.f;
  TraceOut r;
  r.t = 0.f;
  r.b1 = r.b2 = 0.f;
  r.prim = kNoHit;
  r.inst = kNoInstance;
  uint32_t cur_id = kNoInstance;
  bool in_blas = false;
  TwoTierStack st;
  st.ring = lds_address(stk);
  st.spill_wave = wave_spill(acc.spill, cap);
  st.cap = static_cast<uint32_t>(cap);
  stack_reset(st);
  int32_t node = kTravDone, leaf = 0;
  const auto on_full = [&] { atomicOr(overflow, 1u); };
  const LeafTasks tk = leaf_tasks(tsk);
  for (;;) {
    const uint64_t idle = __ballot(slot == kNoHit);
    const uint32_t n_idle = mask_count(idle);
    if (!drained && n_idle >= kRefill) {
      uint32_t base = 0, got = 0;
      if (seg_fetch_k(in, n_seg, home, seg_done, n_idle, base, got)) {
        const uint32_t rank = prefix_count(idle);
        if (slot == kNoHit && rank < got) {
          slot = base + rank;
          float tmax;
          load(slot, ow, dw, tmin, tmax);
          rb = Nodes::setup(grid_of(acc.space.org, acc.space.step[0]), ow, dw);
          in_blas = false;
          r.t = tmax;
          r.prim = kNoHit;
          r.inst = kNoInstance;
          stack_reset(st);
          node = 0;
          leaf = 0;
        }
      } else {
        drained = true;
      }
    }
    if (!__any(slot != kNoHit)) break;
    // inner nodes of either level, as in trace_queue; only mesh leaves are parked
    const uint64_t meshes = __ballot(in_blas);
    for (uint64_t walk = __ballot(node >= 0);;) {
      if (lane_bit(walk)) {
        const uint64_t inner = __ballot(node >= 0);  // the others hold a popped mesh leaf
        const int32_t top = stack_top(st);
        const NodeHits v = Nodes::visit(in_blas ? blas : tlas, max(node, 0), rb, tmin, r.t);
        if (STATS && node >= 0) {
          stats.nodes++;
          if (in_blas) touch(acc.touch_nodes, static_cast<uint32_t>(node) / Nodes::kBytes);
        }
        const uint64_t h0 = __ballot(v.n0 <= v.f0) | ~inner, h1 = __ballot(v.n1 <= v.f1) & inner;
        const int32_t c0 = lane_bit(inner) ? v.c0 : node;
        const uint64_t both = h0 & h1, first1 = (both & __ballot(v.n1 < v.n0)) | ~h0;
        const int32_t nearc = lane_bit(first1) ? v.c1 : c0, farc = lane_bit(first1) ? c0 : v.c1;
        const uint64_t park = (h0 | h1) & __ballot(nearc < 0) & __ballot(leaf == 0) & meshes;
        stack_above(st, farc);
        leaf = lane_bit(park) ? nearc : leaf;
        const uint64_t pop = ~(h0 | h1) | (park & ~both);
        node = lane_bit(park) ? farc : nearc;
        node = lane_bit(pop) ? top : node;
        stack_step<STATS>(st, both & ~park, pop, stats, on_full);
      }
      const uint64_t no_leaf = __ballot(leaf == 0), searching = walk & no_leaf;
      walk = __ballot(node >= 0) | (no_leaf & meshes & __ballot(node > kTravExit));
      if (walk == 0 || mask_count(searching) <= kSearchBreakSpread) break;
    }
    // mesh leaves (the parked one, and `node` when it is one; both in the current
    // instance), spread over the wave. Task hits that beat the ray's best under the
    // (t, inst, prim) order compete; the phase's (t, prim) minimum of those becomes the best.
    bool hit = false;
    const bool node_leaf = in_blas && node < 0 && node > kTravExit;
    const uint32_t ca = leaf != 0 ? (~static_cast<uint32_t>(leaf) & 7u) : 0u;
    const uint32_t cb = node_leaf ? (~static_cast<uint32_t>(node) & 7u) : 0u;
    bool better;
    unsigned long long kf;
    if (leaf_phase<STATS, true>(tk, tris, lane, ~static_cast<uint32_t>(leaf) >> 3, ca, ~static_cast<uint32_t>(node) >> 3,
                                cb, rb.o, rs, tmin, r.t, r.prim, r.inst, cur_id, better, kf, stats,
                                acc.touch_tris) &&
        (leaf != 0 || node_leaf)) {
      if (better) {  // the barycentrics stay in tk.bary[lane] until the ray finishes
        r.t = key_t(kf);
        r.prim = static_cast<uint32_t>(kf);
        r.inst = cur_id;
        hit = ANY;
      }
      leaf = 0;
      if (node_leaf) {
        node = stack_top(st);
        stack_step<STATS>(st, 0ull, ~0ull, stats, on_full);
      }
    }
    // change of space: leave the instance at its marker, then enter the next one at a
    // top-level leaf (the rest of the leaf and the marker go on the stack)
    const bool leaves = leaf == 0 && node == kTravExit;
    if (leaves) {
      in_blas = false;
      node = stack_top(st);
      stack_step<STATS>(st, 0ull, ~0ull, stats, on_full);
    }
    const bool enters = !in_blas && node < 0 && node > kTravExit;
    if (leaves || enters) {
      V3 o = ow, d = dw;
      NodeGrid space = grid_of(acc.space.org, acc.space.step[0]);
      if (enters) {
        const uint32_t c = ~static_cast<uint32_t>(node);
        const uint32_t first = c >> 3, cnt = c & 7u;
        if (cnt > 1u) {
          stack_above(st, static_cast<int32_t>(~(((first + 1u) << 3) | (cnt - 1u))));
          stack_step<STATS>(st, ~0ull, 0ull, stats, on_full);
        }
        stack_above(st, kTravExit);
        stack_step<STATS>(st, ~0ull, 0ull, stats, on_full);
        const TlasInstance& ins = acc.inst[first];
        o = xform_point(ins.w2o, ow);
        d = xform_vector(ins.w2o, dw);
        space = grid_of(ins.org, ins.step);
        rs = ray_shear(d);
        cur_id = ins.id;
        in_blas = true;
        node = static_cast<int32_t>(ins.blas_root);
        if (STATS) stats.nodes++;
      }
      rb = Nodes::setup(space, o, d);
    }
    if (slot != kNoHit && (hit || (node == kTravDone && leaf == 0))) {
      r.b1 = r.b2 = 0.f;
      if (r.prim != kNoHit) {
        const float2 bb = tk.bary[lane];
        r.b1 = bb.x;
        r.b2 = bb.y;
      }
      finish(slot, r, hit || r.prim != kNoHit);
      slot = kNoHit;
      node = kTravDone;
      leaf = 0;
    }
  }
}

// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_zero_counters(uint32_t* ctr) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < static_cast<uint32_t>(kNumCounters)) ctr[i] = 0u;
}

// A frame's counters before their first use, by RayGen's threads: the plain words and one
// word per segment line, but for the primary queue's, which primary_counts writes.
__device__ __forceinline__ void reset_counters(uint32_t* ctr) {
  constexpr uint32_t kWords = kCtrSegBase + (kNumCounters - kCtrSegBase) / kLine;
  constexpr uint32_t kPrimary = seg_ctr(kSegExt, 0);
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < kWords; i += gridDim.x * kBlock) {
    const uint32_t w = i < static_cast<uint32_t>(kCtrSegBase) ? i : kCtrSegBase + (i - kCtrSegBase) * kLine;
    if (w < kPrimary || w >= kPrimary + kSegs * kLine) ctr[w] = 0u;
  }
}

// The plain counter words as the host reads them after a frame, with the totals per depth of
// the extension and shadow queues, into (pinned host) memory. One block.
__device__ __forceinline__ void report_counters(const uint32_t* ctr, uint32_t cap, uint32_t* out) {
  static_assert(kCtrSegBase == kBlock && kCtrExt == 0 && kCtrShadow == kMaxDepth, "a word per thread");
  const uint32_t t = threadIdx.x;
  uint32_t v = ctr[t];
  if (t < 2u * kMaxDepth) {
    const uint32_t* c = ctr + seg_ctr(t < kMaxDepth ? kSegExt : kSegShadow, static_cast<int>(t % kMaxDepth));
    v = 0u;
    for (uint32_t sgm = 0; sgm < kSegs; ++sgm) {
      const uint32_t n = c[sgm * kLine];
      v += n < cap ? n : cap;
    }
  }
  out[t] = v;
}
__global__ __launch_bounds__(kBlock) void k_report_counters(const uint32_t* ctr, uint32_t cap, uint32_t* out) {
  report_counters(ctr, cap, out);
}

// Device to pinned host memory, both 16-byte aligned. Bound by the host link, which few waves
// fill: 32, 64 and 128 blocks bring a 33 MB image over in the same time.
constexpr uint32_t kCopyBlocks = 64;
__global__ __launch_bounds__(kBlock) void k_copy_out(const uint4* __restrict__ src, uint4* __restrict__ dst, uint32_t bytes) {
  const uint32_t n = bytes / 16;
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) dst[i] = src[i];
  const uint32_t t = n * 16 + threadIdx.x;
  if (blockIdx.x == 0 && t < bytes) reinterpret_cast<uint8_t*>(dst)[t] = reinterpret_cast<const uint8_t*>(src)[t];
}

// Distinct items a launch read: set bits of its touch bitmap, which is cleared for the
// next launch.
__global__ __launch_bounds__(kBlock) void k_touch_count(uint32_t* bits, uint32_t words, unsigned long long* out) {
  uint32_t n = 0;
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < words; i += gridDim.x * kBlock) {
    n += static_cast<uint32_t>(__popc(bits[i]));
    bits[i] = 0u;
  }
  wave_add_stat(out, n);
}

// Primary-ray slot of path p: segment p / per, in order (no atomics).
__device__ __forceinline__ uint32_t primary_slot(uint32_t p, uint32_t per, uint32_t cap) {
  return (p / per) * cap + p % per;
}

// Writes the primary-queue counts (one lane per segment).
__device__ __forceinline__ void primary_counts(uint32_t n_paths, uint32_t per, uint32_t* cnt) {
  if (blockIdx.x == 0 && threadIdx.x < kSegs) {
    const uint32_t lo = threadIdx.x * per;
    cnt[threadIdx.x * kLine] = n_paths > lo ? (n_paths - lo < per ? n_paths - lo : per) : 0u;
  }
}

// Stores a primary ray; a camera sample with zero weight is stored with tmax = -1, so
// the traversal rejects it at the root and Shade skips it.
__device__ __forceinline__ void store_primary(const RayQueue& q, uint32_t s, uint32_t p, const PathState& ps,
                                              bool alive, float eps) {
  q.o_tmin[s] = make_float4(ps.o.x, ps.o.y, ps.o.z, eps);
  q.d_tmax[s] = make_float4(ps.d.x, ps.d.y, ps.d.z, alive ? 1e30f : -1.f);
  q.t_pdf[s] = make_float4(ps.T.x, ps.T.y, ps.T.z, ps.pdf);
  q.meta[s] = (p << 2) | ps.flags;
}

// Path whose primary ray RayGen thread t writes to slot t's place in the queue: the
// frame's paths sample by sample, each sample's pixels in 8x8 tiles (row-major tiles over
// the largest region with sides a multiple of 8, then the remaining bottom rows and right
// columns row by row; a bijection on [0, W*H)), so that the 64 rays of a fetched batch
// are a square of neighbouring pixels rather than 64 pixels of a row: the lanes of a wave
// share more nodes on every load. Results are per path, whatever the queue order.
__device__ __forceinline__ uint32_t tiled_path(uint32_t t, uint32_t W, uint32_t H) {
  const uint32_t npix = W * H;
  const uint32_t smp = t / npix, j = t - smp * npix;
  const uint32_t W8 = W & ~7u, H8 = H & ~7u, core = W8 * H8;
  uint32_t x, y;
  if (j < core) {
    const uint32_t tile = j >> 6, k = j & 63u, tiles_x = W8 >> 3;
    x = (tile % tiles_x) * 8u + (k & 7u);
    y = (tile / tiles_x) * 8u + (k >> 3);
  } else {
    uint32_t r = j - core;
    const uint32_t bottom = (H - H8) * W;
    if (r < bottom) {
      y = H8 + r / W;
      x = r % W;
    } else {  // reached only when W8 < W
      r -= bottom;
      const uint32_t wr = W - W8;
      y = r / wr;
      x = W8 + r % wr;
    }
  }
  return smp * npix + y * W + x;
}

__global__ __launch_bounds__(kBlock) void k_raygen(RenderParams rp, uint32_t n_paths, uint32_t per, uint32_t cap,
                                                    RayQueue q, FrameBuffers fb, uint32_t* ctr) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  reset_counters(ctr);
  primary_counts(n_paths, per, ctr + seg_ctr(kSegExt, 0));
  if (t < n_paths) {
    const uint32_t p = tiled_path(t, rp.width, rp.height);
    PathState ps;
    const bool alive = raygen(rp, p, ps);
    fb.radiance[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!alive) {  // Shade never sees this path: its first-hit AOVs are zero
      fb.path_aov_a[p] = make_float4(0.f, 0.f, 0.f, 0.f);
      fb.path_aov_n[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    store_primary(q, primary_slot(t, per, cap), p, ps, alive, rp.eps);
  }
}


// The calling wave's stack ring (this lane's first slot) and leaf-task area in the
// traversal kernels' dynamic LDS: the block's rings, then its task areas.
__device__ __forceinline__ uint32_t* wave_ring(uint32_t* lds) {
  return lds + (threadIdx.x >> 6) * kRingEntries * 64 + lane_id();
}
__device__ __forceinline__ uint32_t* wave_tasks(uint32_t* lds) {
  return lds + kWavesPerBlock * kRingEntries * 64 + (threadIdx.x >> 6) * kTaskWords;
}

// A ray from its (origin, tmin) and (direction, tmax) records.
struct RayLoad {
  const float4* o_tmin;
  const float4* d_tmax;
  uint32_t stride;
  __device__ __forceinline__ void operator()(uint32_t slot, V3& o, V3& d, float& tmin, float& tmax) const {
    const float4 a = o_tmin[static_cast<size_t>(slot) * stride];
    const float4 b = d_tmax[static_cast<size_t>(slot) * stride];
    o = v3(a.x, a.y, a.z);
    d = v3(b.x, b.y, b.z);
    tmin = a.w;
    tmax = b.w;
  }
};

// A bounce's emission list into the path radiance, before the block's share of the bounce's
// shadow rays: a path ends where it emits, so no path of the list has a shadow ray of this
// bounce, and the radiance of every path is summed in vertex order. The blocks of a grid
// deal the segments out; the next entry is read while the last one is added. A launch of
// its own had waited, on the second stream, for CUs that Extend of the next bounce already
// filled (37 us a bounce of a 256 x 256 x 16 frame). With the counters reset in RayGen and
// reported by Finalize, six launches and a copy fewer: 0.517 -> 0.484 ms a 640 x 360 frame
// of four bounces, 0.80 -> 0.77 ms a 256 x 256 x 16 one.
__device__ __forceinline__ void add_emission(const float4* __restrict__ emit, const uint32_t* __restrict__ cnt,
                                             uint32_t cap, float4* radiance) {
  for (uint32_t sgm = blockIdx.x % kSegs; sgm < kSegs; sgm += gridDim.x) {
    const uint32_t c = cnt[sgm * kLine];
    const uint32_t n = c < cap ? c : cap;
    const uint32_t first = segment_place(blockIdx.x, kSegs) * kBlock, step = segment_blocks(sgm, gridDim.x, kSegs) * kBlock;
    const float4* seg = emit + static_cast<size_t>(sgm) * cap;
    uint32_t i = first + threadIdx.x;
    float4 e = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < n) e = seg[i];
    while (i < n) {
      const float4 cur = e;
      i += step;
      if (i < n) e = seg[i];
      const uint32_t path = __float_as_uint(cur.w);
      float4 L = radiance[path];
      L.x += cur.x;
      L.y += cur.y;
      L.z += cur.z;
      radiance[path] = L;
    }
  }
}

// Single-level scenes: Extend and Shadow through trace_queue, held to 72 VGPRs (two spilled,
// 12 bytes of scratch, with 32-byte nodes), 7 waves per SIMD. They are bound by throughput, not latency (the texture data path is 91 % busy and
// VALU issue above its 4-cycle rate): 6 and 5 waves measured 11.98 and 12.01 ms a soup
// frame against 11.82.
template <class Nodes, bool STATS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_extend_sl(DevAccel acc, RayQueue q, HitBuf h, SegIn in, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  st.nodes = 0;
  st.tests = 0;
  st.spills = 0;
  trace_queue<Nodes, false, STATS>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st,
      RayLoad{q.o_tmin, q.d_tmax, q.stride},
      [&](uint32_t slot, const TraceOut& r, bool) {
        h.thit[slot] = make_float4(r.t, r.b1, r.b2, __uint_as_float(r.prim));
      });
  if (STATS) {
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 0]), st.nodes);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 2]), st.tests);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 8]), st.spills);
  }
}

template <class Nodes, bool STATS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_shadow_sl(DevAccel acc, ShadowQueue sq, float4* radiance, SegIn in,
                                                       const uint32_t* emit_cnt, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  add_emission(sq.emit, emit_cnt, in.cap, radiance);
  TraceOut st;
  st.nodes = 0;
  st.tests = 0;
  st.spills = 0;
  trace_queue<Nodes, true, STATS>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st,
      RayLoad{sq.o_tmin, sq.d_tmax, 1u},
      [&](uint32_t slot, const TraceOut&, bool occluded) {
        if (!occluded) {
          const float4 c = sq.contrib[slot];
          const uint32_t path = __float_as_uint(c.w);
          float4 L = radiance[path];
          L.x += c.x;
          L.y += c.y;
          L.z += c.z;
          radiance[path] = L;
        }
      });
  if (STATS) {
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 4]), st.nodes);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 6]), st.tests);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 10]), st.spills);
  }
}

// Two-level scenes: Extend and Shadow through trace_queue2, at 92 to 96 VGPRs, 5 waves per SIMD:
// 11.8 ms per 4K frame of 1000 instances on 32-byte nodes, against 12.5 at 6 waves and 13.2 at 7
// (spilled registers) and 11.9 at 4. On 48-byte nodes, 1280x720x4: 1000 spheres 2.71 ms, 2.91 at
// 6 waves, 2.72 at 4; 300 on a ground plane 4.87, 5.13, 4.87.
template <class Nodes, bool STATS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_extend_tl(DevAccel acc, RayQueue q, HitBuf h, SegIn in, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  st.nodes = 0;
  st.tests = 0;
  st.spills = 0;
  trace_queue2<Nodes, false, STATS>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st,
      RayLoad{q.o_tmin, q.d_tmax, q.stride},
      [&](uint32_t slot, const TraceOut& r, bool) {
        h.thit[slot] = make_float4(r.t, r.b1, r.b2, __uint_as_float(r.prim));
        h.inst[slot] = r.inst;
      });
  if (STATS) {
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 0]), st.nodes);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 2]), st.tests);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 8]), st.spills);
  }
}

template <class Nodes, bool STATS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_shadow_tl(DevAccel acc, ShadowQueue sq, float4* radiance, SegIn in,
                                                       const uint32_t* emit_cnt, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  add_emission(sq.emit, emit_cnt, in.cap, radiance);
  TraceOut st;
  st.nodes = 0;
  st.tests = 0;
  st.spills = 0;
  trace_queue2<Nodes, true, STATS>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st,
      RayLoad{sq.o_tmin, sq.d_tmax, 1u},
      [&](uint32_t slot, const TraceOut&, bool occluded) {
        if (!occluded) {
          const float4 c = sq.contrib[slot];
          const uint32_t path = __float_as_uint(c.w);
          float4 L = radiance[path];
          L.x += c.x;
          L.y += c.y;
          L.z += c.z;
          radiance[path] = L;
        }
      });
  if (STATS) {
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 4]), st.nodes);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 6]), st.tests);
    wave_add_stat(reinterpret_cast<unsigned long long*>(&ctr[kCtrStats + 10]), st.spills);
  }
}


// Any-hit ray queries: one byte per ray.
template <class Nodes>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_occluded_sl(
    DevAccel acc, RayQueue q, uint8_t* occluded, SegIn in, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  trace_queue<Nodes, true, false>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st, RayLoad{q.o_tmin, q.d_tmax, q.stride},
      [&](uint32_t slot, const TraceOut&, bool hit) { occluded[slot] = hit ? 1 : 0; });
}

template <class Nodes>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_occluded_tl(
    DevAccel acc, RayQueue q, uint8_t* occluded, SegIn in, uint32_t* ctr) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  trace_queue2<Nodes, true, false>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st, RayLoad{q.o_tmin, q.d_tmax, q.stride},
      [&](uint32_t slot, const TraceOut&, bool hit) { occluded[slot] = hit ? 1 : 0; });
}

// A caller's ray records as a depth-0 queue: checks them (origin and direction finite,
// bounds not NaN, tmin not negative: the traversal's box tests are conservative for those),
// gives an invalid ray an empty interval and reports the first. The counters the query uses
// are reset first: by the block itself when it is the only one, else by k_ray_reset.
__device__ __forceinline__ void ray_reset(uint32_t t, uint32_t n, uint32_t per, uint32_t* ctr) {
  if (t < kSegs) {
    const uint64_t first = static_cast<uint64_t>(t) * per;
    ctr[seg_ctr(kSegExt, 0) + t * kLine] = first >= n ? 0u : (n - first < per ? static_cast<uint32_t>(n - first) : per);
    ctr[seg_ctr(kSegWorkExt, 0) + t * kLine] = 0u;
  }
  if (t == kSegs) {
    ctr[kCtrOverflow] = 0u;
    ctr[kCtrBadRay] = ctr[kCtrBadRay + 1] = 0xffffffffu;
  }
}
__global__ __launch_bounds__(64) void k_ray_reset(uint32_t n, uint32_t per, uint32_t* ctr) {
  ray_reset(threadIdx.x, n, per, ctr);
}
__global__ __launch_bounds__(kBlock) void k_ray_check(const float4* src, float4* rec, uint32_t n, uint32_t per, uint32_t* ctr) {
  if (gridDim.x == 1) {
    ray_reset(threadIdx.x, n, per, ctr);
    __syncthreads();
  }
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
    const float4 a = src[2 * i];
    float4 b = src[2 * i + 1];
    const float inf = __builtin_huge_valf();
    const bool finite = __builtin_fabsf(a.x) < inf && __builtin_fabsf(a.y) < inf && __builtin_fabsf(a.z) < inf &&
                        __builtin_fabsf(b.x) < inf && __builtin_fabsf(b.y) < inf && __builtin_fabsf(b.z) < inf &&
                        a.w == a.w && b.w == b.w;
    const bool bad = !finite || !(a.w >= 0.f);
    if (bad) {
      atomicMin(reinterpret_cast<unsigned long long*>(ctr + kCtrBadRay), 2ull * i + (finite ? 1ull : 0ull));
      b = make_float4(0.f, 0.f, 1.f, -1.f);
    }
    if (src != rec || bad) {
      rec[2 * i] = bad ? make_float4(0.f, 0.f, 0.f, 0.f) : a;
      rec[2 * i + 1] = b;
    }
  }
}

// Per-wave LDS list of Shade's pending work: queue slots whose ray needs shading, with
// the ray's (direction, tmax) and hit records already read when the slot was fetched.
constexpr uint32_t kShadeList = 128;
struct ShadeList {
  uint32_t slot[kShadeList];
  float4 dir[kShadeList];
  float4 hit[kShadeList];
};

// DEBUG: the render modes of render_modes.h instead of the path-tracing step.
// Slots are fetched 64 at a time; a ray that left the scene adds nothing when the sky
// is off (path tracing), so only the slots that hit are listed (a miss at depth 0 still
// writes its pixel's zero albedo and normal), and the wave shades 64 listed slots at a
// time: in the 1M soup 18% of the rays miss (35% at the second bounce), lanes that the
// per-slot loop left idle through the whole shading step. Held to 3 waves per SIMD (150
// VGPRs with one material set; the allocator could otherwise take more than 170, 2 waves;
// 4 waves spill 20 bytes per lane and measured 1% slower).
// SEP: the material-set mode of shade_impl (0, 1 or 2), fixed per launch from
// RenderParams::separate_sampling.
template <bool DEBUG, int SEP>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_shade(SceneView sv, const Material* sampling_mats, RenderParams rp,
                                                   RayQueue q, HitBuf h, RayQueue qn, ShadowQueue sq,
                                                   FrameBuffers fb, SegIn in, uint32_t* next_cnt,
                                                   uint32_t* shadow_cnt, uint32_t* emit_cnt, uint32_t* ctr,
                                                   uint32_t depth, uint32_t two_level,
                                                   const SkyParams* __restrict__ sky) {
  // sv.sky again, as a restrict kernel argument: nothing the kernel writes can alias it, so
  // its fields are read with scalar loads where they are used
  sv.sky = sky;
  __builtin_assume(sv.tri_rec != nullptr && sv.alias != nullptr);
  __shared__ ShadeList lists[kWavesPerBlock];
  ShadeList& L = lists[threadIdx.x >> 6];
  const uint32_t lane = lane_id();
  const uint32_t npix = rp.width * rp.height;
  const uint32_t n_seg = seg_counts(in), home = block_home();
  const bool keep_misses = DEBUG || sv.sky->enabled != 0u;
  uint64_t done = seg_empty(n_seg, home, gridDim.x >= kSegs);
  uint32_t pend = 0;  // listed slots (wave-uniform)
  bool more = true;
  for (;;) {
    while (more && pend < 64u) {
      uint32_t slot0, n_valid;
      more = seg_fetch(in, n_seg, home, done, slot0, n_valid);
      if (!more) break;
      const uint32_t slot = slot0 + lane;
      float4 b = make_float4(0.f, 0.f, 0.f, -1.f), hh = make_float4(0.f, 0.f, 0.f, 0.f);
      if (lane < n_valid) {
        b = q.d_tmax[slot];
        hh = h.thit[slot];
      }
      // a dead primary ray has tmax < 0 and is skipped
      const bool live = b.w >= 0.f;
      const bool work = live && (keep_misses || __float_as_uint(hh.w) != kNoHit);
      if (live && !work && depth == 0) {
        const uint32_t path = q.meta[slot] >> 2;
        fb.path_aov_a[path] = make_float4(0.f, 0.f, 0.f, 0.f);
        fb.path_aov_n[path] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      const uint64_t m = __ballot(work);
      if (work) {
        const uint32_t k = pend + prefix_count(m);
        L.slot[k] = slot;
        L.dir[k] = b;
        L.hit[k] = hh;
      }
      pend += static_cast<uint32_t>(__popcll(m));
    }
    if (pend == 0u) break;  // drained
    const uint32_t take = pend < 64u ? pend : 64u;
    ShadeOut out;
    out.has_ext = 0;
    out.has_shadow = 0;
    uint32_t path = 0;
    bool emits = false;
    if (lane < take) {
      const uint32_t slot = L.slot[lane];
      const float4 a = q.o_tmin[slot];
      const float4 b = L.dir[lane];
      const float4 tp = q.t_pdf[slot];
      const uint32_t meta = q.meta[slot];
      const float4 hh = L.hit[lane];
      const uint32_t hinst = two_level ? h.inst[slot] : kNoInstance;
      PathState ps;
      ps.o = v3(a.x, a.y, a.z);
      ps.d = v3(b.x, b.y, b.z);
      ps.T = v3(tp.x, tp.y, tp.z);
      ps.pdf = tp.w;
      ps.flags = meta & 3u;
      ps.path = meta >> 2;
      path = ps.path;
      Hit hit;
      hit.t = hh.x;
      hit.b1 = hh.y;
      hit.b2 = hh.z;
      hit.prim = __float_as_uint(hh.w);
      hit.inst = hinst;
      if (DEBUG) shade_debug(sv, rp, ps, hit, depth, out);
      else shade<SEP>(sv, sampling_mats, rp, ps, hit, depth, out);
      emits = !is_black(out.L);
      if (depth == 0) {
        fb.path_aov_a[path] = make_float4(out.albedo.x, out.albedo.y, out.albedo.z, out.vdepth);
        fb.path_aov_n[path] = make_float4(out.normal.x, out.normal.y, out.normal.z, 0.f);
      }
    }
    // emission (emitter hits, the sky) to the emission list: the path radiance belongs to
    // the previous bounce's shadow launch, which may still run
    const uint64_t mL = __ballot(emits);
    if (mL != 0ull) {
      const uint32_t sl = seg_append(emit_cnt, in.cap, home, mL, &ctr[kCtrOverflow]);
      if (emits && sl != kNoHit) sq.emit[sl] = make_float4(out.L.x, out.L.y, out.L.z, __uint_as_float(path));
    }
    // move the unprocessed tail (at most 63 slots, all at or above `take`) to the front
    if (take == 64u && lane + 64u < pend) {
      L.slot[lane] = L.slot[lane + 64u];
      L.dir[lane] = L.dir[lane + 64u];
      L.hit[lane] = L.hit[lane + 64u];
    }
    pend -= take;
    const bool ext = out.has_ext != 0;
    const bool shw = out.has_shadow != 0;
    const uint64_t me = __ballot(ext);
    const uint64_t ms = __ballot(shw);
    const uint32_t se = seg_append(next_cnt, in.cap, home, me, &ctr[kCtrOverflow]);
    const uint32_t ss = seg_append(shadow_cnt, in.cap, home, ms, &ctr[kCtrOverflow]);
    if (ext && se != kNoHit) {
      const uint32_t s = se;
      qn.o_tmin[s] = make_float4(out.next.o.x, out.next.o.y, out.next.o.z, rp.eps);
      qn.d_tmax[s] = make_float4(out.next.d.x, out.next.d.y, out.next.d.z, 1e30f);
      qn.t_pdf[s] = make_float4(out.next.T.x, out.next.T.y, out.next.T.z, out.next.pdf);
      qn.meta[s] = (path << 2) | out.next.flags;
    }
    if (shw && ss != kNoHit) {
      const uint32_t s = ss;
      sq.o_tmin[s] = make_float4(out.s_o.x, out.s_o.y, out.s_o.z, rp.eps);
      sq.d_tmax[s] = make_float4(out.s_d.x, out.s_d.y, out.s_d.z, out.s_tmax);
      sq.contrib[s] = make_float4(out.s_contrib.x, out.s_contrib.y, out.s_contrib.z, __uint_as_float(path));
    }
  }
}

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// Per pixel, in sample order: the frame's radiance into the accumulator (mean colour),
// and its first-hit AOVs into their sums (means over the accumulated samples: the
// denoiser's guide images, anti-aliased like the colour).
// The grid's last block reports the frame's counters instead.
__global__ __launch_bounds__(kBlock) void k_finalize(RenderParams rp, const float4* radiance, FrameBuffers fb,
                                                      uint32_t reset, uint32_t aov_reset, uint32_t aov_count,
                                                      const uint32_t* ctr, uint32_t cap, uint32_t* report) {
  if (blockIdx.x == gridDim.x - 1) {
    report_counters(ctr, cap, report);
    return;
  }
  const uint32_t pix = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t npix = rp.width * rp.height;
  if (pix >= npix) return;
  float sx = 0.f, sy = 0.f, sz = 0.f;
  float4 sa = make_float4(0.f, 0.f, 0.f, 0.f), sn = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t s = 0; s < rp.spp; ++s) {
    const size_t i = static_cast<size_t>(s) * npix + pix;
    const float4 L = radiance[i];
    sx += L.x;
    sy += L.y;
    sz += L.z;
    sa = add4(sa, fb.path_aov_a[i]);
    sn = add4(sn, fb.path_aov_n[i]);
  }
  float4 acc = reset ? make_float4(0.f, 0.f, 0.f, 0.f) : fb.accum[pix];
  acc.x += sx;
  acc.y += sy;
  acc.z += sz;
  acc.w += static_cast<float>(rp.spp);
  fb.accum[pix] = acc;
  const float inv = acc.w > 0.f ? 1.f / acc.w : 0.f;
  fb.color[pix] = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, 1.f);
  if (!aov_reset) {
    sa = add4(fb.aov_sum_a[pix], sa);
    sn = add4(fb.aov_sum_n[pix], sn);
  }
  fb.aov_sum_a[pix] = sa;
  fb.aov_sum_n[pix] = sn;
  const float ia = 1.f / static_cast<float>(aov_count);
  fb.albedo[pix] = make_float4(sa.x * ia, sa.y * ia, sa.z * ia, 1.f);
  fb.normal[pix] = make_float4(sn.x * ia, sn.y * ia, sn.z * ia, sa.w * ia);
}

__global__ __launch_bounds__(kBlock) void k_tonemap(const float4* src, uint32_t n, TonemapParams tp,
                                                     uchar4* dst) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 c = src[i];
  dst[i] = make_uchar4(static_cast<unsigned char>(tonemap_u8(tp, c.x)), static_cast<unsigned char>(tonemap_u8(tp, c.y)),
                       static_cast<unsigned char>(tonemap_u8(tp, c.z)), 255);
}

// ------------------------------------------------------------------------------------
// Adjoint (path-replay backpropagation). Gradient records live in fixed slots
// r = depth * paths + path, so their values never depend on queue order; the reduction
// below sums them in slot order.
__global__ __launch_bounds__(kBlock) void k_raygen_adj(RenderParams rp, uint32_t n_paths, uint32_t per, uint32_t cap,
                                                        RayQueue q, AdjBuffers ab, uint32_t* ctr) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  reset_counters(ctr);
  primary_counts(n_paths, per, ctr + seg_ctr(kSegExt, 0));
  if (t < n_paths) {
    const uint32_t p = tiled_path(t, rp.width, rp.height);
    PathState ps;
    const bool alive = raygen(rp, p, ps);
    for (uint32_t d = 0; d < ab.depth; ++d) ab.rec_key[static_cast<size_t>(d) * ab.n_paths + p] = kNoHit;
    store_primary(q, primary_slot(t, per, cap), p, ps, alive, rp.eps);
  }
}


// The adjoint's Shade. Held to 168 VGPRs, 3 waves per SIMD (2 waves: 4 % slower step). VALU
// issue fills four fifths of its time, gathers by path (records, remaining radiance, pending
// derivatives: ~250 bytes a vertex) the rest: 1.29 ms a bounce of 512 x 512 x 64 paths, 1.40
// before a vertex's derivatives shared their terms and came as twelve numbers of fifteen.
template <int SEP>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_shade_adj(SceneView sv, const Material* sampling_mats, RenderParams rp,
                                                       RayQueue q, HitBuf h, RayQueue qn, ShadowQueue sq,
                                                       AdjBuffers ab, SegIn in, uint32_t* next_cnt,
                                                       uint32_t* shadow_cnt, uint32_t* ctr, uint32_t depth,
                                                       uint32_t two_level, const SkyParams* __restrict__ sky) {
  sv.sky = sky;  // scalar loads of the sky's fields, as in k_shade
  __builtin_assume(sv.tri_rec != nullptr && sv.alias != nullptr);
  const uint32_t lane = lane_id();
  const uint32_t npix = rp.width * rp.height;
  const float inv_spp = 1.f / static_cast<float>(rp.spp);
  const uint32_t n_seg = seg_counts(in), home = wave_home();
  uint64_t done = seg_empty(n_seg);
  uint32_t slot0, n_valid;
  while (seg_fetch(in, n_seg, home, done, slot0, n_valid)) {
    const uint32_t slot = slot0 + lane;
    ShadeOut out;
    AdjOut adj;
    out.has_ext = 0;
    out.has_shadow = 0;
    uint32_t path = 0;
    const float4 b = lane < n_valid ? q.d_tmax[slot] : make_float4(0.f, 0.f, 0.f, -1.f);
    if (b.w >= 0.f) {
      const float4 a = q.o_tmin[slot];
      const float4 tp = q.t_pdf[slot];
      const uint32_t meta = q.meta[slot];
      const float4 hh = h.thit[slot];
      PathState ps;
      ps.o = v3(a.x, a.y, a.z);
      ps.d = v3(b.x, b.y, b.z);
      ps.T = v3(tp.x, tp.y, tp.z);
      ps.pdf = tp.w;
      ps.flags = meta & 3u;
      ps.path = meta >> 2;
      path = ps.path;
      const uint32_t pix = path % npix;
      const V3 delta = v3(ab.dldi[pix * 3 + 0] * inv_spp, ab.dldi[pix * 3 + 1] * inv_spp, ab.dldi[pix * 3 + 2] * inv_spp);
      float4 lr = depth > 0 ? ab.lrem[path] : ab.radiance[path];
      // continuation gradient of the previous vertex (which had a record and sent this
      // ray on): the radiance still unaccounted for arrived through its sampled direction
      if (depth > 0) {
        const size_t np = ab.n_paths, r = static_cast<size_t>(depth - 1) * np + path;
        const uint32_t key = ab.rec_key[r];
        float4 a4 = ab.rec_a[r];
        float a1 = ab.rec_b[r];
        const float4 c = ab.contrib[path];
        const float4* pp = ab.pend + path;
        const float4 p0 = pp[0], p1 = pp[np], p2 = pp[2 * np];
        if (key & kRecUnlit) {  // no light reached it: the record holds nothing yet
          ab.rec_key[r] = key ^ kRecUnlit;
          a4 = make_float4(0.f, 0.f, 0.f, 0.f);
          a1 = 0.f;
        } else {
          lr.x -= c.x;
          lr.y -= c.y;
          lr.z -= c.z;
        }
        const BsdfGrad prev = {{p0.x, p0.y, p0.z}, {p0.w, p1.x, p1.y}, {p1.z, p1.w, p2.x}, {p2.y, p2.z, p2.w}};
        float g[kNumParams];
        continuation_grad(prev, delta, v3(lr.x, lr.y, lr.z), g);
        ab.rec_a[r] = make_float4(a4.x + g[0], a4.y + g[1], a4.z + g[2], a4.w + g[3]);
        ab.rec_b[r] = a1 + g[4];
      }
      Hit hit;
      hit.t = hh.x;
      hit.b1 = hh.y;
      hit.b2 = hh.z;
      hit.prim = __float_as_uint(hh.w);
      hit.inst = two_level ? h.inst[slot] : kNoInstance;
      shade_adjoint<SEP, 2>(sv, sampling_mats, rp, ps, hit, depth, delta, out, adj);
      if (adj.mat != kNoHit) {
        const size_t r = static_cast<size_t>(depth) * ab.n_paths + path;
        ab.rec_key[r] = out.has_shadow ? adj.mat : adj.mat | kRecUnlit;
        if (out.has_shadow) {  // as if light arrives; an occluded shadow ray marks the key
          ab.rec_a[r] = make_float4(adj.nee_g[0], adj.nee_g[1], adj.nee_g[2], adj.nee_g[3]);
          ab.rec_b[r] = adj.nee_g[4];
        }
      }
      if (out.has_ext) {  // (a path that emits here ends: nothing is left of its radiance)
        ab.lrem[path] = lr;
        if (out.has_shadow) ab.contrib[path] = make_float4(out.s_contrib.x, out.s_contrib.y, out.s_contrib.z, 0.f);
        float4* pp = ab.pend + path;
        const size_t np = ab.n_paths;
        const BsdfGrad& e = adj.rel;
        pp[0] = make_float4(e.own[0], e.own[1], e.own[2], e.tint[0]);
        pp[np] = make_float4(e.tint[1], e.tint[2], e.rough[0], e.rough[1]);
        pp[2 * np] = make_float4(e.rough[2], e.metal[0], e.metal[1], e.metal[2]);
      }
    }
    const bool ext = out.has_ext != 0;
    const bool shw = out.has_shadow != 0;
    const uint64_t me = __ballot(ext);
    const uint64_t ms = __ballot(shw);
    const uint32_t se = seg_append(next_cnt, in.cap, home, me, &ctr[kCtrOverflow]);
    const uint32_t ss = seg_append(shadow_cnt, in.cap, home, ms, &ctr[kCtrOverflow]);
    if (ext && se != kNoHit) {
      const uint32_t s = se;
      qn.o_tmin[s] = make_float4(out.next.o.x, out.next.o.y, out.next.o.z, rp.eps);
      qn.d_tmax[s] = make_float4(out.next.d.x, out.next.d.y, out.next.d.z, 1e30f);
      qn.t_pdf[s] = make_float4(out.next.T.x, out.next.T.y, out.next.T.z, out.next.pdf);
      qn.meta[s] = (path << 2) | out.next.flags;
    }
    if (shw && ss != kNoHit) {
      const uint32_t s = ss;
      sq.o_tmin[s] = make_float4(out.s_o.x, out.s_o.y, out.s_o.z, rp.eps);
      sq.d_tmax[s] = make_float4(out.s_d.x, out.s_d.y, out.s_d.z, out.s_tmax);
      ab.s_path[s] = path;
    }
  }
}

// Shadow rays of the adjoint, through the render's own traversal. Shade has written the
// vertex's record as if light arrives; an occluded ray marks its key, and the next vertex's
// Shade and the reduction go by that. (Records written and the path's radiance updated here,
// by whichever lanes had just finished, held the whole wave at their loads: 1.05 ms a bounce
// of 512 x 512 x 64 paths beside Extend, now 0.84.)
__device__ __forceinline__ void finish_shadow_adj(const AdjBuffers& ab, uint32_t depth, uint32_t slot, bool occluded) {
  if (occluded) atomicOr(&ab.rec_key[static_cast<size_t>(depth) * ab.n_paths + ab.s_path[slot]], kRecUnlit);
}

template <class Nodes>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_shadow_adj_sl(
    DevAccel acc, ShadowQueue sq, AdjBuffers ab, SegIn in, uint32_t* ctr, uint32_t depth) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  trace_queue<Nodes, true, false>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st, RayLoad{sq.o_tmin, sq.d_tmax, 1u},
      [&](uint32_t slot, const TraceOut&, bool occluded) { finish_shadow_adj(ab, depth, slot, occluded); });
}

template <class Nodes>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_shadow_adj_tl(
    DevAccel acc, ShadowQueue sq, AdjBuffers ab, SegIn in, uint32_t* ctr, uint32_t depth) {
  extern __shared__ uint32_t lds[];
  TraceOut st;
  trace_queue2<Nodes, true, false>(
      acc, in, wave_ring(lds), wave_tasks(lds), &ctr[kCtrOverflow], st, RayLoad{sq.o_tmin, sq.d_tmax, 1u},
      [&](uint32_t slot, const TraceOut&, bool occluded) { finish_shadow_adj(ab, depth, slot, occluded); });
}

// Deterministic reduction of records into per-material gradients, materials
// [mat_lo, mat_lo + n_mat). Block b owns records [b R/B, (b+1) R/B); each of its waves
// a contiguous quarter, 64 records at a time, one per lane: lanes whose records have the
// same material are linked in lane order (a ballot per bit of the key finds them), the
// chains are summed by pointer jumping, and each chain's first lane adds its sum to the
// wave's private LDS accumulator, every material by one lane; then the block adds its
// four accumulators in wave order. The order of the additions is fixed and no float
// atomics are used: results are bitwise reproducible. Bound by reading the records (24 B
// each); adding them one by one, five lanes at a time, took 4.0 ms for the 67 M records of
// 512 x 512 x 64 spp at depth 4.
__global__ __launch_bounds__(kBlock) void k_grad_reduce(const uint32_t* __restrict__ rec_key,
                                                         const float4* __restrict__ rec_a,
                                                         const float* __restrict__ rec_b, uint64_t R, uint32_t mat_lo,
                                                         uint32_t n_mat, uint32_t key_bits, float* partial) {
  extern __shared__ float acc_lds[];
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  const uint32_t P = n_mat * kNumParams;
  float* acc = acc_lds + wave * P;
  for (uint32_t i = lane; i < P; i += 64) acc[i] = 0.f;
  const uint64_t b0 = R * blockIdx.x / gridDim.x, b1 = R * (blockIdx.x + 1) / gridDim.x;
  const uint64_t w0 = b0 + (b1 - b0) * wave / kWavesPerBlock, w1 = b0 + (b1 - b0) * (wave + 1) / kWavesPerBlock;
  const uint64_t above = lane == 63 ? 0ull : ~0ull << (lane + 1);
  for (uint64_t base = w0; base < w1; base += 64) {
    const uint64_t r = base + lane;
    const uint32_t key = r < w1 ? rec_key[r] - mat_lo : kNoHit;  // kNoHit - mat_lo stays out of range
    const bool in = key < n_mat;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    float b = 0.f;
    if (in) {
      a = rec_a[r];
      b = rec_b[r];
    }
    uint64_t same = __ballot(in);  // lanes with this lane's key
    if (same == 0ull) continue;
    for (uint32_t bit = 0; bit < key_bits; ++bit) {
      const bool one = (key >> bit) & 1u;
      const uint64_t m = __ballot(one);
      same &= one ? m : ~m;
    }
    const bool head = in && prefix_count(same) == 0u;
    int next = in && (same & above) != 0ull ? static_cast<int>(__builtin_ctzll(same & above)) : -1;
    while (__any(next >= 0)) {
      const int j = next >= 0 ? next : static_cast<int>(lane);
      const float ax = __shfl(a.x, j), ay = __shfl(a.y, j), az = __shfl(a.z, j), aw = __shfl(a.w, j), bb = __shfl(b, j);
      const int nn = __shfl(next, j);
      if (next >= 0) {
        a.x += ax;
        a.y += ay;
        a.z += az;
        a.w += aw;
        b += bb;
        next = nn;
      }
    }
    if (head) {
      float* t = acc + key * kNumParams;
      t[0] += a.x;
      t[1] += a.y;
      t[2] += a.z;
      t[3] += a.w;
      t[4] += b;
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < P; i += kBlock) {
    float t = acc_lds[i];
    for (int w = 1; w < kWavesPerBlock; ++w) t += acc_lds[w * P + i];
    partial[static_cast<size_t>(blockIdx.x) * P + i] = t;
  }
}

// Sum of the blocks' partial gradients, in a fixed order: a block takes 16 parameters,
// sixteen threads each (thread t of a parameter the partials t, t + 16, ..., so that 16
// neighbouring parameters are read together), then adds the sixteen sums pairwise. A thread's
// loads go sixteen at a time (one after the other: 21 us for 512 materials; now 6).
__global__ __launch_bounds__(kBlock) void k_grad_final(const float* __restrict__ partial, uint32_t n_blocks, uint32_t P,
                                                        float* out) {
  __shared__ float sum[kBlock];
  const uint32_t i = blockIdx.x * 16u + (threadIdx.x & 15u), part = threadIdx.x >> 4;
  float t = 0.f;
  for (uint32_t b0 = 0; b0 < n_blocks; b0 += 256u) {
    float v[16];
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) {
      const uint32_t b = b0 + part + 16u * k;
      v[k] = i < P && b < n_blocks ? partial[static_cast<size_t>(b) * P + i] : 0.f;
    }
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) t += v[k];
  }
  sum[threadIdx.x] = t;
  for (uint32_t s = 128u; s >= 16u; s >>= 1) {
    __syncthreads();
    if (threadIdx.x < s) sum[threadIdx.x] += sum[threadIdx.x + s];
  }
  if (threadIdx.x < 16u && i < P) out[i] = sum[threadIdx.x];
}

size_t ring_lds_bytes() { return static_cast<size_t>(kRingEntries) * 64u * 4u * kWavesPerBlock; }
// queue traversals: rings, then each wave's leaf-task area
size_t trace_lds_bytes() { return ring_lds_bytes() + static_cast<size_t>(kTaskWords) * 4u * kWavesPerBlock; }

}  // namespace

// Calls f with the node layout of an acceleration structure.
template <class F>
auto with_nodes(const DevAccel& acc, F f) {
  return acc.node_bytes == Nodes32::kBytes ? f(Nodes32{}) : f(Nodes48{});
}

int trace_blocks_per_cu(const DevAccel& acc) {
  return with_nodes(acc, [&](auto nodes) {
    using N = decltype(nodes);
    int a = 0, b = 0;
    hipError_t ea, eb;
    if (acc.two_level) {
      ea = hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, k_extend_tl<N, false>, kBlock, trace_lds_bytes());
      eb = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_shadow_tl<N, false>, kBlock, trace_lds_bytes());
    } else {
      ea = hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, k_extend_sl<N, false>, kBlock, trace_lds_bytes());
      eb = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_shadow_sl<N, false>, kBlock, trace_lds_bytes());
    }
    if (ea != hipSuccess) a = 4;
    if (eb != hipSuccess) b = 4;
    const int m = a < b ? a : b;
    return m > 0 ? m : 1;
  });
}

// The queue traversals address their LDS rings as 4 KiB-aligned blocks from LDS
// address 0: they must have no static LDS, which would move dynamic LDS up.
template <class N>
static bool no_static_lds() {
  const void* ks[] = {reinterpret_cast<const void*>(k_extend_sl<N, false>), reinterpret_cast<const void*>(k_extend_sl<N, true>),
                      reinterpret_cast<const void*>(k_shadow_sl<N, false>), reinterpret_cast<const void*>(k_shadow_sl<N, true>),
                      reinterpret_cast<const void*>(k_extend_tl<N, false>), reinterpret_cast<const void*>(k_extend_tl<N, true>),
                      reinterpret_cast<const void*>(k_shadow_tl<N, false>), reinterpret_cast<const void*>(k_shadow_tl<N, true>),
                      reinterpret_cast<const void*>(k_shadow_adj_sl<N>), reinterpret_cast<const void*>(k_shadow_adj_tl<N>),
                      reinterpret_cast<const void*>(k_occluded_sl<N>), reinterpret_cast<const void*>(k_occluded_tl<N>)};
  for (const void* k : ks) {
    hipFuncAttributes a{};
    if (hipFuncGetAttributes(&a, k) != hipSuccess || a.sharedSizeBytes != 0) return false;
  }
  return true;
}

bool traversal_lds_check() { return no_static_lds<Nodes32>() && no_static_lds<Nodes48>(); }

void launch_zero_counters(uint32_t* ctr, hipStream_t stream) {
  hipLaunchKernelGGL(k_zero_counters, dim3((kNumCounters + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, ctr);
}

void launch_copy_out(const void* src, void* dst, uint32_t bytes, hipStream_t stream) {
  const uint32_t blocks = std::min<uint32_t>((bytes / 16 + kBlock - 1) / kBlock, kCopyBlocks);
  hipLaunchKernelGGL(k_copy_out, dim3(blocks ? blocks : 1), dim3(kBlock), 0, stream, static_cast<const uint4*>(src),
                     static_cast<uint4*>(dst), bytes);
}

void launch_tonemap(const float4* src, uint32_t n, const TonemapParams& tp, uchar4* dst, hipStream_t stream) {
  hipLaunchKernelGGL(k_tonemap, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, src, n, tp, dst);
}

void launch_report_counters(const uint32_t* ctr, uint32_t cap, uint32_t* report, hipStream_t stream) {
  hipLaunchKernelGGL(k_report_counters, dim3(1), dim3(kBlock), 0, stream, ctr, cap, report);
}

void launch_touch_count(uint32_t* bits, uint32_t words, unsigned long long* out, hipStream_t stream) {
  const uint32_t blocks = (words + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_touch_count, dim3(blocks < 1024 ? (blocks ? blocks : 1) : 1024), dim3(kBlock), 0, stream, bits,
                     words, out);
}

void launch_raygen(const RenderParams& rp, uint32_t n_paths, uint32_t cap, RayQueue q, const FrameBuffers& fb,
                   uint32_t* ctr, hipStream_t stream) {
  const uint32_t blocks = (n_paths + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_raygen, dim3(blocks), dim3(kBlock), 0, stream, rp, n_paths, prim_per_seg(n_paths), cap, q,
                     fb, ctr);
}

void launch_extend(const DevAccel& acc, RayQueue q, HitBuf h, SegIn in, uint32_t* ctr, int grid, bool stats,
                   hipStream_t stream) {
  with_nodes(acc, [&](auto nodes) {
    using N = decltype(nodes);
    const auto k = acc.two_level ? (stats ? k_extend_tl<N, true> : k_extend_tl<N, false>)
                                 : (stats ? k_extend_sl<N, true> : k_extend_sl<N, false>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), trace_lds_bytes(), stream, acc, q, h, in, ctr);
  });
}

void launch_ray_queue(const float4* src, float4* rec, uint32_t n, uint32_t per, uint32_t* ctr, hipStream_t stream) {
  // one block takes up to four rays a thread (one launch less: 8 us of a query of 64 rays);
  // beyond that a block per 256 rays, up to a grid that covers the device several times
  const uint32_t blocks = n <= 4 * kBlock ? 1u : std::min<uint32_t>((n + 0ull + kBlock - 1) / kBlock, 1u << 16);
  if (blocks > 1) hipLaunchKernelGGL(k_ray_reset, dim3(1), dim3(64), 0, stream, n, per, ctr);
  hipLaunchKernelGGL(k_ray_check, dim3(blocks), dim3(kBlock), 0, stream, src, rec, n, per, ctr);
}

void launch_occluded(const DevAccel& acc, RayQueue q, uint8_t* occluded, SegIn in, uint32_t* ctr, int grid,
                     hipStream_t stream) {
  with_nodes(acc, [&](auto nodes) {
    using N = decltype(nodes);
    const auto k = acc.two_level ? k_occluded_tl<N> : k_occluded_sl<N>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), trace_lds_bytes(), stream, acc, q, occluded, in, ctr);
  });
}

void launch_shade(const SceneView& sv, const Material* sampling_mats, const RenderParams& rp, RayQueue q,
                  HitBuf h, RayQueue qn, ShadowQueue sq, FrameBuffers fb, SegIn in, uint32_t* next_cnt,
                  uint32_t* shadow_cnt, uint32_t* emit_cnt, uint32_t* ctr, uint32_t depth, int grid,
                  hipStream_t stream) {
  const auto k = rp.mode != kModePathTracing     ? k_shade<true, -1>
                 : rp.separate_sampling == 0u ? k_shade<false, 0>
                 : rp.separate_sampling == 1u ? k_shade<false, 1>
                                              : k_shade<false, 2>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), 0, stream, sv, sampling_mats, rp, q, h, qn, sq, fb, in, next_cnt,
                     shadow_cnt, emit_cnt, ctr, depth, sv.instances ? 1u : 0u, sv.sky);
}

void launch_shadow(const DevAccel& acc, ShadowQueue sq, float4* radiance, SegIn in, const uint32_t* emit_cnt,
                   uint32_t* ctr, int grid, bool stats, hipStream_t stream) {
  with_nodes(acc, [&](auto nodes) {
    using N = decltype(nodes);
    const auto k = acc.two_level ? (stats ? k_shadow_tl<N, true> : k_shadow_tl<N, false>)
                                 : (stats ? k_shadow_sl<N, true> : k_shadow_sl<N, false>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), trace_lds_bytes(), stream, acc, sq, radiance, in, emit_cnt, ctr);
  });
}

void launch_finalize(const RenderParams& rp, const float4* radiance, FrameBuffers fb, uint32_t reset,
                     uint32_t aov_reset, uint32_t aov_count, const uint32_t* ctr, uint32_t cap, uint32_t* report,
                     hipStream_t stream) {
  const uint32_t npix = rp.width * rp.height;
  hipLaunchKernelGGL(k_finalize, dim3((npix + kBlock - 1) / kBlock + 1), dim3(kBlock), 0, stream, rp, radiance, fb,
                     reset, aov_reset, aov_count, ctr, cap, report);
}


void launch_raygen_adj(const RenderParams& rp, uint32_t n_paths, uint32_t cap, RayQueue q, const AdjBuffers& ab,
                       uint32_t* ctr, hipStream_t stream) {
  const uint32_t blocks = (n_paths + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_raygen_adj, dim3(blocks), dim3(kBlock), 0, stream, rp, n_paths, prim_per_seg(n_paths), cap, q,
                     ab, ctr);
}

void launch_shade_adj(const SceneView& sv, const Material* sampling_mats, const RenderParams& rp, RayQueue q,
                      HitBuf h, RayQueue qn, ShadowQueue sq, const AdjBuffers& ab, SegIn in, uint32_t* next_cnt,
                      uint32_t* shadow_cnt, uint32_t* ctr, uint32_t depth, int grid, hipStream_t stream) {
  const auto k = rp.separate_sampling == 0u ? k_shade_adj<0> : rp.separate_sampling == 1u ? k_shade_adj<1> : k_shade_adj<2>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), 0, stream, sv, sampling_mats, rp, q, h, qn, sq, ab, in, next_cnt,
                     shadow_cnt, ctr, depth, sv.instances ? 1u : 0u, sv.sky);
}

void launch_shadow_adj(const DevAccel& acc, ShadowQueue sq, const AdjBuffers& ab, SegIn in, uint32_t* ctr,
                       uint32_t depth, int grid, hipStream_t stream) {
  with_nodes(acc, [&](auto nodes) {
    using N = decltype(nodes);
    const auto k = acc.two_level ? k_shadow_adj_tl<N> : k_shadow_adj_sl<N>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), trace_lds_bytes(), stream, acc, sq, ab, in, ctr, depth);
  });
}

void launch_grad_reduce(const AdjBuffers& ab, uint32_t mat_lo, uint32_t n_mat, float* partial, float* out,
                        hipStream_t stream) {
  const uint32_t P = n_mat * kNumParams;
  uint32_t key_bits = 0;
  while (key_bits < 32u && (n_mat - 1u) >> key_bits) ++key_bits;
  hipLaunchKernelGGL(k_grad_reduce, dim3(kGradBlocks), dim3(kBlock), P * 4 * kWavesPerBlock, stream, ab.rec_key,
                     ab.rec_a, ab.rec_b, static_cast<uint64_t>(ab.n_records), mat_lo, n_mat, key_bits, partial);
  hipLaunchKernelGGL(k_grad_final, dim3((P + 15) / 16), dim3(kBlock), 0, stream, partial,
                     static_cast<uint32_t>(kGradBlocks), P, out);
}

}  // namespace trt
