// U-Net denoiser kernels for gfx950: BF16 activations/weights, FP32 accumulation on
// MFMA (v_mfma_f32_32x32x16_bf16), NHWC tensors.
//
// Replaces the OptiX AI denoiser the reference invokes (Tracer/Optix/Denoiser.cpp:36-42,
// 101-112; closed vendor code) with a project-trained U-Net.
//
// Convolution = implicit GEMM: M = output pixels, N = output channels, K = 9 taps x Cin.
// MFMA operand layouts (checked on the device): for 32x32x16, lane l holds A row l%32,
// k = 8*(l/32)..+7 and B column l%32, k = 8*(l/32)..+7; accumulator register r holds
// row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#include <hip/hip_runtime.h>

#include "denoiser.h"
#include "dn_limits.h"

namespace trt {
namespace dn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
  // round to nearest even (no NaNs occur here)
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(r >> 16);
}

constexpr int kTileH = 8, kTileW = 16;          // output pixels per workgroup
constexpr int kPatchH = kTileH + 2, kPatchW = kTileW + 2;

// ------------------------------------------------------------------------------------
// 3x3 'same' convolution as an implicit GEMM (M = pixels, N = output channels,
// K = 9 taps x Cin), input and weights staged through LDS per 32-channel chunk.
//
// Input: `x` [N][H][W][cx] bf16, optionally preceded (in channel order) by `coarse`
// [N][H/2][W/2][c1] bf16 read with nearest upsampling, so a decoder convolution reads
// [upsample(coarse) | skip] without materialising the concatenation. Cin = c1 + cx;
// c1, cx multiples of 32, or Cin = 16 without coarse. Weights [Cout][9][Cin] bf16.
//
// Workgroup = 4 waves over a (8 MB) x 16 pixel tile and 32 NB output channels (one
// channel group); wave w owns MB m-blocks of 2 x 16 pixels (rows 2(w MB + m) + 0..1)
// and all NB n-blocks, so every A fragment feeds NB MFMAs and every B fragment MB.
// The next chunk's global loads are issued before the current chunk's MFMAs.
struct ConvArgs {
  const uint16_t* x;
  const uint16_t* coarse;
  int c1, cx;
  const uint16_t* w;
  const float* bias;  // nullable
  void* y;            // bf16 or fp32 [N][H][W][cout]; unused by kEpiRadiance
  int cout;
  uint16_t* pooled;     // kEpiReluPool: 2x2 average of the bf16 output [N][H/2][W/2][cout]
  const uint16_t* feat; // kEpiRadiance: input features [N][H][W][16]
  float4* radiance;     // kEpiRadiance: expm1(max(feat[0..2] + y[0..2], 0)), alpha 1
  int N, H, W;
  int groups;  // cout / (32 NB)
};

typedef unsigned v4u32_t __attribute__((ext_vector_type(4)));
// third dword of a raw buffer resource on gfx9 parts (32-bit data format, no swizzle)
constexpr int kBufFlags = 0x00020000;
constexpr int kOOB = static_cast<int>(kBufOutside);  // buffer offset past every range

// two floats -> packed bf16 (round to nearest even), low half first
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// LDS layouts, in 16-byte slots. A 128-bit LDS read serves each half-wave (32 lanes) at
// once and is conflict-free when their 32 slots are distinct modulo 32. A-fragment
// reads take 16 consecutive patch positions of two consecutive rows: 5 slots per
// position (odd, so 16 positions are distinct mod 32) and a row pitch of 112 slots
// (= 16 mod 32, so the second row fills the other 16 residues). B-fragment reads take
// 32 consecutive output channels 37 slots apart (odd).
constexpr int kPosStride = 40;           // bf16 per staged position (32 + 8 padding)
constexpr int kRowPitch = 112 * 8;       // bf16 per staged patch row (18 positions + padding)
constexpr int kWStride = 9 * 32 + 8;     // bf16 per staged output channel

// LDS of a k_conv workgroup; one spare 16-byte slot at the end of patch and wl takes the
// stores of idle threads.
template <int MB, int NB, int EPI>
struct ConvLds {
  static constexpr int TH = 8 * MB, PH = TH + 2, PW = kTileW + 2;
  static constexpr int OS = 32 * NB + 8;                             // bf16 per pixel in the output staging
  static constexpr int OWAVE = (EPI == kEpiF32 ? 8 : MB * 32 * OS);  // output staging per wave (bf16)
  alignas(16) uint16_t patch[PH * kRowPitch + 8];
  alignas(16) uint16_t wl[32 * NB * kWStride + 8];
  alignas(16) uint16_t ob[4 * OWAVE];
  alignas(16) float bl[32 * NB];
};

// The workgroup `block` of `blocks` (a multiple of 8).
template <int MB, int NB, int EPI, bool SC, bool C16>
__device__ __forceinline__ void conv_block(const ConvArgs& a, unsigned block, unsigned blocks, ConvLds<MB, NB, EPI>& lds) {
  using L = ConvLds<MB, NB, EPI>;
  constexpr int TH = L::TH, PH = L::PH, PW = L::PW, NPOS = PH * PW, OS = L::OS, OWAVE = L::OWAVE;
  constexpr int PLOADS = (NPOS * 4 + 255) / 256;
  constexpr int WLOADS = (32 * NB * 9 * 4 + 255) / 256;
  constexpr int PARTS = 4 * NB;                                   // 16-byte parts per staged pixel
  constexpr int FLUSH = (MB * 32 * PARTS) / 64;                   // 16-byte stores per lane per tile
  uint16_t *const patch = lds.patch, *const wl = lds.wl, *const ob = lds.ob;
  float* const bl = lds.bl;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = a.H, W = a.W, Cin = a.c1 + a.cx, Cout = a.cout;
  constexpr int gs = C16 ? 1 : 2;    // log2 of 16-byte groups per staged position
  constexpr int cc = 8 << gs;        // channels per chunk (Cin = 16 is one 16-channel chunk)
  constexpr int KS = cc / 16;        // MFMA k-steps per tap
  constexpr int NK = 9 * KS;         // MFMA k-steps per chunk
  const int nchunks = Cin / cc;      // 1 when SC (single chunk)
  const int tiles_x = W / kTileW, tiles_y = (H + TH - 1) / TH;
  const int total = tiles_x * tiles_y * a.N * a.groups;
  // Persistent workgroups. Workgroups are dealt round-robin over the 8 XCDs, so XCD
  // x = block % 8 gets one contiguous range of items (neighbouring tiles share
  // their halo rows in that XCD's L2); its workgroups stride through the range by
  // `per`, a multiple of the group count, so one workgroup keeps one channel group.
  // Item order: channel group fastest, then tile column, tile row, image.
  const int per = static_cast<int>(blocks) >> 3, xcd = static_cast<int>(block) & 7;
  const int q = total >> 3, rem = total & 7;
  const int begin = xcd * q + (xcd < rem ? xcd : rem);
  const int end = begin + q + (xcd < rem ? 1 : 0);
  const int first = begin + (static_cast<int>(block) >> 3);
  if (first >= end) return;
  struct Step {
    int it, ch;  // item, input-channel chunk
    int x0, y0, co0, n;
  };
  auto set_item = [&](Step& s, int it) __attribute__((always_inline)) {
    s.it = it;
    it = it < end ? it : end - 1;  // past the end: stage the last item again (discarded)
    const int g = it % a.groups;
    it /= a.groups;
    const int tx = it % tiles_x;
    it /= tiles_x;
    s.x0 = tx * kTileW;
    s.y0 = (it % tiles_y) * TH;
    s.n = it / tiles_y;
    s.co0 = g * 32 * NB;
  };
  auto advance = [&](Step s) __attribute__((always_inline)) {
    if (++s.ch == nchunks) {
      s.ch = 0;
      set_item(s, s.it + per);
    }
    return s;
  };

  f32x16 acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[m][j] = f32x16{};

  // Staging: global -> registers -> LDS, the patch two steps ahead (two register sets),
  // the weights (reloaded per step unless SC) and features one step ahead, through
  // buffer loads: a buffer resource per image, per-thread byte offsets fixed for the
  // kernel (relative to the tile's corner), and out-of-range offsets reading zero (the
  // padding of the 'same' convolution). Every thread issues the same loads on every
  // step and none sits in a branch, so the wait before each LDS store counts exactly
  // the loads issued after it. Idle threads store to the spare slot.
  int pyx[PLOADS];  // patch position: row | column << 8
  uint32_t prel[PLOADS], crel[PLOADS];
  int plds[PLOADS];
  uint32_t pidle = 0;
#pragma unroll
  for (int k = 0; k < PLOADS; ++k) {
    const int i = tid + k * 256;
    const int pos = i >> gs, gi = i & ((1 << gs) - 1), py = pos / PW, px = pos - py * PW;
    const bool ok = i < (NPOS << gs);
    pidle |= (ok ? 1u : 0u) << k;
    pyx[k] = py | (px << 8);
    prel[k] = (static_cast<uint32_t>(py * W + px) * a.cx + gi * 8) * 2;
    crel[k] = static_cast<uint32_t>(((py + 1) >> 1) * (W >> 1) + ((px + 1) >> 1)) * a.c1 * 2 + (gi * 8) * 2;
    plds[k] = ok ? py * kRowPitch + px * kPosStride + gi * 8 : PH * kRowPitch;
  }
  u32x4 prA[PLOADS], prB[PLOADS], wr[WLOADS];
  float br = 0.f;
  uint2 fr_next = make_uint2(0u, 0u), fr_cur = make_uint2(0u, 0u);  // kEpiRadiance features
  const uint32_t img_bytes = static_cast<uint32_t>(H) * W * a.cx * 2;
  const uint32_t cimg_bytes = static_cast<uint32_t>(H >> 1) * (W >> 1) * a.c1 * 2;
  auto load_patch = [&](u32x4(&pr)[PLOADS], const Step& s) __attribute__((always_inline)) {
    const int c0 = s.ch * cc;
    const bool coarse = c0 < a.c1;  // chunk of the nearest-upsampled coarse input
    const uint16_t* base = coarse ? a.coarse + static_cast<size_t>(s.n) * (H >> 1) * (W >> 1) * a.c1 + c0
                                  : a.x + static_cast<size_t>(s.n) * H * W * a.cx + (c0 - a.c1);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(base), static_cast<short>(0), coarse ? cimg_bytes : img_bytes, kBufFlags);
    // byte offset of the patch corner (row y0 - 1, column x0 - 1)
    const uint32_t corner = coarse ? static_cast<uint32_t>(((s.y0 >> 1) - 1) * (W >> 1) + ((s.x0 >> 1) - 1)) * a.c1 * 2
                                   : static_cast<uint32_t>((s.y0 - 1) * W + (s.x0 - 1)) * a.cx * 2;
    const bool interior = __builtin_amdgcn_readfirstlane(
        s.y0 >= 1 && s.y0 + PH - 1 <= H && s.x0 >= 1 && s.x0 + PW - 1 <= W ? 1 : 0);
    uint32_t okm = pidle;  // bit k: load k reads image data (else the zero padding)
    if (!interior) {       // uniform branch; it only narrows the mask
      uint32_t m = 0;
#pragma unroll
      for (int k = 0; k < PLOADS; ++k) {
        const int yy = s.y0 + (pyx[k] & 0xff) - 1, xx = s.x0 + ((pyx[k] >> 8) & 0xff) - 1;
        const bool ok = static_cast<unsigned>(yy) < static_cast<unsigned>(H) &&
                        static_cast<unsigned>(xx) < static_cast<unsigned>(W);
        m |= (ok ? 1u : 0u) << k;
      }
      okm &= m;
    }
#pragma unroll
    for (int k = 0; k < PLOADS; ++k) {
      uint32_t r0 = prel[k], r1 = crel[k];
      asm volatile("" : "+v"(r0), "+v"(r1));  // keep the per-load select a register select
      const int off = (okm >> k) & 1u ? static_cast<int>(corner + (coarse ? r1 : r0)) : kOOB;
      pr[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
  };
  int wrel[WLOADS];
#pragma unroll
  for (int k = 0; k < WLOADS; ++k) {
    const int i = tid + k * 256;
    const int qq = i >> gs, co = qq / 9, tap = qq - co * 9;
    wrel[k] = i < (32 * NB * 9 << gs) ? ((co * 9 + tap) * Cin + (i & ((1 << gs) - 1)) * 8) * 2 : kOOB;
  }
  const uint32_t w_bytes = static_cast<uint32_t>(Cout) * 9 * Cin * 2;
  auto load_weights = [&](const Step& s) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.w), static_cast<short>(0), w_bytes, kBufFlags);
    const int base = (s.co0 * 9 * Cin + s.ch * cc) * 2;
#pragma unroll
    for (int k = 0; k < WLOADS; ++k)
      wr[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, wrel[k] == kOOB ? kOOB : base + wrel[k], 0, 0));
    br = a.bias ? a.bias[s.co0 + (tid & (32 * NB - 1))] : 0.f;
  };
  auto load_feat = [&](const Step& s) __attribute__((always_inline)) {  // kEpiRadiance: features 0..3
    const int pi = lane & 31, yy = s.y0 + 2 * (wave * MB + (lane >> 5) % MB) + (pi >> 4);
    const size_t p = (static_cast<size_t>(s.n) * H + (yy < H ? yy : 0)) * W + s.x0 + (pi & 15);
    fr_next = *reinterpret_cast<const uint2*>(a.feat + p * 16);
  };
  auto store_patch = [&](const u32x4(&pr)[PLOADS]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < PLOADS; ++k) *reinterpret_cast<u32x4*>(patch + plds[k]) = pr[k];
  };
  auto store_weights = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < WLOADS; ++k) {
      const int i = tid + k * 256;
      const int qq = i >> gs, co = qq / 9, tap = qq - co * 9;
      const int o = i < (32 * NB * 9 << gs) ? co * kWStride + tap * 32 + (i & ((1 << gs) - 1)) * 8 : 32 * NB * kWStride;
      *reinterpret_cast<u32x4*>(wl + o) = wr[k];
    }
    if (tid < 32 * NB) bl[tid] = br;
  };
  // Output of a finished tile, staged per wave in LDS by the epilogue ([pixel][channel]
  // bf16) and written one step later with 16-byte buffer stores (rows past the image
  // fall outside the buffer and are dropped), so that the stores are issued before the
  // following loads (one in-order counter tracks both) and never delay the wait for
  // them. The 2x2 pooling reads the staged bf16 values back.
  uint16_t* obw = ob + wave * OWAVE;
  uint32_t orel[FLUSH];
#pragma unroll
  for (int k = 0; k < FLUSH; ++k) {
    const int c = lane + 64 * k, px = c / PARTS, part = c - px * PARTS, pi = px & 31;
    orel[k] = (static_cast<uint32_t>((2 * (wave * MB + (px >> 5)) + (pi >> 4)) * W + (pi & 15)) * Cout + part * 8) * 2;
  }
  const uint32_t out_bytes = static_cast<uint32_t>(H) * W * Cout * 2;
  auto flush = [&](const Step& s) __attribute__((always_inline)) {
    if (EPI == kEpiRadiance) {
      if (lane < 32 * MB) {
        const int pi = lane & 31, yy = s.y0 + 2 * (wave * MB + (lane >> 5)) + (pi >> 4);
        const float4 y = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(obw) + lane * 4);
        if (yy < H) {
          float4 o;
          o.x = expm1f(fmaxf(bf2f(static_cast<uint16_t>(fr_cur.x & 0xffffu)) + y.x, 0.f));
          o.y = expm1f(fmaxf(bf2f(static_cast<uint16_t>(fr_cur.x >> 16)) + y.y, 0.f));
          o.z = expm1f(fmaxf(bf2f(static_cast<uint16_t>(fr_cur.y & 0xffffu)) + y.z, 0.f));
          o.w = 1.f;
          a.radiance[(static_cast<size_t>(s.n) * H + yy) * W + s.x0 + (pi & 15)] = o;
        }
      }
      return;
    }
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        static_cast<uint16_t*>(a.y) + static_cast<size_t>(s.n) * H * W * Cout + s.co0, static_cast<short>(0),
        out_bytes, kBufFlags);
    const uint32_t corner = static_cast<uint32_t>(s.y0 * W + s.x0) * Cout * 2;
#pragma unroll
    for (int k = 0; k < FLUSH; ++k) {
      const int c = lane + 64 * k, px = c / PARTS, part = c - px * PARTS;
      const u32x4 v = *reinterpret_cast<const u32x4*>(obw + px * OS + part * 8);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u32_t, v), rs, static_cast<int>(corner + orel[k]), 0, 0);
    }
    if (EPI == kEpiReluPool) {  // H even: pooled rows are whole
      const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
          a.pooled + static_cast<size_t>(s.n) * (H >> 1) * (W >> 1) * Cout + s.co0, static_cast<short>(0),
          out_bytes >> 2, kBufFlags);
      for (int c = lane; c < MB * 8 * PARTS; c += 64) {
        const int pq = c / PARTS, part = c - pq * PARTS, m = pq >> 3, px = 2 * (pq & 7);
        const int yy = s.y0 + 2 * (wave * MB + m);
        const uint16_t* src = obw + (m * 32 + px) * OS + part * 8;
        const u32x4 v00 = *reinterpret_cast<const u32x4*>(src), v01 = *reinterpret_cast<const u32x4*>(src + OS);
        const u32x4 v10 = *reinterpret_cast<const u32x4*>(src + 16 * OS);
        const u32x4 v11 = *reinterpret_cast<const u32x4*>(src + 17 * OS);
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          // two channels per dword; top pair + bottom pair as in a stand-alone pooling
          const float lo = (__uint_as_float(v00[d] << 16) + __uint_as_float(v01[d] << 16)) +
                           (__uint_as_float(v10[d] << 16) + __uint_as_float(v11[d] << 16));
          const float hi = (__uint_as_float(v00[d] & 0xffff0000u) + __uint_as_float(v01[d] & 0xffff0000u)) +
                           (__uint_as_float(v10[d] & 0xffff0000u) + __uint_as_float(v11[d] & 0xffff0000u));
          o[d] = pack_bf16(0.25f * lo, 0.25f * hi);
        }
        const uint32_t off = (static_cast<uint32_t>((yy >> 1) * (W >> 1) + (s.x0 >> 1) + (px >> 1)) * Cout + part * 8) * 2;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u32_t, o), rp, static_cast<int>(off), 0, 0);
      }
    }
  };

  const int l32 = lane & 31, khalf = (lane >> 5) * 8;
  bool pend = false;
  Step pend_step;
  // one step on the patch staged in `pr`: stage it, write the previous tile, issue the
  // loads of the following steps, then MFMAs and the epilogue of a finished tile
  auto step = [&](u32x4(&pr)[PLOADS], const Step& s0, const Step& s1, const Step& s2, bool valid)
                  __attribute__((always_inline)) {
    __syncthreads();
    store_patch(pr);
    if (!SC) store_weights();
    __syncthreads();
    if (pend) {
      flush(pend_step);
      pend = false;
    }
    if (EPI == kEpiRadiance) fr_cur = fr_next;
    if (!SC) load_weights(s1);
    if (EPI == kEpiRadiance) load_feat(s1);  // single-chunk: step s1 is the next item
    // issue order = wait order: nothing of the next step's loads may move behind these
    __builtin_amdgcn_sched_barrier(0);
    load_patch(pr, s2);
    // MFMA with the weights as A (rows = output channels) and the patch as B (columns =
    // pixels): accumulator register r of lane l then holds pixel l % 32 of the m-block
    // and channel 8 (r / 4) + 4 (l / 32) + r % 4 of the n-block, i.e. four runs of four
    // consecutive channels of one pixel. Fragments are read from LDS two k-steps ahead
    // of the MFMAs that use them (three register sets), so LDS latency overlaps MFMAs.
    bf16x8 af[3][MB], bf[3][NB];
    auto frag = [&](int k, int buf) __attribute__((always_inline)) {
      const int tap = k / KS, ks = (k % KS) * 16, ky = tap / 3, kx = tap % 3;
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int row = 2 * (wave * MB + m) + (l32 >> 4) + ky, col = (l32 & 15) + kx;
        af[buf][m] = *reinterpret_cast<const bf16x8*>(patch + row * kRowPitch + col * kPosStride + ks + khalf);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j)
        bf[buf][j] = *reinterpret_cast<const bf16x8*>(wl + (j * 32 + l32) * kWStride + tap * 32 + ks + khalf);
    };
    frag(0, 0);
    frag(1, 1);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if (k + 2 < NK) frag(k + 2, (k + 2) % 3);
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[k % 3][j], af[k % 3][m], acc[m][j], 0, 0, 0);
    }
    if (valid && s0.ch == nchunks - 1) {
      const int pi = l32, h4 = 4 * (lane >> 5);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int yy = s0.y0 + 2 * (wave * MB + m) + (pi >> 4);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const int col = j * 32 + 8 * qd + h4;  // first of four channels
            const float4 bb = *reinterpret_cast<const float4*>(bl + col);
            float v0 = acc[m][j][4 * qd] + bb.x, v1 = acc[m][j][4 * qd + 1] + bb.y;
            float v2 = acc[m][j][4 * qd + 2] + bb.z, v3 = acc[m][j][4 * qd + 3] + bb.w;
            if (EPI == kEpiRelu || EPI == kEpiReluPool) {
              v0 = fmaxf(v0, 0.f);
              v1 = fmaxf(v1, 0.f);
              v2 = fmaxf(v2, 0.f);
              v3 = fmaxf(v3, 0.f);
            }
            if (EPI == kEpiF32) {
              if (yy < H)
                *reinterpret_cast<float4*>(static_cast<float*>(a.y) +
                                           ((static_cast<size_t>(s0.n) * H + yy) * W + s0.x0 + (pi & 15)) * Cout +
                                           s0.co0 + col) = make_float4(v0, v1, v2, v3);
            } else if (EPI == kEpiRadiance) {
              if (j == 0 && qd == 0 && h4 == 0)
                *reinterpret_cast<float4*>(reinterpret_cast<float*>(obw) + (m * 32 + pi) * 4) =
                    make_float4(v0, v1, v2, v3);
            } else {
              uint2 o;
              o.x = pack_bf16(v0, v1);
              o.y = pack_bf16(v2, v3);
              *reinterpret_cast<uint2*>(obw + (m * 32 + pi) * OS + col) = o;
            }
          }
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[m][j] = f32x16{};
      }
      if (EPI != kEpiF32) {
        pend = true;
        pend_step = s0;
      }
    }
  };

  // step cursors: s0 is computed now, s1 and s2 follow. The loop runs pairs of steps
  // (register sets A, B) with its only exit test at the end; an odd last step is a B
  // step that computes a repeat of the last staged data and discards it.
  const int n_steps = ((end - first + per - 1) / per) * nchunks;
  Step s0;
  s0.ch = 0;
  set_item(s0, first);
  Step s1 = advance(s0), s2 = advance(s1);
  if (SC) {  // weights and bias once
    load_weights(s0);
    __syncthreads();
    store_weights();
  } else {
    load_weights(s0);
  }
  if (EPI == kEpiRadiance) load_feat(s0);
  __builtin_amdgcn_sched_barrier(0);
  load_patch(prA, s0);
  __builtin_amdgcn_sched_barrier(0);
  load_patch(prB, s1);
  for (int k = 0; k < n_steps; k += 2) {
    step(prA, s0, s1, s2, true);
    s0 = s1;
    s1 = s2;
    s2 = advance(s2);
    step(prB, s0, s1, s2, k + 1 < n_steps);
    s0 = s1;
    s1 = s2;
    s2 = advance(s2);
  }
  if (pend) flush(pend_step);
}

template <int MB, int NB, int EPI, bool SC, bool C16>
__global__ __launch_bounds__(256) void k_conv(ConvArgs a) {
  __shared__ ConvLds<MB, NB, EPI> lds;
  conv_block<MB, NB, EPI, SC, C16>(a, blockIdx.x, gridDim.x, lds);
}

// ------------------------------------------------------------------------------------
// Weight gradient: dW[co][tap][ci] = sum_p dZ[p][co] X[p + s(tap)][ci] (X optionally
// [upsample(coarse) | X] as in the forward convolution), as an MFMA GEMM
// with M = co (32-block), N = ci (32-block), K = pixels. Each workgroup covers kWgradTiles
// consecutive 8x16 pixel tiles and writes its partial sums to
// partial[chunk][co][tap][ci]; a fixed-order reduction over chunks follows.
// Blocks: n_chunks x (Cout/32 * ceil(Cin/32)); wave w handles the taps of kernel row w.
//
// The fragments hold eight consecutive pixels of one channel, while the tensors have the
// channels together, so staging transposes: a thread loads 8 channels of four neighbouring
// pixels (16 bytes each), exchanges halves in registers and writes eight 8-byte runs of
// pixels to LDS as [channel][row][pixel]. A wave then reads one aligned run of ten pixels of
// an input row and forms the three horizontally shifted fragments of its kernel row from it
// in registers. The loads of the next kWgAhead tiles are in flight while a tile is
// multiplied: training crops leave at most a block per CU, so a chunk's time is its tiles'
// load latency. (Element by element staging took 220 us a layer on average at 8 x 128 x 128;
// one tile ahead, through loads in branches, 24 us; now 16 us, with two tiles ahead as with
// three.)
constexpr int kWgThreads = 192;
constexpr int kWgAhead = 2;                   // tiles whose loads are in flight
constexpr int kWgRow = 24;                    // LDS pixels per staged input row (18 used)
constexpr int kWgXs = kPatchH * kWgRow + 8;   // bf16 per channel: an odd number of 16-byte slots
constexpr int kWgZs = kTileH * kTileW + 8;
constexpr int kWgXItems = kPatchH * 5 * 4;    // rows x pixel quads x channel octets (dZ: 8 x 4 x 4 = 128)
constexpr int kWgItems = 2;                   // per thread

struct WgradArgs {
  const uint16_t *x, *coarse, *dz;
  float* partial;
  int c1, N, H, W, cin, cout, chunks;
};
struct WgradLds {
  alignas(16) uint16_t xs[32 * kWgXs];  // [ci][row][pixel]
  alignas(16) uint16_t zs[32 * kWgZs];  // [co][row][pixel]
};
__device__ __forceinline__ void wgrad_block(const WgradArgs& a, int chunk, int channels, WgradLds& lds) {
  uint16_t *const xs = lds.xs, *const zs = lds.zs;
  const uint16_t *const X = a.x, *const coarse = a.coarse, *const dZ = a.dz;
  const int c1 = a.c1, N = a.N, H = a.H, W = a.W, Cin = a.cin, Cout = a.cout;
  const int tid = threadIdx.x, lane = tid & 63, ky = tid >> 6;
  const int ci_blocks = (Cin + 31) / 32;
  const int cb = channels / ci_blocks, ib = channels - cb * ci_blocks;
  const int tiles_x = W / kTileW, tiles_y = (H + kTileH - 1) / kTileH;
  const int tiles_img = tiles_x * tiles_y;
  const int first = chunk * kWgradTiles;
  const int last = min(first + kWgradTiles, tiles_img * N);
  const bool up = ib * 32 < c1;  // this input block comes from the upsampled coarse tensor
  const int cx = Cin - c1;
  // Two items per thread (a quad of pixels, an octet of channels): item 0 of the input patch,
  // item 1 of dZ (waves 0 and 1) or the rest of the patch (wave 2). Every thread issues the
  // same eight buffer loads on every tile, padding and idle ones past the buffer's end (they
  // return zero): with loads in branches the wait before a tile's stores could not tell how
  // many later ones are in flight and drained them all.
  int py[kWgItems], px[kWgItems], to[kWgItems];  // first pixel, place in LDS
  uint32_t rel[kWgItems][4];                     // byte offsets from the tile's corner
  const bool z1 = __builtin_amdgcn_readfirstlane(ky) < 2;          // item 1 is one of dZ
  bool have[kWgItems];
#pragma unroll
  for (int k = 0; k < kWgItems; ++k) {
    const bool z = k == 1 && z1;
    const int i = k == 0 || z ? tid : kWgThreads + tid - 128;  // of the patch or of dZ
    const int part = i & 3, g = i >> 2, quads = z ? 4 : 5;
    const int row = g / quads, quad = g - row * quads;
    have[k] = z ? true : i < kWgXItems && ib * 32 + part * 8 < Cin;
    py[k] = z ? row : row - 1;
    px[k] = z ? quad * 4 : quad * 4 - 1;
    to[k] = i < kWgXItems ? part * 8 * (z ? kWgZs : kWgXs) + row * (z ? kTileW : kWgRow) + quad * 4 : -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int y = py[k], x = px[k] + q;
      rel[k][q] = z    ? static_cast<uint32_t>(y * W + x) * Cout * 2 + part * 16
                  : up ? static_cast<uint32_t>((y >> 1) * (W >> 1) + (x >> 1)) * c1 * 2 + part * 16
                       : static_cast<uint32_t>(y * W + x) * cx * 2 + part * 16;
    }
  }
  const uint32_t x_bytes = up ? static_cast<uint32_t>((H >> 1) * (W >> 1)) * c1 * 2 : static_cast<uint32_t>(H * W) * cx * 2;
  const uint32_t z_bytes = static_cast<uint32_t>(H * W) * Cout * 2;
  u32x4 stage[kWgAhead][kWgItems][4];
  auto load_tile = [&](u32x4(&stage)[kWgItems][4], int tile) __attribute__((always_inline)) {
    const int n = tile / tiles_img, tr = tile - n * tiles_img;
    const int ty = tr / tiles_x, y0 = ty * kTileH, x0 = (tr - ty * tiles_x) * kTileW;
    const uint16_t* xb = up ? coarse + static_cast<size_t>(n) * (H >> 1) * (W >> 1) * c1 + ib * 32
                            : X + static_cast<size_t>(n) * H * W * cx + (ib * 32 - c1);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(xb), static_cast<short>(0), x_bytes, kBufFlags);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(dZ) + static_cast<size_t>(n) * H * W * Cout + cb * 32, static_cast<short>(0), z_bytes, kBufFlags);
    const uint32_t xc = up ? static_cast<uint32_t>((y0 >> 1) * (W >> 1) + (x0 >> 1)) * c1 * 2
                           : static_cast<uint32_t>(y0 * W + x0) * cx * 2;
    const uint32_t zc = static_cast<uint32_t>(y0 * W + x0) * Cout * 2;
#pragma unroll
    for (int k = 0; k < kWgItems; ++k) {
      const bool row_ok = have[k] && static_cast<unsigned>(y0 + py[k]) < static_cast<unsigned>(H);
      const uint32_t corner = k == 1 && z1 ? zc : xc;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int x = px[k] + q;
        const bool ok = row_ok && x <= kTileW && static_cast<unsigned>(x0 + x) < static_cast<unsigned>(W);
        const int off = ok ? static_cast<int>(corner + rel[k][q]) : kOOB;
        stage[k][q] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(k == 1 && z1 ? rz : rx, off, 0, 0));
      }
    }
  };
  auto store_tile = [&](const u32x4(&stage)[kWgItems][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kWgItems; ++k) {
      const bool z = k == 1 && z1;
      if (to[k] < 0) continue;
      uint16_t* dst = (z ? zs : xs) + to[k];
      const int pitch = z ? kWgZs : kWgXs;
#pragma unroll
      for (int c = 0; c < 4; ++c) {  // channels 2c, 2c + 1 in the halves of dword c
        uint2 lo, hi;
        lo.x = __builtin_amdgcn_perm(stage[k][1][c], stage[k][0][c], 0x05040100u);
        lo.y = __builtin_amdgcn_perm(stage[k][3][c], stage[k][2][c], 0x05040100u);
        hi.x = __builtin_amdgcn_perm(stage[k][1][c], stage[k][0][c], 0x07060302u);
        hi.y = __builtin_amdgcn_perm(stage[k][3][c], stage[k][2][c], 0x07060302u);
        *reinterpret_cast<uint2*>(dst + (2 * c) * pitch) = lo;
        *reinterpret_cast<uint2*>(dst + (2 * c + 1) * pitch) = hi;
      }
    }
  };
  f32x16 acc[3] = {f32x16{}, f32x16{}, f32x16{}};
  const int khalf = (lane >> 5) * 8;
  const uint16_t* zrow = zs + (lane & 31) * kWgZs + khalf;
  const uint16_t* xrow = xs + (lane & 31) * kWgXs + ky * kWgRow + khalf;
#pragma unroll
  for (int t = 0; t < kWgAhead; ++t)
    if (first + t < last) load_tile(stage[t], first + t);
#pragma unroll
  for (int t = 0; t < kWgradTiles; ++t) {
    if (first + t >= last) break;
    __syncthreads();
    store_tile(stage[t % kWgAhead]);
    __syncthreads();
    if (t + kWgAhead < kWgradTiles && first + t + kWgAhead < last) load_tile(stage[t % kWgAhead], first + t + kWgAhead);
#pragma unroll
    for (int row = 0; row < kTileH; ++row) {  // K-step = 16 pixels of one tile row
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(zrow + row * kTileW);
      const u32x4 x0 = *reinterpret_cast<const u32x4*>(xrow + row * kWgRow);
      const uint32_t x4 = *reinterpret_cast<const uint32_t*>(xrow + row * kWgRow + 8);
      const u32x4 x1 = {__builtin_amdgcn_alignbyte(x0[1], x0[0], 2), __builtin_amdgcn_alignbyte(x0[2], x0[1], 2),
                        __builtin_amdgcn_alignbyte(x0[3], x0[2], 2), __builtin_amdgcn_alignbyte(x4, x0[3], 2)};
      const u32x4 x2 = {x0[1], x0[2], x0[3], x4};
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, x0), acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, x1), acc[1], 0, 0, 0);
      acc[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, x2), acc[2], 0, 0, 0);
    }
  }
  // write partial: rows = co (A rows), cols = ci (B cols)
  const size_t wsize = static_cast<size_t>(Cout) * 9 * Cin;
  float* out = a.partial + chunk * wsize;
  const int ci = ib * 32 + (lane & 31);
  if (ci >= Cin) return;
#pragma unroll
  for (int kx = 0; kx < 3; ++kx)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int co = cb * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      out[(static_cast<size_t>(co) * 9 + ky * 3 + kx) * Cin + ci] = acc[kx][r];
    }
}
__global__ __launch_bounds__(kWgThreads) void k_wgrad(WgradArgs a) {
  __shared__ WgradLds lds;
  wgrad_block(a, blockIdx.x, blockIdx.y, lds);
}

// A layer's input gradient (a convolution of dZ) and its weight gradient in one launch: they
// are independent and, at the sizes of training crops, each is a chain of load latencies
// that leaves most of the chip idle (8 x 128 x 128: 12 and 16 us a layer on average one after
// the other, 20 us together). The last conv_blocks workgroups convolve; the wave that the
// weight gradient has no use for ends. With 32 output channels a group (NB = 1) held to 3 waves
// per SIMD, 157 VGPRs, which two tiles ahead in the weight gradient allow (a step at 8 x 128 x
// 128: 0.79 ms; with three tiles ahead at 2 waves 0.82; convolution first 0.80); with 64 the
// convolution's 55 KB of LDS leave room for 2, of 179 VGPRs and 48 accumulators.
template <int MB, int NB, bool SC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_conv_wgrad(ConvArgs c, unsigned conv_blocks,
                                                                                           WgradArgs w) {
  __shared__ union {
    ConvLds<MB, NB, kEpiF32> conv;
    WgradLds wgrad;
  } lds;
  const unsigned wgrad_blocks = gridDim.x - conv_blocks;
  if (blockIdx.x >= wgrad_blocks) {
    conv_block<MB, NB, kEpiF32, SC, false>(c, blockIdx.x - wgrad_blocks, conv_blocks, lds.conv);
  } else if (threadIdx.x < kWgThreads) {
    const int b = static_cast<int>(blockIdx.x);
    wgrad_block(w, b % w.chunks, b / w.chunks, lds.wgrad);
  }
}

// out[i] = sum over chunks c (in order) of partial[c][i], all loads in flight (one after the
// other they were bound by their latency: 36 us a layer on average at 8 x 128 x 128).
// Up to kReduceDirect chunks a thread adds one output's in registers. Beyond, a block takes
// kReduceOuts outputs: its threads bring 128 chunks at a time into LDS and kReduceOuts of
// them add them in order.
// A layer's two sums share a launch: the first blocks reduce the biases' (256 chunks, the
// longest chain), the others the weights'.
constexpr int kReduceOuts = 32, kReduceChunks = 128, kReduceDirect = 32;
struct ChunkSum {
  const float* partial;
  int n_chunks;
  size_t n;
  float* out;
};
struct LayerSums {
  ChunkSum weights, biases;
  unsigned first, blocks;
};
struct ReduceLds {
  float v[kReduceChunks * kReduceOuts];
};
template <int kThreads>
__device__ __forceinline__ void reduce_block(const LayerSums& sums, unsigned block, ReduceLds& l) {
  float* const lds = l.v;
  const ChunkSum r = block < sums.first ? sums.biases : sums.weights;
  if (block >= sums.first) block -= sums.first;
  if (r.n_chunks <= kReduceDirect) {
    const size_t i = static_cast<size_t>(block) * kThreads + threadIdx.x;
    if (i >= r.n) return;
    float v[kReduceDirect];
#pragma unroll
    for (int c = 0; c < kReduceDirect; ++c) v[c] = c < r.n_chunks ? r.partial[static_cast<size_t>(c) * r.n + i] : 0.f;
    float t = 0.f;
#pragma unroll
    for (int c = 0; c < kReduceDirect; ++c)
      if (c < r.n_chunks) t += v[c];
    r.out[i] = t;
    return;
  }
  constexpr int kParts = kThreads / kReduceOuts, kEach = kReduceChunks / kParts;
  const int o = threadIdx.x & (kReduceOuts - 1), part = threadIdx.x / kReduceOuts;
  const size_t i = static_cast<size_t>(block) * kReduceOuts + o;
  float t = 0.f;
  for (int c0 = 0; c0 < r.n_chunks; c0 += kReduceChunks) {
    const int m = min(kReduceChunks, r.n_chunks - c0);
    float v[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
      const int c = part + kParts * k;
      v[k] = c < m && i < r.n ? r.partial[static_cast<size_t>(c0 + c) * r.n + i] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; ++k) lds[(part + kParts * k) * kReduceOuts + o] = v[k];
    __syncthreads();
    if (part == 0) {
      int c = 0;
      for (; c + 8 <= m; c += 8) {
        float u[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) u[k] = lds[(c + k) * kReduceOuts + o];
#pragma unroll
        for (int k = 0; k < 8; ++k) t += u[k];
      }
      for (; c < m; ++c) t += lds[c * kReduceOuts + o];
    }
  }
  if (part == 0 && i < r.n) r.out[i] = t;
}
__global__ __launch_bounds__(256) void k_reduce_chunks(LayerSums sums) {
  __shared__ ReduceLds lds;
  reduce_block<256>(sums, blockIdx.x, lds);
}

// dZ = bf16(dY * (Y > 0)) (ReLU backward; Y is the post-activation output, null for a
// linear layer) and the bias gradient's partial sums: block b takes pixels
// [b*P/B, (b+1)*P/B), stages their dZ in LDS and adds it per channel in pixel order. Bound by
// its 8 bytes a value and, at training crops, by the latency of one block per CU. (As two
// kernels the sums re-read dZ with C threads a block: 40 + 7 us a layer on average at
// 8 x 128 x 128, plus 6 launches that wrote the gathered gradients; as one of 256 threads
// 10 us and 6.5 for the sums of the layer above in a launch of their own; now 11 for both.)
// dY is formed on the way from what the layers above left:
//   kGradPlain  gradient of this tensor
//   kGradUp     gradient g of [upsample(this) | skip] at twice the side: the 2x2 sum
//   kGradSkip   this tensor's skip share of such a gradient g, plus a quarter of the
//               gradient `pooled` of its 2x2 pooling
constexpr int kBiasElems = 16384;  // bf16 staged at a time
struct GradSrc {
  const float* g;
  const float* pooled;  // kGradSkip
  int kind;
  int H, W;    // of this tensor
  int gc, c0;  // channels of g, first channel of this tensor's share
};
__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
// p: pixel over all images (below 2^31: a gradient tensor of that many would not fit the GPU)
__device__ __forceinline__ float4 grad4(const GradSrc& s, int C, unsigned p, int c) {
  if (s.kind == kGradPlain) return *reinterpret_cast<const float4*>(s.g + static_cast<size_t>(p) * C + c);
  const unsigned W = static_cast<unsigned>(s.W);
  const size_t row = p / W;  // over all images
  const unsigned x = p % W;
  if (s.kind == kGradUp) {
    const float* q = s.g + (2 * row * 2 * W + 2 * x) * s.gc + c;
    const size_t down = static_cast<size_t>(2 * W) * s.gc;
    return add4(add4(*reinterpret_cast<const float4*>(q), *reinterpret_cast<const float4*>(q + s.gc)),
                add4(*reinterpret_cast<const float4*>(q + down), *reinterpret_cast<const float4*>(q + down + s.gc)));
  }
  const float4 k = *reinterpret_cast<const float4*>(s.g + static_cast<size_t>(p) * s.gc + s.c0 + c);
  // H is even: the rows of an image pair up
  const float4 h = *reinterpret_cast<const float4*>(s.pooled + ((row >> 1) * (W >> 1) + (x >> 1)) * C + c);
  return make_float4(k.x + 0.25f * h.x, k.y + 0.25f * h.y, k.z + 0.25f * h.z, k.w + 0.25f * h.w);
}

// The blocks from kBiasBlocks on add up the parameter gradients of the layer above, whose
// partial sums the previous launch left.
constexpr int kBiasThreads = 512;
__global__ __launch_bounds__(kBiasThreads) void k_relu_bias(GradSrc src, const uint16_t* __restrict__ Y,
                                                   uint16_t* __restrict__ dZ, size_t P, int C,
                                                   float* __restrict__ partial, LayerSums above) {
  __shared__ union {
    alignas(16) uint16_t z[kBiasElems];
    ReduceLds reduce;
  } u;
  if (blockIdx.x >= kBiasBlocks) {
    reduce_block<kBiasThreads>(above, blockIdx.x - kBiasBlocks, u.reduce);
    return;
  }
  uint16_t* const lds = u.z;
  const size_t p0 = P * blockIdx.x / kBiasBlocks, p1 = P * (blockIdx.x + 1) / kBiasBlocks;
  const int pixels = kBiasElems / C, octets = C / 8;
  float t = 0.f;
  for (size_t p = p0; p < p1; p += pixels) {
    const int m = static_cast<int>(p1 - p < static_cast<size_t>(pixels) ? p1 - p : pixels);
    __syncthreads();
#pragma unroll 4
    for (int i = threadIdx.x; i < m * octets; i += kBiasThreads) {
      const int q = static_cast<int>(static_cast<unsigned>(i) / static_cast<unsigned>(octets)), c = (i - q * octets) * 8;
      const unsigned pq = static_cast<unsigned>(p) + static_cast<unsigned>(q);
      const float4 g0 = grad4(src, C, pq, c), g1 = grad4(src, C, pq, c + 4);
      const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
      const size_t at = (p + q) * C + c;
      u32x4 y = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // ones
      if (Y) y = *reinterpret_cast<const u32x4*>(Y + at);
      u32x4 z;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t lo = __uint_as_float(y[k] << 16) > 0.f ? f2bf(g[2 * k]) : 0u;
        const uint32_t hi = __uint_as_float(y[k] & 0xffff0000u) > 0.f ? f2bf(g[2 * k + 1]) : 0u;
        z[k] = lo | (hi << 16);
      }
      *reinterpret_cast<u32x4*>(dZ + at) = z;
      *reinterpret_cast<u32x4*>(lds + i * 8) = z;
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < C) {
      int q = 0;
      for (; q + 16 <= m; q += 16) {
        float u[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) u[k] = bf2f(lds[(q + k) * C + threadIdx.x]);
#pragma unroll
        for (int k = 0; k < 16; ++k) t += u[k];
      }
      for (; q < m; ++q) t += bf2f(lds[q * C + threadIdx.x]);
    }
  }
  if (static_cast<int>(threadIdx.x) < C) partial[static_cast<size_t>(blockIdx.x) * C + threadIdx.x] = t;
}

// Input features (16 channels, 10 used): log(1+radiance) rgb, albedo rgb (clamped to
// [0,1]), normal xyz, log(1+view depth); from the renderer's per-pixel buffers.
__global__ void k_features(const float4* __restrict__ color, const float4* __restrict__ albedo,
                           const float4* __restrict__ normal, uint16_t* __restrict__ out, size_t P) {
  const size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const float4 c = color[p], a = albedo[p], nd = normal[p];
  float f[16];
  f[0] = log1pf(fmaxf(c.x, 0.f));
  f[1] = log1pf(fmaxf(c.y, 0.f));
  f[2] = log1pf(fmaxf(c.z, 0.f));
  f[3] = fminf(fmaxf(a.x, 0.f), 1.f);
  f[4] = fminf(fmaxf(a.y, 0.f), 1.f);
  f[5] = fminf(fmaxf(a.z, 0.f), 1.f);
  f[6] = nd.x;
  f[7] = nd.y;
  f[8] = nd.z;
  f[9] = log1pf(fmaxf(nd.w, 0.f));
  for (int k = 10; k < 16; ++k) f[k] = 0.f;
  uint16_t* o = out + p * 16;
  for (int k = 0; k < 16; ++k) o[k] = f2bf(f[k]);
}

// denoised = (1 - b) denoised + b noisy (OptiX's blend factor, Tracer/Optix/Denoiser.cpp:108)
__global__ void k_blend(float4* __restrict__ den, const float4* __restrict__ color, float b, size_t P) {
  const size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const float4 d = den[p], c = color[p];
  den[p] = make_float4(fmaf(b, c.x - d.x, d.x), fmaf(b, c.y - d.y, d.y), fmaf(b, c.z - d.z, d.z), d.w);
}

// training target: log(1+radiance) of the reference image
__global__ void k_target(const float4* __restrict__ color, float* __restrict__ out, size_t P) {
  const size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const float4 c = color[p];
  out[p * 3 + 0] = log1pf(fmaxf(c.x, 0.f));
  out[p * 3 + 1] = log1pf(fmaxf(c.y, 0.f));
  out[p * 3 + 2] = log1pf(fmaxf(c.z, 0.f));
}

// crop gather: batch item b copies a (S x S) window at (x0, y0) of dataset image idx
__global__ void k_gather_crop(const uint16_t* __restrict__ feat, const float* __restrict__ tgt, int Hs, int Ws,
                              const int4* __restrict__ crops, int S, uint16_t* __restrict__ fo, float* __restrict__ to) {
  const int b = blockIdx.y;
  const int4 cr = crops[b];  // (image, x0, y0, flip)
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<size_t>(S) * S) return;
  const int y = static_cast<int>(i / S), x = static_cast<int>(i % S);
  const int sx = cr.w ? cr.y + (S - 1 - x) : cr.y + x;
  const size_t src = (static_cast<size_t>(cr.x) * Hs + cr.z + y) * Ws + sx;
  const size_t dst = static_cast<size_t>(b) * S * S + i;
  const uint4* fs = reinterpret_cast<const uint4*>(feat + src * 16);
  uint4* fd = reinterpret_cast<uint4*>(fo + dst * 16);
  fd[0] = fs[0];
  fd[1] = fs[1];
  if (cr.w) {  // mirrored crop: flip the normal's x component sign bit (channel 6)
    uint16_t* h = fo + dst * 16;
    h[6] ^= 0x8000u;
  }
  to[dst * 3 + 0] = tgt[src * 3 + 0];
  to[dst * 3 + 1] = tgt[src * 3 + 1];
  to[dst * 3 + 2] = tgt[src * 3 + 2];
}

// L1 loss in log space. The network predicts a correction added to the noisy input
// (feature channels 0..2 = log(1 + radiance)): prediction = x + y over the first 3 of
// 32 output channels. Partial sums of |x + y - t| per block and dOut = sign(x + y - t) /
// (3 P); the padding channels of dOut stay zero as allocated (writing them too was most of
// the kernel's traffic). L1 keeps the firefly pixels of many-emitter scenes
// from dominating the gradient (with an L2 loss the network trained on the soup and the
// instanced scene reached relMSE 0.0125 at 8 spp on a held-out soup view; with L1,
// 0.0085).
__global__ void k_loss(const float* __restrict__ Y, const uint16_t* __restrict__ X, const float* __restrict__ T,
                       size_t P, float* __restrict__ dY, float* __restrict__ partial) {
  __shared__ float red[256];
  const size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (p < P) {
    const float inv = 1.f / (3.f * static_cast<float>(P));
    float g[3];
    for (int c = 0; c < 3; ++c) {
      const float d = (bf2f(X[p * 16 + c]) + Y[p * 32 + c]) - T[p * 3 + c];
      l += fabsf(d);
      g[c] = (d > 0.f ? inv : (d < 0.f ? -inv : 0.f));
    }
    *reinterpret_cast<float4*>(dY + p * 32) = make_float4(g[0], g[1], g[2], 0.f);
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The data-gradient convolution is a 3x3 convolution of dZ with the spatially flipped,
// channel-transposed kernel Wd[ci][tap][co] = W[co][8 - tap][ci]: where parameter i of the
// network goes in the flipped copy (-1: a bias, or a layer without one).
__device__ __forceinline__ int flipped_index(const WeightTable& t, int i) {
  for (int l = 0; l < t.n; ++l) {
    const int r = i - t.off[l], k = 9 * t.cin[l];
    if (r < 0 || r >= k * t.cout[l]) continue;
    const int co = r / k, tap = (r - co * k) / t.cin[l], ci = r - co * k - tap * t.cin[l];
    return t.off[l] + (ci * 9 + (8 - tap)) * t.cout[l] + co;
  }
  return -1;
}

// Adam (Kingma & Ba 2015) on fp32 master weights; the bf16 copy and the flipped bf16 copy
// are refreshed in the same pass (a launch per layer for the flips cost 3 us each).
__global__ void k_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v, const float* __restrict__ g,
                       uint16_t* __restrict__ wb, uint16_t* __restrict__ wd, WeightTable table, int n, float lr,
                       float b1, float b2, float c1, float c2, float eps) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  const uint16_t h = f2bf(wi);
  wb[i] = h;
  const int f = flipped_index(table, i);
  if (f >= 0) wd[f] = h;
}

// bf16 copies of the weights (plain and flipped) without an update
__global__ void k_weights_bf16(const float* __restrict__ w, uint16_t* __restrict__ wb, uint16_t* __restrict__ wd,
                               WeightTable table, int n) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= n) return;
  const uint16_t h = f2bf(w[i]);
  wb[i] = h;
  const int f = flipped_index(table, i);
  if (f >= 0) wd[f] = h;
}

inline unsigned blocks_for(size_t n, unsigned b = 256) { return static_cast<unsigned>((n + b - 1) / b); }

}  // namespace dn

using namespace dn;

// Persistent grid: as many workgroups as fit on the device at once (occupancy of the
// instantiation x CUs), a multiple of 8 (one share per XCD) whose per-XCD share is a
// multiple of the channel-group count, so a workgroup keeps one group's weights. `beside`:
// workgroups of other work in the same launch, which get up to half of the room.
template <typename K>
static unsigned persistent_blocks(K kernel, long items, int groups, long beside = 0) {
  static thread_local int cus = 0, dev = -1;
  int d = 0;
  (void)hipGetDevice(&d);
  if (d != dev) {
    dev = d;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d) != hipSuccess || cus <= 0) cus = 256;
  }
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, 256, 0) != hipSuccess || occ <= 0) occ = 1;
  const long fit = long(cus) * occ;
  long per = (fit - beside > fit / 2 ? fit - beside : fit / 2) / 8;
  per = per / groups * groups;
  if (per < groups) per = groups;
  const long need = (items + 7) / 8;
  if (per > need) per = (need + groups - 1) / groups * groups;
  return static_cast<unsigned>(per * 8);
}

template <int MB, int NB, int EPI>
static void launch_conv_epi(const ConvArgs& a, long items, hipStream_t s) {
  const int cin = a.c1 + a.cx;
  if (cin == 16) {
    const unsigned blocks = persistent_blocks(k_conv<MB, NB, EPI, true, true>, items, a.groups);
    hipLaunchKernelGGL((k_conv<MB, NB, EPI, true, true>), dim3(blocks), dim3(256), 0, s, a);
  } else if (cin == 32) {
    const unsigned blocks = persistent_blocks(k_conv<MB, NB, EPI, true, false>, items, a.groups);
    hipLaunchKernelGGL((k_conv<MB, NB, EPI, true, false>), dim3(blocks), dim3(256), 0, s, a);
  } else {
    const unsigned blocks = persistent_blocks(k_conv<MB, NB, EPI, false, false>, items, a.groups);
    hipLaunchKernelGGL((k_conv<MB, NB, EPI, false, false>), dim3(blocks), dim3(256), 0, s, a);
  }
}

template <int MB, int NB>
static void launch_conv(const ConvArgs& a, int epi, long items, hipStream_t s) {
  switch (epi) {
    case kEpiRelu: launch_conv_epi<MB, NB, kEpiRelu>(a, items, s); break;
    case kEpiF32: launch_conv_epi<MB, NB, kEpiF32>(a, items, s); break;
    case kEpiReluPool: launch_conv_epi<MB, NB, kEpiReluPool>(a, items, s); break;
    default: launch_conv_epi<MB, NB, kEpiRadiance>(a, items, s); break;
  }
}

// Tile shape per layer: 16-row tiles (MB = 2) unless that leaves < 1024 tiles, then
// 8-row tiles with 64-channel groups (NB = 2) when Cout is a multiple of 64.
struct ConvPlan {
  ConvArgs a;
  int MB, NB;
  long items;
};
static bool plan_conv(const DnConv& c, ConvPlan& p) {
  const int Cin = c.c1 + c.cx;
  const bool shape_ok = (Cin == 16 && c.c1 == 0) || (c.c1 % 32 == 0 && c.cx % 32 == 0 && Cin > 0);
  if (!shape_ok || c.cout % 32 || c.W % kTileW || c.H <= 0 || c.N <= 0) return false;
  if ((c.epi == kEpiReluPool || c.c1) && c.H % 2) return false;
  if (c.epi == kEpiRadiance && c.cout < 4) return false;
  if (c.c1 && !c.coarse) return false;
  if (!dn_load_ok(c.H, c.W, c.cx) || !dn_load_ok(c.H / 2, c.W / 2, c.c1)) return false;
  if (c.epi == kEpiRadiance && Cin > 32) return false;  // feature prefetch assumes one chunk
  const long tiles16 = long(c.W / kTileW) * ((c.H + 15) / 16) * c.N;
  const int MB = p.MB = tiles16 >= 1024 ? 2 : 1;
  const long tiles = long(c.W / kTileW) * ((c.H + 8 * MB - 1) / (8 * MB)) * c.N;
  if ((c.epi == kEpiRelu || c.epi == kEpiReluPool) && !dn_store_ok(c.H, c.W, c.cout, 8 * MB)) return false;
  const int NB = p.NB = MB == 1 && c.cout % 64 == 0 ? 2 : 1;  // MB = NB = 2 would need > 100 KB of LDS
  ConvArgs& a = p.a;
  a.x = c.x;
  a.coarse = c.coarse;
  a.c1 = c.c1;
  a.cx = c.cx;
  a.w = c.w;
  a.bias = c.bias;
  a.y = c.y;
  a.cout = c.cout;
  a.pooled = c.pooled;
  a.feat = c.feat;
  a.radiance = c.radiance;
  a.N = c.N;
  a.H = c.H;
  a.W = c.W;
  a.groups = c.cout / (32 * NB);
  p.items = tiles * a.groups;
  return true;
}

bool dn_conv(const DnConv& c, hipStream_t s) {
  ConvPlan p;
  if (!plan_conv(c, p)) return false;
  if (p.MB == 2) {
    launch_conv<2, 1>(p.a, c.epi, p.items, s);
  } else {
    if (p.NB == 2) launch_conv<1, 2>(p.a, c.epi, p.items, s); else launch_conv<1, 1>(p.a, c.epi, p.items, s);
  }
  return true;
}

bool dn_conv3x3(const uint16_t* X, const uint16_t* Wt, const float* bias, void* Y, int N, int H, int W, int Cin,
                int Cout, bool relu, bool out_f32, hipStream_t s) {
  if (relu == out_f32) return false;  // bf16 + ReLU or fp32 linear
  DnConv c;
  c.x = X;
  c.cx = Cin;
  c.w = Wt;
  c.bias = bias;
  c.y = Y;
  c.cout = Cout;
  c.N = N;
  c.H = H;
  c.W = W;
  c.epi = relu ? kEpiRelu : kEpiF32;
  return dn_conv(c, s);
}

int dn_wgrad_chunks(int N, int H, int W) {
  const int tiles = (W / kTileW) * ((H + kTileH - 1) / kTileH) * N;
  return (tiles + kWgradTiles - 1) / kWgradTiles;
}

static LayerSums layer_sums(const DnSums& p, int threads) {
  if (!p.wpartial) return LayerSums{};
  const auto blocks = [&](int chunks, size_t n) {
    return blocks_for(n, static_cast<unsigned>(chunks <= kReduceDirect ? threads : kReduceOuts));
  };
  const unsigned first = blocks(kBiasBlocks, p.cout);
  return LayerSums{ChunkSum{p.wpartial, p.chunks, p.n_weights, p.dW},
                   ChunkSum{p.bpartial, kBiasBlocks, static_cast<size_t>(p.cout), p.db}, first,
                   first + blocks(p.chunks, p.n_weights)};
}

void dn_relu_bias(const DnGrad& grad, const uint16_t* Y, uint16_t* dZ, int N, int H, int W, int Cout, float* bpartial,
                  const DnSums& above, hipStream_t s) {
  const GradSrc src{grad.g, grad.pooled, grad.kind, H, W, grad.gc, grad.c0};
  const LayerSums sums = layer_sums(above, kBiasThreads);
  hipLaunchKernelGGL(k_relu_bias, dim3(kBiasBlocks + sums.blocks), dim3(kBiasThreads), 0, s, src, Y, dZ,
                     static_cast<size_t>(N) * H * W, Cout, bpartial, sums);
}

void dn_sums(const DnSums& p, hipStream_t s) {
  const LayerSums sums = layer_sums(p, 256);
  if (sums.blocks) hipLaunchKernelGGL(k_reduce_chunks, dim3(sums.blocks), dim3(256), 0, s, sums);
}

template <int MB, int NB, bool SC>
static void launch_conv_wgrad(const ConvPlan& p, const WgradArgs& w, unsigned wblocks, hipStream_t s) {
  const unsigned blocks = persistent_blocks(k_conv_wgrad<MB, NB, SC>, p.items, p.a.groups, wblocks);
  hipLaunchKernelGGL((k_conv_wgrad<MB, NB, SC>), dim3(blocks + wblocks), dim3(256), 0, s, p.a, blocks, w);
}

// One launch for the two where the convolution has 8-row tiles, which is where either leaves
// compute units idle; each alone, with its own registers and occupancy, above.
bool dn_conv_wgrad(const uint16_t* X, const uint16_t* coarse, int c1, const uint16_t* dZ, int N, int H, int W, int Cin,
                   int Cout, float* wpartial, const uint16_t* Wd, float* gout, hipStream_t s) {
  const WgradArgs w{X, coarse, dZ, wpartial, c1, N, H, W, Cin, Cout, dn_wgrad_chunks(N, H, W)};
  if (!dn_load_ok(H, W, Cin - c1) || !dn_load_ok(H / 2, W / 2, c1) || !dn_load_ok(H, W, Cout)) return false;
  const unsigned channels = (Cout / 32) * ((Cin + 31) / 32), wblocks = w.chunks * channels;
  DnConv c;
  ConvPlan p;
  if (gout) {
    c.x = dZ;
    c.cx = Cout;
    c.w = Wd;
    c.y = gout;
    c.cout = Cin;
    c.N = N;
    c.H = H;
    c.W = W;
    c.epi = kEpiF32;
    if (!plan_conv(c, p)) return false;
    if (p.MB == 1) {
      if (p.NB == 2) launch_conv_wgrad<1, 2, false>(p, w, wblocks, s);
      else if (Cout == 32) launch_conv_wgrad<1, 1, true>(p, w, wblocks, s);
      else launch_conv_wgrad<1, 1, false>(p, w, wblocks, s);
      return true;
    }
  }
  hipLaunchKernelGGL(k_wgrad, dim3(w.chunks, channels), dim3(kWgThreads), 0, s, w);
  return !gout || dn_conv(c, s);
}
void dn_features(const float4* color, const float4* albedo, const float4* normal, uint16_t* out, size_t P,
                 hipStream_t s) {
  hipLaunchKernelGGL(k_features, dim3(blocks_for(P)), dim3(256), 0, s, color, albedo, normal, out, P);
}
void dn_blend(float4* den, const float4* color, float b, size_t P, hipStream_t s) {
  hipLaunchKernelGGL(k_blend, dim3(blocks_for(P)), dim3(256), 0, s, den, color, b, P);
}
void dn_target(const float4* color, float* out, size_t P, hipStream_t s) {
  hipLaunchKernelGGL(k_target, dim3(blocks_for(P)), dim3(256), 0, s, color, out, P);
}
void dn_gather_crop(const uint16_t* feat, const float* tgt, int Hs, int Ws, const int4* crops, int B, int S,
                    uint16_t* fo, float* to, hipStream_t s) {
  hipLaunchKernelGGL(k_gather_crop, dim3(blocks_for(static_cast<size_t>(S) * S), B), dim3(256), 0, s, feat, tgt, Hs,
                     Ws, crops, S, fo, to);
}
int dn_loss(const float* Y, const uint16_t* X, const float* T, size_t P, float* dY, float* partial, hipStream_t s) {
  const unsigned nb = blocks_for(P);
  hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, s, Y, X, T, P, dY, partial);
  return static_cast<int>(nb);
}
void dn_adam(float* w, float* m, float* v, const float* g, uint16_t* wb, uint16_t* wd, const WeightTable& table, size_t n,
             float lr, float b1, float b2, float c1, float c2, float eps, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(n)), dim3(256), 0, s, w, m, v, g, wb, wd, table, static_cast<int>(n), lr, b1,
                     b2, c1, c2, eps);
}

void dn_weights_bf16(const float* w, uint16_t* wb, uint16_t* wd, const WeightTable& table, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_weights_bf16, dim3(blocks_for(n)), dim3(256), 0, s, w, wb, wd, table, static_cast<int>(n));
}

}  // namespace trt
