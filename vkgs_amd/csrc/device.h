// Device-only helpers shared by the kernels of the plain and the batched
// paths: the Gaussian falloff of the raster, the wave digit match of the
// radix ranking, and the pair emission of binning.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace vkgs {

// exp(-q / 2) as v_exp_f32 (exp2) of q * (-log2(e) / 2).  Halving the float
// log2(e) is exact, so this equals exp2((-q / 2) * log2(e)) bit for bit while
// saving a multiply.
__device__ __forceinline__ float gauss_falloff(float q) {
  constexpr float kNegHalfLog2e = -0.5f * 1.44269504088896340736f;
  return __builtin_amdgcn_exp2f(q * kNegHalfLog2e);
}

// Load and store through a pointer known to address device (global) memory:
// for a pointer read from memory (a field of a table in HBM) the compiler
// cannot always infer the address space and falls back to flat accesses,
// which also count against the LDS wait counter.
__device__ __forceinline__ float ld_global(const float* p) { return *(const __attribute__((address_space(1))) float*)p; }
__device__ __forceinline__ float4 ld_global(const float4* p) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  const v4 v = *(const __attribute__((address_space(1))) v4*)p;
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st_global(float* p, float v) { *(__attribute__((address_space(1))) float*)p = v; }
__device__ __forceinline__ void st_global(float4* p, const float4& v) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  *(__attribute__((address_space(1))) v4*)p = v4{v.x, v.y, v.z, v.w};
}

// Number of set bits of m below this lane.
__device__ __forceinline__ uint32_t mbcnt(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Mask of the lanes whose kBits-bit digit equals this lane's (valid lanes
// only): per bit one ballot and m &= ~(ballot ^ this lane's bit broadcast).
template <int kBits>
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
  const uint64_t m0 = __ballot(valid);
  uint32_t lo = (uint32_t)m0, hi = (uint32_t)(m0 >> 32);
#pragma unroll
  for (int b = 0; b < kBits; ++b) {
    const uint32_t sel = (uint32_t)((int32_t)(d << (31 - b)) >> 31);  // bit b of d, all ones or zero
    const uint64_t bb = __ballot(sel != 0u);
    // m &= ~(bb ^ sel): v_bitop3 with m as the middle operand and the
    // symmetric bb / sel on either side, truth table 0x84
    lo = __builtin_amdgcn_bitop3_b32((uint32_t)bb, lo, sel, 0x84);
    hi = __builtin_amdgcn_bitop3_b32((uint32_t)(bb >> 32), hi, sel, 0x84);
  }
  return ((uint64_t)hi << 32) | lo;
}

// Splats covering more tiles than this are emitted by a whole wave.
constexpr uint32_t kEmitSerial = 8;

__device__ __forceinline__ uint32_t lane_u32(uint32_t x, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, (int)lane);
}

// Segments of large splats' pair runs, written by a later launch whose waves
// take one each (emit_segments_kernel).  In depth order the splats nearest to
// the camera sit together, so a few waves held nearly all of a frame's large
// splats (1M splats at 1600x900: the emit took 58 us and all but a handful of
// its waves were done in 10; 3839x2159: 316 us).  The segments live in the
// tile sort's key buffer that the emit does not write: a segment takes 32
// bytes and stands for more than kQueueAbove pairs (4 bytes of that buffer
// each), so they fit; where they should not, the wave writes the pairs itself.
struct EmitQueue {
  uint4* segs;      // two words of four per segment
  uint32_t* count;  // zeroed before the emit
  uint32_t cap;
};
constexpr uint32_t kSegPairs = 512;   // pairs of a segment (more from 64 segments a splat up)
constexpr uint32_t kQueueAbove = 64;  // splats of more tiles are queued ...
constexpr uint32_t kQueueWave = 2048; // ... where their wave has more pairs than this to write

// i / w and the remainder by a float reciprocal, for quotients up to 2^20
// (tile rows; the quotient is then off by at most one before the correction).
__device__ __forceinline__ void row_col(uint32_t i, uint32_t w, float inv_w, uint32_t& row, uint32_t& col) {
  row = (uint32_t)((float)i * inv_w);
  int32_t c = (int32_t)(i - row * w);
  if (c < 0) {
    --row;
    c += (int32_t)w;
  } else if (c >= (int32_t)w) {
    ++row;
    c -= (int32_t)w;
  }
  col = (uint32_t)c;
}

// Emits the pairs of one splat per lane: c tiles of rectangle r (tile x in
// r.x's low/high 16 bits, tile y in r.y's) as keys key_base + ty * tiles_x + tx
// at o, o + 1, ... in row-major tile order; pairs at or beyond max_pairs are
// dropped (the caller flags the overflow).  The value of the i-th pair is val,
// or, with kIndexValues, q0 + i: a second numbering of the pairs (the
// caller's q0 per splat), which a later pass uses to find each pair after the
// sort (clamped to max_pairs - 1 on overflow, so readers stay in bounds).  Lanes
// with up to kEmitSerial tiles write their own pairs (a lane's few stores cost
// less than finding owners).  The larger splats' pairs are then numbered
// across the wave and written 64 at a time, each lane finding the splat of its
// pair: the wave's steps follow the pairs it has, not the splats (one splat per
// step, most of its lanes idle, took 93 us for 7.3M pairs of 19 tiles a splat).
// A wave with too many of them queues its largest splats.  Every lane of the
// wave must call this (c = 0 for lanes without a splat); tiles_x is the same
// in every lane unless kIndexValues.
template <bool kIndexValues = false>
__device__ __forceinline__ void emit_pairs_wave(uint32_t c, uint64_t o, TileRect r, uint32_t val, uint32_t key_base,
                                                uint32_t tiles_x, uint64_t max_pairs, uint32_t* __restrict__ keys,
                                                uint32_t* __restrict__ vals, const EmitQueue& queue,
                                                uint64_t q0 = 0) {
  __shared__ uint32_t s_owner[256 / kWave][kWave];  // per wave: the lane whose run starts at a place of the step
  const bool big = c > kEmitSerial;
  if (c != 0 && !big) {
    const uint32_t tx0 = r.x & 0xffffu, tx1 = r.x >> 16, ty0 = r.y & 0xffffu, ty1 = r.y >> 16;
    uint64_t j = o, q = q0;
    for (uint32_t ty = ty0; ty <= ty1; ++ty)
      for (uint32_t tx = tx0; tx <= tx1; ++tx, ++j, ++q) {
        if (j < max_pairs) {
          keys[j] = key_base + ty * tiles_x + tx;
          vals[j] = kIndexValues ? (uint32_t)(q < max_pairs ? q : max_pairs - 1) : val;
        }
      }
  }
  uint32_t cb = big && o < max_pairs ? c : 0u;
  if (__ballot(cb != 0) == 0) return;
  const uint32_t lane = __lane_id();
  const uint32_t w = (r.x >> 16) - (r.x & 0xffffu) + 1u;
  const uint32_t first = key_base + (r.y & 0xffffu) * tiles_x + (r.x & 0xffffu);
  const uint32_t o32 = (uint32_t)o, v32 = kIndexValues ? (uint32_t)q0 : val;
  auto inclusive = [&](uint32_t x) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)x, d, kWave);
      if ((int)lane >= d) x += t;
    }
    return x;
  };
  uint32_t incl = inclusive(cb);
  uint32_t total = lane_u32(incl, kWave - 1);
  if (total > kQueueWave) {
    if (cb > kQueueAbove) {
      const uint32_t n = (uint32_t)(max_pairs - o < cb ? max_pairs - o : cb);
      const uint32_t per = ((n + 63u) / 64u + 63u) & ~63u;
      const uint32_t len = per > kSegPairs ? per : kSegPairs;
      const uint32_t ns = (n + len - 1u) / len;
      const uint32_t at = atomicAdd(queue.count, ns);
      const bool fits = at < queue.cap && ns <= queue.cap - at;
      for (uint32_t s = 0; s < ns && at + s < queue.cap; ++s) {
        const uint32_t i0 = s * len, m = n - i0 < len ? n - i0 : len;
        queue.segs[2 * (size_t)(at + s)] = make_uint4(i0, fits ? m : 0u, w, first);
        queue.segs[2 * (size_t)(at + s) + 1] = make_uint4(tiles_x, o32, v32, 0u);
      }
      if (fits) cb = 0;
    }
    incl = inclusive(cb);
    total = lane_u32(incl, kWave - 1);
  }
  const uint32_t start = incl - cb;
  const float inv_w = __builtin_amdgcn_rcpf((float)w);
  uint32_t* own = s_owner[threadIdx.x / kWave];
  const uint64_t upto = ~0ull >> (kWave - 1 - lane);  // this lane and those below it
  uint32_t carry = 0;                                 // the lane whose run crosses into this step
  for (uint32_t base = 0; base < total; base += kWave) {
    own[lane] = 0xffffffffu;
    __builtin_amdgcn_wave_barrier();  // a wave's LDS operations complete in order
    if (cb != 0 && start - base < (uint32_t)kWave) own[start - base] = lane;
    __builtin_amdgcn_wave_barrier();
    const uint32_t v = own[lane];
    const uint64_t starts = __ballot(v != 0xffffffffu);
    const uint64_t mine = starts & upto;
    const int from = mine ? 63 - (int)__builtin_clzll(mine) : (int)lane;
    const uint32_t near = (uint32_t)__shfl((int)v, from, kWave);
    const int src = (int)(mine ? near : carry);
    if (starts) carry = lane_u32(v, 63u - (uint32_t)__builtin_clzll(starts));
    const uint32_t p = base + lane;
    const uint32_t i = p - (uint32_t)__shfl((int)start, src, kWave);
    const uint32_t sw = (uint32_t)__shfl((int)w, src, kWave), sf = (uint32_t)__shfl((int)first, src, kWave);
    const uint32_t so = (uint32_t)__shfl((int)o32, src, kWave), sv = (uint32_t)__shfl((int)v32, src, kWave);
    const float si = __shfl(inv_w, src, kWave);
    const uint32_t stx = kIndexValues ? (uint32_t)__shfl((int)tiles_x, src, kWave) : tiles_x;
    uint32_t row, col;
    row_col(i, sw, si, row, col);
    const uint64_t j = (uint64_t)so + i;
    if (p < total && j < max_pairs) {
      keys[j] = sf + row * stx + col;
      const uint64_t q = (uint64_t)sv + i;
      vals[j] = kIndexValues ? (uint32_t)(q < max_pairs ? q : max_pairs - 1) : sv;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace vkgs
