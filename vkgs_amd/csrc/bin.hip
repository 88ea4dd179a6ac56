// Two-level tile binning for gfx950: depth-ordered splats to per-tile lists
// without a (tile, splat) pair sort.
//
// Supertiles are 16 x 16 tiles.  Level one moves the splats, in depth order, to
// the lists of the supertiles they touch (about 1.1 per splat where a splat
// touches two tiles); level two moves each supertile's items, in order, to the
// lists of its tiles.  Both are stable counting passes over at most 512 and 256
// lists, so a tile's list keeps the depth order: the list a stable sort of
// (tile, splat) pairs by tile gives, bit for bit.  Against that sort (emit the
// pairs, two or three radix passes of three launches, mark the ranges), pairs
// are formed once, in the last kernel, and the tile ranges fall out of the
// counts: 5-6 launches instead of 10-13, and 6M splats with 10.1M pairs move
// 0.35 GB instead of 0.6.  Binning and pair sort together, before and after:
// 5k splats at 320x240 32 -> 21 us, 100k at 1600x900 77 -> 43, 6M 207 -> 166,
// 2.3M at 3839x2159 240 -> 175 (12M pairs).  The counting kernels are bound by
// their reads and launch latency, the moving ones by the masks' LDS traffic.
//
//   super_count : per chunk of splats, items per supertile (and the pair total)
//   super_scan  : per supertile, offsets over the chunks (grids above kRawGrid)
//   super_move  : (slot, rectangle inside the supertile) to its supertile's list
//   tile_count  : per chunk of one supertile's items, pairs per tile
//   tile_scan   : the tiles' list ranges, in row-major tile order, and the counts of
//                 the longest-first schedule
//   tile_move   : slots to the tiles' lists
//
// A workgroup ranks 512 entries at a time by 64-bit masks of its waves (see
// Ranker), which needs no ordered atomics.
//
// Where the pairs outgrow max_pairs, the first max_pairs of the draw order are kept
// (a splat's in row-major tile order), as by emitting them into a buffer of that
// size: super_move cuts the splats there, and everything after it sees only what
// is kept, so every list is whole or cut at the same place in every run and all
// max_pairs positions of the lists are written.
#pragma clang fp contract(off)

#include "common.h"
#include "device.h"
#include "kernels.h"
#include "sort.h"

namespace vkgs {
namespace {

constexpr int kT = 512;  // threads, and entries ranked at a time
constexpr int kW = kT / kWave;
constexpr uint32_t kSuperShift = 4;
constexpr uint32_t kSuperTiles = 1u << (2 * kSuperShift);
constexpr uint32_t kMaxSupers = 512;
constexpr uint32_t kMaxLines = 128;   // their columns and rows together
constexpr uint32_t kStage = 2048;     // entries reordered in LDS before they are stored
constexpr uint32_t kRawGrid = 256;    // chunks whose counts the movers sum themselves
constexpr uint32_t kMaxGrid = 1024;
static_assert(2 * kMaxGrid <= kStage, "find_cut holds the chunks' pairs there");
constexpr uint32_t kMaxChunks = 4096;  // of level two
// A chunk of level two reads the counts of its supertile's chunks before it, so its
// time grows with their number and falls with its own steps: where a supertile has
// more than kManyChunks, as in views from afar, chunks take 3 sqrt(its items) instead.
// 1M splats in 1162 tiles: binning 173 us without, 87 with it (78 by the pair sort); 6M
// in 378 tiles 324, 226 (197); 300k in 199 tiles 60, 52 (59).
constexpr uint32_t kManyChunks = 64;
constexpr uint32_t kXcds = 8;         // consecutive workgroups go round the dies

// Chunk b of `live` chunks, dealt so that each die takes consecutive ones (a
// list's runs of consecutive chunks are adjacent and then meet in one L2).
__device__ __forceinline__ uint32_t deal(uint32_t b, uint32_t live) {
  if (b >= live) return b;
  const uint32_t die = b % kXcds, q = live / kXcds, r = live % kXcds;
  return die * q + min(die, r) + b / kXcds;
}

struct Chunk {
  uint32_t id, live, begin, end;
};

__device__ __forceinline__ uint32_t chunk_subs(uint32_t n, uint32_t grid) {  // 512-entry parts per chunk
  return ((n + kT - 1) / kT + grid - 1) / grid;
}

__device__ __forceinline__ Chunk chunk_of(uint32_t n) {
  const uint32_t sub = (n + kT - 1) / kT, per = chunk_subs(n, gridDim.x);
  Chunk c;
  c.live = per ? (sub + per - 1) / per : 0u;
  c.id = deal(blockIdx.x, c.live);
  const uint64_t size = (uint64_t)per * kT, begin = (uint64_t)c.id * size;
  c.begin = (uint32_t)(begin < n ? begin : n);
  c.end = (uint32_t)(begin + size < n ? begin + size : n);
  return c;
}

// Exclusive scan over the workgroup; s_tmp holds kW words.
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* s_tmp, uint32_t* total) {
  const uint32_t lane = __lane_id(), w = threadIdx.x / kWave;
  uint32_t inc = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, d, kWave);
    if ((int)lane >= d) inc += t;
  }
  if (lane == kWave - 1) s_tmp[w] = inc;
  __syncthreads();
  uint32_t off = 0, all = 0;
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    const uint32_t t = s_tmp[i];
    off += (uint32_t)i < w ? t : 0u;
    all += t;
  }
  __syncthreads();
  *total = all;
  return off + inc - v;
}

// The lists an entry goes to: cells [x0, x1] x [y0, y1] of a grid `stride` wide.
struct Cells {
  uint32_t x0, x1, y0, y1;
  bool any;
};

template <typename F>
__device__ __forceinline__ void for_cells(const Cells& c, uint32_t stride, F&& f) {
  if (!c.any) return;
  for (uint32_t y = c.y0; y <= c.y1; ++y)
    for (uint32_t x = c.x0; x <= c.x1; ++x) f(y * stride + x, x, y);
}

// Depth-ordered input: values slot | packed rectangle << 32, or rectangles with
// their tile counts and (optionally) the slot order.
struct PackedItems {
  const uint64_t* val64;
  RectBits rb;
  __device__ void load(uint32_t k, uint32_t& slot, TileRect& r, uint32_t& c) const {
    const uint64_t v = val64[k];
    slot = (uint32_t)v;
    r = unpack_rect((uint32_t)(v >> 32), rb, &c);
  }
};
struct RectItems {
  const TileRect* rect;
  const uint32_t* cnt;
  const uint32_t* order;
  __device__ void load(uint32_t k, uint32_t& slot, TileRect& r, uint32_t& c) const {
    r = rect[k];
    c = cnt[k];
    slot = order ? order[k] : k;
  }
};

__device__ __forceinline__ Cells super_cells(const TileRect& r, uint32_t c) {
  return Cells{(r.x & 0xffffu) >> kSuperShift, (r.x >> 16) >> kSuperShift, (r.y & 0xffffu) >> kSuperShift,
               (r.y >> 16) >> kSuperShift, c != 0};
}

// Words of the level-one results at `table`: item offsets of the supertiles
// (S + 1), their first chunks (S + 1), items per chunk, supertile totals (S).
struct Table {
  uint32_t* p;
  uint32_t S;
  __device__ uint32_t* offsets() const { return p; }
  __device__ uint32_t* chunks() const { return p + S + 1; }
  __device__ uint32_t* per_chunk() const { return p + 2 * S + 2; }
  __device__ uint32_t* totals() const { return p + 2 * S + 3; }
};

template <typename Items>
__global__ __launch_bounds__(kT) void super_count_kernel(Items in, const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                         uint32_t supers_x, uint32_t S, uint32_t* __restrict__ hist,
                                                         uint32_t* __restrict__ d_pairs,
                                                         uint32_t* __restrict__ status,
                                                         uint32_t* __restrict__ clear, uint32_t n_clear) {
  // the chunks' pairs, two words each, follow their rows of items in hist (see find_cut)
  constexpr uint32_t kCopies = 4;
  __shared__ uint32_t s_h[kMaxSupers * kCopies];
  __shared__ uint64_t s_sum[kW];
  const uint32_t n = min(*d_count, max_n), tid = threadIdx.x;
  const Chunk ch = chunk_of(n);
  for (uint32_t i = blockIdx.x * kT + tid; i < n_clear; i += gridDim.x * kT) clear[i] = 0u;
  if (ch.begin >= ch.end) return;  // workgroup-uniform
  for (uint32_t i = tid; i < S * kCopies; i += kT) s_h[i] = 0u;
  __syncthreads();
  uint32_t pairs = 0;  // (at most 2^13 entries of 2^17 tiles)
  for (uint32_t k = ch.begin + tid; k < ch.end; k += kT) {
    uint32_t slot, c;
    TileRect r;
    in.load(k, slot, r, c);
    pairs += c;
    for_cells(super_cells(r, c), supers_x,
              [&](uint32_t s, uint32_t, uint32_t) { atomicAdd(&s_h[s * kCopies + tid % kCopies], 1u); });
  }
  uint64_t sum = pairs;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) sum += __shfl_xor((unsigned long long)sum, d, kWave);
  if (__lane_id() == 0) s_sum[tid / kWave] = sum;
  __syncthreads();
  if (tid == 0) {
    uint64_t all = 0;
    for (int i = 0; i < kW; ++i) all += s_sum[i];
    const uint32_t low = (uint32_t)all;
    const uint32_t old = all ? atomicAdd(d_pairs, low) : 0u;
    if (all >> 32 || old + low < old) *status = 1u;  // the total passed 2^32: more than max_pairs, whatever its low word
    uint32_t* p = hist + (size_t)gridDim.x * S + 2 * ch.id;
    p[0] = low;
    p[1] = (uint32_t)(all >> 32);
  }
  if (tid < S) {
    uint32_t v = 0;
#pragma unroll
    for (uint32_t j = 0; j < kCopies; ++j) v += s_h[tid * kCopies + j];
    hist[gridDim.x <= kRawGrid ? (size_t)ch.id * S + tid : (size_t)tid * gridDim.x + ch.id] = v;
  }
}

// Exclusive offsets of one supertile's counts over the chunks, in place.
__global__ __launch_bounds__(256) void super_scan_kernel(uint32_t* __restrict__ hist, uint32_t grid,
                                                         const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                         Table table) {
  __shared__ uint32_t s_w[4];
  const uint32_t n = min(*d_count, max_n);
  const uint32_t sub = (n + kT - 1) / kT, per = chunk_subs(n, grid);
  const uint32_t live = per ? (sub + per - 1) / per : 0u;  // at most kMaxGrid = 4 words a thread
  uint32_t* row = hist + (size_t)blockIdx.x * grid;
  const uint32_t first = threadIdx.x * 4, lane = __lane_id(), w = threadIdx.x / kWave;
  uint32_t x[4], s = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x[j] = first + j < live ? row[first + j] : 0u;
    s += x[j];
  }
  uint32_t inc = s;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, d, kWave);
    if ((int)lane >= d) inc += t;
  }
  if (lane == kWave - 1) s_w[w] = inc;
  __syncthreads();
  uint32_t run = inc - s, all = 0;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    run += i < w ? s_w[i] : 0u;
    all += s_w[i];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (first + j < live) row[first + j] = run;
    run += x[j];
  }
  if (threadIdx.x == 0) table.totals()[blockIdx.x] = all;
}

// The position of the r-th set bit of m (r below its population).
__device__ __forceinline__ uint32_t select_bit(uint64_t m, uint32_t r) {
  uint32_t at = 0, x = (uint32_t)m;
  const uint32_t low = (uint32_t)__popc(x);
  if (r >= low) {
    r -= low;
    at = 32u;
    x = (uint32_t)(m >> 32);
  }
#pragma unroll
  for (uint32_t h = 16; h > 0; h >>= 1) {
    const uint32_t c = (uint32_t)__popc(x & ((1u << h) - 1u));
    const bool up = r >= c;
    r -= up ? c : 0u;
    at += up ? h : 0u;
    x = up ? x >> h : x;
  }
  return at;
}

// Ranks 512 entries at a time into the lists of a grid `cols` wide (at most kD
// lists, kLines columns and rows together) and stores them.  Per wave and list a
// 64-bit mask says which of the wave's entries go there; a list's entries then
// follow from the masks' populations.
//  - Steps whose entries go to at most kFewCells lists each: an entry sets its
//    bit in the mask of each of its lists, and where the step has at most kStage
//    list entries every lane walks its own lists, the entries are reordered in LDS
//    and stored in runs.
//  - Steps with larger rectangles: a list's mask is the AND of one per column and
//    one per row, in whose lines the entries set their bits.
//  - Steps with larger rectangles or more list entries number the entries of all
//    lists and let each lane find the list and the set bit of its numbers, so that
//    a wave's work follows the entries and not its largest rectangle (100k splats
//    of 15 tiles each, the last kernel: 39 us with every lane walking its own
//    lists, 21 so; 6M splats of 2 tiles: 76 us by cell masks, 81 by lines, whose
//    few words every lane of a wave hits).
// base[] holds the lists' next positions and is advanced; the masks are zero
// before and after.
//  - Steps with more than kManyTotal go list by list instead, a wave's entries of
//    one list in one store: about 10 instructions a wave and list whatever its
//    entries, against about 85 per 64 list entries (the sum breaks even near 20,000
//    of the 131,072 that 512 whole-supertile rectangles have).
constexpr uint32_t kFewCells = 16;
constexpr uint32_t kManyTotal = 20000;

template <uint32_t kD, uint32_t kLines>
struct Ranker {
  static constexpr uint32_t kRow = kLines > kD ? kLines : kD;
  uint64_t mask[kW][kRow];  // per list, or (lines) per column, then per row
  uint16_t pre[kW][kD];     // a list's entries in the waves before
  uint32_t base[kD], start[kD];
  uint32_t word[kStage], meta[kStage];
  uint32_t tmp[kW];
  uint32_t large[2];  // whether the step's (by parity) entries hold large rectangles

  static __device__ bool is_large(const Cells& c) {
    return c.any && (c.x1 - c.x0 + 1u) * (c.y1 - c.y0 + 1u) > kFewCells;
  }
  __device__ void clear() {
    for (uint32_t i = threadIdx.x; i < kW * kRow; i += kT) (&mask[0][0])[i] = 0ull;
  }
  __device__ uint64_t of(bool lines, uint32_t w, uint32_t d, uint32_t x, uint32_t y, uint32_t cols) const {
    return lines ? mask[w][x] & mask[w][cols + y] : mask[w][d];
  }

  // All steps of a chunk: load(first, entry) gives this lane's entry of the 512
  // from `first` on (any = false past the end).  A step's entries are loaded
  // while the step before it runs.
  struct Entry {
    Cells cells;
    uint32_t slot;
    TileRect rect;
  };
  template <typename Load, typename Extra, typename Put>
  __device__ void run(uint32_t begin, uint32_t end, uint32_t lists, uint32_t cols, float inv_cols, Load&& load,
                      Extra&& extra, Put&& put) {
    if (threadIdx.x < 2) large[threadIdx.x] = 0u;
    clear();
    __syncthreads();
    Entry e = load(begin);
    if (is_large(e.cells)) large[0] = 1u;
    __syncthreads();
    uint32_t parity = 0;
    for (uint32_t at = begin; at < end; at += kT, parity ^= 1u) {
      Entry next = {};
      if (at + kT < end) next = load(at + kT);
      step(large[parity] != 0u, e, lists, cols, inv_cols, extra, put);
      if (threadIdx.x == 0) large[parity] = 0u;
      if (is_large(next.cells)) large[parity ^ 1u] = 1u;
      __syncthreads();
      e = next;
    }
  }

  // lists: their number; extra(rect, x, y): 16 bits stored with a slot; put(position, slot, extra)
  template <typename Extra, typename Put>
  __device__ void step(bool lines, const Entry& entry, uint32_t lists, uint32_t cols, float inv_cols, Extra&& extra,
                       Put&& put) {
    const uint32_t tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    const unsigned long long bit = 1ull << lane;
    const Cells& cells = entry.cells;
    const TileRect rect = entry.rect;
    const uint32_t slot = entry.slot;
    if (lines) {
      if (cells.any) {
        for (uint32_t x = cells.x0; x <= cells.x1; ++x)
          atomicOr(reinterpret_cast<unsigned long long*>(&mask[w][x]), bit);
        for (uint32_t y = cells.y0; y <= cells.y1; ++y)
          atomicOr(reinterpret_cast<unsigned long long*>(&mask[w][cols + y]), bit);
      }
    } else {
      for_cells(cells, cols, [&](uint32_t d, uint32_t, uint32_t) {
        atomicOr(reinterpret_cast<unsigned long long*>(&mask[w][d]), bit);
      });
    }
    __syncthreads();
    uint32_t count = 0;
    if (tid < lists) {
      uint32_t x, y;
      row_col(tid, cols, inv_cols, y, x);
#pragma unroll
      for (int i = 0; i < kW; ++i) {
        pre[i][tid] = (uint16_t)count;
        count += (uint32_t)__popcll(of(lines, i, tid, x, y, cols));
      }
    }
    uint32_t total;
    const uint32_t at = block_exclusive(count, tmp, &total);
    if (tid < kD) start[tid] = at;
    __syncthreads();
    if (!lines && total <= kStage) {
      for_cells(cells, cols, [&](uint32_t d, uint32_t x, uint32_t y) {
        const uint32_t p = start[d] + pre[w][d] + (uint32_t)__popcll(mask[w][d] & (bit - 1ull));
        word[p] = slot;
        meta[p] = d | (extra(rect, x, y) << 16);
      });
      __syncthreads();
      for (uint32_t p = tid; p < total; p += kT) {
        const uint32_t m = meta[p], d = m & 0xffffu;
        put(base[d] + p - start[d], word[p], m >> 16);
      }
    } else if (total > kManyTotal) {
      // list by list: a wave stores its entries of one list at a time
      for (uint32_t d0 = 0; d0 < lists; d0 += kWave) {
        const uint32_t d = d0 + lane;
        uint32_t x, y, at_d = 0;
        row_col(d, cols, inv_cols, y, x);
        uint64_t m = 0;
        if (d < lists) {
          m = of(lines, w, d, x, y, cols);
          at_d = base[d] + pre[w][d];
        }
        uint64_t todo = __ballot(m != 0);
        while (todo) {
          const uint32_t l = (uint32_t)__builtin_ctzll(todo);
          todo &= todo - 1;
          const uint64_t mine = ((uint64_t)lane_u32((uint32_t)(m >> 32), l) << 32) | lane_u32((uint32_t)m, l);
          const uint32_t pos = lane_u32(at_d, l) + mbcnt(mine);
          const uint32_t lx = lane_u32(x, l), ly = lane_u32(y, l);
          if (mine & bit) put(pos, slot, extra(rect, lx, ly));
        }
      }
    } else {
      word[tid] = slot;
      meta[tid] = rect.x;
      meta[kT + tid] = rect.y;
      __syncthreads();
      for (uint32_t p = tid; p < total; p += kT) {
        uint32_t d = 0;  // the last list that starts at or before p
#pragma unroll
        for (uint32_t h = kD / 2; h > 0; h >>= 1)
          if (start[d + h] <= p) d += h;
        uint32_t r = p - start[d], i = 0;
        const uint32_t pos = base[d] + r;
#pragma unroll
        for (uint32_t h = kW / 2; h > 0; h >>= 1)
          if (pre[i + h][d] <= r) i += h;
        r -= pre[i][d];
        uint32_t x, y;
        row_col(d, cols, inv_cols, y, x);
        const uint32_t e = i * kWave + select_bit(of(lines, i, d, x, y, cols), r);
        put(pos, word[e], extra(TileRect{meta[e], meta[kT + e]}, x, y));
      }
    }
    __syncthreads();
    if (tid < kD) base[tid] += count;
    clear();
  }
};

// The rectangle's part inside supertile (sx, sy): x0, x1, y0, y1 in 4 bits each.
__device__ __forceinline__ uint32_t local_rect(const TileRect& r, uint32_t sx, uint32_t sy) {
  const uint32_t ox = sx << kSuperShift, oy = sy << kSuperShift, top = (1u << kSuperShift) - 1u;
  const uint32_t x0 = r.x & 0xffffu, x1 = r.x >> 16, y0 = r.y & 0xffffu, y1 = r.y >> 16;
  const uint32_t lx0 = x0 > ox ? x0 - ox : 0u, lx1 = min(x1 - ox, top);
  const uint32_t ly0 = y0 > oy ? y0 - oy : 0u, ly1 = min(y1 - oy, top);
  return lx0 | (lx1 << 4) | (ly0 << 8) | (ly1 << 12);
}

// Where the draw order's pairs reach max_pairs: in chunk `chunk`, whose entries
// before position `at` are kept whole.  Of entry `at` the first tiles are kept, as up
// to two rectangles: whole rows of its own, then the start of the next row.  Nothing
// after it is kept.
struct Cut {
  uint32_t chunk, at, pieces;
  TileRect piece[2];
};

// The cut of a frame with more than max_pairs pairs, found by every workgroup for
// itself (such a frame is drawn again with more room).  counts[] gets the kept
// items per supertile of the cut chunk, in LDS as words[] (2 kMaxGrid) and cut;
// chunk_pairs are the chunks' pairs, in 64 bits: whole-frame splats pass 2^32 at 33k.
template <typename Items>
__device__ __forceinline__ void find_cut(const Items& in, uint32_t n, uint32_t live, uint32_t max_pairs,
                                         const uint32_t* __restrict__ chunk_pairs, uint32_t supers_x,
                                         uint32_t lists, uint32_t* words, uint32_t* counts, uint32_t* tmp, Cut* cut) {
  const uint32_t tid = threadIdx.x, size = chunk_subs(n, gridDim.x) * kT;
  for (uint32_t i = tid; i < 2 * kMaxGrid; i += kT) words[i] = i < 2 * live ? chunk_pairs[i] : 0u;
  for (uint32_t i = tid; i < lists; i += kT) counts[i] = 0u;
  __syncthreads();
  if (tid < kWave) {  // the first chunk after which more than max_pairs are reached
    constexpr uint32_t kEach = kMaxGrid / kWave;
    auto pairs_of = [&](uint32_t i) { return words[2 * i] | (uint64_t)words[2 * i + 1] << 32; };
    uint64_t inc = 0;
    for (uint32_t i = 0; i < kEach; ++i) inc += pairs_of(tid * kEach + i);
    const uint64_t own = inc;
    for (uint32_t d = 1; d < (uint32_t)kWave; d <<= 1) {
      const uint64_t t = (uint64_t)__shfl_up((unsigned long long)inc, d, kWave);
      if (tid >= d) inc += t;
    }
    uint64_t run = inc - own;
    if (run <= max_pairs && inc > max_pairs) {
      uint32_t i = tid * kEach;
      while (run + pairs_of(i) <= max_pairs) run += pairs_of(i++);
      cut->chunk = i;
      words[0] = (uint32_t)(max_pairs - run);
    }
  }
  __syncthreads();
  uint32_t room = words[0];
  for (uint32_t first = cut->chunk * size;; first += kT) {  // (ends where the room does, inside the chunk)
    const uint32_t k = first + tid;
    uint32_t slot, c = 0, all;
    TileRect r = {0u, 0u};
    if (k < n) in.load(k, slot, r, c);
    const uint32_t o = block_exclusive(c, tmp, &all);
    auto count = [&](const TileRect& t, uint32_t tiles) {
      for_cells(super_cells(t, tiles), supers_x, [&](uint32_t d, uint32_t, uint32_t) { atomicAdd(&counts[d], 1u); });
    };
    if (o + c <= room) {
      count(r, c);
    } else if (o <= room) {  // one entry
      const uint32_t x0 = r.x & 0xffffu, w = (r.x >> 16) - x0 + 1u, y0 = r.y & 0xffffu;
      const uint32_t rows = (room - o) / w, left = (room - o) % w;
      const TileRect whole = {r.x, y0 | ((y0 + rows - 1u) << 16)};
      const TileRect part = {x0 | ((x0 + left - 1u) << 16), (y0 + rows) | ((y0 + rows) << 16)};
      cut->at = k;
      cut->pieces = (rows ? 1u : 0u) + (left ? 1u : 0u);
      cut->piece[0] = rows ? whole : part;
      cut->piece[1] = part;
      count(whole, rows);
      count(part, left);
    }
    if (all > room || first + kT >= n) break;  // workgroup-uniform
    room -= all;
  }
  __syncthreads();
}

// max_chunks: chunks of level two besides one per supertile.
template <uint32_t kD, typename Items>
__global__ __launch_bounds__(kT, 8) void super_move_kernel(Items in, const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                        uint32_t supers_x, const uint32_t* __restrict__ hist,
                                                        Table table, uint32_t max_chunks, uint32_t max_items,
                                                        const uint32_t* __restrict__ d_pairs,
                                                        const uint32_t* __restrict__ status,
                                                        uint32_t* __restrict__ item_slot,
                                                        uint32_t* __restrict__ item_rect) {
  // max_items: max_pairs, which is at least the kept items
  __shared__ Ranker<kD, kMaxLines> s;
  __shared__ Cut s_cut;
  const uint32_t n = min(*d_count, max_n), tid = threadIdx.x, S = table.S;
  const float inv_cols = __builtin_amdgcn_rcpf((float)supers_x);
  Chunk ch = chunk_of(n);
  if (ch.begin >= ch.end && blockIdx.x != 0) return;  // workgroup-uniform
  uint32_t kept = ch.live, cut_at = 0xffffffffu;  // kept: whole chunks
  if (*d_pairs > max_items || *status != 0u) {
    find_cut(in, n, ch.live, max_items, hist + (size_t)gridDim.x * S, supers_x, S, s.word, s.start, s.tmp, &s_cut);
    kept = s_cut.chunk;
    if (ch.id > kept) return;  // workgroup-uniform (block 0 has chunk 0)
    if (ch.id == kept) {
      cut_at = s_cut.at;
      ch.end = cut_at + s_cut.pieces;
    }
  }
  uint32_t total = 0, before = 0;
  if (gridDim.x <= kRawGrid) {
    // the rows of all chunks, kParts of them at a time
    constexpr uint32_t kParts = kT / kD;
    const uint32_t d = tid % kD, part = tid / kD;
    for (uint32_t b0 = part; b0 < kept; b0 += 8 * kParts) {
      uint32_t h[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t b = b0 + j * kParts;
        h[j] = b < kept && d < S ? hist[(size_t)b * S + d] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        total += h[j];
        before += b0 + j * kParts < ch.id ? h[j] : 0u;
      }
    }
    s.word[tid] = total;
    s.meta[tid] = before;
    __syncthreads();
    total = before = 0;
    if (tid < kD)
#pragma unroll
      for (uint32_t p = 0; p < kParts; ++p) {
        total += s.word[p * kD + tid];
        before += s.meta[p * kD + tid];
      }
  } else if (tid < S) {
    total = kept < ch.live ? hist[(size_t)tid * gridDim.x + kept] : table.totals()[tid];
    before = hist[(size_t)tid * gridDim.x + ch.id];  // (of no use where there are no chunks)
  }
  if (kept < ch.live && tid < S) total += s.start[tid];  // the cut chunk's
  uint32_t all;
  const uint32_t smaller = block_exclusive(tid < S ? total : 0u, s.tmp, &all);
  if (tid < kD) s.base[tid] = smaller + before;
  if (blockIdx.x == 0) {  // the supertiles' item ranges and their chunks
    const uint32_t items = min(all, max_items);
    // items of a chunk: whole steps of 512 where they make enough chunks to
    // fill the GPU, part steps below that
    const uint32_t steps = (items + kT - 1) / kT;
    uint32_t per = steps >= 512u ? (steps + 2047u) / 2048u * kT : steps >= 128u ? kT / 2 : kT / 4;
    if (items > (uint64_t)per * max_chunks) per = ((items + max_chunks - 1) / max_chunks + kT - 1) / kT * kT;
    const uint32_t o = min(smaller, max_items), c = min(smaller + total, max_items) - o;
    uint32_t top = tid < S ? c : 0u;  // the largest supertile's
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) top = max(top, (uint32_t)__shfl_xor((int)top, d, kWave));
    if (tid % kWave == 0) s.tmp[tid / kWave] = top;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kW; ++i) top = max(top, s.tmp[i]);
    __syncthreads();
    if (top > (uint64_t)kManyChunks * per) per = max(per, ((uint32_t)(3.f * sqrtf((float)top)) + kT - 1) / kT * kT);
    uint32_t chunks;
    const uint32_t first = block_exclusive(tid < S ? (c + per - 1) / per : 0u, s.tmp, &chunks);
    if (tid < S) {
      table.offsets()[tid] = o;
      table.chunks()[tid] = first;
    }
    if (tid == 0) {
      table.offsets()[S] = items;
      table.chunks()[S] = chunks;
      *table.per_chunk() = per;
    }
  }
  __syncthreads();
  s.run(
      ch.begin, ch.end, S, supers_x, inv_cols,
      [&](uint32_t first) {
        const uint32_t k = first + tid;
        uint32_t slot = 0, c = 0;
        TileRect r = {0u, 0u};
        if (k < ch.end) in.load(min(k, cut_at), slot, r, c);
        if (k >= cut_at && k < ch.end) r = s_cut.piece[k - cut_at];
        return typename Ranker<kD, kMaxLines>::Entry{super_cells(r, c), slot, r};
      },
      [](const TileRect& t, uint32_t x, uint32_t y) { return local_rect(t, x, y); },
      [&](uint32_t pos, uint32_t v, uint32_t lr) {
        if (pos < max_items) {
          item_slot[pos] = v;
          item_rect[pos] = lr;
        }
      });
}

__device__ __forceinline__ Cells tile_cells(uint32_t lr, bool any) {
  return Cells{lr & 15u, (lr >> 4) & 15u, (lr >> 8) & 15u, lr >> 12, any};
}

// This workgroup's chunk of level two: its supertile and items [begin, end);
// first = the supertile's first chunk, id = this one.  s_find: one word of LDS.
struct ItemChunk {
  uint32_t super, first, id, begin, end;
  bool any;
};

__device__ __forceinline__ ItemChunk item_chunk(const Table& table, uint32_t* s_find) {
  const uint32_t S = table.S, live = table.chunks()[S], per = *table.per_chunk();
  ItemChunk c = {0u, 0u, 0u, 0u, 0u, false};
  if (blockIdx.x >= live) return c;  // workgroup-uniform
  c.any = true;
  c.id = deal(blockIdx.x, live);
  // the last supertile whose first chunk is not after this one (an empty one
  // has its successor's first chunk)
  if (threadIdx.x < S) {
    const uint32_t a = table.chunks()[threadIdx.x], b = table.chunks()[threadIdx.x + 1];
    if (a <= c.id && c.id < b) *s_find = threadIdx.x;
  }
  __syncthreads();
  c.super = *s_find;
  c.first = table.chunks()[c.super];
  const uint32_t o = table.offsets()[c.super], e = table.offsets()[c.super + 1];
  c.begin = o + (c.id - c.first) * per;
  c.end = min(c.begin + per, e);
  return c;
}

// Tile `local` of a supertile in the frame's grid; false outside it.
__device__ __forceinline__ bool frame_tile(uint32_t super, uint32_t local, uint32_t supers_x, uint32_t tiles_x,
                                           uint32_t tiles_y, uint32_t& tile) {
  const uint32_t m = (1u << kSuperShift) - 1u;
  const uint32_t x = ((super % supers_x) << kSuperShift) + (local & m);
  const uint32_t y = ((super / supers_x) << kSuperShift) + (local >> kSuperShift);
  tile = y * tiles_x + x;
  return x < tiles_x && y < tiles_y;
}

// Small rectangles count cell by cell, larger ones by their corners in a
// difference grid that is summed over rows and columns at the end: four adds an
// item whatever its size.
__global__ __launch_bounds__(kT) void tile_count_kernel(Table table, const uint32_t* __restrict__ item_rect,
                                                        uint32_t supers_x, uint32_t tiles_x, uint32_t tiles_y,
                                                        uint32_t* __restrict__ rows, uint32_t* __restrict__ tile_cnt) {
  constexpr uint32_t kCopies = 16, kSide = 1u << kSuperShift, kGrid = kSide + 1u;
  __shared__ uint32_t s_h[kSuperTiles * kCopies];
  __shared__ uint32_t s_diff[kGrid * kGrid];
  __shared__ uint32_t s_find;
  const uint32_t tid = threadIdx.x;
  const ItemChunk ch = item_chunk(table, &s_find);
  if (!ch.any) return;
  for (uint32_t i = tid; i < kSuperTiles * kCopies; i += kT) s_h[i] = 0u;
  for (uint32_t i = tid; i < kGrid * kGrid; i += kT) s_diff[i] = 0u;
  __syncthreads();
  for (uint32_t k = ch.begin + tid; k < ch.end; k += kT) {
    const Cells c = tile_cells(item_rect[k], true);
    if ((c.x1 - c.x0 + 1u) * (c.y1 - c.y0 + 1u) <= 4u) {
      for_cells(c, kSide, [&](uint32_t d, uint32_t, uint32_t) { atomicAdd(&s_h[d * kCopies + tid % kCopies], 1u); });
    } else {
      atomicAdd(&s_diff[c.y0 * kGrid + c.x0], 1u);
      atomicAdd(&s_diff[c.y0 * kGrid + c.x1 + 1u], ~0u);
      atomicAdd(&s_diff[(c.y1 + 1u) * kGrid + c.x0], ~0u);
      atomicAdd(&s_diff[(c.y1 + 1u) * kGrid + c.x1 + 1u], 1u);
    }
  }
  __syncthreads();
  if (tid < kGrid) {
    uint32_t run = 0;
    for (uint32_t x = 0; x < kGrid; ++x) s_diff[tid * kGrid + x] = run += s_diff[tid * kGrid + x];
  }
  __syncthreads();
  if (tid < kGrid) {
    uint32_t run = 0;
    for (uint32_t y = 0; y < kGrid; ++y) s_diff[y * kGrid + tid] = run += s_diff[y * kGrid + tid];
  }
  __syncthreads();
  if (tid < kSuperTiles) {
    uint32_t v = s_diff[(tid / kSide) * kGrid + tid % kSide];
#pragma unroll
    for (uint32_t j = 0; j < kCopies; ++j) v += s_h[tid * kCopies + (j + tid) % kCopies];
    rows[(size_t)ch.id * kSuperTiles + tid] = v;
    uint32_t tile;
    if (v && frame_tile(ch.super, tid, supers_x, tiles_x, tiles_y, tile)) atomicAdd(&tile_cnt[tile], v);
  }
}

// [start, end) of every tile's list, clipped at max_pairs ([0, 0) where empty);
// each workgroup takes kT * 4 tiles and sums the counts before them.
__global__ __launch_bounds__(kT) void tile_scan_kernel(const uint32_t* __restrict__ tile_cnt, uint32_t tiles,
                                                       const uint32_t* __restrict__ d_pairs, uint32_t max_pairs,
                                                       uint32_t* __restrict__ ranges, uint32_t* __restrict__ status,
                                                       uint32_t* __restrict__ order_counts) {
  // the tile schedule's counts of this block's tiles, in copies that spread the
  // crowded buckets over banks (its own launch took 4.5 us more a frame)
  constexpr uint32_t kCopies = 8;
  static_assert(kTileOrderChunk == 4 * kT, "a chunk of the schedule per workgroup");
  __shared__ uint32_t s_order[256 * kCopies];
  __shared__ uint32_t s_tmp[kW];
  const uint32_t tid = threadIdx.x, first = blockIdx.x * kT * 4;
  if (order_counts)
    for (uint32_t i = tid; i < 256 * kCopies; i += kT) s_order[i] = 0u;  // (block_exclusive's barriers follow)
  uint32_t acc = 0;
  const uint4* c4 = reinterpret_cast<const uint4*>(tile_cnt);
  for (uint32_t i = tid; i < first / 4; i += 8 * kT) {  // 8 loads in flight
    uint4 v[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) v[j] = i + j * kT < first / 4 ? c4[i + j * kT] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) acc += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  uint32_t before;
  block_exclusive(acc, s_tmp, &before);
  uint32_t x[4], s = 0;
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t t = first + tid * 4 + j;
    x[j] = t < tiles ? tile_cnt[t] : 0u;
    s += x[j];
  }
  uint32_t all;
  uint32_t run = before + block_exclusive(s, s_tmp, &all);
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t t = first + tid * 4 + j;
    const uint32_t a = min(run, max_pairs), b = min(run + x[j], max_pairs);
    if (t < tiles) {
      reinterpret_cast<uint2*>(ranges)[t] = a < b ? make_uint2(a, b) : make_uint2(0u, 0u);
      if (order_counts) atomicAdd(&s_order[tile_order_key(b - a) * kCopies + tid % kCopies], 1u);
    }
    run += x[j];
  }
  if (order_counts) {  // workgroup-uniform
    __syncthreads();
    if (tid < 256) {
      uint32_t n = 0;
#pragma unroll
      for (uint32_t j = 0; j < kCopies; ++j) n += s_order[tid * kCopies + (j + tid) % kCopies];
      order_counts[blockIdx.x * 256 + tid] = n;
    }
  }
  if (blockIdx.x == 0 && tid == 0 && *d_pairs > max_pairs) *status = 1u;
}

__global__ __launch_bounds__(kT, 8) void tile_move_kernel(Table table, const uint32_t* __restrict__ item_slot,
                                                       const uint32_t* __restrict__ item_rect, uint32_t supers_x,
                                                       uint32_t tiles_x, uint32_t tiles_y,
                                                       const uint32_t* __restrict__ rows,
                                                       const uint32_t* __restrict__ ranges, uint32_t max_pairs,
                                                       uint32_t* __restrict__ vals) {
  __shared__ Ranker<kSuperTiles, 2u << kSuperShift> s;
  __shared__ uint32_t s_find;
  const uint32_t tid = threadIdx.x;
  const ItemChunk ch = item_chunk(table, &s_find);
  if (!ch.any) return;
  {
    // a tile's next position: its list's start + its pairs in the supertile's earlier chunks
    constexpr uint32_t kParts = kT / kSuperTiles;
    const uint32_t d = tid % kSuperTiles, part = tid / kSuperTiles;
    uint32_t before = 0;
    for (uint32_t b0 = ch.first + part; b0 < ch.id; b0 += 8 * kParts) {
      uint32_t h[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t b = b0 + j * kParts;
        h[j] = b < ch.id ? rows[(size_t)b * kSuperTiles + d] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) before += h[j];
    }
    s.word[tid] = before;
    __syncthreads();
    uint32_t tile;
    if (tid < kSuperTiles)
      s.base[tid] = s.word[tid] + s.word[kSuperTiles + tid] +
                    (frame_tile(ch.super, tid, supers_x, tiles_x, tiles_y, tile) ? ranges[2 * (size_t)tile] : 0u);
    __syncthreads();
  }
  s.run(
      ch.begin, ch.end, kSuperTiles, 1u << kSuperShift, 1.f / (float)(1u << kSuperShift),
      [&](uint32_t first) {
        const uint32_t k = first + tid;
        const bool valid = k < ch.end;
        const uint32_t slot = valid ? item_slot[k] : 0u, lr = valid ? item_rect[k] : 0u;
        return Ranker<kSuperTiles, 2u << kSuperShift>::Entry{tile_cells(lr, valid), slot, TileRect{0u, 0u}};
      },
      [](const TileRect&, uint32_t, uint32_t) { return 0u; },
      [&](uint32_t pos, uint32_t v, uint32_t) {
        if (pos < max_pairs) vals[pos] = v;
      });
}

template <typename Items>
hipError_t launch_lists(Items in, const uint32_t* d_count, uint32_t max_n, const RasterShape& rs, uint64_t max_pairs,
                        const TileListBuffers& b, hipStream_t s) {
  const uint32_t sx = ceil_div(rs.tiles_x, 1u << kSuperShift), S = sx * ceil_div(rs.tiles_y, 1u << kSuperShift);
  const uint32_t tiles = rs.tiles_x * rs.tiles_y;
  const uint32_t parts = ceil_div(max_n ? max_n : 1, kT);
  // few chunks where the movers sum their counts, up to four parts a chunk;
  // enough of them to fill the GPU above that
  uint32_t grid = parts <= 4 * kRawGrid ? (parts < kRawGrid ? parts : kRawGrid) : kMaxGrid;
  if (grid > parts) grid = parts;
  if (grid > b.row_words / (S + 2)) grid = b.row_words / (S + 2);  // two rows more: the chunks' pairs
  uint32_t chunks = b.row_words / kSuperTiles - S;  // of level two besides one per supertile
  if (chunks > kMaxChunks) chunks = kMaxChunks;
  const uint32_t few = 8 * parts > 64 ? 8 * parts : 64;
  if (chunks > few) chunks = few;
  const Table table = {b.table, S};
  const uint32_t cap = (uint32_t)max_pairs;
  super_count_kernel<Items><<<grid, kT, 0, s>>>(in, d_count, max_n, sx, S, b.rows, b.pairs, b.status, b.tile_cnt,
                                                tiles);
  if (grid > kRawGrid) super_scan_kernel<<<S, 256, 0, s>>>(b.rows, grid, d_count, max_n, table);
  if (S <= 64)
    super_move_kernel<64, Items><<<grid, kT, 0, s>>>(in, d_count, max_n, sx, b.rows, table, chunks, cap, b.pairs,
                                                     b.status, b.item_slot, b.item_rect);
  else if (S <= 128)
    super_move_kernel<128, Items><<<grid, kT, 0, s>>>(in, d_count, max_n, sx, b.rows, table, chunks, cap, b.pairs,
                                                      b.status, b.item_slot, b.item_rect);
  else if (S <= 256)
    super_move_kernel<256, Items><<<grid, kT, 0, s>>>(in, d_count, max_n, sx, b.rows, table, chunks, cap, b.pairs,
                                                      b.status, b.item_slot, b.item_rect);
  else
    super_move_kernel<512, Items><<<grid, kT, 0, s>>>(in, d_count, max_n, sx, b.rows, table, chunks, cap, b.pairs,
                                                      b.status, b.item_slot, b.item_rect);
  tile_count_kernel<<<chunks + S, kT, 0, s>>>(table, b.item_rect, sx, rs.tiles_x, rs.tiles_y, b.rows, b.tile_cnt);
  tile_scan_kernel<<<ceil_div(tiles, kT * 4), kT, 0, s>>>(b.tile_cnt, tiles, b.pairs, cap, b.ranges, b.status,
                                                             b.order_counts);
  tile_move_kernel<<<chunks + S, kT, 0, s>>>(table, b.item_slot, b.item_rect, sx, rs.tiles_x, rs.tiles_y, b.rows,
                                             b.ranges, cap, b.vals);
  return hipGetLastError();
}

}  // namespace

bool tile_lists_fit(const RasterShape& rs, uint32_t row_words) {
  const uint32_t x = ceil_div(rs.tiles_x, 1u << kSuperShift), y = ceil_div(rs.tiles_y, 1u << kSuperShift);
  return x * y <= kMaxSupers && x + y <= kMaxLines && 2 * x * y <= row_words / kSuperTiles;
}

hipError_t launch_tile_lists_packed(const uint64_t* val64, const RectBits& rb, const uint32_t* d_count, uint32_t max_n,
                                    const RasterShape& rs, uint64_t max_pairs, const TileListBuffers& b,
                                    hipStream_t s) {
  return launch_lists(PackedItems{val64, rb}, d_count, max_n, rs, max_pairs, b, s);
}

hipError_t launch_tile_lists(const TileRect* rect, const uint32_t* cnt, const uint32_t* order, const uint32_t* d_count,
                             uint32_t max_n, const RasterShape& rs, uint64_t max_pairs, const TileListBuffers& b,
                             hipStream_t s) {
  return launch_lists(RectItems{rect, cnt, order}, d_count, max_n, rs, max_pairs, b, s);
}

}  // namespace vkgs
