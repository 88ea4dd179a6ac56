// LSD radix sort (reduce-then-scan) and device-wide exclusive scan for gfx950.
//
// Replaces the reference's external sorter (vrdxCmdSortKeyValueIndirect,
// engine.cc:1218-1219; "reduce-then-scan", DETAILS.md:26-30).  Each pass of
// up to 8 key bits (9 in wide plans) runs two or three kernels:
//   upsweep   : every block counts the digits of its contiguous chunk with
//               one LDS atomic per key into bank-interleaved copies of the
//               histogram, then writes its counts;
//   scan      : one workgroup per digit turns the counts into exclusive offsets
//               (no launch for grids of at most kRawGrid blocks, whose
//               downsweep blocks sum the counts themselves);
//   downsweep : every block walks its chunk in 2048-key sub-tiles, ranks keys
//               stably (wave multisplit: ballots + LDS counters, then a
//               cross-wave prefix), reorders the sub-tile in LDS and writes
//               runs of equal digits contiguously to global memory.
// Sorts of at most kSmallSort pairs (kSmallShort with few bits) are one kernel of one workgroup instead.
// The narrow digit of a key width that is not a multiple of 8 goes first
// unless the caller names another pass (depth keys, see sort.h).  No
// block ever waits on another block, so the sort cannot hang on forward
// progress.  Counts are read from device memory (indirect semantics) or given
// by the host; the grid is fixed by the capacity and each block derives its
// chunk from the count.  Values are 32 or 64 bits.
//
// The exclusive scan is two kernels: block sums, then each block adds the
// sums before it and scans its chunk through LDS.
#pragma clang fp contract(off)

#include "common.h"
#include "device.h"
#include "sort.h"

namespace vkgs {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kIpt = 8;  // keys per thread per sub-tile
constexpr int kTile = kThreads * kIpt;  // keys per sub-tile
constexpr int kMaxBlocks = 1024;
// A scan's apply blocks each sum the partials before them, which stays cheap
// at twice the sort's grid and gives the binning scan more waves in flight
// (6M splats: bin 0.063 -> 0.059 ms; the sort itself is fastest at 1024).
constexpr int kMaxScanBlocks = 2048;
// Grids of up to this many blocks (393,216 pairs) take two launches a pass: every
// downsweep block sums the block counts itself, 4 digits of 64 chunks' rows at a time.
// Sorts of 32 bits, us, with three launches and two: 131k pairs 62, 50; 160k 58, 53;
// 300k 61, 58; 400k 63, 62; 524k 65, 67.  (One digit of 16 rows at a time: 300k 81, 524k
// 107.)
constexpr uint32_t kRawGrid = 192;
// Larger grids whose live count fills at most this many chunks (a pair list far
// shorter than its storage) do the same: their row-scan launch returns at once.
constexpr uint32_t kRawChunks = 64;
// Grids of up to this many blocks (524,288 pairs), which leave compute units idle, run
// 512 threads of 4 keys each: a pass is then a chain of latencies, and the ranking
// rounds of a wave are half as many (300k pairs, 32 bits: 66 us with 256 threads, 61).
constexpr uint32_t kSmallGrid = 256;
constexpr int kSmallGridThreads = 512;
constexpr uint32_t kXcds = 8;  // consecutive workgroups go round the dies

__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  const int lane = __lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t t = __shfl_up(v, d, kWave);
    if (lane >= d) v += t;
  }
  return v;
}

// Exclusive scan across the workgroup; s_tmp holds one word per wave.
template <int kBlock>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_tmp, uint32_t* total) {
  constexpr int kNw = kBlock / kWave;
  const int lane = __lane_id();
  const int w = threadIdx.x / kWave;
  const uint32_t incl = wave_inclusive_scan(v);
  if (lane == kWave - 1) s_tmp[w] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kNw; ++i) {
    const uint32_t t = s_tmp[i];
    off += (i < w) ? t : 0u;
    tot += t;
  }
  __syncthreads();
  *total = tot;
  return off + incl - v;
}

// Contiguous chunk of block blockIdx.x of a scan; chunks are multiples of kTile.
__device__ __forceinline__ void block_range(uint32_t n, uint32_t& begin, uint32_t& end) {
  const uint64_t per = ((uint64_t)n + gridDim.x - 1) / gridDim.x;
  const uint64_t chunk = (per + kTile - 1) / kTile * kTile;
  const uint64_t b = (uint64_t)blockIdx.x * chunk;
  begin = (uint32_t)(b < n ? b : n);
  end = (uint32_t)(b + chunk < n ? b + chunk : n);
}

// The part of n pairs that this workgroup of a sort takes: chunk `id` of `live`
// chunks of whole sub-tiles, [begin, end).  The live chunks are dealt so that
// each die takes consecutive ones: a digit's runs of consecutive chunks are
// adjacent in the output, and their partial lines then meet in one L2 (sorts of 24
// bits, us, as they come and dealt: 600k pairs 67, 64; 2M 96, 92; 3.5M 131, 120; 6.2M
// 186, 182).  Not where that measured slower: single sub-tiles on some three
// workgroups a compute unit (1.3M 79, 83) and chunks of four and more (8M 226, 230).
struct SortChunk {
  uint32_t id, live, begin, end;
};

__device__ __forceinline__ SortChunk sort_chunk(uint32_t n) {
  const uint32_t grid = gridDim.x, b = blockIdx.x;
  const uint32_t sub = (uint32_t)(((uint64_t)n + kTile - 1) / kTile);
  const uint32_t per = (sub + grid - 1) / grid;  // sub-tiles per chunk
  SortChunk c;
  c.live = per ? (sub + per - 1) / per : 0u;
  c.id = b;
  if (b < c.live && (per == 1 ? c.live <= 512 || c.live > 928 : per < 4)) {
    const uint32_t die = b % kXcds, q = c.live / kXcds, r = c.live % kXcds;
    c.id = die * q + min(die, r) + b / kXcds;
  }
  const uint64_t size = (uint64_t)per * kTile, begin = (uint64_t)c.id * size;
  c.begin = (uint32_t)(begin < n ? begin : n);
  c.end = (uint32_t)(begin + size < n ? begin + size : n);
  return c;
}

// Four words by one load.  A caller's storage need not be aligned to more than a word.
typedef uint32_t Words4 __attribute__((ext_vector_type(4), aligned(4)));

// Block counts as one row of digits per chunk, summed by the downsweep itself,
// instead of one row of chunks per digit that a scan launch turns into offsets.
__device__ __forceinline__ bool raw_counts(uint32_t grid, uint32_t live) {
  return grid <= kRawGrid || live <= kRawChunks;
}

// A pass of a pair of passes that the keys' largest value makes unneeded:
// every key's bits from skip_shift up are zero, so that pair would keep the
// order (a stable sort on an all-zero digit), and both of its passes return
// at once.  The pass count still has its parity, so the result lands where
// the full sort would put it.
__device__ __forceinline__ bool pass_skipped(uint32_t key_max, uint32_t skip_shift) {
  return skip_shift < 32 && (key_max >> skip_shift) == 0u;
}

// The keys' maximum for a sort given d_key_max, without atomics: the first
// pass's blocks store their own maxima in block_max (max_mode 1), and block 0
// of the second pass reduces them into *key_max (max_mode 2), before any pass
// that tests it.
enum : uint32_t { kMaxNone = 0, kMaxPerBlock = 1, kMaxReduce = 2 };

// Sort inputs: arrays, or the longest-first schedule of tiles: key tile_order_key
// of the tile's list length, value the tile, so that an ascending stable pass puts
// long lists first.  Lengths within 1/8 of an octave share a bucket, which is fine
// for a schedule.
template <typename T>
struct ArrayInput {
  const T* p;
  __device__ T operator()(uint32_t i) const { return p[i]; }
};
struct IndexInput {
  __device__ uint32_t operator()(uint32_t i) const { return i; }
};
struct TileLengthInput {
  const uint2* ranges;
  __device__ uint32_t operator()(uint32_t i) const {
    const uint2 r = ranges[i];
    return tile_order_key(r.y - r.x);
  }
};

// The count and the keys' maximum (both in flight at once).
__device__ __forceinline__ void load_counts(const uint32_t* d_count, uint32_t max_n, const uint32_t* d_key_max,
                                            uint32_t& n, uint32_t& key_max) {
  const uint32_t c = d_count ? *d_count : max_n;
  key_max = d_key_max ? *d_key_max : 0xffffffffu;
  n = min(c, max_n);
}

template <int kBits, int kT, typename Keys>
__global__ __launch_bounds__(kT) void sort_upsweep(Keys keys, const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                   uint32_t shift, uint32_t* __restrict__ hist,
                                                   const uint32_t* __restrict__ d_key_max, uint32_t skip_shift,
                                                   uint32_t max_mode, uint32_t* __restrict__ block_max,
                                                   uint32_t* __restrict__ key_max) {
  constexpr int kK = 1 << kBits, kN = kTile / kT;
  // a histogram needs no ranking: one LDS atomic per key, into one of kCopies
  // copies of the histogram chosen by lane (lane l counts into copy l %
  // kCopies), bin d of copy j at word kCopies d + j.  Depth keys crowd into few
  // digit values: lanes with the same digit then mostly count into different
  // copies, whose words for that bin sit in different banks.  (8-bit digits:
  // with 4 copies per wave the 4 depth passes took 0.186 ms; with 16
  // interleaved copies 0.168 ms; with 64, 0.193 ms, the clearing and summing
  // costing more.)
  constexpr int kCopies = 4096 / kK < 8 ? 8 : 4096 / kK > 64 ? 64 : 4096 / kK;
  __shared__ uint32_t s_h[kK * kCopies];
  __shared__ uint32_t s_wmax[kT / kWave];
  uint32_t n, top;
  load_counts(d_count, max_n, d_key_max, n, top);
  if (pass_skipped(top, skip_shift)) return;
  const SortChunk c = sort_chunk(n);
  const uint32_t tid = threadIdx.x;
  uint32_t k[kN];
#pragma unroll
  for (int r = 0; r < kN; ++r) {
    const uint32_t i = c.begin + r * kT + tid;
    k[r] = i < c.end ? keys(i) : 0u;  // (0 for the padding: no effect on the maximum)
  }
  uint32_t* h = s_h + (tid % kCopies);
  for (uint32_t i = tid; i < kK * kCopies; i += kT) s_h[i] = 0u;
  __syncthreads();
  const uint32_t mask = kK - 1u;
  uint32_t kmax = 0;
  for (uint32_t base = c.begin; base < c.end; base += kTile) {
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      kmax = max(kmax, k[r]);
      if (base + r * kT + tid < c.end) atomicAdd(&h[((k[r] >> shift) & mask) * kCopies], 1u);
    }
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      const uint32_t i = base + kTile + r * kT + tid;
      k[r] = i < c.end ? keys(i) : 0u;
    }
  }
  if (max_mode == kMaxReduce && blockIdx.x == 0) {
    kmax = 0;
    for (uint32_t b = tid; b < gridDim.x; b += kT) kmax = max(kmax, block_max[b]);
  }
  if (max_mode != kMaxNone) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, d, kWave));
    if (__lane_id() == 0) s_wmax[tid / kWave] = kmax;
  }
  __syncthreads();
  if (max_mode != kMaxNone && tid == 0) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < kT / kWave; ++i) m = max(m, s_wmax[i]);
    if (max_mode == kMaxPerBlock)
      block_max[c.id] = m;
    else if (blockIdx.x == 0)
      *key_max = m;
  }
  if (tid < (uint32_t)kK) {
    // thread d reads its bin's copies rotated by d, so the lanes' reads fall
    // in distinct banks
    uint32_t s = 0;
#pragma unroll 16
    for (int j = 0; j < kCopies; ++j) s += s_h[tid * kCopies + ((j + tid) % kCopies)];
    if (!raw_counts(gridDim.x, c.live))
      hist[(size_t)tid * gridDim.x + c.id] = s;
    else if (c.id < c.live)
      hist[(size_t)c.id * kK + tid] = s;
  }
}

// Exclusive scan of one digit's row hist[d][0..blocks) in place (one workgroup
// per digit); digit_total[d] receives the row sum.
__global__ __launch_bounds__(kThreads) void sort_scan_rows(uint32_t* __restrict__ hist, uint32_t blocks,
                                                           uint32_t* __restrict__ digit_total,
                                                           const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                           const uint32_t* __restrict__ d_key_max,
                                                           uint32_t skip_shift) {
  __shared__ uint32_t s_tmp[kWaves];
  static_assert(kMaxBlocks <= kThreads * 4, "4 words a thread");
  uint32_t* row = hist + (size_t)blockIdx.x * blocks;
  const uint32_t first = threadIdx.x * 4;
  uint32_t x[4];  // in flight beside the count (read after it, a pass of 1.2M pairs took 1 us more)
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = first + j < blocks ? row[first + j] : 0u;
  uint32_t n, top;
  load_counts(d_count, max_n, d_key_max, n, top);
  if (pass_skipped(top, skip_shift)) return;
  const uint32_t sub = (uint32_t)(((uint64_t)n + kTile - 1) / kTile), per = (sub + blocks - 1) / blocks;
  const uint32_t live = per ? (sub + per - 1) / per : 0u;
  if (raw_counts(blocks, live)) return;
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) s += first + j < live ? x[j] : 0u;
  uint32_t all;
  uint32_t run = block_exclusive_scan<kThreads>(s, s_tmp, &all);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (first + j < live) row[first + j] = run;
    run += x[j];
  }
  if (threadIdx.x == 0) digit_total[blockIdx.x] = all;
}

template <int kBits, int kT, typename V, typename Keys, typename Vals>
__global__ __launch_bounds__(kT) void sort_downsweep(Keys kin, Vals vin, uint32_t* __restrict__ kout,
                                                     V* __restrict__ vout, const uint32_t* __restrict__ d_count,
                                                     uint32_t max_n, uint32_t shift,
                                                     const uint32_t* __restrict__ hist,
                                                     const uint32_t* __restrict__ digit_total,
                                                     const uint32_t* __restrict__ d_key_max, uint32_t skip_shift) {
  constexpr int kK = 1 << kBits, kN = kTile / kT, kW = kT / kWave;
  static_assert(kK <= kT, "one digit per thread");
  __shared__ uint32_t s_base[kK];
  __shared__ uint32_t s_wcnt[kW][kK];
  __shared__ uint32_t s_start[kK];
  __shared__ uint32_t s_tmp[kW];
  __shared__ uint32_t s_key[kTile];
  __shared__ V s_val[kTile];

  uint32_t n, top;
  load_counts(d_count, max_n, d_key_max, n, top);
  if (pass_skipped(top, skip_shift)) return;
  const SortChunk ch = sort_chunk(n);
  if (ch.begin >= ch.end) return;  // workgroup-uniform
  const uint32_t tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
  constexpr uint32_t mask = kK - 1u;
  uint32_t k[kN], rank[kN];
  V v[kN];
  auto load = [&](uint32_t base) {
    const uint32_t seg = base + w * (kWave * kN);
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      const uint32_t i = seg + r * kWave + lane;
      const bool valid = i < ch.end;
      k[r] = valid ? kin(i) : 0u;
      v[r] = valid ? vin(i) : V(0);
    }
  };
  load(ch.begin);  // in flight while the digits' offsets are formed
  for (uint32_t i = tid; i < kW * kK; i += kT) s_wcnt[0][i] = 0u;
  {
    // global offset of digit tid for this chunk: keys of smaller digits
    // everywhere plus keys of this digit in earlier chunks
    uint32_t total = 0, before = 0;
    if (raw_counts(gridDim.x, ch.live)) {
      // the rows of all chunks: 4 digits a thread, kParts rows at a time, 8 loads in flight per thread
      constexpr uint32_t kVec = kK < 4 ? 1 : 4, kFly = 8;
      constexpr uint32_t kCols = kK / kVec < 16 ? 16 : kK / kVec, kParts = kT / kCols;
      static_assert(kParts * kK <= kTile, "the parts' sums fit the sub-tile's words");
      const uint32_t d = tid % kCols * kVec, part = tid / kCols;
      uint32_t t[kVec] = {}, f[kVec] = {};
      for (uint32_t b0 = part; b0 < ch.live; b0 += kFly * kParts) {
        uint32_t h[kFly][kVec];
#pragma unroll
        for (uint32_t j = 0; j < kFly; ++j) {
          const uint32_t b = b0 + j * kParts;
          const bool in = b < ch.live && d < (uint32_t)kK;
          if constexpr (kVec == 4) {
            Words4 x = {};
            if (in) x = *reinterpret_cast<const Words4*>(hist + (size_t)b * kK + d);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) h[j][i] = x[i];
          } else {
            h[j][0] = in ? hist[(size_t)b * kK + d] : 0u;
          }
        }
#pragma unroll
        for (uint32_t j = 0; j < kFly; ++j)
#pragma unroll
          for (uint32_t i = 0; i < kVec; ++i) {
            t[i] += h[j][i];
            f[i] += b0 + j * kParts < ch.id ? h[j][i] : 0u;
          }
      }
      uint32_t* s_before = reinterpret_cast<uint32_t*>(s_val);
#pragma unroll
      for (uint32_t i = 0; i < kVec; ++i)
        if (d < (uint32_t)kK) {
          s_key[part * kK + d + i] = t[i];
          s_before[part * kK + d + i] = f[i];
        }
      __syncthreads();
      if (tid < (uint32_t)kK)
#pragma unroll
        for (uint32_t p = 0; p < kParts; ++p) {
          total += s_key[p * kK + tid];
          before += s_before[p * kK + tid];
        }
    } else if (tid < (uint32_t)kK) {
      total = digit_total[tid];
      before = hist[(size_t)tid * gridDim.x + ch.id];
    }
    uint32_t all;
    const uint32_t smaller = block_exclusive_scan<kT>(tid < (uint32_t)kK ? total : 0u, s_tmp, &all);
    if (tid < (uint32_t)kK) s_base[tid] = smaller + before;
  }
  __syncthreads();

  for (uint32_t base = ch.begin; base < ch.end; base += kTile) {
    const uint32_t cnt = min((uint32_t)kTile, ch.end - base);
    const uint32_t seg = base + w * (kWave * kN);
    if (base != ch.begin) load(base);
    // stable rank inside this wave's segment, 64 keys at a time.  The wave
    // owns its counter row, so no atomics: every lane reads its digit's count,
    // then the first lane of each digit group writes count + group size.  LDS
    // operations of one wave complete in issue order, so the reads of a row
    // see the writes of the rows before it and none of its own.
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      const bool valid = seg + r * kWave + lane < ch.end;
      const uint32_t d = (k[r] >> shift) & mask;
      const uint64_t peers = match_digit<kBits>(d, valid);
      const uint32_t below = mbcnt(peers);
      const uint32_t old = valid ? s_wcnt[w][d] : 0u;
      __builtin_amdgcn_wave_barrier();
      if (valid && below == 0) s_wcnt[w][d] = old + (uint32_t)__popcll(peers);
      __builtin_amdgcn_wave_barrier();
      rank[r] = old + below;
    }
    __syncthreads();
    // per digit: exclusive prefix over waves, then over digits
    uint32_t total_d = 0;
    if (tid < (uint32_t)kK) {
#pragma unroll
      for (int i = 0; i < kW; ++i) {
        const uint32_t c = s_wcnt[i][tid];
        s_wcnt[i][tid] = total_d;
        total_d += c;
      }
    }
    uint32_t all;
    const uint32_t start = block_exclusive_scan<kT>(total_d, s_tmp, &all);
    if (tid < (uint32_t)kK) s_start[tid] = start;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      const bool valid = seg + r * kWave + lane < ch.end;
      if (valid) {
        const uint32_t d = (k[r] >> shift) & mask;
        const uint32_t pos = s_start[d] + s_wcnt[w][d] + rank[r];
        if (pos < (uint32_t)kTile) {
          s_key[pos] = k[r];
          s_val[pos] = v[r];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kN; ++j) {
      const uint32_t idx = j * kT + tid;
      if (idx < cnt) {
        const uint32_t kk = s_key[idx];
        const uint32_t d = (kk >> shift) & mask;
        const uint32_t dst = s_base[d] + idx - s_start[d];
        if (dst < n) {
          if (kout) kout[dst] = kk;
          vout[dst] = s_val[idx];
        }
      }
    }
    if (base + kTile >= ch.end) break;  // workgroup-uniform
    __syncthreads();
    if (tid < (uint32_t)kK) s_base[tid] += total_d;
    for (uint32_t i = tid; i < kW * kK; i += kT) s_wcnt[0][i] = 0u;
    __syncthreads();
  }
}

// Scan inputs: plain words, or the tile count of the packed rectangle in the
// high word of 64-bit sort values.
struct LoadWords {
  static constexpr uint32_t kSmallScan = 3u << 13;  // see scan_small
  const uint32_t* p;
  __device__ uint32_t operator()(uint32_t i) const { return p[i]; }
};
struct LoadRectCount {
  static constexpr uint32_t kSmallScan = 1u << 13;
  const uint64_t* v;
  RectBits rb;
  __device__ uint32_t operator()(uint32_t i) const {
    uint32_t c;
    unpack_rect((uint32_t)(v[i] >> 32), rb, &c);
    return c;
  }
};

template <typename Load>
__global__ __launch_bounds__(kThreads) void scan_reduce(Load in, const uint32_t* __restrict__ d_count,
                                                        uint32_t max_n, uint32_t* __restrict__ partial) {
  __shared__ uint32_t s_tmp[kWaves];
  const uint32_t n = d_count ? min(*d_count, max_n) : max_n;
  uint32_t begin, end;
  block_range(n, begin, end);
  uint32_t s = 0;
  for (uint32_t i = begin + threadIdx.x; i < end; i += kThreads) s += in(i);
  uint32_t all;
  block_exclusive_scan<kThreads>(s, s_tmp, &all);
  if (threadIdx.x == 0) partial[blockIdx.x] = all;
}

// partial[] holds the raw per-block sums of scan_reduce: each block adds up
// those of the blocks before it (a few per thread) instead of a separate
// single-workgroup scan launch; the last block also writes *d_total.
template <typename Load>
__global__ __launch_bounds__(kThreads) void scan_apply(Load in, uint32_t* out, const uint32_t* __restrict__ d_count,
                                                       uint32_t max_n, const uint32_t* __restrict__ partial,
                                                       uint32_t* __restrict__ d_total) {
  // the sub-tile passes through LDS so that global loads and stores are
  // lane-strided (coalesced) while each thread scans kIpt consecutive words;
  // index i is stored at i + i / 32, which spreads a thread's run over banks
  __shared__ uint32_t s_tmp[kWaves];
  __shared__ uint32_t s_x[kTile + kTile / 32];
  const uint32_t tid = threadIdx.x;
  const uint32_t n = d_count ? min(*d_count, max_n) : max_n;
  uint32_t begin, end;
  block_range(n, begin, end);
  uint32_t carry;
  {
    uint32_t before = 0;
    for (uint32_t i = tid; i < blockIdx.x; i += kThreads) before += partial[i];
    block_exclusive_scan<kThreads>(before, s_tmp, &carry);
    if (d_total != nullptr && tid == 0 && blockIdx.x == gridDim.x - 1) *d_total = carry + partial[blockIdx.x];
  }
  for (uint32_t base = begin; base < end; base += kTile) {
#pragma unroll
    for (int r = 0; r < kIpt; ++r) {
      const uint32_t i = r * kThreads + tid;
      s_x[i + (i >> 5)] = base + i < end ? in(base + i) : 0u;
    }
    __syncthreads();
    uint32_t x[kIpt];
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < kIpt; ++j) {
      const uint32_t i = tid * kIpt + j;
      x[j] = s_x[i + (i >> 5)];
      s += x[j];
    }
    uint32_t all;
    uint32_t run = carry + block_exclusive_scan<kThreads>(s, s_tmp, &all);
#pragma unroll
    for (int j = 0; j < kIpt; ++j) {
      const uint32_t i = tid * kIpt + j;
      s_x[i + (i >> 5)] = run;
      run += x[j];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kIpt; ++r) {
      const uint32_t i = r * kThreads + tid;
      if (base + i < end) out[base + i] = s_x[i + (i >> 5)];
    }
    __syncthreads();
    carry += all;
  }
}

// A whole scan of at most Load::kSmallScan words in one workgroup, in place of two
// launches.  Bound by the latency of its steps of 8192 words: one step 4.4-4.7 us
// against 9.2-9.7 of two launches, three steps of words 7.1 against 7.1 (and a launch
// less for the host), of packed rectangles 12.4 against 10.1.
constexpr int kSmallScanThreads = 1024;
constexpr int kSmallScanTile = kSmallScanThreads * kIpt;

template <typename Load>
__global__ __launch_bounds__(kSmallScanThreads) void scan_small(Load in, uint32_t* out,
                                                                const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                                uint32_t* __restrict__ d_total) {
  __shared__ uint32_t s_tmp[kSmallScanThreads / kWave];
  __shared__ uint32_t s_x[kSmallScanTile + kSmallScanTile / 32];  // as scan_apply's
  const uint32_t tid = threadIdx.x, n = d_count ? min(*d_count, max_n) : max_n;
  uint32_t carry = 0, next[kIpt];
#pragma unroll
  for (uint32_t r = 0; r < (uint32_t)kIpt; ++r) {
    const uint32_t i = r * kSmallScanThreads + tid;
    next[r] = i < n ? in(i) : 0u;
  }
  for (uint32_t base = 0; base < n; base += kSmallScanTile) {
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)kIpt; ++r) {
      const uint32_t i = r * kSmallScanThreads + tid, k = base + kSmallScanTile + i;
      s_x[i + (i >> 5)] = next[r];
      next[r] = k < n ? in(k) : 0u;
    }
    __syncthreads();
    uint32_t x[kIpt], s = 0, all;
#pragma unroll
    for (uint32_t j = 0; j < (uint32_t)kIpt; ++j) {
      const uint32_t i = tid * kIpt + j;
      x[j] = s_x[i + (i >> 5)];
      s += x[j];
    }
    uint32_t run = carry + block_exclusive_scan<kSmallScanThreads>(s, s_tmp, &all);
#pragma unroll
    for (uint32_t j = 0; j < (uint32_t)kIpt; ++j) {
      const uint32_t i = tid * kIpt + j;
      s_x[i + (i >> 5)] = run;
      run += x[j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)kIpt; ++r) {
      const uint32_t i = r * kSmallScanThreads + tid;
      if (base + i < n) out[base + i] = s_x[i + (i >> 5)];
    }
    __syncthreads();
    carry += all;
  }
  if (d_total != nullptr && tid == 0) *d_total = carry;
}

// A whole sort of at most kSmallSort pairs in one workgroup: the keys and the
// pairs' places in the input go round LDS, digits of up to 9 bits, and the values
// are gathered once at the end.  A wave holds consecutive pairs, 64 a round, and
// ranks a round by ballots against its own counters; the waves' counts are then
// summed per digit.  Bound by its chain of LDS steps and barriers, which beats the
// launches of three passes up to this size: frames at 320x240 and 640x400, us, with
// passes and with this: 100 splats 59, 47; 5k 71, 63; 8192 76, 74.
// Keys of up to two of its digits (18 bits) take it up to 6144 only: 16 bits, us, with
// passes and with this: 5k pairs 27, 25; 6k 27, 27; 7k 28, 29; 8192 28, 32.
constexpr uint32_t kSmallSort = 8192, kSmallShort = 6144;
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
constexpr int kSmallRounds = kSmallSort / kSmallThreads;

template <typename V>
__global__ __launch_bounds__(kSmallThreads) void sort_small(const uint32_t* kin, const V* vin, uint32_t* kout, V* vout,
                                                            const uint32_t* __restrict__ d_count, uint32_t max_n,
                                                            uint32_t key_bits) {
  constexpr uint32_t kDigits = 512;
  __shared__ uint32_t s_key[kSmallSort];
  __shared__ uint16_t s_from[kSmallSort];
  __shared__ uint32_t s_count[kSmallWaves][kDigits];
  __shared__ uint32_t s_base[kDigits], s_sum[kDigits / kWave];
  const uint32_t n = d_count ? min(*d_count, max_n) : max_n;
  if (n == 0) return;
  const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid / kWave;
  const uint32_t rounds = (n + kSmallThreads - 1) / kSmallThreads, first = w * rounds * kWave + lane;
  const uint32_t passes = (key_bits + 8) / 9, width = (key_bits + passes - 1) / passes;
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t key[kSmallRounds], from[kSmallRounds], rank[kSmallRounds];
#pragma unroll
  for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
    from[r] = first + r * kWave;
    key[r] = r < rounds && from[r] < n ? kin[from[r]] : 0u;
  }
  for (uint32_t shift = 0; shift < key_bits; shift += width) {
    const uint32_t bits = min(width, key_bits - shift), mask = (1u << bits) - 1u;
    for (uint32_t i = tid; i < (uint32_t)kSmallWaves * kDigits; i += kSmallThreads) (&s_count[0][0])[i] = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
      if (r >= rounds) break;  // workgroup-uniform
      const bool live = first + r * kWave < n;
      const uint32_t d = (key[r] >> shift) & mask;
      uint64_t same = __ballot(live);
#pragma unroll
      for (uint32_t b = 0; b < 9; ++b) {  // bits above the digit's width are 0 in every lane
        const uint64_t m = __ballot((d >> b) & 1u);
        same &= m ^ (((d >> b) & 1u) - 1ull);
      }
      const uint32_t before = (uint32_t)__popcll(same & below);
      const uint32_t had = s_count[w][d];
      rank[r] = had + before;
      __builtin_amdgcn_wave_barrier();  // a wave's LDS operations complete in order
      if (live && before == 0) s_count[w][d] = had + (uint32_t)__popcll(same);
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // a digit's counts to offsets over the waves, the digits' totals to bases
    uint32_t total = 0, inc = 0;
    if (tid < kDigits) {
#pragma unroll
      for (int v = 0; v < kSmallWaves; ++v) {
        const uint32_t c = s_count[v][tid];
        s_count[v][tid] = total;
        total += c;
      }
      inc = wave_inclusive_scan(total);
      if (lane == kWave - 1) s_sum[w] = inc;
    }
    __syncthreads();
    if (tid < kDigits) {
      uint32_t off = 0;
#pragma unroll
      for (uint32_t v = 0; v < kDigits / kWave; ++v) off += v < w ? s_sum[v] : 0u;
      s_base[tid] = off + inc - total;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
      if (r < rounds && first + r * kWave < n) {
        const uint32_t d = (key[r] >> shift) & mask, at = s_base[d] + s_count[w][d] + rank[r];
        s_key[at] = key[r];
        s_from[at] = (uint16_t)from[r];
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
      const uint32_t i = first + r * kWave;
      if (r < rounds && i < n) {
        key[r] = s_key[i];
        from[r] = s_from[i];
      }
    }
    // (the next pass writes these only after its barriers)
  }
  // the values before any is overwritten: the output may be the input
  V v[kSmallRounds];
#pragma unroll
  for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
    const uint32_t i = first + r * kWave;
    v[r] = r < rounds && i < n ? vin[from[r]] : V(0);
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < (uint32_t)kSmallRounds; ++r) {
    const uint32_t i = first + r * kWave;
    if (r < rounds && i < n) {
      kout[i] = key[r];
      vout[i] = v[r];
    }
  }
}

template <typename V>
__global__ void copy_pairs(const uint32_t* __restrict__ ks, const V* __restrict__ vs, uint32_t* __restrict__ kd,
                           V* __restrict__ vd, const uint32_t* __restrict__ d_count, uint32_t max_n) {
  const uint32_t n = d_count ? min(*d_count, max_n) : max_n;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    kd[i] = ks[i];
    vd[i] = vs[i];
  }
}

__global__ void fill_u32(uint32_t* __restrict__ dst, uint32_t value, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = value;
}

__global__ void set_words(uint32_t* __restrict__ dst, Words16 words, uint32_t n) {
  if (threadIdx.x < n) dst[threadIdx.x] = words.w[threadIdx.x];
}

struct WordChunk {
  uint32_t w[kUploadChunkWords];
};

__global__ __launch_bounds__(256) void set_chunk(uint32_t* __restrict__ dst, WordChunk chunk, uint32_t n,
                                                 uint32_t* __restrict__ clear, uint32_t n_clear) {
  if (threadIdx.x < n_clear) clear[threadIdx.x] = 0u;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = chunk.w[i];
}

}  // namespace

SortPlan sort_plan(uint32_t max_n, uint32_t val_bytes, bool wide) {
  SortPlan p;
  p.max_n = max_n;
  uint32_t tiles = ceil_div(max_n ? max_n : 1, kTile);
  p.blocks = tiles < (uint32_t)kMaxBlocks ? tiles : (uint32_t)kMaxBlocks;
  p.digits = wide && p.blocks <= kSmallGrid ? 512u : 256u;
  size_t off = 0;
  p.off_alt_key = off;
  off = align_up(off + (size_t)max_n * 4, 256);
  p.off_alt_val = off;
  off = align_up(off + (size_t)max_n * val_bytes, 256);
  p.off_hist = off;
  off = align_up(off + (size_t)p.digits * p.blocks * 4, 256);
  p.off_digit_total = off;
  off = align_up(off + p.digits * 4, 256);
  p.off_block_max = off;
  off = align_up(off + (size_t)p.blocks * 4, 256);
  p.bytes = off;
  return p;
}

namespace {

// Digit widths of a sort, first pass first: 8 bits each except the narrow
// pass's remainder; with first_bits (1-7) the first pass that many and the last
// the remainder; a wide plan's 25 to 27 bits in three passes of 8 or 9.
struct Digits {
  uint32_t width[5] = {};
  uint32_t passes = 0;
};

Digits digits_of(const SortPlan& plan, uint32_t key_bits, uint32_t narrow_pass, uint32_t first_bits) {
  Digits d;
  if (plan.digits > 256 && key_bits > 24 && key_bits <= 27) {
    d.passes = 3;
    for (uint32_t p = 0; p < 3; ++p) d.width[p] = key_bits - 24 > 2 - p ? 9u : 8u;
  } else if (first_bits > 0 && first_bits < 8 && key_bits > first_bits) {
    d.passes = 1 + (key_bits - first_bits + 7) / 8;
    for (uint32_t p = 0; p < d.passes; ++p) d.width[p] = p == 0 ? first_bits : 8u;
    d.width[d.passes - 1] = key_bits - first_bits - 8 * (d.passes - 2);
  } else {
    d.passes = (key_bits + 7) / 8;
    const uint32_t narrow_at = narrow_pass < d.passes ? narrow_pass : d.passes - 1;
    for (uint32_t p = 0; p < d.passes; ++p) d.width[p] = p == narrow_at ? key_bits - 8 * (d.passes - 1) : 8u;
  }
  return d;
}

struct PassArgs {
  const uint32_t* d_count;
  uint32_t shift, skip_shift, max_mode;
  uint32_t* d_key_max;  // nullptr: no pass is skipped
};

// One pass: the counts (unless counted), the row scan (larger grids) and the move.
template <int kBits, int kT, typename V, typename Keys, typename Vals>
void sort_pass(const SortPlan& plan, Keys kin, Vals vin, uint32_t* kout, V* vout, const PassArgs& a, char* base,
               hipStream_t stream, bool counted = false) {
  uint32_t* hist = reinterpret_cast<uint32_t*>(base + plan.off_hist);
  uint32_t* digit_total = reinterpret_cast<uint32_t*>(base + plan.off_digit_total);
  uint32_t* block_max = reinterpret_cast<uint32_t*>(base + plan.off_block_max);
  if (!counted)
    sort_upsweep<kBits, kT, Keys><<<plan.blocks, kT, 0, stream>>>(kin, a.d_count, plan.max_n, a.shift, hist,
                                                                 a.d_key_max, a.skip_shift, a.max_mode, block_max,
                                                                 a.d_key_max);
  if (plan.blocks > kRawGrid)
    sort_scan_rows<<<1u << kBits, kThreads, 0, stream>>>(hist, plan.blocks, digit_total, a.d_count, plan.max_n,
                                                         a.d_key_max, a.skip_shift);
  sort_downsweep<kBits, kT, V, Keys, Vals><<<plan.blocks, kT, 0, stream>>>(
      kin, vin, kout, vout, a.d_count, plan.max_n, a.shift, hist, digit_total, a.d_key_max, a.skip_shift);
}

template <typename V>
hipError_t sort_launch(const SortPlan& plan, const uint32_t* d_count, uint32_t* keys, V* vals, uint32_t key_bits,
                       void* storage, hipStream_t stream, bool input_in_alt = false, uint32_t narrow_pass = 0,
                       uint32_t* d_key_max = nullptr, uint32_t first_bits = 0) {
  if (key_bits > 32) key_bits = 32;
  char* base = static_cast<char*>(storage);
  uint32_t* alt_k = reinterpret_cast<uint32_t*>(base + plan.off_alt_key);
  V* alt_v = reinterpret_cast<V*>(base + plan.off_alt_val);
  if (plan.max_n == 0) return hipSuccess;
  if (key_bits == 0) {
    if (input_in_alt) copy_pairs<V><<<1024, 256, 0, stream>>>(alt_k, alt_v, keys, vals, d_count, plan.max_n);
    return hipGetLastError();
  }
  uint32_t* src_k = input_in_alt ? alt_k : keys;
  V* src_v = input_in_alt ? alt_v : vals;
  if (plan.max_n <= (key_bits <= 18 ? kSmallShort : kSmallSort)) {
    sort_small<V><<<1, kSmallThreads, 0, stream>>>(src_k, src_v, keys, vals, d_count, plan.max_n, key_bits);
    return hipGetLastError();
  }
  uint32_t* dst_k = input_in_alt ? keys : alt_k;
  V* dst_v = input_in_alt ? vals : alt_v;
  const Digits digits = digits_of(plan, key_bits, narrow_pass, first_bits);
  // with d_key_max and four passes, passes 0 and 1 find the keys' maximum and
  // passes 2 and 3 run only if it has a bit at or above pass 2's shift (as a
  // pair, so the result stays where four passes put it)
  const bool skipping = d_key_max && digits.passes == 4;
  const uint32_t pair_shift = digits.width[0] + digits.width[1];  // shift of pass 2
  PassArgs a = {d_count, 0u, 32u, kMaxNone, skipping ? d_key_max : nullptr};
  for (uint32_t pass = 0; pass < digits.passes; ++pass) {
    a.skip_shift = skipping && pass >= 2 ? pair_shift : 32u;
    a.max_mode = !skipping ? kMaxNone : pass == 0 ? kMaxPerBlock : pass == 1 ? kMaxReduce : kMaxNone;
    const ArrayInput<uint32_t> kin{src_k};
    const ArrayInput<V> vin{src_v};
    const bool small = plan.blocks <= kSmallGrid;
    switch (digits.width[pass]) {
#define VKGS_PASS(B)                                                                                  \
  case B:                                                                                             \
    if (small)                                                                                        \
      sort_pass<B, kSmallGridThreads, V>(plan, kin, vin, dst_k, dst_v, a, base, stream);                    \
    else                                                                                              \
      sort_pass<B, kThreads, V>(plan, kin, vin, dst_k, dst_v, a, base, stream);                       \
    break;
      VKGS_PASS(1)
      VKGS_PASS(2)
      VKGS_PASS(3)
      VKGS_PASS(4)
      VKGS_PASS(5)
      VKGS_PASS(6)
      VKGS_PASS(7)
      VKGS_PASS(8)
#undef VKGS_PASS
      case 9:  // wide plans only, which are small
        sort_pass<9, kSmallGridThreads, V>(plan, kin, vin, dst_k, dst_v, a, base, stream);
        break;
    }
    a.shift += digits.width[pass];
    uint32_t* tk = src_k;
    V* tv = src_v;
    src_k = dst_k;
    src_v = dst_v;
    dst_k = tk;
    dst_v = tv;
  }
  if (src_k != keys) copy_pairs<V><<<1024, 256, 0, stream>>>(src_k, src_v, keys, vals, d_count, plan.max_n);
  return hipGetLastError();
}

}  // namespace

hipError_t sort_kv_launch(const SortPlan& plan, const uint32_t* d_count, uint32_t* keys, uint32_t* vals,
                          uint32_t key_bits, void* storage, hipStream_t stream, uint32_t narrow_pass,
                          uint32_t* d_key_max, uint32_t first_bits, bool input_in_alt) {
  return sort_launch<uint32_t>(plan, d_count, keys, vals, key_bits, storage, stream, input_in_alt, narrow_pass,
                               d_key_max, first_bits);
}

uint32_t sort_passes(uint32_t key_bits) { return ((key_bits > 32 ? 32 : key_bits) + 7) / 8; }

bool sort_is_wide(const SortPlan& plan, uint32_t key_bits) {
  return plan.digits > 256 && key_bits > 24 && key_bits <= 27;
}

void sort_alt_buffers(const SortPlan& plan, void* storage, uint32_t** keys, uint32_t** vals) {
  char* base = static_cast<char*>(storage);
  *keys = reinterpret_cast<uint32_t*>(base + plan.off_alt_key);
  *vals = reinterpret_cast<uint32_t*>(base + plan.off_alt_val);
}

hipError_t sort_kv_from_alt_launch(const SortPlan& plan, const uint32_t* d_count, uint32_t* keys, uint32_t* vals,
                                   uint32_t key_bits, void* storage, hipStream_t stream) {
  return sort_launch<uint32_t>(plan, d_count, keys, vals, key_bits, storage, stream, true);
}

hipError_t sort_kv64_launch(const SortPlan& plan, const uint32_t* d_count, uint32_t* keys, uint64_t* vals,
                            uint32_t key_bits, void* storage, hipStream_t stream, uint32_t narrow_pass,
                            uint32_t* d_key_max, uint32_t first_bits, bool input_in_alt) {
  return sort_launch<uint64_t>(plan, d_count, keys, vals, key_bits, storage, stream, input_in_alt, narrow_pass,
                               d_key_max, first_bits);
}

uint32_t* sort_tile_order_counts(const SortPlan& plan, void* storage) {
  static_assert(kTileOrderChunk == (uint32_t)kTile, "a chunk of the pass is one sub-tile");
  if (plan.blocks > kRawGrid) return nullptr;  // up to there every block's chunk is one sub-tile
  return reinterpret_cast<uint32_t*>(static_cast<char*>(storage) + plan.off_hist);
}

hipError_t sort_tile_order_launch(const SortPlan& plan, const uint32_t* ranges, uint32_t* order, void* storage,
                                  hipStream_t stream, bool counted) {
  if (plan.max_n == 0) return hipSuccess;
  char* base = static_cast<char*>(storage);
  const PassArgs a = {nullptr, 0u, 32u, kMaxNone, nullptr};
  const TileLengthInput keys{reinterpret_cast<const uint2*>(ranges)};
  uint32_t* no_keys = nullptr;
  if (plan.blocks <= kSmallGrid)
    sort_pass<8, kSmallGridThreads, uint32_t>(plan, keys, IndexInput{}, no_keys, order, a, base, stream, counted);
  else
    sort_pass<8, kThreads, uint32_t>(plan, keys, IndexInput{}, no_keys, order, a, base, stream);
  return hipGetLastError();
}

ScanPlan scan_plan(uint32_t max_n) {
  ScanPlan p;
  p.max_n = max_n;
  uint32_t tiles = ceil_div(max_n ? max_n : 1, kTile);
  p.blocks = tiles < (uint32_t)kMaxScanBlocks ? tiles : (uint32_t)kMaxScanBlocks;
  p.off_partial = 0;
  p.bytes = align_up((size_t)p.blocks * 4, 256);
  return p;
}

namespace {

template <typename Load>
hipError_t scan_launch(const ScanPlan& plan, Load in, uint32_t* out, const uint32_t* d_count, uint32_t* d_total,
                       void* storage, hipStream_t stream) {
  if (plan.max_n <= Load::kSmallScan) {
    scan_small<Load><<<1, kSmallScanThreads, 0, stream>>>(in, out, d_count, plan.max_n, d_total);
    return hipGetLastError();
  }
  uint32_t* partial = reinterpret_cast<uint32_t*>(static_cast<char*>(storage) + plan.off_partial);
  scan_reduce<Load><<<plan.blocks, kThreads, 0, stream>>>(in, d_count, plan.max_n, partial);
  scan_apply<Load><<<plan.blocks, kThreads, 0, stream>>>(in, out, d_count, plan.max_n, partial, d_total);
  return hipGetLastError();
}

}  // namespace

hipError_t scan_exclusive_launch(const ScanPlan& plan, const uint32_t* in, uint32_t* out, const uint32_t* d_count,
                                 uint32_t* d_total, void* storage, hipStream_t stream) {
  return scan_launch(plan, LoadWords{in}, out, d_count, d_total, storage, stream);
}

hipError_t scan_rect_counts_launch(const ScanPlan& plan, const uint64_t* val64, const RectBits& rb, uint32_t* out,
                                   const uint32_t* d_count, uint32_t* d_total, void* storage, hipStream_t stream) {
  return scan_launch(plan, LoadRectCount{val64, rb}, out, d_count, d_total, storage, stream);
}

hipError_t fill_u32_launch(uint32_t* dst, uint32_t value, size_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  size_t blocks = (n + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  fill_u32<<<(uint32_t)blocks, 256, 0, stream>>>(dst, value, n);
  return hipGetLastError();
}

hipError_t upload_launch(void* dst, const void* src, size_t bytes, hipStream_t stream, uint32_t* clear,
                         uint32_t n_clear) {
  if (bytes % 4 != 0 || n_clear > 256 || (n_clear && bytes == 0)) return hipErrorInvalidValue;
  const uint32_t* s = static_cast<const uint32_t*>(src);
  uint32_t* d = static_cast<uint32_t*>(dst);
  for (size_t off = 0; off < bytes / 4; off += kUploadChunkWords) {
    const uint32_t n = (uint32_t)(bytes / 4 - off < kUploadChunkWords ? bytes / 4 - off : kUploadChunkWords);
    WordChunk c;
    for (uint32_t i = 0; i < n; ++i) c.w[i] = s[off + i];
    set_chunk<<<1, 256, 0, stream>>>(d + off, c, n, clear, off == 0 ? n_clear : 0u);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t set_words_launch(uint32_t* dst, const Words16& words, uint32_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  if (n > 16) return hipErrorInvalidValue;
  set_words<<<1, 64, 0, stream>>>(dst, words, n);
  return hipGetLastError();
}

}  // namespace vkgs
