// Row sorts for stablehlo.sort and chlo.top_k on gfx950.
//
// Replaces the reference's MLX sort / argsort / take_along_axis chain
// (reference: src/backend/mlx_metal/api.cc:3248-3347, dispatched from
// execution_node_indexing.zig:83-88 and execution_node_indexing_order.zig:
// 12-72, which sorts ascending and reverses for GT comparators). Here a
// descending order is an ascending sort of the inverted key image, so equal
// keys keep their positions' order in both directions (a stable sort, as
// StableHLO's is_stable and XLA's TopK ask).
//
// Kernels:
//  * sort_block: one workgroup sorts up to kSortTile words of a row in LDS by
//    merging: 16 words a thread by a register network, then runs of 16, 32,
//    ... by merge path, and keeps the first `keep` words or writes the results.
//  * merge_runs: merges neighbouring sorted runs of a row from HBM.
//  * topk_select: the first k <= 256 words of a chunk, without sorting it.
//  * merge_pieces: the first k words of rows whose positions a word does not
//    hold (2^30 and more), from those of their pieces.
//  * sort_local, bitonic_global, sort_write: a bitonic network over padded
//    rows in one buffer, for a caller whose fixed scratch block does not hold
//    the two buffers merging needs, and for whole sorts of such rows.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"
#include "kernels/sort.h"

namespace pjrtx {
namespace {

constexpr uint64_t kSentinel = ~0ull;  // sorts after every word (positions are < 2^31)
constexpr int kLocalThreads = 512;

struct LocalPass {
  // Source: raw keys of operand 0 (list == nullptr) or a list of words.
  const void* keys = nullptr;
  SortRows r;
  const uint64_t* list = nullptr;
  int64_t row_len = 0;        // words of a padded row
  int64_t blocks_per_row = 1;
  int64_t k_first = 2, k_last = 2, j_first = 1;
  uint64_t* dst = nullptr;
};

__device__ __forceinline__ uint32_t load_key(const void* keys, int64_t e, int bits) {
  if (bits == 32) return static_cast<const uint32_t*>(keys)[e];
  if (bits == 16) return static_cast<const uint16_t*>(keys)[e];
  return static_cast<const uint8_t*>(keys)[e];
}

// Order-preserving image of a key (ascending), inverted for descending: the
// key XOR one mask where its top bit is set and another where it is not, and
// for FLOAT compares one image for every NaN and one for both zeros. No branch
// per element.
struct KeyMap {
  uint32_t mask = 0, neg = 0, pos = 0, nan_over = 0, zero_keep = 0, nan_image = 0;
  int shift = 0;
};
__host__ __device__ __forceinline__ KeyMap key_map(const SortRows& r) {
  KeyMap m;
  m.mask = r.key_bits == 32 ? 0xffffffffu : ((1u << r.key_bits) - 1u);
  const uint32_t sign = 1u << (r.key_bits - 1), flip = r.descending ? m.mask : 0u;
  const bool fl = r.key_class == kSortKeyFloat, total = fl || r.key_class == kSortKeyTotal;
  m.neg = (total ? m.mask : r.key_class == kSortKeySigned ? sign : 0u) ^ flip;
  m.pos = (r.key_class == kSortKeyUnsigned ? 0u : sign) ^ flip;
  m.nan_over = fl ? r.inf_bits : 0xffffffffu;  // larger magnitudes are NaNs, after +inf
  m.zero_keep = fl ? 0u : 0xffffffffu;         // -0 == +0
  m.nan_image = m.mask ^ flip;
  m.shift = 32 - r.key_bits;
  return m;
}
__device__ __forceinline__ uint32_t key_image(uint32_t v, const KeyMap& m) {
  const uint32_t mag = v & (m.mask >> 1);
  v = mag == 0 ? v & m.zero_keep : v;
  const uint32_t neg = (uint32_t)((int32_t)(v << m.shift) >> 31);
  const uint32_t img = v ^ ((neg & m.neg) | (~neg & m.pos));
  return mag > m.nan_over ? m.nan_image : img;
}

template <typename T>
__device__ __forceinline__ void copy_elem(const void* src, void* dst, int64_t s, int64_t d) {
  static_cast<T*>(dst)[d] = static_cast<const T*>(src)[s];
}

// Result i of `row` comes from position `pos` of the same row.
__device__ __forceinline__ void gather_one(const SortGather& g, const SortRows& r, int64_t row, int64_t i,
                                           int64_t pos) {
  const int64_t outer = row / r.inner, j = row - outer * r.inner;
  const int64_t s = (outer * r.n + pos) * r.inner + j;
  const int64_t d = (outer * g.out_n + i) * r.inner + j;
  for (int o = 0; o < g.count; ++o) {
    if (!g.src[o]) {
      switch (g.elem_bytes[o]) {
        case 1: static_cast<uint8_t*>(g.dst[o])[d] = (uint8_t)pos; break;
        case 2: static_cast<uint16_t*>(g.dst[o])[d] = (uint16_t)pos; break;
        case 4: static_cast<uint32_t*>(g.dst[o])[d] = (uint32_t)pos; break;
        default: static_cast<uint64_t*>(g.dst[o])[d] = (uint64_t)pos; break;
      }
      continue;
    }
    switch (g.elem_bytes[o]) {
      case 1: copy_elem<uint8_t>(g.src[o], g.dst[o], s, d); break;
      case 2: copy_elem<uint16_t>(g.src[o], g.dst[o], s, d); break;
      case 4: copy_elem<uint32_t>(g.src[o], g.dst[o], s, d); break;
      default: copy_elem<uint64_t>(g.src[o], g.dst[o], s, d); break;
    }
  }
  if (g.index_dst) static_cast<int32_t*>(g.index_dst)[d] = static_cast<int32_t>(pos);
}

__global__ void __launch_bounds__(kLocalThreads) sort_local_kernel(LocalPass p) {
  __shared__ uint64_t s[kSortBlock];
  const int64_t row = blockIdx.x / p.blocks_per_row;
  const int64_t blk = blockIdx.x - row * p.blocks_per_row;
  const int64_t base = blk * kSortBlock;
  const int64_t outer = row / p.r.inner, j0 = row - outer * p.r.inner;
  const int64_t row0 = outer * p.r.n * p.r.inner + j0;
  constexpr int kBatch = kSortBlock / kLocalThreads;
  const KeyMap map = key_map(p.r);
  uint64_t w[kBatch];
#pragma unroll
  for (int q = 0; q < kBatch; ++q) {
    const int64_t idx = base + q * kLocalThreads + (int)threadIdx.x;
    if (p.list) w[q] = p.list[row * p.row_len + idx];
    else if (idx < p.r.n)
      w[q] = (static_cast<uint64_t>(key_image(load_key(p.keys, row0 + idx * p.r.inner, p.r.key_bits), map)) << 32) |
             static_cast<uint64_t>(idx);
    else w[q] = kSentinel;
  }
#pragma unroll
  for (int q = 0; q < kBatch; ++q) s[q * kLocalThreads + (int)threadIdx.x] = w[q];
  __syncthreads();
  for (int64_t k = p.k_first; k <= p.k_last; k <<= 1) {
    // Within a block only bit log2(k) of the row position matters: it is the
    // block's (base & k) when k >= kSortBlock, else the position's own bit.
    const bool block_up = k < kSortBlock || (base & k) == 0;
    const int kb = k < kSortBlock ? static_cast<int>(k) : 0;
    for (int64_t jj = (k == p.k_first ? p.j_first : k >> 1); jj > 0; jj >>= 1) {
      const int j = static_cast<int>(jj);
      for (int t = threadIdx.x; t < kSortBlock / 2; t += kLocalThreads) {
        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
        const int l = i | j;
        const bool up = block_up == ((i & kb) == 0);
        const uint64_t a = s[i], b = s[l];
        if ((a > b) == up) {
          s[i] = b;
          s[l] = a;
        }
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int q = 0; q < kBatch; ++q)
    p.dst[row * p.row_len + base + q * kLocalThreads + (int)threadIdx.x] = s[q * kLocalThreads + (int)threadIdx.x];
}

__global__ void bitonic_global_kernel(uint64_t* a, int64_t rows, int64_t p, int64_t k, int64_t j) {
  const int64_t half = p >> 1;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= rows * half) return;
  const int64_t row = t / half, tt = t - row * half;
  const int64_t i = ((tt & ~(j - 1)) << 1) | (tt & (j - 1));
  const int64_t l = i | j;
  const bool up = (i & k) == 0;
  uint64_t* r = a + row * p;
  const uint64_t x = r[i], y = r[l];
  if ((x > y) == up) {
    r[i] = y;
    r[l] = x;
  }
}

__global__ void sort_write_kernel(const uint64_t* list, int64_t list_stride, SortRows r, SortGather g) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= r.rows * g.out_n) return;
  const int64_t row = t / g.out_n, i = t - row * g.out_n;
  gather_one(g, r, row, i, static_cast<int64_t>(list[row * list_stride + i] & 0xffffffffu));
}

// ------------------------------------------------------------ merge sort
// A word is the 32-bit key image over 30 bits of position, 62 bits, held as a
// double: with the top two bits zero it is a finite non-negative double whose
// order is the word's, so a compare-exchange is one v_min_f64 and one
// v_max_f64 (a 64-bit integer one is a compare and four selects).
constexpr int kGroup = 8;           // words loaded together
constexpr int kSortThreads = 512;   // sort_block's largest workgroup, 16 words a thread
constexpr int kSortTile = 16 * kSortThreads;
constexpr int kMergeThreads = 512;
constexpr int kMergeItems = 8;
constexpr int kMergeTile = kMergeItems * kMergeThreads;
constexpr int64_t kWordRows = int64_t{1} << 30;  // positions a word holds
constexpr uint64_t kWordEnd = (uint64_t{1} << 62) - 1;  // after every word

__device__ __forceinline__ double as_word(uint64_t u) { return __builtin_bit_cast(double, u); }
__device__ __forceinline__ uint64_t word_bits(double w) { return __builtin_bit_cast(uint64_t, w); }
__device__ __forceinline__ double make_word(uint32_t image, int64_t pos) {
  return as_word(((uint64_t)image << 30) | (uint64_t)pos);
}
__device__ __forceinline__ int64_t word_pos(double w) { return (int64_t)(word_bits(w) & (uint64_t)(kWordRows - 1)); }
__device__ __forceinline__ uint32_t word_image(double w) { return (uint32_t)(word_bits(w) >> 30); }

__device__ __forceinline__ void order2(double& a, double& b) {
  double lo, hi;
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  a = lo;
  b = hi;
}
// The words in ascending order (Batcher's odd-even merge sort, 1968: 19 / 63
// compare-exchanges for 8 / 16 words).
template <int N>
__device__ __forceinline__ void sort_words(double (&w)[N]) {
#pragma unroll
  for (int p = 1; p < N; p *= 2)
#pragma unroll
    for (int k = p; k >= 1; k /= 2)
#pragma unroll
      for (int j = k % p; j + k < N; j += 2 * k)
#pragma unroll
        for (int i = 0; i < k; ++i)
          if (i + j + k < N && (i + j) / (2 * p) == (i + j + k) / (2 * p)) order2(w[i + j], w[i + j + k]);
}
// An ascending then descending sequence of N words in ascending order.
template <int N>
__device__ __forceinline__ void merge_words(double (&w)[N]) {
#pragma unroll
  for (int d = N / 2; d > 0; d >>= 1)
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (!(i & d)) order2(w[i], w[i | d]);
}

// LDS slot of word i: one word of padding per eight, so that threads storing
// eight neighbouring words each hit different banks.
__device__ __forceinline__ int slot(int i) { return i + (i >> 3); }
constexpr size_t words_lds(int n) { return (size_t)(n + n / 8) * 8; }

// Words of A[0, la) among the first d of A and B[0, lb) merged (A first on
// ties); a and b are the runs' first LDS word indices.
__device__ __forceinline__ int merge_split(const double* s, int a, int la, int b, int lb, int d) {
  int lo = max(0, d - lb), hi = min(d, la);
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s[slot(a + mid)] <= s[slot(b + d - 1 - mid)]) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The thread's N merged words from diagonal d: na from A at a0, the rest from
// B at b0, read as one ascending and descending sequence.
template <int N>
__device__ __forceinline__ void merge_take(const double* s, int a0, int na, int b0, double (&w)[N]) {
  const int b1 = b0 + N - 1;
#pragma unroll
  for (int i = 0; i < N; ++i) w[i] = s[slot(i < na ? a0 + i : b1 - i)];
  merge_words(w);
}

// Raw key of an image (images are invertible except for kSortKeyFloat).
__device__ __forceinline__ uint32_t key_of_image(uint32_t img, const SortRows& r) {
  const uint32_t mask = r.key_bits == 32 ? 0xffffffffu : ((1u << r.key_bits) - 1u);
  const uint32_t sign = 1u << (r.key_bits - 1);
  if (r.descending) img = ~img & mask;
  if (r.key_class == kSortKeySigned) return img ^ sign;
  if (r.key_class == kSortKeyUnsigned) return img;
  return (img & sign) ? img ^ sign : ~img & mask;
}

// Result i of `row` from a sorted word.
__device__ __forceinline__ void write_result(const SortGather& g, const SortRows& r, int64_t row, int64_t i, double w) {
  const int64_t pos = word_pos(w);
  const int64_t outer = r.inner == 1 ? row : row / r.inner, j = row - outer * r.inner;
  const int64_t from = (outer * r.n + pos) * r.inner + j;
  const int64_t d = (outer * g.out_n + i) * r.inner + j;
  for (int o = 0; o < g.count; ++o) {
    uint64_t v = 0;
    if (!g.src[o]) {
      v = (uint64_t)pos;
    } else if (o == 0 && r.key_class != kSortKeyFloat) {
      v = key_of_image(word_image(w), r);
    } else {
      switch (g.elem_bytes[o]) {
        case 1: v = static_cast<const uint8_t*>(g.src[o])[from]; break;
        case 2: v = static_cast<const uint16_t*>(g.src[o])[from]; break;
        case 4: v = static_cast<const uint32_t*>(g.src[o])[from]; break;
        default: v = static_cast<const uint64_t*>(g.src[o])[from]; break;
      }
    }
    switch (g.elem_bytes[o]) {
      case 1: static_cast<uint8_t*>(g.dst[o])[d] = (uint8_t)v; break;
      case 2: static_cast<uint16_t*>(g.dst[o])[d] = (uint16_t)v; break;
      case 4: static_cast<uint32_t*>(g.dst[o])[d] = (uint32_t)v; break;
      default: static_cast<uint64_t*>(g.dst[o])[d] = v; break;
    }
  }
  if (g.index_dst) static_cast<int32_t*>(g.index_dst)[d] = static_cast<int32_t>(pos);
}

// Where a pass reads a row's words: the raw keys, or a list of words.
struct WordSource {
  const void* keys = nullptr;
  const double* list = nullptr;
  int64_t len = 0;      // words of a row
  int64_t stride = 0;   // list: words from one row to the next
  int vec = 0;          // keys: 16-byte loads (inner == 1, rows 16-byte aligned)
  int near = 0;         // keys: a thread's eight are neighbours
};

// The images of the thread's eight of keys [base, base + 8 threads) of a row
// (any of them, since a word carries its position): key e is at position
// base + key_at(src, tid, threads, e), past the row when that is >= src.len.
__device__ __forceinline__ int key_at(const WordSource& src, int tid, int threads, int e) {
  return src.vec || src.near ? tid * kGroup + e : tid + e * threads;
}
__device__ __forceinline__ void load_images(const WordSource& src, const SortRows& r, const KeyMap& map, int64_t row,
                                            int64_t base, int tid, int threads, uint32_t (&img)[kGroup]) {
  const int64_t end = src.len;
  uint32_t raw[kGroup];
  if (src.vec) {
    // Eight neighbouring keys: one 16-byte load of 16-bit keys, two of 32-bit.
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const int64_t pos = base + (int64_t)tid * kGroup;
    const char* from = static_cast<const char*>(src.keys) + (row * r.n + pos) * (r.key_bits / 8);
    // n is a multiple of the load: a load lies inside the row or past it.
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const u32x4 v0 = pos < end ? *reinterpret_cast<const u32x4*>(from) : zero;
    if (r.key_bits == 32) {
      const u32x4 v1 = pos + 4 < end ? *reinterpret_cast<const u32x4*>(from + 16) : zero;
#pragma unroll
      for (int e = 0; e < kGroup; ++e) raw[e] = e < 4 ? v0[e & 3] : v1[e & 3];
    } else {
#pragma unroll
      for (int e = 0; e < kGroup; ++e) raw[e] = (v0[e >> 1] >> ((e & 1) * 16)) & 0xffffu;
    }
  } else {
    const int64_t outer = row / r.inner, j = row - outer * r.inner;
    const int64_t row0 = outer * r.n * r.inner + j;
#pragma unroll
    for (int e = 0; e < kGroup; ++e) {
      const int64_t i = base + key_at(src, tid, threads, e);
      raw[e] = i < end ? load_key(src.keys, row0 + i * r.inner, r.key_bits) : 0u;
    }
  }
#pragma unroll
  for (int e = 0; e < kGroup; ++e) img[e] = key_image(raw[e], map);
}

// The thread's eight of words [base, base + 8 threads) of a row.
__device__ __forceinline__ void load_words(const WordSource& src, const SortRows& r, int64_t row, int64_t base, int tid,
                                           int threads, double (&w)[kGroup]) {
  if (src.list) {
    const double* p = src.list + row * src.stride;
#pragma unroll
    for (int e = 0; e < kGroup; ++e) {
      const int64_t i = base + e * threads + tid;
      w[e] = i < src.len ? p[i] : as_word(kWordEnd);
    }
    return;
  }
  uint32_t img[kGroup];
  load_images(src, r, key_map(r), row, base, tid, threads, img);
#pragma unroll
  for (int e = 0; e < kGroup; ++e) {
    const int64_t i = base + key_at(src, tid, threads, e);
    w[e] = i < src.len ? make_word(img[e], i) : as_word(kWordEnd);
  }
}

// Orders the wave's own LDS writes before its reads (a wave's LDS operations
// run in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct BlockPass {
  SortRows r;
  WordSource src;
  int64_t blocks_per_row = 1;
  double* dst = nullptr;      // the first `keep` words of each block; null: the results
  int64_t keep = 0, dst_stride = 0;
  SortGather g;
};

// One block of N blockDim words. A merge round finds each thread's split of
// the pair's two runs (a binary search), then reads its N words in one LDS
// latency and merges them in registers. Rounds within a wave's words need no
// barrier. Bound by instruction issue, most of it the searches (which is why
// a thread holds 16 words and not 8 in long rows). Whole sorts with
// positions, bitonic blocks and passes before -> now: [4096, 1024] 118 -> 42 us,
// [64, 32000] 187 -> 57, [64, 128256] bf16 735 -> 212, [1, 2^20] 329 -> 116.
template <int N>
__global__ void __launch_bounds__(kSortThreads) sort_block_kernel(BlockPass p) {
  extern __shared__ double sw[];
  __shared__ int part[kSortThreads + 1];
  const int64_t row = blockIdx.x / p.blocks_per_row;
  const int64_t blk = blockIdx.x - row * p.blocks_per_row;
  const int threads = (int)blockDim.x, tid = (int)threadIdx.x;
  const int64_t base = blk * (threads * N);
  double w[N];
#pragma unroll
  for (int q = 0; q < N / kGroup; ++q) {
    double g[kGroup];
    load_words(p.src, p.r, row, base + q * threads * kGroup, tid, threads, g);
#pragma unroll
    for (int e = 0; e < kGroup; ++e) w[q * kGroup + e] = g[e];
  }
  sort_words(w);
  const int mine = tid * N;
  // The words of a short row lie in the first threads: one run holds them all
  // before the block is sorted.
  int words = p.src.near ? (int)p.src.len : threads * N;
  if constexpr (N == kGroup) {
    if (p.src.near && p.g.out_n <= N) {
      // The first eight of two threads' sorted eights: the smaller of one
      // ascending and the other descending, which is bitonic.
      for (int d = 1; d * N < words; d *= 2) {
        double o[N];
#pragma unroll
        for (int e = 0; e < N; ++e) o[e] = __shfl_xor(w[N - 1 - e], d, 64);
#pragma unroll
        for (int e = 0; e < N; ++e) asm("v_min_f64 %0, %0, %1" : "+v"(w[e]) : "v"(o[e]));
        merge_words(w);
      }
      words = 0;  // thread 0 has them
    }
  }
#pragma unroll
  for (int e = 0; e < N; ++e) sw[slot(mine + e)] = w[e];
  for (int run = N; run < words; run *= 2) {
    const bool wave = 2 * run <= 64 * N;
    if (wave) wave_sync();
    else __syncthreads();
    const int pair = mine & ~(2 * run - 1), d = mine - pair;
    const int a = merge_split(sw, pair, run, pair + run, run, d);
    int a1;
    if (wave) {
      a1 = __shfl_down(a, 1, 64);
    } else {
      part[tid] = a;
      __syncthreads();
      a1 = part[tid + 1];
    }
    if (d + N == 2 * run) a1 = run;
    merge_take(sw, pair + a, a1 - a, pair + run + d - a, w);
    if (wave) wave_sync();
    else __syncthreads();
#pragma unroll
    for (int e = 0; e < N; ++e) sw[slot(mine + e)] = w[e];
  }
  __syncthreads();
  if (p.dst) {
    double* dst = p.dst + row * p.dst_stride + blk * p.keep;
    const int64_t n = min(p.keep, p.dst_stride - blk * p.keep);
    for (int i = tid; i < n; i += threads) dst[i] = sw[slot(i)];
  } else {
    for (int i = tid; i < p.g.out_n; i += threads) write_result(p.g, p.r, row, i, sw[slot(i)]);
  }
}

struct MergePass {
  SortRows r;
  const double* src = nullptr;
  double* dst = nullptr;       // null: the results (one pair a row)
  int64_t len = 0, run = 0;    // words of a row (the rows' stride), sorted run length
  int64_t tiles_per_row = 1;
  SortGather g;
};

// Words of A[0, la) among the first d merged, in HBM: the wave's lanes probe
// 64 points of the range at a time.
__device__ int64_t merge_split_wave(const double* A, int64_t la, const double* B, int64_t lb, int64_t d) {
  int64_t lo = max((int64_t)0, d - lb), hi = min(d, la);
  const int lane = (int)__lane_id();
  while (lo < hi) {
    const int64_t step = (hi - lo + 63) / 64, mid = lo + lane * step;
    const bool take = mid < hi && A[mid] <= B[d - 1 - mid];
    const int n = __popcll(__ballot(take));  // true up to the split, then false
    const int64_t from = lo;
    if (n == 0) hi = lo;
    else {
      lo = from + (n - 1) * step + 1;
      hi = min(from + n * step, hi);
    }
  }
  return lo;
}

// Output words [tile, tile + kMergeTile) of a pair of runs: the tile's parts
// of both runs are staged in LDS and merged as in sort_block.
__global__ void __launch_bounds__(kMergeThreads) merge_runs_kernel(MergePass p) {
  __shared__ double sw[kMergeTile + kMergeTile / 8];
  __shared__ int part[kMergeThreads + 1];
  __shared__ int64_t ends[2];
  const int64_t row = blockIdx.x / p.tiles_per_row;
  const int64_t t0 = (blockIdx.x - row * p.tiles_per_row) * kMergeTile;
  // Runs are multiples of the tile: a tile lies in one pair.
  const int64_t pair = t0 / (2 * p.run) * (2 * p.run);
  const double* A = p.src + row * p.len + pair;
  const double* B = A + p.run;
  const int64_t la = min(p.run, p.len - pair), lb = max((int64_t)0, min(p.run, p.len - pair - p.run));
  const int64_t d0 = t0 - pair, d1 = min(d0 + kMergeTile, la + lb);
  const int tid = (int)threadIdx.x, wave = tid >> 6;
  if (wave < 2) {
    const int64_t e = merge_split_wave(A, la, B, lb, wave == 0 ? d0 : d1);
    if ((tid & 63) == 0) ends[wave] = e;
  }
  __syncthreads();
  const int64_t a0 = ends[0], b0 = d0 - a0;
  const int na = (int)(ends[1] - a0), n = (int)(d1 - d0), nb = n - na;
#pragma unroll
  for (int e = 0; e < kMergeItems; ++e) {
    const int i = e * kMergeThreads + tid;
    if (i < n) sw[slot(i)] = i < na ? A[a0 + i] : B[b0 + i - na];
  }
  __syncthreads();
  const int d = min(tid * kMergeItems, n);
  const int a = merge_split(sw, 0, na, na, nb, d);
  part[tid] = a;
  __syncthreads();
  const int d_end = min(d + kMergeItems, n), a1 = d_end == n ? na : part[tid + 1];
  // The last thread with words may have fewer than its share: its B part then
  // starts later in the sequence, behind ends of the order.
  double w[kMergeItems];
  const int take_a = a1 - a, take_b = d_end - d - take_a;
#pragma unroll
  for (int i = 0; i < kMergeItems; ++i) {
    const int k = kMergeItems - 1 - i;
    w[i] = i < take_a ? sw[slot(a + i)] : k < take_b ? sw[slot(na + d - a + k)] : as_word(kWordEnd);
  }
  merge_words(w);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kMergeItems; ++e)
    if (d + e < d_end) sw[slot(d + e)] = w[e];
  __syncthreads();
  if (p.dst) {
    double* dst = p.dst + row * p.len + t0;
    for (int i = tid; i < n; i += kMergeThreads) dst[i] = sw[slot(i)];
  } else {
    for (int i = tid; i < n && t0 + i < p.g.out_n; i += kMergeThreads) write_result(p.g, p.r, row, t0 + i, sw[slot(i)]);
  }
}

// ---------------------------------------------------------------- top-k
// The first `need` <= 256 words of a chunk of 256 * kShare * 8 words. Threads
// (or, for 16-bit keys, groups of one, two or four) take the least of their
// words; the need-th smallest of these, T, has at least `need` words at or
// below it, and usually little more: only those are ranked, by counting, which
// also orders them. No network over the chunk, no histogram: one pass over the
// keys in registers. Larger groups give fewer values to rank (64 for need <= 56)
// and a few more candidates.
constexpr int kTopkThreads = 256;
constexpr int kTopkMax = 256;
struct TopkPass {
  SortRows r;
  WordSource src;
  int64_t blocks_per_row = 1;
  int need = 0;
  int group = 1;           // topk_half: threads per group, at least `need` groups
  double* dst = nullptr;   // `need` words of each block; null: the results
  SortGather g;
};
struct TopkLds {
  double least[2 * kTopkThreads];
  double bound;
  uint32_t bound_image;
  int count;
};

// The candidates' ranks (distinct words): rank k is result k. The threads of a
// candidate count over a segment of the list each, eight words at a time; the
// list holds kTopkPad more words than candidates, filled with ends.
constexpr int kTopkPad = 64;
__device__ __forceinline__ void topk_rank(const TopkPass& p, int64_t row, int64_t blk, int tid, int m, double* cand) {
  double* dst = p.dst ? p.dst + (row * p.blocks_per_row + blk) * p.need : nullptr;
  const int lg = m <= 32 ? 3 : m <= 64 ? 2 : m <= 128 ? 1 : 0;
  const int seg = (((m + (1 << lg) - 1) >> lg) + 7) & ~7;  // at most 63 words past m in all
  if (tid < (seg << lg) - m) cand[m + tid] = as_word(kWordEnd);
  __syncthreads();
  const int sub = tid & ((1 << lg) - 1);
  for (int c = tid >> lg; c < m; c += kTopkThreads >> lg) {
    const double x = cand[c];
    const double* part = cand + sub * seg;
    int k = 0;
    for (int i = 0; i < seg; i += 8) {
      double z[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) z[e] = part[i + e];
#pragma unroll
      for (int e = 0; e < 8; ++e) k += z[e] < x ? 1 : 0;
    }
    if (lg > 0) k += __shfl_xor(k, 1, 64);
    if (lg > 1) k += __shfl_xor(k, 2, 64);
    if (lg > 2) k += __shfl_xor(k, 4, 64);
    if (sub == 0 && k < p.need) {
      if (dst) dst[k] = x;
      else write_result(p.g, p.r, row, k, x);
    }
  }
  if (dst)
    for (int i = m + tid; i < p.need; i += kTopkThreads) dst[i] = as_word(kWordEnd);
}

// The words at or below T of 256 threads' kShare * 8 words each: T is the
// need-th smallest of the threads' own least words, so at most need * 8 *
// kShare words go to `cand`. Returns how many. Where `need` is most of the
// threads, the least of each half of a thread's words are taken: the 256th of
// 256 is the largest of them, with many words below it ([64, 8192] f32, k =
// 256: 105 us, 27 with halves). The longer count costs 5 us a round: at 200 of
// 256 it is the slower one ([17, 54716] 32 and 40).
template <int kShare>
__device__ __forceinline__ int topk_bound(const double (&w)[kShare][kGroup], int need, int tid, TopkLds& lds, double* cand) {
  const double end = as_word(kWordEnd);
  double half[2] = {end, end};
#pragma unroll
  for (int q = 0; q < kShare; ++q)
#pragma unroll
    for (int e = 0; e < kGroup; ++e) asm("v_min_f64 %0, %0, %1" : "+v"(half[e & 1]) : "v"(w[q][e]));
  const double lo = half[0] < half[1] ? half[0] : half[1];
  const bool halves = need > kTopkThreads * 7 / 8;
  if (halves) {
    lds.least[2 * tid] = half[0];
    lds.least[2 * tid + 1] = half[1];
  } else {
    lds.least[tid] = lo;
  }
  if (tid == 0) {
    lds.bound = as_word(kWordEnd - 1);  // fewer than `need` of them hold words: all words
    lds.count = 0;
  }
  __syncthreads();
  if (halves) {
    int rank[2] = {0, 0};
#pragma unroll 8
    for (int i = 0; i < 2 * kTopkThreads; ++i) {
      const double x = lds.least[i];
      rank[0] += x < half[0] ? 1 : 0;
      rank[1] += x < half[1] ? 1 : 0;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (rank[h] == need - 1 && half[h] < end) lds.bound = half[h];
  } else {
    int rank = 0;
#pragma unroll 8
    for (int i = 0; i < kTopkThreads; ++i) rank += lds.least[i] < lo ? 1 : 0;
    if (rank == need - 1 && lo < end) lds.bound = lo;
  }
  __syncthreads();
  const double T = lds.bound;
  if (lo <= T) {
#pragma unroll
    for (int q = 0; q < kShare; ++q)
#pragma unroll
      for (int e = 0; e < kGroup; ++e)
        if (w[q][e] <= T) cand[atomicAdd(&lds.count, 1)] = w[q][e];
  }
  __syncthreads();
  return lds.count;
}

// The candidates again where they are many: m words in `cand`. Rows and lists
// in some order can give every thread words of like rank (lists of 256 words
// put word k of each in thread k: T is then near the last of them all, and
// ranking by counting is quadratic). A thread takes words a golden ratio of the
// list apart, which are of many ranks in any such order.
template <int kShare>
__device__ __forceinline__ int topk_again(int m, int need, int tid, TopkLds& lds, double* cand) {
  if (m <= 2 * need + kTopkThreads / 2) return m;
  int bits = 8;
  while ((1 << bits) < m) ++bits;  // m <= 256 * 8 * kShare
  const uint32_t each = 1u << (bits - 8), step = (0x9e3779b1u >> (32 - bits)) | 1u, mask = (1u << bits) - 1u;
  double w[kShare][kGroup];
#pragma unroll
  for (int q = 0; q < kShare; ++q)
#pragma unroll
    for (int e = 0; e < kGroup; ++e) {
      const uint32_t j = q * kGroup + e, c = ((tid * each + j) * step) & mask;
      w[q][e] = j < each && (int)c < m ? cand[c] : as_word(kWordEnd);
    }
  __syncthreads();
  return topk_bound<kShare>(w, need, tid, lds, cand);
}

// Any source.
template <int kShare>
__device__ __forceinline__ int topk_words(const TopkPass& p, int64_t row, int64_t blk, int tid, TopkLds& lds, double* cand) {
  double w[kShare][kGroup];
#pragma unroll
  for (int q = 0; q < kShare; ++q)
    load_words(p.src, p.r, row, (blk * kShare + q) * (kTopkThreads * kGroup), tid, kTopkThreads, w[q]);
  return topk_again<kShare>(topk_bound<kShare>(w, p.need, tid, lds, cand), p.need, tid, lds, cand);
}

template <int kShare>
__global__ void __launch_bounds__(kTopkThreads) topk_select_kernel(TopkPass p) {
  extern __shared__ double cand[];  // need * kShare * kGroup + kTopkPad words
  __shared__ TopkLds lds;
  const int64_t row = blockIdx.x / p.blocks_per_row;
  const int64_t blk = blockIdx.x - row * p.blocks_per_row;
  const int m = topk_words<kShare>(p, row, blk, (int)threadIdx.x, lds, cand);
  topk_rank(p, row, blk, (int)threadIdx.x, m, cand);
}

// 16-bit keys (not FLOAT-compared) in 16-byte aligned rows: the images, the
// least of them and the test against T two keys an instruction, on packed
// 16-bit integers. T is the least image with `need` groups at or below it, so
// every key of T's image is a candidate; the few candidates are read again and
// made words. Many candidates (ties, or neighbouring keys that are all large)
// are bounded again as words.
// [64, 128256] bf16, k = 50: 69 us with bitonic blocks, 25 on words, 20 now
// (both launches).
template <int kShare>
__global__ void __launch_bounds__(kTopkThreads) topk_half_kernel(TopkPass p) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  typedef short ss2 __attribute__((ext_vector_type(2)));
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int kPairs = 4 * kShare;  // packed registers a thread
  constexpr int kChunk = kTopkThreads * kShare * kGroup;
  extern __shared__ double cand[];  // need * kShare * kGroup + kTopkPad words
  __shared__ TopkLds lds;
  const int64_t row = blockIdx.x / p.blocks_per_row;
  const int64_t blk = blockIdx.x - row * p.blocks_per_row;
  const int tid = (int)threadIdx.x;
  const int64_t base = blk * kChunk;
  const int keys = (int)min((int64_t)kChunk, p.src.len - base);  // a multiple of 8
  const uint16_t* from = static_cast<const uint16_t*>(p.src.keys) + row * p.r.n + base;
  const KeyMap map = key_map(p.r);
  const uint32_t neg2 = map.neg * 0x10001u, pos2 = map.pos * 0x10001u;
  u32x4 v[kShare];
#pragma unroll
  for (int q = 0; q < kShare; ++q) {
    const int at = q * (kTopkThreads * kGroup) + tid * kGroup;
    v[q] = *reinterpret_cast<const u32x4*>(from + (at < keys ? at : 0));
  }
  uint32_t img[kPairs];
  us2 least2 = {0xffff, 0xffff};
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {
    const bool in = (j / 4) * (kTopkThreads * kGroup) + tid * kGroup < keys;
    const uint32_t raw = v[j / 4][j % 4];
    const uint32_t sign = __builtin_bit_cast(uint32_t, (ss2)(__builtin_bit_cast(ss2, raw) >> 15));
    img[j] = in ? raw ^ ((sign & neg2) | (~sign & pos2)) : 0xffffffffu;
    least2 = __builtin_elementwise_min(least2, __builtin_bit_cast(us2, img[j]));
  }
  uint32_t lo = min((uint32_t)least2[0], (uint32_t)least2[1]);
  for (int d = 1; d < p.group; d *= 2) lo = min(lo, (uint32_t)__shfl_xor((int)lo, d, 64));
  uint32_t* least = reinterpret_cast<uint32_t*>(lds.least);
  if (tid % p.group == 0) least[tid / p.group] = lo;
  if (tid == 0) {
    lds.bound_image = 0xffffu;
    lds.count = 0;
  }
  __syncthreads();
  int le = 0;
#pragma unroll 4
  for (int i = 0; i < kTopkThreads / p.group; i += 4) {
    const u32x4 x = *reinterpret_cast<const u32x4*>(least + i);
    le += (x[0] <= lo ? 1 : 0) + (x[1] <= lo ? 1 : 0) + (x[2] <= lo ? 1 : 0) + (x[3] <= lo ? 1 : 0);
  }
  if (le >= p.need) atomicMin(&lds.bound_image, lo);
  __syncthreads();
  const uint32_t T = lds.bound_image;
  const us2 T2 = {(unsigned short)T, (unsigned short)T}, one = {1, 1};
  // Bit kPairs - 1 - j of the low half: pair j's low key is above T; of the
  // high half, its high key.
  uint32_t above = 0;
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {
    const us2 over = __builtin_elementwise_sub_sat(__builtin_bit_cast(us2, img[j]), T2);
    above = (above << 1) | __builtin_bit_cast(uint32_t, (us2)__builtin_elementwise_min(over, one));
  }
  uint32_t bits = ~above & (((1u << kPairs) - 1u) * 0x10001u);
#pragma unroll
  for (int q = 0; q < kShare; ++q)
    if (q * (kTopkThreads * kGroup) + tid * kGroup >= keys) bits &= ~((0xfu << (kPairs - 4 - 4 * q)) * 0x10001u);
  const int room = p.need * kShare * kGroup;
  int to = bits ? atomicAdd(&lds.count, __popc(bits)) : 0;
  while (bits) {
    const int k = __ffs(bits) - 1;
    bits &= bits - 1;
    const int j = kPairs - 1 - (k & 15);
    const int at = (j >> 2) * (kTopkThreads * kGroup) + tid * kGroup + (j & 3) * 2 + (k >> 4);
    if (to < room) reinterpret_cast<int*>(cand + to)[0] = at;
    ++to;
  }
  __syncthreads();
  int m = lds.count;
  if (m > room) {
    __syncthreads();
    m = topk_words<kShare>(p, row, blk, tid, lds, cand);
  } else {
    // Every candidate's key in one round of loads.
    for (int c = tid; c < m; c += kTopkThreads) {
      const int at = reinterpret_cast<const int*>(cand + c)[0];
      cand[c] = make_word(key_image(from[at], map), base + at);
    }
    __syncthreads();
    m = topk_again<kShare>(m, p.need, tid, lds, cand);
  }
  topk_rank(p, row, blk, tid, m, cand);
}

// A row's results from the sorted first words of its pieces, whose words hold
// positions within the piece: a word's rank is its own index plus the words
// ahead of it in every other piece (equal keys of earlier pieces come first).
struct PieceMerge {
  SortRows r;
  SortGather g;
  const double* list = nullptr;  // [piece][row][out_n]
  int pieces = 0;
  int64_t piece_len = 0;         // of all but the last
};
__global__ void merge_pieces_kernel(PieceMerge p) {
  const int64_t k = p.g.out_n, t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= p.pieces * p.r.rows * k) return;
  const int piece = static_cast<int>(t / (p.r.rows * k));
  const int64_t row = t / k % p.r.rows, i = t % k;
  const auto words = [&](int q) { return min(k, min(p.piece_len, p.r.n - q * p.piece_len)); };
  if (i >= words(piece)) return;
  const double w = p.list[t];
  int64_t rank = i;
  for (int q = 0; q < p.pieces && rank < k; ++q) {
    if (q == piece) continue;
    const double* other = p.list + (q * p.r.rows + row) * k;
    int64_t lo = 0, hi = words(q);
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      const uint32_t x = word_image(other[mid]);
      if (x < word_image(w) || (x == word_image(w) && q < piece)) lo = mid + 1;
      else hi = mid;
    }
    rank += lo;
  }
  if (rank < k) gather_one(p.g, p.r, row, rank, piece * p.piece_len + word_pos(w));
}

int64_t pow2_at_least(int64_t v) {
  int64_t p = 1;
  while (p < v) p <<= 1;
  return p;
}

void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail(Code::kInternal, strformat("%s launch failed: %s", what, hipGetErrorString(e)));
}

void local(hipStream_t s, const LocalPass& p, int64_t rows) {
  const int64_t grid = rows * p.blocks_per_row;
  PJRTX_CHECK(grid > 0 && grid < (int64_t{1} << 31), Code::kUnimplemented, "sort: too many rows");
  hipLaunchKernelGGL(sort_local_kernel, dim3(static_cast<unsigned>(grid)), dim3(kLocalThreads), 0, s, p);
  check_launch("sort_local");
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The kernels a row's sort takes and their scratch.
enum SortPath {
  kPathTopk,    // topk_select rounds
  kPathKeep,    // sort_block rounds that keep the first out_n words of a block
  kPathMerge,   // sort_block, then merge_runs
  kPathBitonic  // padded rows in one buffer
};
struct Layout {
  SortPath path = kPathMerge;
  int share = 1;               // topk: eight-word groups a thread
  int pieces = 1;              // topk / keep: parts a row is taken in
  int64_t piece_len = 0;       // elements of all but the last
  int64_t len1 = 0;            // topk / keep: list length after a piece's round one
  int64_t p = 0;               // bitonic: padded row length
  size_t bytes = 0;
};

// Words a topk thread holds (in eights): a row that one chunk holds goes to
// one launch; else enough workgroups for the GPU (1024), then long chunks,
// whose lists are shorter.
int topk_share(const SortRows& r, int64_t len) {
  for (int one = 1; one <= 4; one *= 2)
    if (len <= kTopkThreads * kGroup * one) return one;
  int share = 4;
  while (share > 1 && r.rows * ceil_div(len, kTopkThreads * kGroup * share) < 1024) share /= 2;
  return share;
}
int64_t topk_blocks(int share, int64_t len) { return ceil_div(len, kTopkThreads * kGroup * share); }

Layout layout_of(const SortRows& r, int64_t out_n, int64_t max_bytes) {
  Layout L;
  const auto bitonic = [&] {
    L.path = kPathBitonic;
    L.p = std::max<int64_t>(pow2_at_least(r.n), kSortBlock);
    L.bytes = static_cast<size_t>(r.rows * L.p) * 8;
    return L;
  };
  // Short rows are sorted whole: a bound costs its 256 counts however few the
  // words are. us bounded / sorted: [256, 64] k = 20 8.5 / 5.7, [256, 500] k =
  // 5 7.9 / 8.5, k = 50 8.8 / 8.4, k = 250 26 / 9.6, [4096, 500] k = 50 42 / 15;
  // longer ones [256, 1000] k = 20 8.2 / 9.9, bf16 k = 64 10.9 / 9.9,
  // [17, 2047] k = 256 22 / 15.
  const bool whole = r.n <= 64 * kGroup || (r.n <= 1024 && out_n > 40) || (r.n <= 2048 && out_n > kTopkThreads / 2);
  const bool topk = out_n < r.n && out_n <= kTopkMax && !whole, keep = r.n > kSortTile && out_n <= kSortTile / 2;
  if (r.n >= kWordRows && !topk && !keep) return bitonic();
  L.piece_len = r.n < kWordRows ? std::max<int64_t>(r.n, 1) : kWordRows / 2;
  L.pieces = static_cast<int>(ceil_div(r.n, L.piece_len));
  const size_t merged = L.pieces > 1 ? static_cast<size_t>(L.pieces * r.rows * out_n) * 8 : 0;
  if (topk) {
    L.path = kPathTopk;
    // Longer chunks, whose lists are shorter, where those of the best do not fit.
    for (L.share = topk_share(r, L.piece_len);; L.share *= 2) {
      const int64_t blocks = topk_blocks(L.share, L.piece_len);
      L.len1 = blocks * out_n;
      L.bytes = blocks > 1 ? static_cast<size_t>(2 * r.rows * L.len1) * 8 + merged : 0;
      if (static_cast<int64_t>(L.bytes) <= max_bytes || L.share == 4) break;
    }
  } else if (keep) {
    L.path = kPathKeep;
    L.len1 = ceil_div(L.piece_len, kSortTile) * out_n;
    L.bytes = static_cast<size_t>(2 * r.rows * L.len1) * 8 + merged;
  } else {
    // One buffer per side of a merge round; the last round writes the results.
    L.bytes = r.n <= kSortTile ? 0 : static_cast<size_t>((r.n <= 2 * kSortTile ? 1 : 2) * r.rows * r.n) * 8;
    if (static_cast<int64_t>(L.bytes) > max_bytes) return bitonic();
  }
  return L;
}

unsigned grid_of(int64_t rows, int64_t per_row) {
  const int64_t grid = rows * per_row;
  PJRTX_CHECK(grid > 0 && grid < (int64_t{1} << 31), Code::kUnimplemented, "sort: too many rows");
  return static_cast<unsigned>(grid);
}

// Blocks of `words` <= kSortTile words. A whole row of one wave's words (512)
// is merged only as far as it goes ([1024, 8] f32 argsort 8.8 us with all six
// rounds, 4.1 so), and rows of up to 2048 words by threads of 8, whose rounds
// are shorter ([16, 1000] 18.1 us with 16 a thread, 13.2 with 8; [4096, 1000] 45
// and 42, but [4096, 4000] 128 and 134).
void sort_blocks(hipStream_t s, BlockPass p, int64_t words) {
  p.src.near = !p.src.list && p.blocks_per_row == 1 && words <= 64 * kGroup;
  const int n = words <= 2048 ? kGroup : 16;
  const int threads = static_cast<int>(std::max<int64_t>(64, pow2_at_least(ceil_div(words, n))));
  const dim3 grid(grid_of(p.r.rows, p.blocks_per_row));
  if (n == kGroup) hipLaunchKernelGGL((sort_block_kernel<kGroup>), grid, dim3(threads), words_lds(threads * n), s, p);
  else hipLaunchKernelGGL((sort_block_kernel<16>), grid, dim3(threads), words_lds(threads * n), s, p);
  check_launch("sort_block");
}

void topk_blocks_launch(hipStream_t s, TopkPass p, int share) {
  const dim3 grid(grid_of(p.r.rows, p.blocks_per_row)), block(kTopkThreads);
  const size_t lds = static_cast<size_t>(p.need * share * kGroup + kTopkPad) * 8;
  p.group = p.need <= 56 ? 4 : p.need <= 112 ? 2 : 1;
  // As many groups as `need` hold words, or the bound takes them all (bf16 [9,
  // 576] k = 20 14.7 us, 8.6 so).
  const int64_t holding = std::min<int64_t>(kTopkThreads, ceil_div(p.src.len, kGroup));
  while (p.group > 1 && holding / p.group < p.need) p.group /= 2;
  const bool half = !p.src.list && p.src.vec && p.r.key_bits == 16 && p.r.key_class != kSortKeyFloat;
#define PJRTX_TOPK(SHARE)                                                                  \
  if (half) hipLaunchKernelGGL((topk_half_kernel<SHARE>), grid, block, lds, s, p);         \
  else hipLaunchKernelGGL((topk_select_kernel<SHARE>), grid, block, lds, s, p)
  if (share == 1) { PJRTX_TOPK(1); }
  else if (share == 2) { PJRTX_TOPK(2); }
  else { PJRTX_TOPK(4); }
#undef PJRTX_TOPK
  check_launch("topk_select");
}

WordSource key_source(const SortRows& r, const void* keys) {
  WordSource src;
  src.keys = keys;
  src.len = r.n;
  src.vec = r.inner == 1 && r.key_bits >= 16 && (r.n * r.key_bits / 8) % 16 == 0 && reinterpret_cast<uintptr_t>(keys) % 16 == 0;
  return src;
}

// The first out_n words of every row of `src` (kPathTopk, kPathKeep), as the
// results or, with `dst`, as a list of out_n words a row (ends after the last
// of fewer). `lists` holds two lists of len1 words a row.
void first_words(hipStream_t s, const SortRows& r, const WordSource& src, const SortGather& g, const Layout& L,
                 double* lists, double* dst) {
  double *a = lists, *b = lists + r.rows * L.len1;
  if (L.path == kPathTopk) {
    TopkPass p;
    p.r = r;
    p.src = src;
    p.need = static_cast<int>(g.out_n);
    p.g = g;
    int share = L.share;
    for (;;) {
      p.blocks_per_row = topk_blocks(share, p.src.len);
      const bool last = p.blocks_per_row == 1;
      p.dst = last ? dst : a;
      topk_blocks_launch(s, p, share);
      if (last) return;
      p.src.list = a;
      p.src.len = p.src.stride = p.blocks_per_row * p.need;
      share = topk_share(r, p.src.len);
      std::swap(a, b);
    }
  }
  BlockPass p;
  p.r = r;
  p.src = src;
  p.g = g;
  p.keep = g.out_n;
  while (p.src.len > kSortTile) {
    p.blocks_per_row = ceil_div(p.src.len, kSortTile);
    p.dst = a;
    p.dst_stride = p.blocks_per_row * p.keep;
    sort_blocks(s, p, kSortTile);
    p.src.list = a;
    p.src.len = p.src.stride = p.dst_stride;
    std::swap(a, b);
  }
  p.blocks_per_row = 1;
  p.dst = dst;
  p.dst_stride = p.keep;
  sort_blocks(s, p, dst ? std::max(p.src.len, p.keep) : p.src.len);
}

}  // namespace

size_t sort_scratch_bytes(const SortRows& r, int64_t out_n, int64_t max_bytes) {
  return layout_of(r, out_n, max_bytes).bytes;
}

void sort_rows(hipStream_t s, const SortRows& r, const void* keys, const SortGather& g, void* scratch, int64_t max_bytes) {
  if (r.rows == 0 || r.n == 0 || g.out_n == 0) return;
  PJRTX_CHECK(r.n < (int64_t{1} << 31) && g.out_n <= r.n, Code::kInvalidArgument, "sort: row length out of range");
  PJRTX_CHECK(r.key_bits == 8 || r.key_bits == 16 || r.key_bits == 32, Code::kUnimplemented,
              "sort: keys wider than 32 bits are not supported");
  const Layout L = layout_of(r, g.out_n, max_bytes);
  if (L.pieces > 1) {
    PJRTX_CHECK(r.inner == 1, Code::kInternal, "sort: a row in pieces must be contiguous");
    // Each piece's first out_n words, through the same two lists.
    double* const lists = static_cast<double*>(scratch);
    PieceMerge m;
    m.r = r;
    m.g = g;
    m.pieces = L.pieces;
    m.piece_len = L.piece_len;
    double* const merged = lists + 2 * r.rows * L.len1;
    m.list = merged;
    for (int q = 0; q < L.pieces; ++q) {
      WordSource src = key_source(r, static_cast<const char*>(keys) + q * L.piece_len * (r.key_bits / 8));
      src.len = std::min(L.piece_len, r.n - q * L.piece_len);
      first_words(s, r, src, g, L, lists, merged + q * r.rows * g.out_n);
    }
    const unsigned grid = grid_of(ceil_div(L.pieces * r.rows * g.out_n, 256), 1);
    hipLaunchKernelGGL(merge_pieces_kernel, dim3(grid), dim3(256), 0, s, m);
    check_launch("merge_pieces");
    return;
  }
  const WordSource src = key_source(r, keys);
  if (L.path == kPathTopk || L.path == kPathKeep) {
    first_words(s, r, src, g, L, static_cast<double*>(scratch), nullptr);
    return;
  }
  if (L.path == kPathMerge) {
    double *a = static_cast<double*>(scratch), *b = a + r.rows * r.n;
    BlockPass p;
    p.r = r;
    p.src = src;
    p.g = g;
    if (r.n <= kSortTile) {
      sort_blocks(s, p, r.n);
      return;
    }
    p.blocks_per_row = ceil_div(r.n, kSortTile);
    p.dst = a;
    p.keep = kSortTile;
    p.dst_stride = r.n;
    sort_blocks(s, p, kSortTile);
    MergePass m;
    m.r = r;
    m.g = g;
    m.len = r.n;
    m.tiles_per_row = ceil_div(r.n, kMergeTile);
    for (m.run = kSortTile; m.run < r.n; m.run *= 2) {
      m.src = a;
      m.dst = 2 * m.run >= r.n ? nullptr : b;
      hipLaunchKernelGGL(merge_runs_kernel, dim3(grid_of(r.rows, m.tiles_per_row)), dim3(kMergeThreads), 0, s, m);
      check_launch("merge_runs");
      std::swap(a, b);
    }
    return;
  }
  // Bitonic network over L.p words per row: LDS passes for partner distances
  // below kSortBlock, global passes for the rest.
  uint64_t* buf = static_cast<uint64_t*>(scratch);
  LocalPass p;
  p.keys = keys;
  p.r = r;
  p.row_len = L.p;
  p.blocks_per_row = L.p / kSortBlock;
  p.k_first = 2, p.k_last = kSortBlock, p.j_first = 1;
  p.dst = buf;
  local(s, p, r.rows);
  const int64_t pairs = r.rows * (L.p / 2);
  PJRTX_CHECK((pairs + 255) / 256 < (int64_t{1} << 31), Code::kUnimplemented, "sort: too large");
  for (int64_t k = 2 * kSortBlock; k <= L.p; k <<= 1) {
    for (int64_t j = k >> 1; j >= kSortBlock; j >>= 1) {
      hipLaunchKernelGGL(bitonic_global_kernel, dim3(static_cast<unsigned>((pairs + 255) / 256)), dim3(256), 0, s, buf,
                         r.rows, L.p, k, j);
      check_launch("bitonic_global");
    }
    LocalPass m = p;
    m.list = buf;
    m.k_first = k, m.k_last = k, m.j_first = kSortBlock / 2;
    local(s, m, r.rows);
  }
  const int64_t outs = r.rows * g.out_n;
  hipLaunchKernelGGL(sort_write_kernel, dim3(static_cast<unsigned>((outs + 255) / 256)), dim3(256), 0, s, buf, L.p, r,
                     g);
  check_launch("sort_write");
}

}  // namespace pjrtx
