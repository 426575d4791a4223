// MFMA GEMM for bf16 / f16 with f32 accumulation, either layout of either
// operand, in block tiles from 32 x 64 to 256 x 256.
//
// gemm_tile: C[b] = A[b] * B[b], A K-contiguous ([M][K]) or M-contiguous
// ([K][M]), B K-contiguous ([N][K]) or N-contiguous ([K][N]).
//  * 64-deep k-tiles go from global memory straight into LDS (lds_dma16, 16
//    bytes a lane, 1 KB an instruction), kStages of them; the loads of tile
//    kt + kStages are issued when tile kt's last fragments are in registers.
//  * One barrier per k-tile, placed before the tile's last 16-deep slab: by
//    then every wave holds its last-slab fragments in registers and has read
//    all of the tile, so the barrier both publishes tile kt + 1 and frees
//    tile kt's stage.
//  * v_mfma_f32_32x32x16; the next slab's fragments are read while the
//    current one multiplies.
//  * A K-contiguous operand's stage is rows of 64 elements (eight 16-byte
//    chunks), chunk c of row r stored at c ^ ((r >> 1) & 7): the fragment
//    reads of 32 consecutive rows hit distinct banks. An M- or N-contiguous
//    operand's stage is 64 k rows of kT elements (tile width), and its
//    fragments come from transposing reads (ds_read_b64_tr_b16: lane j of a
//    16-lane group gets element j & 3 of the 8-byte pieces lanes
//    4 e + (j >> 2) address, e = 0..3; lanes addressing 4 consecutive k rows
//    x 16 columns return 4 consecutive k of one column, half a fragment);
//    chunk c of row k is stored at c ^ 4 (k & 3) (c ^ 4 ((k >> 1) & 1) for
//    64-wide tiles, two rows to 256 bytes), so the 4 rows x 64 bytes a
//    half-wave reads hit distinct banks. A load places lane L's 16 bytes at
//    slot L of its 1 KB, so the swizzle is applied on the global side.
//  * Rows past M or N and k past K read as zero: the lane part of every
//    load's offset is what the buffer range check covers, the k-tile part
//    moves the resource's base and shortens its range, and lanes whose chunk
//    lies past K (or whose columns past M / N) get an offset beyond it.
//  * Tiles with at most 64 x 64 outputs a wave read a whole k-tile's fragments
//    while the tile before multiplies (one LDS latency a k-tile); where WK
//    waves share a sub-tile each takes 4 / WK of the slabs, which divides the
//    fragment reads, and the sums meet through LDS once at the end.
//
// Measured on MI355X, bf16, B N-contiguous, executes back to back on the same
// operands (before: one 256 x 256 kernel whose loads were waited for a tile
// early, and 128 x 128 tiles transposed through 2-byte LDS stores); operands
// that change from call to call come from HBM and take up to 8 us more:
//   8192 x 8192 x 8192    256 x 256 tiles   887 -> 807 us (807-846 with the clock; 1300-1360 TFLOP/s)
//   1000 x 2048 x 5632    128 x 256         148 -> 37 us
//   512 x 2048 x 5632     128 x 128          98 -> 23 us
//   512 x 5632 x 2048     64 x 64           233 -> 25 us
//   512 x 2048 x 2048     64 x 64            91 -> 12.4 us
//   64 x 4096 x 4096      64 x 64, k-split  170 -> 13 us
// What bounds it: the large tile, power (the clock drops to about 1.6 GHz)
// and LDS reads; the small ones, the loads (a 64 x 64 k-tile brings 16 KB per
// CU, 0.157 us alone, against 0.073 us of matrix work) and the issue slots of
// one wave per SIMD.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels/dot.h"
#include "kernels/lds_dma.h"

namespace pjrtx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
typedef __attribute__((address_space(3))) uint16_t lds_u16;

constexpr int BK = 64;

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

template <bool kF16>
__device__ __forceinline__ uint16_t to_half(float f) {
  if constexpr (kF16) return __builtin_bit_cast(uint16_t, (_Float16)f);
  return to_bf16(f);
}

template <bool kF16>
__device__ __forceinline__ float from_half(uint16_t h) {
  if constexpr (kF16) return (float)__builtin_bit_cast(_Float16, h);
  return __builtin_bit_cast(float, (uint32_t)h << 16);
}

// Eight 16-bit sums a + v.
template <bool kF16>
__device__ __forceinline__ u32x4 add8(const u32x4& v, const u32x4& a) {
  u32x4 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float lo = from_half<kF16>((uint16_t)a[q]) + from_half<kF16>((uint16_t)v[q]);
    const float hi = from_half<kF16>((uint16_t)(a[q] >> 16)) + from_half<kF16>((uint16_t)(v[q] >> 16));
    o[q] = (uint32_t)to_half<kF16>(lo) | (uint32_t)to_half<kF16>(hi) << 16;
  }
  return o;
}

template <bool kF16>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (kF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}

// s_waitcnt vmcnt(n) alone, and vmcnt(n) lgkmcnt(0).
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
constexpr int wait_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

// One operand's k-tiles: kKC K-contiguous rows, or k rows of kT columns.
// kT: rows (or columns) of the block tile; kLW waves issue the loads.
template <bool kKC, int kT, int kLW>
struct Operand {
  static constexpr int kElems = kT * BK;            // elements per stage
  static constexpr int kLoads = kT / 8 / kLW;       // 1 KB loads per load wave and tile
  static constexpr int kRowsPerLoad = kKC ? 8 : 512 / kT;  // stage rows one load fills
  static_assert(kT % (8 * kLW) == 0, "loads divide evenly over the load waves");

  uint64_t base;
  uint64_t bytes;      // valid bytes from base
  uint64_t step;       // bytes from one k-tile to the next
  uint32_t off[kLoads];
  uint32_t tail;       // OR-ed into a K-contiguous operand's offsets at the last k-tile

  static __device__ __forceinline__ int swz(int k, int chunk) {
    if (kT < 64) return chunk;  // four rows to 256 bytes
    return kT >= 128 ? chunk ^ ((k & 3) << 2) : chunk ^ (((k >> 1) & 1) << 2);
  }

  // P: the operand's block rows (columns) start, `n` of them valid.
  __device__ __forceinline__ void init(const uint16_t* P, int64_t ld, int n, int K, int ktail, int wave, int lane) {
    base = reinterpret_cast<uint64_t>(P);
    if constexpr (kKC) {
      bytes = (uint64_t)((int64_t)(n - 1) * ld + (K + 7) / 8 * 8) * 2;  // whole chunks
      step = BK * 2;
      const int r = lane >> 3, slot = lane & 7;
      // Every load of a wave starts at a row that is a multiple of 8; the
      // swizzle depends on row % 16 = 8 (first row / 8 odd) + r.
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int row = (i * kLW + wave) * 8 + r;
        const int chunk = slot ^ ((row >> 1) & 7);
        off[i] = (uint32_t)(row * ld * 2 + chunk * 16);
      }
      // kLW is even or 1: with an even count the wave's rows keep their
      // parity, so one tail mask serves all its loads.
      static_assert(kLW % 2 == 0, "an even number of load waves");
      const int chunk0 = slot ^ ((((wave & 1) * 8 + r) >> 1) & 7);
      tail = chunk0 * 8 >= ktail ? 0x80000000u : 0u;
    } else {
      bytes = (uint64_t)((int64_t)(K - 1) * ld + (n + 7) / 8 * 8) * 2;
      step = (uint64_t)ld * (BK * 2);
      tail = 0;
      constexpr int kChunks = kT / 8;  // per k row
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int k = (i * kLW + wave) * kRowsPerLoad + lane / kChunks;
        const int chunk = swz(k, lane % kChunks);
        off[i] = (uint32_t)(k * ld * 2 + chunk * 16) | (chunk * 8 >= n ? 0x80000000u : 0u);
      }
    }
  }
  __device__ __forceinline__ lds_rsrc rsrc(int kt) const {
    const uint64_t d = step * (uint64_t)kt, b = base + d, left = bytes - d;
    return lds_rsrc{(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, left < 0x7fffffffu ? (uint32_t)left : 0x7fffffffu,
                    0x00020000u};
  }
  // Load i of the tile behind `r` into the stage whose first byte is `lds`.
  __device__ __forceinline__ void load(const lds_rsrc& r, int i, bool last, uint32_t lds, int wave) const {
    const uint32_t o = kKC ? off[i] | (last ? tail : 0u) : off[i];
    lds_dma16(r, o, 0u, lds + (uint32_t)(i * kLW + wave) * 1024u);
  }
};

// Fragment addresses of one operand: 32 rows (columns) x 16 k, for the KS
// slabs from slab0 on.
template <bool kKC, int kT, int KS>
struct FragReader {
  int off[KS][kKC ? 1 : 2];
  __device__ __forceinline__ void init(int first, int slab0, int lane) {
    if constexpr (kKC) {
      const int fr = lane & 31, fh = lane >> 5;
#pragma unroll
      for (int s = 0; s < KS; ++s) off[s][0] = (first + fr) * BK + (((2 * (slab0 + s) + fh) ^ ((fr >> 1) & 7)) << 3);
    } else {
      // Lane L (16-lane group g = L / 16, e = (L % 16) / 4, c = L % 4) of
      // transposing read h addresses k row 16 slab + 8 (g / 2) + 4 h + e,
      // columns first + 16 (g % 2) + 4 c .. + 3.
      const int g = lane >> 4, e = (lane >> 2) & 3, c = lane & 3;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = 16 * (slab0 + s) + 8 * (g >> 1) + 4 * h + e;
          const int chunk = first / 8 + 2 * (g & 1) + (c >> 1);
          off[s][h] = k * kT + (Operand<kKC, kT, 2>::swz(k, chunk) << 3) + 4 * (c & 1);
        }
    }
  }
  // Block j: 32 j rows (columns) further.
  __device__ __forceinline__ u32x4 read(const uint16_t* stage, int s, int j) const {
    if constexpr (kKC) {
      return *reinterpret_cast<const u32x4*>(stage + off[s][0] + j * 32 * BK);
    } else {
      // 32 columns are four chunks: the swizzle flips chunk bits 2 and 3, so
      // block j's address is the first block's with chunk bits 2.. XOR j.
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)((lds_u16*)(stage + (off[s][0] ^ (j << 5)))));
      const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)((lds_u16*)(stage + (off[s][1] ^ (j << 5)))));
      const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
      return u32x4{l2[0], l2[1], h2[0], h2[1]};
    }
  }
};

// kOut: 2 (bits of the input type) or 4 (f32, or a k-split's f32 partials).
// WM x WN x WK waves: WK waves share an output sub-tile, each multiplying
// 4 / WK of a k-tile's slabs.
template <bool kF16, int kOut, bool kAK, bool kBKc, int TM, int TN, int WM, int WN, int WK, int kStages, int kLW>
__global__ void __launch_bounds__(WM * WN * WK * 64) gemm_tile(GemmGroup p, const uint16_t* __restrict__ A) {
  constexpr int kWaves = WM * WN * WK, WTM = TM / WM, WTN = TN / WN, MI = WTM / 32, NJ = WTN / 32, KS = 4 / WK;
  // Fragments of a whole k-tile fit in registers twice over: they are read
  // while the tile before multiplies. Otherwise a slab at a time.
  constexpr bool kWhole = MI * NJ <= 4;
  using OpA = Operand<kAK, TM, kLW>;
  using OpB = Operand<kBKc, TN, kLW>;
  constexpr int STAGE = (TM + TN) * BK;
  constexpr int kLoads = OpA::kLoads + OpB::kLoads;
  __shared__ __attribute__((aligned(1024))) uint16_t smem[kStages * STAGE];

  // Consecutive workgroup ids go to the 8 XCDs in turn: each XCD gets a
  // contiguous run of tiles, walked 8 tile rows at a time so that B k-tiles
  // are reused from its L2.
  const int tiles_m = (p.M + TM - 1) / TM, tiles_n = p.tiles_n;
  const int per_batch = tiles_m * tiles_n;
  const int total = gridDim.x;
  const int xcd = blockIdx.x & 7;
  const int unit = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  const int split = unit / (per_batch * p.batch);
  const int bt = unit - split * (per_batch * p.batch);
  const int b = bt / per_batch;
  const int t = bt - b * per_batch;
  const int gsize = 8 * tiles_n;
  const int g = t / gsize;
  const int first_m = g * 8;
  const int gm = min(tiles_m - first_m, 8);
  const int tm = first_m + (t - g * gsize) % gm;
  const int tn = (t - g * gsize) / gm;
  int mi = 0;
#pragma unroll
  for (int i = 1; i < kMaxGemmMembers; ++i)
    if (i < p.count && tn >= p.m[i].tile0) mi = i;
  const GemmMember mb = p.m[mi];
  const int N = mb.N;
  const int m0 = tm * TM, n0 = (tn - mb.tile0) * TN;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = WK == 1 ? 0 : wave % WK;
  const int wm = wave / WK / WN, wn = wave / WK % WN;

  // This split's k-tiles [kt0, kt0 + nk).
  const int nk_all = (p.K + BK - 1) / BK;
  const int kt0 = split * p.split_tiles;
  const int nk = min(p.split_tiles, nk_all - kt0);
  const int ktail = p.K - (nk_all - 1) * BK;
  OpA oa;
  OpB ob;
  oa.init(A + (int64_t)b * p.a_batch_stride + (kAK ? (int64_t)m0 * p.lda : (int64_t)m0), p.lda, min(TM, p.M - m0), p.K,
          ktail, wave, lane);
  ob.init(static_cast<const uint16_t*>(mb.B) + (int64_t)b * mb.b_batch_stride + (kBKc ? (int64_t)n0 * mb.ldb : (int64_t)n0),
          mb.ldb, min(TN, N - n0), p.K, ktail, wave, lane);
  const uint32_t lds0 = lds_offset(smem);

  FragReader<kAK, TM, KS> ra;
  FragReader<kBKc, TN, KS> rb;
  ra.init(wm * WTM, wk * KS, lane);
  rb.init(wn * WTN, wk * KS, lane);
  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  auto load_one = [&](const lds_rsrc& xa, const lds_rsrc& xb, int q, bool last, uint32_t stage) {
    if (q < OpA::kLoads) oa.load(xa, q, last, stage, wave);
    else ob.load(xb, q - OpA::kLoads, last, stage + OpA::kElems * 2, wave);
  };
  auto load_tile = [&](int kt, int stage) {
    const bool last = kt0 + kt == nk_all - 1;
    const lds_rsrc xa = oa.rsrc(kt0 + kt), xb = ob.rsrc(kt0 + kt);
#pragma unroll
    for (int q = 0; q < kLoads; ++q) load_one(xa, xb, q, last, lds0 + (uint32_t)stage * (STAGE * 2));
  };

  // Tile indices past the last reload it into the free stage, so the load
  // waves' counts stay uniform.
  auto prologue = [&](auto loader) {
    if constexpr (decltype(loader)::value) {
#pragma unroll
      for (int s = 0; s < kStages; ++s) load_tile(min(s, nk - 1), s);
      __builtin_amdgcn_s_waitcnt(wait_vm(kLoads * (kStages - 1)));
    }
    __builtin_amdgcn_s_barrier();
  };
  // Own loads of the next tile landed and own reads of this one done, then
  // everyone's.
  auto next_tile = [&](auto loader) {
    if constexpr (decltype(loader)::value) __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(kLoads * (kStages - 2)));
    else __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(63));
    __builtin_amdgcn_s_barrier();
  };
  // Whole k-tiles of fragments, double-buffered in registers: tile kt + 1's
  // are read (one LDS latency a tile) while tile kt multiplies.
  auto run_whole = [&](auto loader) {
    constexpr bool kL = decltype(loader)::value;
    u32x4 fa[2][KS][MI], fb[2][KS][NJ];
    auto read = [&](int stage, int buf) {
      const uint16_t* sa = smem + stage * STAGE;
      const uint16_t* sb = sa + OpA::kElems;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[buf][s][i] = ra.read(sa, s, i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) fb[buf][s][j] = rb.read(sb, s, j);
      }
    };
    int cur = 0;
    auto body = [&](int kt, auto bufc) {
      constexpr int buf = decltype(bufc)::value;
      next_tile(loader);
      const int nxt = cur + 1 == kStages ? 0 : cur + 1;
      read(nxt, buf ^ 1);
      // Nothing of the next tile moves up here and nothing of this one down:
      // the multiplications below are what covers the reads above.
      __builtin_amdgcn_sched_barrier(0);
      const int kn = min(kt + kStages, nk - 1);
      const bool last = kt0 + kn == nk_all - 1;
      const lds_rsrc xa = oa.rsrc(kt0 + kn), xb = ob.rsrc(kt0 + kn);
      const uint32_t stage = lds0 + (uint32_t)cur * (STAGE * 2);
      constexpr int kMul = KS * MI * NJ, kPer = (kLoads + kMul - 1) / kMul;
#pragma unroll
      for (int q = 0; q < kMul; ++q) {
        const int sl = q / (MI * NJ), i = q / NJ % MI, j = q % NJ;
        acc[i][j] = mfma32<kF16>(fa[buf][sl][i], fb[buf][sl][j], acc[i][j]);
        if constexpr (kL) {
#pragma unroll
          for (int e = q * kPer; e < (q + 1) * kPer && e < kLoads; ++e) load_one(xa, xb, e, last, stage);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      cur = nxt;
    };
    prologue(loader);
    read(0, 0);
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      body(kt, std::integral_constant<int, 0>{});
      body(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) body(kt, std::integral_constant<int, 0>{});
  };
  // A slab at a time: the next slab's fragments are read while the current
  // one multiplies, and the last slab's multiplications cover the barrier.
  auto run_slabs = [&](auto loader) {
    constexpr bool kL = decltype(loader)::value;
    u32x4 fa[2][MI], fb[2][NJ];
    auto read_slab = [&](int stage, int s, int buf) {
      const uint16_t* sa = smem + stage * STAGE;
      const uint16_t* sb = sa + OpA::kElems;
      fa[buf][0] = ra.read(sa, s, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) fb[buf][j] = rb.read(sb, s, j);
#pragma unroll
      for (int i = 1; i < MI; ++i) fa[buf][i] = ra.read(sa, s, i);
    };
    prologue(loader);
    read_slab(0, 0, 0);
    int cur = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int nxt = cur + 1 == kStages ? 0 : cur + 1;
#pragma unroll
      for (int s = 0; s + 1 < KS; ++s) {
        read_slab(cur, s + 1, (s + 1) & 1);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i][j] = mfma32<kF16>(fa[s & 1][i], fb[s & 1][j], acc[i][j]);
        // Fragment reads spread between the MFMAs.
        constexpr int kReads = MI * (kAK ? 1 : 2) + NJ * (kBKc ? 1 : 2);
        constexpr int kEach = (kReads + MI * NJ - 1) / (MI * NJ), kPairs = kReads / kEach;
#pragma unroll
        for (int q = 0; q < kPairs; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x100, kEach, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        if constexpr (kPairs * kEach < kReads) __builtin_amdgcn_sched_group_barrier(0x100, kReads - kPairs * kEach, 0);
        if constexpr (kPairs < MI * NJ) __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ - kPairs, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      next_tile(loader);
      read_slab(nxt, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      const int kn = min(kt + kStages, nk - 1);
      const bool last = kt0 + kn == nk_all - 1;
      const lds_rsrc xa = oa.rsrc(kt0 + kn), xb = ob.rsrc(kt0 + kn);
      const uint32_t stage = lds0 + (uint32_t)cur * (STAGE * 2);
      constexpr int kPer = (kLoads + MI * NJ - 1) / (MI * NJ);
#pragma unroll
      for (int q = 0; q < MI * NJ; ++q) {
        acc[q / NJ][q % NJ] = mfma32<kF16>(fa[(KS - 1) & 1][q / NJ], fb[(KS - 1) & 1][q % NJ], acc[q / NJ][q % NJ]);
        if constexpr (kL) {
#pragma unroll
          for (int e = q * kPer; e < (q + 1) * kPer && e < kLoads; ++e) load_one(xa, xb, e, last, stage);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      cur = nxt;
    }
  };
  auto run = [&](auto loader) {
    if constexpr (kWhole) run_whole(loader);
    else run_slabs(loader);
  };
  if constexpr (kLW == kWaves) {
    run(std::true_type{});
  } else {
    if (wave < kLW) run(std::true_type{});
    else run(std::false_type{});
  }
  // The reloads of the last tile have landed before the stages are reused.
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
  __syncthreads();

  // WK waves hold partial sums of one sub-tile: wave k of them keeps 32 x 32
  // blocks k, k + WK, ... and adds the others' sums of those, in wave order.
  constexpr int kBlocks = MI * NJ / WK;
  f32x16 own[kBlocks];
  static_assert(MI * NJ % WK == 0, "blocks divide over the waves of a k-tile");
  static_assert(kWaves * (MI * NJ - kBlocks) * 4096 <= kStages * STAGE * 2, "the exchanged blocks fit in the stages");
  if constexpr (WK == 1) {
#pragma unroll
    for (int q = 0; q < kBlocks; ++q) own[q] = acc[q / NJ][q % NJ];
  } else {
    // Block q of wave w for wave o = q % WK, slot (w, o - (o > w)) * ...:
    // float4 groups of 64 lanes.
    f32x4* ex = reinterpret_cast<f32x4*>(smem);
    const int grp = wave / WK * WK;
    auto slot = [&](int from, int to, int i) {
      return ((((grp + from) * (WK - 1) + (to > from ? to - 1 : to)) * kBlocks + i) * 4) * 64 + lane;
    };
#pragma unroll
    for (int q = 0; q < MI * NJ; ++q)
      if (q % WK != wk) {
        const int at = slot(wk, q % WK, q / WK);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          ex[at + e * 64] = f32x4{acc[q / NJ][q % NJ][4 * e], acc[q / NJ][q % NJ][4 * e + 1],
                                  acc[q / NJ][q % NJ][4 * e + 2], acc[q / NJ][q % NJ][4 * e + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
#pragma unroll
      for (int w = 0; w < WK; ++w) {
        f32x16 part;
        if (w == wk) {
#pragma unroll
          for (int c = 0; c < WK; ++c)
            if (c == wk) part = acc[(i * WK + c) / NJ][(i * WK + c) % NJ];
        } else {
          const int at = slot(w, wk, i);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x4 v = ex[at + e * 64];
#pragma unroll
            for (int r = 0; r < 4; ++r) part[4 * e + r] = v[r];
          }
        }
        if (w == 0) own[i] = part;
        else own[i] += part;
      }
    }
    if constexpr (kOut == 2) __syncthreads();  // the exchange is read before the staging below
  }

  // Epilogue: lane L holds rows 8 (r / 4) + 4 (L / 32) + r % 4, column L % 32
  // of each 32 x 32 block.
  const int fr = lane & 31, fh = lane >> 5;
  const int wrow0 = wm * WTM, wcol0 = wn * WTN;
  if constexpr (kOut == 2) {
    // The tile is staged through LDS and written a row segment of 16 lanes at
    // a time, 16 bytes a lane.
    constexpr int kCh = TN / 8;  // 16-byte chunks per staged row
    auto at = [&](int row, int ch) { return row * TN + ((ch ^ ((row >> 1) & 7)) << 3); };
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      const int q = i * WK + wk, bi = q / NJ, bj = q % NJ;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = wrow0 + bi * 32 + (r >> 2) * 8 + fh * 4 + (r & 3), col = wcol0 + bj * 32 + fr;
        smem[at(row, col >> 3) + (col & 7)] = to_half<kF16>(own[i][r]);
      }
    }
    __syncthreads();
    uint16_t* Cb = static_cast<uint16_t*>(mb.C) + (int64_t)b * p.M * N;
    const uint16_t* add = static_cast<const uint16_t*>(mb.add) + (mb.add_ld ? (int64_t)b * p.M * N : 0);
    const bool vec = N % 8 == 0;
#pragma unroll
    for (int tt = 0; tt < TM * kCh / (kWaves * 64); ++tt) {
      const int c = tid + kWaves * 64 * tt;
      const int row = c / kCh, ch = c % kCh;
      const int m = m0 + row, n = n0 + ch * 8;
      if (m >= p.M || n >= N) continue;
      u32x4 v = *reinterpret_cast<const u32x4*>(&smem[at(row, ch)]);
      if (vec) {
        if (mb.add) v = add8<kF16>(v, *reinterpret_cast<const u32x4*>(add + m * mb.add_ld + n));
        *reinterpret_cast<u32x4*>(Cb + (int64_t)m * N + n) = v;
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (n + q < N) {
            uint16_t x = (uint16_t)(v[q >> 1] >> ((q & 1) * 16));
            if (mb.add) x = to_half<kF16>(from_half<kF16>(add[m * mb.add_ld + n + q]) + from_half<kF16>(x));
            Cb[(int64_t)m * N + n + q] = x;
          }
      }
    }
  } else {
    float* Cb = static_cast<float*>(mb.C) + ((int64_t)split * p.batch + b) * p.M * N;
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      const int q = i * WK + wk, bi = q / NJ, bj = q % NJ;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wrow0 + bi * 32 + (r >> 2) * 8 + fh * 4 + (r & 3);
        const int n = n0 + wcol0 + bj * 32 + fr;
        if (m < p.M && n < N) Cb[(int64_t)m * N + n] = own[i][r];
      }
    }
  }
}

// C[i] = (add +) the sum over the k-splits of their f32 partials, in split
// order; one grid row per member.
struct SplitSum {
  int splits = 1, count = 1;
  struct {
    const float* part = nullptr;
    void* C = nullptr;
    const void* add = nullptr;
    int64_t n = 0, N = 1, add_ld = 0;
  } m[kMaxGemmMembers];
};
template <int kOutKind>  // 0 bf16, 1 f16, 2 f32
__global__ void __launch_bounds__(256) splitk_reduce(SplitSum p) {
  constexpr bool f16 = kOutKind == 1;
  const auto& mb = p.m[blockIdx.y];
  const int64_t n = mb.n;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  const float* part = mb.part;
  const uint16_t* add = static_cast<const uint16_t*>(mb.add);
  if (mb.N % 4 == 0) {
    f32x4 s = *reinterpret_cast<const f32x4*>(part + i);
#pragma unroll 4
    for (int k = 1; k < p.splits; ++k) s += *reinterpret_cast<const f32x4*>(part + (int64_t)k * n + i);
    if constexpr (kOutKind == 2) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(mb.C) + i) = s;
    } else {
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = to_half<f16>(s[e]);
      if (add) {
        const uint16_t* a = add + (mb.add_ld ? i : i % mb.N);
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = to_half<f16>(from_half<f16>(a[e]) + from_half<f16>(h[e]));
      }
      *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(mb.C) + i) =
          u32x2{(uint32_t)h[0] | (uint32_t)h[1] << 16, (uint32_t)h[2] | (uint32_t)h[3] << 16};
    }
    return;
  }
  for (int64_t j = i; j < min(i + 4, n); ++j) {
    float s = part[j];
    for (int k = 1; k < p.splits; ++k) s += part[(int64_t)k * n + j];
    if constexpr (kOutKind == 2) {
      static_cast<float*>(mb.C)[j] = s;
    } else {
      uint16_t h = to_half<f16>(s);
      if (add) h = to_half<f16>(from_half<f16>(add[mb.add_ld ? j : j % mb.N]) + from_half<f16>(h));
      static_cast<uint16_t*>(mb.C)[j] = h;
    }
  }
}

template <bool kF16>
__global__ void __launch_bounds__(256) add_rows16(uint16_t* __restrict__ C, const uint16_t* __restrict__ add, int64_t total,
                                                  int64_t n, int64_t add_ld) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < total) C[i] = to_half<kF16>(from_half<kF16>(add[add_ld ? i : i % n]) + from_half<kF16>(C[i]));
}

// out[b][r] = in[b][r] (cols 16-bit elements, any alignment) in rows of ldp
// elements, a multiple of 8, filled up with zeros.
__global__ void __launch_bounds__(256) pad_rows16(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                  int64_t bs, int64_t rows, int64_t rs, int64_t cols, int64_t ldp) {
  const int64_t chunks = ldp / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * chunks) return;
  const int64_t r = i / chunks, c = (i - r * chunks) * 8;
  const uint16_t* src = in + (int64_t)blockIdx.y * bs + r * rs;
  u32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = c + 2 * e < cols ? src[c + 2 * e] : 0u, hi = c + 2 * e + 1 < cols ? src[c + 2 * e + 1] : 0u;
    v[e] = lo | hi << 16;
  }
  *reinterpret_cast<u32x4*>(out + ((int64_t)blockIdx.y * rows + r) * ldp + c) = v;
}

void check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail(Code::kInternal, strformat("%s launch failed: %s", what, hipGetErrorString(e)));
}

// The block tiles. us_tile and us_edge: measured microseconds of one 64-deep
// k-tile of a workgroup that has its CU to itself (co-resident workgroups of
// the smaller tiles share the CU's rate, so theirs add up), and of a
// workgroup's start and end (first loads, epilogue); resident: workgroups a
// CU holds (LDS).
struct Tile {
  int tm, tn;
  float us_tile, us_edge;
  int resident;
};
constexpr Tile kTiles[kGemmTiles] = {
    {256, 256, 1.30f, 7.0f, 1}, {128, 256, 0.66f, 4.7f, 1}, {128, 128, 0.39f, 3.7f, 1},
    {64, 128, 0.31f, 2.5f, 2},  {64, 64, 0.22f, 1.8f, 2},   {32, 64, 0.20f, 1.8f, 3},
};
constexpr int kCus = 256;
constexpr int kMinSplitTiles = 4;  // k-tiles a split must have

int64_t tile_columns(const GemmGroup& g, const Tile& t) {
  int64_t n = 0;
  for (int i = 0; i < g.count; ++i) n += (g.m[i].N + t.tn - 1) / t.tn;
  return n;
}
int64_t tiles_of(const GemmGroup& g, const Tile& t) {
  return (int64_t)((g.M + t.tm - 1) / t.tm) * tile_columns(g, t) * g.batch;
}

template <bool kF16, int kOut, bool kAK, bool kBKc>
void launch_cfg(hipStream_t s, int cfg, unsigned grid, const GemmGroup& g, const uint16_t* A) {
#define PJRTX_TILE(TM, TN, WM, WN, WK, ST, LW)                                                             \
  hipLaunchKernelGGL((gemm_tile<kF16, kOut, kAK, kBKc, TM, TN, WM, WN, WK, ST, LW>), dim3(grid),           \
                     dim3(WM * WN * WK * 64), 0, s, g, A)
  switch (cfg) {
    case 0: PJRTX_TILE(256, 256, 2, 4, 1, 2, 4); break;
    case 1: PJRTX_TILE(128, 256, 2, 4, 1, 3, 8); break;
    case 2: PJRTX_TILE(128, 128, 2, 2, 2, 4, 8); break;
    case 3: PJRTX_TILE(64, 128, 2, 2, 1, 3, 4); break;
    case 4: PJRTX_TILE(64, 64, 1, 2, 2, 5, 4); break;
    default: PJRTX_TILE(32, 64, 1, 1, 2, 4, 2); break;
  }
#undef PJRTX_TILE
}

template <bool kF16, int kOut>
void launch_layout(hipStream_t s, int cfg, unsigned grid, const GemmGroup& g, const void* A, bool a_kmajor, bool b_kmajor) {
  const uint16_t* a = static_cast<const uint16_t*>(A);
  if (a_kmajor) {
    if (b_kmajor) launch_cfg<kF16, kOut, true, true>(s, cfg, grid, g, a);
    else launch_cfg<kF16, kOut, true, false>(s, cfg, grid, g, a);
  } else {
    if (b_kmajor) launch_cfg<kF16, kOut, false, true>(s, cfg, grid, g, a);
    else launch_cfg<kF16, kOut, false, false>(s, cfg, grid, g, a);
  }
}

}  // namespace

bool gemm_fits(const GemmGroup& g, bool a_kmajor, bool b_kmajor) {
  // A load's lane offset (a block of K-contiguous rows, or 64 k rows) stays
  // below 2^31 bytes; 16-byte chunks are aligned.
  const int64_t limit = int64_t(1) << 30;
  const auto ok = [&](int64_t ld, int64_t bs, bool kc, int64_t len) {
    return ld % 8 == 0 && bs % 8 == 0 && (kc ? 256 : BK) * ld < limit && ld >= len;
  };
  bool fits = g.M > 0 && g.K > 0 && g.count >= 1 && g.count <= kMaxGemmMembers &&
              ok(g.lda, g.a_batch_stride, a_kmajor, a_kmajor ? g.K : g.M);
  for (int i = 0; i < g.count && fits; ++i)
    fits = g.m[i].N > 0 && ok(g.m[i].ldb, g.m[i].b_batch_stride, b_kmajor, b_kmajor ? g.K : g.m[i].N);
  // Workgroups (splits only of few tiles) and their ids stay below 2^31.
  return fits && tiles_of(g, kTiles[kGemmTiles - 1]) < (int64_t(1) << 30);
}

GemmPlan plan_gemm(const GemmGroup& g, int64_t max_workspace) {
  const int64_t nk = (g.K + BK - 1) / BK;
  const int64_t forced = env_int("PJRTX_GEMM_TILE", -1);
  const int64_t big_min = env_int("PJRTX_BIG_GEMM_MIN_TILES", 0);
  int64_t n_all = 0;
  for (int i = 0; i < g.count; ++i) n_all += g.m[i].N;
  const int64_t out_bytes = int64_t(4) * g.batch * g.M * n_all;
  GemmPlan best;
  double best_us = 1e30;
  for (int c = 0; c < kGemmTiles; ++c) {
    const Tile& t = kTiles[c];
    const int64_t tiles = tiles_of(g, t);
    if (forced >= 0 && forced < kGemmTiles && c != forced) continue;
    if (forced < 0 && big_min > 0 && g.M >= 256 && n_all >= 256 && tiles_of(g, kTiles[0]) >= big_min && c != 0) continue;
    for (int64_t want = 1; want <= 64; want += want < 8 ? 1 : want / 4) {
      const int64_t per = (nk + want - 1) / want, splits = (nk + per - 1) / per;
      if (splits != want) continue;
      if (splits > 1 && (per < kMinSplitTiles || splits * (double)out_bytes > (double)max_workspace)) break;
      // Every round of kCus workgroups multiplies its k-tiles; the splits'
      // partials are written, then read by a second launch (2.5 us and the
      // bytes at 6 TB/s).
      const int64_t rounds = (tiles * splits + kCus - 1) / kCus;
      double us = 2.0 + (double)rounds * per * t.us_tile + (double)((rounds + t.resident - 1) / t.resident) * t.us_edge;
      if (splits > 1) us += 2.5 + 2.0 * splits * (double)out_bytes / 6e6;
      if (us < best_us) {
        best_us = us;
        best.cfg = c;
        best.splits = static_cast<int>(splits);
        best.split_tiles = static_cast<int>(per);
      }
      if (tiles * splits >= 2 * kCus) break;
    }
  }
  best.workspace = best.splits > 1 ? (size_t)best.splits * out_bytes : 0;
  return best;
}

void launch_gemm(hipStream_t s, GemmGroup g, const GemmPlan& plan, const void* A, bool a_kmajor, bool b_kmajor, bool f16,
                 int out_bytes, float* workspace) {
  const Tile& t = kTiles[plan.cfg];
  const int64_t grid = tiles_of(g, t) * plan.splits;
  PJRTX_CHECK(grid > 0 && grid < (int64_t(1) << 31) && (plan.splits == 1 || workspace), Code::kInternal, "gemm: bad plan");
  g.split_tiles = plan.split_tiles;
  g.tiles_n = 0;
  SplitSum sum;
  sum.splits = plan.splits;
  sum.count = g.count;
  int64_t most = 0;
  for (int i = 0; i < g.count; ++i) {
    GemmMember& m = g.m[i];
    PJRTX_CHECK(!m.add || out_bytes == 2, Code::kInternal, "gemm: an addend needs a 16-bit result");
    PJRTX_CHECK(!m.add || m.add_ld == 0 || m.add_ld == m.N, Code::kInternal, "gemm: an addend's rows are not the product's");
    m.tile0 = g.tiles_n;
    g.tiles_n += (m.N + t.tn - 1) / t.tn;
    if (plan.splits > 1) {
      const int64_t n = (int64_t)g.batch * g.M * m.N;
      sum.m[i] = {workspace, m.C, m.add, n, m.N, m.add_ld};
      m.C = workspace;
      m.add = nullptr;
      workspace += n * plan.splits;
      most = std::max(most, n);
    }
  }
  const unsigned gr = static_cast<unsigned>(grid);
  const bool half_out = plan.splits == 1 && out_bytes == 2;
  if (half_out) {
    if (f16) launch_layout<true, 2>(s, plan.cfg, gr, g, A, a_kmajor, b_kmajor);
    else launch_layout<false, 2>(s, plan.cfg, gr, g, A, a_kmajor, b_kmajor);
  } else {
    if (f16) launch_layout<true, 4>(s, plan.cfg, gr, g, A, a_kmajor, b_kmajor);
    else launch_layout<false, 4>(s, plan.cfg, gr, g, A, a_kmajor, b_kmajor);
  }
  if (plan.splits > 1) {
    const dim3 sg(static_cast<unsigned>((most + 1023) / 1024), static_cast<unsigned>(g.count)), block(256);
    if (out_bytes == 4) hipLaunchKernelGGL((splitk_reduce<2>), sg, block, 0, s, sum);
    else if (f16) hipLaunchKernelGGL((splitk_reduce<1>), sg, block, 0, s, sum);
    else hipLaunchKernelGGL((splitk_reduce<0>), sg, block, 0, s, sum);
  }
  check("gemm_tile");
}

void launch_add_rows16(hipStream_t s, void* C, const void* add, int64_t rows, int64_t n, int64_t add_ld, bool f16) {
  const int64_t total = rows * n;
  if (total == 0) return;
  PJRTX_CHECK((total + 255) / 256 < (int64_t(1) << 31), Code::kInternal, "add_rows16: grid too large");
  const dim3 grid(static_cast<unsigned>((total + 255) / 256)), block(256);
  uint16_t* c = static_cast<uint16_t*>(C);
  const uint16_t* a = static_cast<const uint16_t*>(add);
  if (f16) hipLaunchKernelGGL((add_rows16<true>), grid, block, 0, s, c, a, total, n, add_ld);
  else hipLaunchKernelGGL((add_rows16<false>), grid, block, 0, s, c, a, total, n, add_ld);
  check("add_rows16");
}

void launch_pad_rows16(hipStream_t s, const void* in, void* out, int64_t batch, int64_t bs, int64_t rows, int64_t rs,
                       int64_t cols, int64_t ldp) {
  if (batch == 0 || rows == 0 || ldp == 0) return;
  const int64_t blocks = (rows * (ldp / 8) + 255) / 256;
  PJRTX_CHECK(blocks < (int64_t(1) << 31), Code::kInternal, "pad_rows16: grid too large");
  constexpr int64_t kMost = 65535;  // batches a launch's grid holds
  for (int64_t b = 0; b < batch; b += kMost)
    hipLaunchKernelGGL(pad_rows16, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(std::min(kMost, batch - b))),
                       dim3(256), 0, s, static_cast<const uint16_t*>(in) + b * bs,
                       static_cast<uint16_t*>(out) + b * rows * ldp, bs, rows, rs, cols, ldp);
  check("pad_rows16");
}

}  // namespace pjrtx
