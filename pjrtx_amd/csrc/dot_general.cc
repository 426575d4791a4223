// dot_general: StableHLO dimension numbers -> batched GEMM / GEMV launch.
//
// Output dims follow StableHLO (batch..., lhs free..., rhs free...), the same
// order the reference produces (reference: src/backend/mlx_metal/api.cc:
// 1562-1577, 3429-3492). Each operand is viewed as [batch][rows][K] or
// [batch][K][cols] with uniform strides when its dimension groups can be
// merged; otherwise it is first copied into that canonical layout.
#include <algorithm>
#include <map>

#include "blaslt.h"
#include "kernels/dot.h"
#include "kernels/library.h"
#include "runtime.h"

namespace pjrtx {

namespace {

struct OperandView {
  int64_t batch = 1, free = 1, k = 1;
  int64_t bs = 0, fs = 0, ks = 0;  // strides (elements); 0 when the group is empty
  bool ok = true;                  // groups mergeable into single strides
};

// Merges a group of dims (in the given order) into one (size, stride). False
// where the group has no one stride; the size is set all the same.
bool merge(const Dims& dims, const int64_t* strides, const std::vector<int64_t>& group, int64_t* size, int64_t* stride) {
  *size = 1;
  *stride = 0;
  if (group.empty()) return true;
  *stride = strides[group.back()];
  for (const int64_t d : group) *size *= dims[d];
  int64_t outer = -1;  // the non-unit dim before d: d follows it where d's extent is its stride
  for (const int64_t d : group) {
    if (dims[d] == 1) continue;
    if (outer >= 0 && strides[outer] != strides[d] * dims[d]) return false;
    outer = d;
    *stride = strides[d];
  }
  return true;
}

OperandView view_of(const TensorType& t, const Dims& batch, const Dims& contract) {
  int64_t st[kMaxRank];
  int64_t s = 1;
  for (int i = t.rank() - 1; i >= 0; --i) {
    st[i] = s;
    s *= t.dims[i];
  }
  std::vector<int64_t> b(batch.begin(), batch.end()), c(contract.begin(), contract.end()), f;
  for (int d = 0; d < t.rank(); ++d)
    if (std::find(b.begin(), b.end(), d) == b.end() && std::find(c.begin(), c.end(), d) == c.end()) f.push_back(d);
  OperandView v;
  const bool bo = merge(t.dims, st, b, &v.batch, &v.bs), fo = merge(t.dims, st, f, &v.free, &v.fs),
             co = merge(t.dims, st, c, &v.k, &v.ks);
  v.ok = bo && fo && co;
  return v;
}

// Both operands of a product as the block tiles read them: K-contiguous as it
// is, else M- or N-contiguous. `ready` is false where an operand is neither.
struct DotLayout {
  bool ready = false, a_kmajor = false, b_kmajor = false;
};
DotLayout layout_of(const OperandView& a, const OperandView& b) {
  DotLayout l;
  l.a_kmajor = a.ks == 1 || a.k == 1;
  l.b_kmajor = (b.ks == 1 || b.k == 1) && !(b.fs == 1 && b.free != 1);
  l.ready = a.ok && b.ok && (l.a_kmajor || a.fs == 1 || a.free == 1) && (l.b_kmajor || b.fs == 1 || b.free == 1);
  return l;
}

// True where every 16-byte piece of the operand's rows lies on a 16-byte
// boundary (of an aligned base) and inside the operand: an operand with rows
// that do not is copied into padded ones.
bool whole_rows(const OperandView& v, bool kmajor) {
  const int64_t rows = kmajor ? v.free : v.k, cols = kmajor ? v.k : v.free, ld = kmajor ? v.fs : v.ks;
  return (rows == 1 || ld % 8 == 0) && (v.batch == 1 || v.bs % 8 == 0) && (cols % 8 == 0 || (!kmajor && rows > 1));
}

int64_t round8(int64_t n) { return (n + 7) / 8 * 8; }

GemmParams gemm_params(const OperandView& a, const OperandView& b, const DotLayout& l) {
  GemmParams g;
  g.batch = static_cast<int>(a.batch);
  g.M = static_cast<int>(a.free);
  g.N = static_cast<int>(b.free);
  g.K = static_cast<int>(a.k);
  // One row only: its stride is not used; a multiple of 8.
  g.lda = l.a_kmajor ? (a.free == 1 ? round8(a.k) : a.fs) : (a.k == 1 ? round8(a.free) : a.ks);
  g.ldb = l.b_kmajor ? (b.free == 1 ? round8(b.k) : b.fs) : (b.k == 1 ? round8(b.free) : b.ks);
  g.ldc = b.free;
  g.a_batch_stride = a.batch == 1 ? 0 : a.bs;
  g.b_batch_stride = a.batch == 1 ? 0 : b.bs;
  return g;
}
GemmGroup gemm_group(const GemmParams& g) {
  GemmGroup gg;
  gg.batch = g.batch;
  gg.M = g.M;
  gg.K = g.K;
  gg.lda = g.lda;
  gg.a_batch_stride = g.a_batch_stride;
  gg.m[0].N = g.N;
  gg.m[0].ldb = g.ldb;
  gg.m[0].b_batch_stride = g.b_batch_stride;
  return gg;
}

// Decode rows that contract a short ragged K go to the tiles with padded rows:
// the GEMV walks K's rows one at a time. us GEMV / tiles: 4 x 44 x 512 9.4 /
// 6.7, 6 x 58 x 16 16.4 / 6.7, three batches of 7 x 73 x 896 19 / 7.
bool short_ragged_rows(const OperandView& a) { return a.free >= 2 && a.free <= 8 && a.k % 8 != 0 && a.k <= 128; }

// True where one launch of the scalar kernel is faster than the launches the
// matrix-core kernels take for this 16-bit product with its copies and pads.
// Measured: 2.2 us + 0.19 a contracted element (its loads are a chain), or + 2 us
// a million results + 0.42 a million multiplications (0.66 where neighbouring
// results read B rows apart), against 4.1 us for the tiles with 0.75 a million
// results (of whole 64 x 64 tiles), 6.3 for the GEMV of decode rows (3.7 with one
// row) and 2.6 for every launch before or after them.
// us scalar / padded: [256, 256] K = 9 3.9 / 9.4, K = 28 7.2 / 9.5, K = 44 10.2
// / 9.5; [1000, 520] K = 5 4.5 / 7.2, K = 20 8.1 / 7.4; [4096, 512] K = 5 10.4 /
// 8.3. `add_apart`: an addend the tiles would add in place.
bool scalar_is_faster(OperandView a, OperandView b, bool a_aligned, bool b_aligned, bool add_apart) {
  const int64_t M = a.free, N = b.free, K = a.k, batch = a.batch;
  int extra = 0;  // launches the scalar kernel does without (an operand with no one stride is copied for it, too)
  for (OperandView* v : {&a, &b})
    if (!v->ok) {
      *v = OperandView{v->batch, v->free, v->k, v->free * v->k, v->k, 1, true};
      (v == &a ? a_aligned : b_aligned) = true;
    }
  const bool gemv = M <= 8 && !short_ragged_rows(a);
  if (a.ks != 1 && K != 1 && gemv) {
    a = OperandView{batch, M, K, M * K, K, 1, true};
    a_aligned = true;
    ++extra;
  }
  const DotLayout l = layout_of(a, b);
  if (!l.ready) return false;
  const bool b_whole = b_aligned && whole_rows(b, l.b_kmajor);
  double other = 4.1;
  if (gemv && (a.ks == 1 || K == 1) && b_whole && (l.b_kmajor || N % 8 == 0) &&
      (!l.b_kmajor || (a_aligned && (M == 1 || a.fs % 8 == 0) && (batch == 1 || a.bs % 8 == 0)))) {
    if (extra == 0 && (K % 8 == 0 || M == 1)) return false;
    other = M == 1 ? 3.7 : 6.3;
    add_apart = false;  // the GEMV's result is added to in another launch as well
  } else {
    extra += !(a_aligned && whole_rows(a, l.a_kmajor)) + !b_whole;
    if (extra == 0 && K % 8 == 0) return false;
    other += 0.75e-6 * 4096 * static_cast<double>(batch) * ((M + 63) / 64) * ((N + 63) / 64);
  }
  const double results = static_cast<double>(batch) * M * N;
  const double chain = std::max(3.8, 2.2 + 0.19 * K);
  const double stream = 2.2 + results * (2e-6 + K * (b.fs == 1 || N == 1 ? 0.42e-6 : 0.66e-6));
  return std::max(chain, stream) + (add_apart ? 2.6 : 0.0) < other + 2.6 * extra;
}

// Decode rows with few and ragged N-contiguous columns: B is transposed for the
// K-contiguous GEMV, which spreads each column's K over lanes, where padded rows
// would go to the tiles and their k-splits. us transposed / padded: 1 x 2048 x
// 33 6.8 / 12.0, x 257 8.8 / 12.7, x 1001 15.5 / 15.4; 3 x 4096 x 257 14.8 /
// 15.9; 8 x 4096 x 33 19.2 / 13.3; with K = 256 they are equal.
bool few_ragged_columns(const OperandView& a, const OperandView& b) {
  return b.ok && a.batch == 1 && a.free <= 4 && b.free <= 512 && b.free % 8 != 0 && b.k >= 512 && b.k % 8 == 0 && b.ks != 1;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Copies `t` into a canonical [batch][free][k] (or [batch][k][free] when
// k_inner is false) row-major buffer.
MemRef canonicalize(Device* dev, const TensorType& t, const Dims& batch, const Dims& contract, const void* src,
                    bool k_inner) {
  int64_t st[kMaxRank];
  int64_t s = 1;
  for (int i = t.rank() - 1; i >= 0; --i) {
    st[i] = s;
    s *= t.dims[i];
  }
  std::vector<int64_t> order(batch.begin(), batch.end()), f;
  for (int d = 0; d < t.rank(); ++d)
    if (std::find(batch.begin(), batch.end(), d) == batch.end() &&
        std::find(contract.begin(), contract.end(), d) == contract.end())
      f.push_back(d);
  if (k_inner) {
    order.insert(order.end(), f.begin(), f.end());
    order.insert(order.end(), contract.begin(), contract.end());
  } else {
    order.insert(order.end(), contract.begin(), contract.end());
    order.insert(order.end(), f.begin(), f.end());
  }
  BoxCopy b;
  b.rank = t.rank();
  int64_t ds = 1;
  for (int i = b.rank - 1; i >= 0; --i) {
    const int64_t d = order[i];
    b.dims[i] = t.dims[d];
    b.src_stride[i] = st[d];
    b.dst_stride[i] = ds;
    ds *= t.dims[d];
  }
  MemRef out = dev->allocate(t.bytes());
  launch_box_copy(dev->stream(), b, src, out->ptr, static_cast<int>(dtype_size(t.dtype)));
  return out;
}

}  // namespace

// Workgroups of the one-pass GEMV for a single product with N columns.
int single_wide_tiles(int64_t N) {
  GemvGroup one;
  one.count = 1;
  one.m[0].N = static_cast<int>(N);
  return gemv_wide_tiles(one);
}

// Row stride of a product's addend (GemmMember::add_ld). The product is
// [batch][M][N] with N all of the right operand's free dims, whatever their
// number, and so is an addend of the result's shape; a bias is one row for all.
int64_t dot_addend_stride(const Program& prog, const Op& dot, bool row) {
  return row ? 0 : view_of(prog.type(dot.operands[1]), dot.rhs_batch, dot.rhs_contract).free;
}

std::string describe_dot(const Program& prog, const Op& dot, bool add) {
  OperandView a = view_of(prog.type(dot.operands[0]), dot.lhs_batch, dot.lhs_contract);
  OperandView b = view_of(prog.type(dot.operands[1]), dot.rhs_batch, dot.rhs_contract);
  const bool a_copied = !a.ok, b_copied = !b.ok || few_ragged_columns(a, b);
  const bool scalar = scalar_is_faster(a, b, true, true, add);
  for (OperandView* v : {&a, &b})
    if (v == &a ? a_copied : b_copied) *v = OperandView{v->batch, v->free, v->k, v->free * v->k, v->k, 1, true};
  const DotLayout l = layout_of(a, b);
  const auto one = [](bool copied, const OperandView& v, bool kmajor) {
    return copied ? "\"copied\"" : !whole_rows(v, kmajor) ? "\"padded\"" : "\"read\"";
  };
  // With the strides padding gives.
  const auto taken = [](OperandView v, bool kmajor) {
    if (!whole_rows(v, kmajor)) {
      const int64_t rows = kmajor ? v.free : v.k, ld = round8(kmajor ? v.k : v.free);
      v = OperandView{v.batch, v.free, v.k, rows * ld, kmajor ? ld : 1, kmajor ? 1 : ld, true};
    }
    return v;
  };
  const bool tiles = gemm_fits(gemm_group(gemm_params(taken(a, l.a_kmajor), taken(b, l.b_kmajor), l)), l.a_kmajor, l.b_kmajor);
  return std::string("\"operands\":[") + one(a_copied, a, l.a_kmajor) + "," + one(b_copied, b, l.b_kmajor) +
         "],\"block_tiles\":" + (tiles ? "true" : "false") + ",\"scalar\":" + (scalar ? "true" : "false");
}

// Writes the product to the dot's result, plus `add` (GemmMember::add, its
// row stride add_ld) where the block tiles run it; returns whether they did.
bool run_dot_general(Device* dev, const Program& prog, const Op& op, std::vector<MemRef>& vals, const void* add,
                     int64_t add_ld) {
  const TensorType& lt = prog.type(op.operands[0]);
  const TensorType& rt = prog.type(op.operands[1]);
  const TensorType& ot = prog.type(op.results[0]);
  PJRTX_CHECK(lt.rank() <= kMaxRank && rt.rank() <= kMaxRank, Code::kUnimplemented, "dot_general: rank too large");
  PJRTX_CHECK(op.lhs_batch.size() == op.rhs_batch.size() && op.lhs_contract.size() == op.rhs_contract.size(),
              Code::kInvalidArgument, "dot_general: dimension numbers do not pair up");
  for (size_t i = 0; i < op.lhs_batch.size(); ++i)
    PJRTX_CHECK(lt.dims[op.lhs_batch[i]] == rt.dims[op.rhs_batch[i]], Code::kInvalidArgument, "dot_general: batch size mismatch");
  for (size_t i = 0; i < op.lhs_contract.size(); ++i)
    PJRTX_CHECK(lt.dims[op.lhs_contract[i]] == rt.dims[op.rhs_contract[i]], Code::kInvalidArgument,
                "dot_general: contracting size mismatch");
  PJRTX_CHECK(lt.dtype == rt.dtype, Code::kUnimplemented, "dot_general: mixed operand types");

  OperandView a = view_of(lt, op.lhs_batch, op.lhs_contract);
  OperandView b = view_of(rt, op.rhs_batch, op.rhs_contract);
  const int64_t batch = a.batch, M = a.free, N = b.free, K = a.k;
  void* out = vals[op.results[0]]->ptr;
  if (ot.elements() == 0) return true;
  const void* A = vals[op.operands[0]]->ptr;
  const void* B = vals[op.operands[1]]->ptr;
  const bool low_precision = lt.dtype == DType::kBF16 || lt.dtype == DType::kF16;
  const bool out_ok = ot.dtype == lt.dtype || ot.dtype == DType::kF32;
  if (K == 0) {  // empty contraction: zeros
    launch_zero(dev->stream(), out, ot.elements() * static_cast<int64_t>(dtype_size(ot.dtype)));
    return false;
  }
  if (low_precision && out_ok && !scalar_is_faster(a, b, aligned16(A), aligned16(B), add != nullptr)) {
    const bool f16 = lt.dtype == DType::kF16;
    const int out_kind = ot.dtype == DType::kBF16 ? 0 : (ot.dtype == DType::kF16 ? 1 : 2);
    MemRef a_copy, b_copy, a_pad, b_pad;
    // Copies the call makes must fit a fixed block (allocation-free execute)
    // where one is installed; those that would not take the strided fallback.
    const auto fits = [&](int64_t bytes) { return scratch_left(dev) >= bytes + 4096; };
    // (An M-contiguous A goes to the GEMV kernels and to rows too long for
    // 32-bit offsets as a copy.)
    const bool gemv_rows = M <= 8 && !short_ragged_rows(a);
    if ((!a.ok || (a.ks != 1 && K != 1 && (gemv_rows || a.ks >= int64_t(1) << 23))) && fits(lt.bytes())) {
      a_copy = canonicalize(dev, lt, op.lhs_batch, op.lhs_contract, A, true);
      A = a_copy->ptr;
      a = OperandView{batch, M, K, M * K, K, 1, true};
    }
    if ((!b.ok || few_ragged_columns(a, b)) && fits(rt.bytes())) {
      b_copy = canonicalize(dev, rt, op.rhs_batch, op.rhs_contract, B, true);  // [batch][N][K]
      B = b_copy->ptr;
      b = OperandView{batch, N, K, N * K, K, 1, true};
    }
    const auto aligned_rows = [&](const void* p, const OperandView& v, bool kc) { return aligned16(p) && whole_rows(v, kc); };
    const auto pad = [&](const void** p, OperandView* v, bool kc, MemRef* mem) {
      const int64_t rows = kc ? v->free : v->k, cols = kc ? v->k : v->free, ldp = round8(cols);
      if (rows * (ldp / 8) >= (int64_t(1) << 38) || !fits(batch * rows * ldp * 2)) return false;
      *mem = dev->allocate(static_cast<size_t>(batch * rows * ldp) * 2);
      const int64_t rs = kc ? (v->fs ? v->fs : cols) : (v->ks ? v->ks : cols);
      launch_pad_rows16(dev->stream(), *p, (*mem)->ptr, batch, v->bs, rows, rs, cols, ldp);
      *p = (*mem)->ptr;
      v->bs = rows * ldp;
      (kc ? v->fs : v->ks) = ldp;
      (kc ? v->ks : v->fs) = 1;
      return true;
    };
    const DotLayout lay = layout_of(a, b);
    const bool a_kmajor = lay.a_kmajor, b_kmajor = lay.b_kmajor;
    bool ready = lay.ready;
    // Decode rows: W streamed once. (K may be any length for an N-contiguous
    // W; a K-contiguous one needs 16-byte rows.)
    if (ready && gemv_rows && (a.ks == 1 || K == 1) && aligned_rows(B, b, b_kmajor) && (b_kmajor || N % 8 == 0) &&
        (!b_kmajor || (aligned16(A) && (M == 1 || a.fs % 8 == 0) && (batch == 1 || a.bs % 8 == 0)))) {
      if (batch == 1 && !b_kmajor && N < (int64_t(1) << 30) &&
          gemv_wide_fits(static_cast<int>(M), static_cast<int>(K), single_wide_tiles(N))) {
        GemvGroup g;
        g.count = 1;
        g.M = static_cast<int>(M);
        g.K = static_cast<int>(K);
        g.ldx = a.fs ? a.fs : K;
        g.out_kind = out_kind;
        g.m[0].W = B;
        g.m[0].Y = out;
        g.m[0].N = static_cast<int>(N);
        g.m[0].ldw = b.ks ? b.ks : N;
        g.m[0].ldy = N;
        launch_gemv_wide(dev->stream(), g, A, f16);
        return false;
      }
      GemvParams g;
      g.batch = static_cast<int>(batch);
      g.M = static_cast<int>(M);
      g.N = static_cast<int>(N);
      g.K = static_cast<int>(K);
      g.ldx = a.fs ? a.fs : K;
      g.ldw = b_kmajor ? (b.fs ? b.fs : K) : (b.ks ? b.ks : N);
      g.ldy = N;
      g.x_bs = a.bs;
      g.w_bs = b.bs;
      g.y_bs = M * N;
      g.out_kind = out_kind;
      MemRef part;
      bool room = true;
      if (!b_kmajor) {
        plan_gemv_split(&g);
        const int64_t bytes = batch * g.ksplit * M * N * 4;
        if (g.ksplit > 1 && !(room = fits(bytes))) g.ksplit = 1;
        if (g.ksplit > 1) part = dev->allocate(static_cast<size_t>(bytes));
      }
      if (room) {
        launch_gemv(dev->stream(), g, A, B, out, part ? static_cast<float*>(part->ptr) : nullptr, f16, b_kmajor);
        return false;
      }
    }
    if (ready && !aligned_rows(A, a, a_kmajor)) ready = pad(&A, &a, a_kmajor, &a_pad);
    if (ready && !aligned_rows(B, b, b_kmajor)) ready = pad(&B, &b, b_kmajor, &b_pad);
    if (ready) {
      const GemmParams g = gemm_params(a, b, lay);
      if (a_kmajor && K % 8 == 0 && (b_kmajor || N % 8 == 0) && blaslt_wanted(g) &&
          blaslt_gemm(dev, g, A, B, out, f16, b_kmajor, out_kind == 2 ? 4 : 2))
        return false;
      GemmGroup gg = gemm_group(g);
      gg.m[0].B = B;
      gg.m[0].C = out;
      const bool fuse = add && out_kind != 2 && aligned16(add) && aligned16(out);
      if (fuse) gg.m[0].add = add;
      gg.m[0].add_ld = add_ld;
      if (gemm_fits(gg, a_kmajor, b_kmajor)) {
        // Partials of a k-split: at most 64 MiB, and what a fixed block has left.
        const int64_t left = std::max<int64_t>(0, std::min<int64_t>(int64_t(64) << 20, scratch_left(dev) - 4096));
        const GemmPlan plan = plan_gemm(gg, left);
        MemRef ws;
        if (plan.workspace) ws = dev->allocate(plan.workspace);
        launch_gemm(dev->stream(), gg, plan, A, a_kmajor, b_kmajor, f16, out_kind == 2 ? 4 : 2,
                    ws ? static_cast<float*>(ws->ptr) : nullptr);
        return fuse;
      }
      if (a_kmajor && K % 8 == 0 && (b_kmajor || N % 8 == 0)) {
        launch_mfma_gemm(dev->stream(), g, A, B, out, f16, b_kmajor, out_kind == 2 ? 4 : 2);
        return false;
      }
    }
  }
  // Scalar fallback with general strides.
  if (!a.ok) {
    MemRef c = canonicalize(dev, lt, op.lhs_batch, op.lhs_contract, A, true);
    vals.push_back(c);  // keep alive until the step ends
    A = c->ptr;
    a = OperandView{batch, M, K, M * K, K, 1, true};
  }
  if (!b.ok) {
    MemRef c = canonicalize(dev, rt, op.rhs_batch, op.rhs_contract, B, true);
    vals.push_back(c);
    B = c->ptr;
    b = OperandView{batch, N, K, N * K, K, 1, true};
  }
  FmaGemmParams f;
  f.batch = batch;
  f.M = M;
  f.N = N;
  f.K = K;
  f.a_bs = a.bs;
  f.a_ms = a.fs;
  f.a_ks = a.ks;
  f.b_bs = b.bs;
  f.b_ns = b.fs;
  f.b_ks = b.ks;
  f.row_lanes = op.dot_swapped;
  launch_fma_gemm(dev->stream(), f, A, B, out, lt.dtype, ot.dtype);
  return false;
}

// A dot whose result only feeds `add(dot, x)`: out = x + round(dot) as the
// one-pass GEMV's epilogue, or, when that kernel does not apply to these
// buffers, the dot into a temporary followed by the elementwise add.
// `row`: x is one row added to every row of the product (a bias).
void run_dot_residual(Device* dev, const Program& prog, const Op& op, std::vector<MemRef>& vals, int add, int out,
                      bool row) {
  const TensorType& lt = prog.type(op.operands[0]);
  const TensorType& rt = prog.type(op.operands[1]);
  const TensorType& ot = prog.type(op.results[0]);
  const void* A = vals[op.operands[0]]->ptr;
  const void* W = vals[op.operands[1]]->ptr;
  const bool ok = !row && lt.rank() == 2 && rt.rank() == 2 && op.lhs_batch.empty() && op.lhs_contract == Dims{1} &&
                  op.rhs_contract == Dims{0} && (lt.dtype == DType::kBF16 || lt.dtype == DType::kF16) &&
                  rt.dtype == lt.dtype && ot.dtype == lt.dtype && lt.dims[1] % 8 == 0 && rt.dims[1] % 8 == 0 &&
                  aligned16(W) && rt.dims[1] < (int64_t(1) << 30) &&
                  gemv_wide_fits(static_cast<int>(lt.dims[0]), static_cast<int>(lt.dims[1]), single_wide_tiles(rt.dims[1]));
  if (ok) {
    GemvGroup g;
    g.count = 1;
    g.M = static_cast<int>(lt.dims[0]);
    g.K = static_cast<int>(lt.dims[1]);
    g.ldx = lt.dims[1];
    g.out_kind = lt.dtype == DType::kF16 ? 1 : 0;
    g.m[0].W = W;
    g.m[0].Y = vals[out]->ptr;
    g.m[0].add = vals[add]->ptr;
    g.m[0].N = static_cast<int>(rt.dims[1]);
    g.m[0].ldw = rt.dims[1];
    g.m[0].ldy = rt.dims[1];
    launch_gemv_wide(dev->stream(), g, A, lt.dtype == DType::kF16);
    return;
  }
  if (ot.dtype == DType::kBF16 || ot.dtype == DType::kF16) {
    // The block tiles add in their epilogue; any other kernel's product is
    // added to in place.
    const int64_t ld = dot_addend_stride(prog, op, row), n = dot_addend_stride(prog, op, false);
    PJRTX_CHECK(prog.type(add).elements() == (row ? n : ot.elements()), Code::kInternal,
                "dot_general: an addend of another size than the product's");
    vals[op.results[0]] = vals[out];
    const bool added = run_dot_general(dev, prog, op, vals, vals[add]->ptr, ld);
    vals[op.results[0]].reset();
    if (!added && n > 0)
      launch_add_rows16(dev->stream(), vals[out]->ptr, vals[add]->ptr, ot.elements() / n, n, ld, ot.dtype == DType::kF16);
    return;
  }
  vals[op.results[0]] = dev->allocate(ot.bytes());
  run_dot_general(dev, prog, op, vals, nullptr, 0);
  launch_add(dev->stream(), vals[add]->ptr, vals[op.results[0]]->ptr, vals[out]->ptr, ot.elements(), ot.dtype);
  vals[op.results[0]].reset();
}

// A group of more than 8 rows as one launch of the block tiles (the members'
// tile columns side by side fill the GPU better than each alone); false when
// they do not take some member's layout.
static bool run_gemm_group(Device* dev, const Program& prog, const std::vector<int>& ops, std::vector<MemRef>& vals) {
  const Op& first = prog.ops.at(ops.at(0));
  const TensorType& lt = prog.type(first.operands[0]);
  if (ops.size() > static_cast<size_t>(kMaxGemmMembers) || lt.rank() != 2 || lt.dims[0] <= 8 || lt.dims[1] == 0) return false;
  const void* A = vals[first.operands[0]]->ptr;
  const DType ot = prog.type(first.results[0]).dtype;
  if ((lt.dtype != DType::kBF16 && lt.dtype != DType::kF16) || (ot != lt.dtype && ot != DType::kF32)) return false;
  GemmGroup g;
  g.M = static_cast<int>(lt.dims[0]);
  g.K = static_cast<int>(lt.dims[1]);
  g.lda = lt.dims[1];
  g.count = static_cast<int>(ops.size());
  if (!aligned16(A) || lt.dims[1] % 8 != 0) return false;
  for (size_t i = 0; i < ops.size(); ++i) {
    const Op& op = prog.ops.at(ops[i]);
    const TensorType& rt = prog.type(op.operands[1]);
    const void* B = vals[op.operands[1]]->ptr;
    void* C = vals[op.results[0]]->ptr;
    if (op.operands[0] != first.operands[0] || rt.rank() != 2 || op.lhs_contract != Dims{1} || op.rhs_contract != Dims{0} ||
        rt.dtype != lt.dtype || prog.type(op.results[0]).dtype != ot || rt.dims[1] % 8 != 0 || !aligned16(B) || !aligned16(C))
      return false;
    g.m[i].B = B;
    g.m[i].C = C;
    g.m[i].N = static_cast<int>(rt.dims[1]);
    g.m[i].ldb = rt.dims[1];
  }
  if (!gemm_fits(g, true, false)) return false;
  const int64_t left = std::max<int64_t>(0, std::min<int64_t>(int64_t(64) << 20, scratch_left(dev) - 4096));
  const GemmPlan plan = plan_gemm(g, left);
  MemRef ws;
  if (plan.workspace) ws = dev->allocate(plan.workspace);
  launch_gemm(dev->stream(), g, plan, A, true, false, lt.dtype == DType::kF16, ot == DType::kF32 ? 4 : 2,
              ws ? static_cast<float*>(ws->ptr) : nullptr);
  return true;
}

// A dot group (planner: dots sharing one LHS): one gemv_wide launch when
// every member is a decode-shaped product over the same X with an
// N-contiguous weight; otherwise the members run one by one.
void run_dot_group(Device* dev, const Program& prog, const std::vector<int>& ops, std::vector<MemRef>& vals) {
  if (run_gemm_group(dev, prog, ops, vals)) return;
  GemvGroup g;
  bool ok = ops.size() >= 1 && ops.size() <= static_cast<size_t>(kMaxGemvMembers);
  const void* X = nullptr;
  DType in_t = DType::kInvalid;
  int tiles = 0;
  for (size_t i = 0; i < ops.size() && ok; ++i) {
    const Op& op = prog.ops.at(ops[i]);
    const TensorType& lt = prog.type(op.operands[0]);
    const TensorType& rt = prog.type(op.operands[1]);
    const TensorType& ot = prog.type(op.results[0]);
    ok = op.kind == OpKind::kDotGeneral && lt.rank() == 2 && rt.rank() == 2 && op.lhs_batch.empty() &&
         op.lhs_contract == Dims{1} && op.rhs_contract == Dims{0} && (lt.dtype == DType::kBF16 || lt.dtype == DType::kF16) &&
         rt.dtype == lt.dtype && (ot.dtype == lt.dtype || ot.dtype == DType::kF32);
    if (!ok) break;
    const int64_t M = lt.dims[0], K = lt.dims[1], N = rt.dims[1];
    const int out_kind = ot.dtype == DType::kBF16 ? 0 : (ot.dtype == DType::kF16 ? 1 : 2);
    const void* A = vals[op.operands[0]]->ptr;
    const void* W = vals[op.operands[1]]->ptr;
    ok = M >= 1 && M <= 4 && K % 8 == 0 && N % 8 == 0 && aligned16(A) && aligned16(W) && N < (int64_t(1) << 30) &&
         M * K <= kGemvWideMaxX;
    if (i == 0) {
      X = A;
      in_t = lt.dtype;
      g.M = static_cast<int>(M);
      g.K = static_cast<int>(K);
      g.ldx = K;
      g.out_kind = out_kind;
    } else {
      ok = ok && A == X && lt.dtype == in_t && g.M == M && g.K == K && g.out_kind == out_kind;
    }
    if (!ok) break;
    GemvMember& m = g.m[i];
    m.W = W;
    m.Y = vals[op.results[0]]->ptr;
    m.N = static_cast<int>(N);
    m.ldw = N;
    m.ldy = N;
  }
  if (ok) {
    g.count = static_cast<int>(ops.size());
    tiles = gemv_wide_tiles(g);
  }
  if (ok && gemv_wide_fits(g.M, g.K, tiles)) {
    launch_gemv_wide(dev->stream(), g, X, in_t == DType::kF16);
    return;
  }
  for (int oi : ops) run_dot_general(dev, prog, prog.ops.at(oi), vals, nullptr, 0);
}

// transpose(dot_general(a, b)) that only moves b's free dims before a's is
// dot_general(b, a) (the weight gradient as jax.vjp lowers it): the product is
// written where the transpose would put it. Same sums, same rounding.
// Decode-shaped products (8 rows or fewer on either side) keep their
// orientation, which the GEMV kernels need.
bool fold_dot_transpose(Program* prog) {
  std::map<int, size_t> producer;
  std::map<int, int> uses;
  for (size_t i = 0; i < prog->ops.size(); ++i) {
    for (int r : prog->ops[i].results) producer[r] = i;
    for (int v : prog->ops[i].operands) uses[v]++;
  }
  for (int r : prog->results) uses[r]++;
  bool changed = false;
  for (Op& t : prog->ops) {
    if (t.kind != OpKind::kTranspose) continue;
    auto it = producer.find(t.operands[0]);
    if (it == producer.end() || uses[t.operands[0]] != 1) continue;
    const Op& d = prog->ops[it->second];
    if (d.kind != OpKind::kDotGeneral || d.operands.size() != 2 || d.results.size() != 1) continue;
    const TensorType& dt = prog->type(d.results[0]);
    const int64_t nb = static_cast<int64_t>(d.lhs_batch.size());
    const int64_t nl = prog->type(d.operands[0]).rank() - nb - static_cast<int64_t>(d.lhs_contract.size());
    const int64_t nr = prog->type(d.operands[1]).rank() - nb - static_cast<int64_t>(d.rhs_contract.size());
    if (nb + nl + nr != dt.rank() || static_cast<int64_t>(t.dims.size()) != dt.rank()) continue;
    bool swaps = nl > 0 && nr > 0;
    int64_t m = 1, n = 1;
    for (int64_t i = 0; i < dt.rank() && swaps; ++i) {
      const int64_t want = i < nb ? i : i < nb + nr ? i + nl : i - nr;
      swaps = t.dims[i] == want;
      if (i >= nb) (i < nb + nl ? m : n) *= dt.dims[i];
    }
    if (!swaps || m <= 8 || n <= 8) continue;
    Op r = d;
    std::swap(r.operands[0], r.operands[1]);
    std::swap(r.lhs_batch, r.rhs_batch);
    std::swap(r.lhs_contract, r.rhs_contract);
    r.results = t.results;
    r.dot_swapped = !d.dot_swapped;
    t = std::move(r);
    changed = true;
  }
  return changed;
}

}  // namespace pjrtx
