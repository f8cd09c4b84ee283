// RMSNorm forward and backward: row passes that read each operand from HBM
// once.
//
// Fast path (at least one 16-byte pack and at most 1024*16 of them): a row is
// held in registers by TPR lanes, each owning VPT packs (contiguous per
// wave in the one-shot forward, else strided by TPR) so a wave's loads are
// contiguous. TPR = 64 is one wavefront per row (several
// rows per block, sum of squares by wave shuffles alone); TPR = NTB is the
// whole block (a wave reduction plus one LDS exchange). Rows that are not whole
// packs, or not on 16-byte boundaries, take the same kernels with accesses across
// those boundaries and a last pack that ends with the row (rmsnorm_rows.h);
// narrower or wider rows a one-block-per-row kernel that loops over the row twice.
//
// Forward launches one block per row group, the even and the odd XCDs each
// sweeping one half of the rows, except for row counts that fit in a few waves
// of resident blocks: there a persistent grid takes rows in grid stride with w
// in registers and the next row prefetched (measured faster on MI355X for such
// short launches, slower for long ones).
//
// Backward is a persistent grid (a few blocks per CU): block b takes rows
// b, b + G, b + 2G, ... (G = grid size; the blocks together sweep the tensors
// front to back, which measured 13% faster than contiguous runs of rows per
// block) with w and its running dw / dbias columns in registers, prefetching
// the next row's x and dy while the current row's dot product is reduced.
// Blocks leave one fp32 partial row each (the rows of a block's wavefront
// slots are combined through LDS first), and a column reduction sums the
// partials in a fixed order, so dw is deterministic.
//
// Types: T is x's type (and dx's); W is the weight's, which is also the type
// of the bias, of y and of dy, and of dw / dbias: W = T, or fp32 with a 16-bit
// x (torch's promotion of a 16-bit normalised row times an fp32 weight gives
// an fp32 result, unrounded).
#include <mutex>

#include "rmsnorm_rows.h"

namespace pk {
namespace {

// Any row width, any alignment: one block per row, two passes over x.
template <typename T, typename W, int MODE>
__global__ __launch_bounds__(kThreads) void rmsnorm_fwd_any(const T* __restrict__ x, const W* __restrict__ w,
                                                            const W* __restrict__ bias, const T* __restrict__ res,
                                                            T* __restrict__ s_out, float offset, W* __restrict__ y,
                                                            float* __restrict__ rstd, int64_t rows, int cols,
                                                            float eps, float inv_cols) {
  constexpr bool BIAS = MODE == kBias;
  __shared__ float red[kThreads / 64];
  const int64_t row = blockIdx.x;
  const T* xr = x + row * cols;
  float ss = 0.f;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    float f = to_f32(xr[c]);
    if constexpr (MODE == kAdd) {
      const T sv = from_f32<T>(f + to_f32(res[row * cols + c]));
      s_out[row * cols + c] = sv;  // re-read below by this same thread
      f = to_f32(sv);
    }
    ss += f * f;
  }
  ss = row_sum<kThreads, kThreads>(ss, red);
  const float r = 1.0f / sqrtf(ss * inv_cols + eps);
  if (rstd != nullptr && threadIdx.x == 0) rstd[row] = r;
  W* yr = y + row * cols;
  const T* sr = MODE == kAdd ? s_out + row * cols : xr;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    const float wv = MODE == kAdd ? to_f32(from_f32<W>(to_f32(w[c]) + offset)) : to_f32(w[c]);
    yr[c] = fwd_elem<T, W, BIAS>(to_f32(sr[c]), r, wv, BIAS ? to_f32(bias[c]) : 0.f);
  }
}

// Any row width: block b walks rows b, b + G, ..., one column per thread per
// step, one partial row per block.
template <typename T, typename W, int MODE>
__global__ __launch_bounds__(kThreads) void rmsnorm_bwd_any(const T* __restrict__ x, const W* __restrict__ w,
                                                            const float* __restrict__ rstd,
                                                            const W* __restrict__ dy, const T* __restrict__ ds,
                                                            float offset, T* __restrict__ dx,
                                                            float* __restrict__ dw_part,
                                                            float* __restrict__ db_part, int64_t rows, int cols,
                                                            float inv_cols) {
  constexpr bool BIAS = MODE == kBias;
  constexpr bool ADD = MODE == kAdd;
  const bool has_ds = ADD && ds != nullptr;
  // weight as the forward used it: w, or w + offset rounded to its type
  auto wc = [&](int c) { return ADD ? to_f32(from_f32<W>(to_f32(w[c]) + offset)) : to_f32(w[c]); };
  __shared__ float red[kThreads / 64];
  float* dwp = dw_part + (int64_t)blockIdx.x * cols;
  float* dbp = BIAS ? db_part + (int64_t)blockIdx.x * cols : nullptr;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    dwp[c] = 0.f;
    if constexpr (BIAS) dbp[c] = 0.f;
  }
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const float r = rstd[row];
    const T* xr = x + row * cols;
    const W* gr = dy + row * cols;
    float dot = 0.f;
    for (int c = threadIdx.x; c < cols; c += kThreads) dot += to_f32(gr[c]) * wc(c) * (to_f32(xr[c]) * r);
    dot = row_sum<kThreads, kThreads>(dot, red) * inv_cols;
    T* dxr = dx + row * cols;
    for (int c = threadIdx.x; c < cols; c += kThreads) {
      const float g = to_f32(gr[c]);
      const float n = to_f32(xr[c]) * r;
      float d = r * (g * wc(c) - n * dot);
      if (has_ds) d += to_f32(ds[row * cols + c]);
      dxr[c] = from_f32<T>(d);
      dwp[c] += g * n;  // column c is only ever touched by this thread
      if constexpr (BIAS) dbp[c] += g;
    }
  }
}

template <typename T, typename W, int MODE> int bwd_any_resident() {
  static const int n = resident_per_cu(rmsnorm_bwd_any<T, W, MODE>, kThreads, 0);
  return n;
}

template <typename T, typename W, int MODE> int fwd(const FwdArgs& a, const char* who) {
  const bool aligned = aligned16(a.x) && aligned16(a.w) && aligned16(a.y) && (MODE != kBias || aligned16(a.b)) &&
                       (MODE != kAdd || (aligned16(a.res) && aligned16(a.s_out)));
  const Plan p = plan_for(a.cols, sizeof(T), aligned, false);
  if (p.vec && p.aln)
    fwd_vec<T, W, MODE, true>(a, p);
  else if (p.vec)
    Ragged<T, W, MODE>::fwd(a, p);
  else
    hipLaunchKernelGGL((rmsnorm_fwd_any<T, W, MODE>), dim3(a.rows), dim3(kThreads), 0, a.s,
                       static_cast<const T*>(a.x), static_cast<const W*>(a.w), static_cast<const W*>(a.b),
                       static_cast<const T*>(a.res), static_cast<T*>(a.s_out), a.offset, static_cast<W*>(a.y),
                       a.rstd, a.rows, a.cols, a.eps, 1.0f / (float)a.cols);
  return launched(who);
}

// Persistent backward grid: every resident block slot of the device, never
// more blocks than the rows need.
template <typename T, typename W, int MODE> int64_t bwd_blocks(int64_t rows, const Plan& p) {
  const int64_t rpb = p.vec ? p.ntb / p.tpr : 1;
  const int per_cu = !p.vec  ? bwd_any_resident<T, W, MODE>()
                     : p.aln ? bwd_vec_resident<T, W, MODE, true>(p)
                             : Ragged<T, W, MODE>::resident(p);
  const int64_t want = (rows + rpb - 1) / rpb;
  const int64_t cap = (int64_t)cu_count() * per_cu;
  return want < cap ? want : cap;
}

template <typename T, typename W, int MODE> int bwd(const BwdArgs& a, const char* who) {
  const bool aligned = aligned16(a.x) && aligned16(a.w) && aligned16(a.dy) && aligned16(a.dx) &&
                       (a.ds == nullptr || aligned16(a.ds));
  const Plan p = plan_for(a.cols, sizeof(T), aligned, true);
  const int64_t blocks = bwd_blocks<T, W, MODE>(a.rows, p);
  if (p.vec && p.aln)
    bwd_vec<T, W, MODE, true>(a, p, blocks);
  else if (p.vec)
    Ragged<T, W, MODE>::bwd(a, p, blocks);
  else
    hipLaunchKernelGGL((rmsnorm_bwd_any<T, W, MODE>), dim3(blocks), dim3(kThreads), 0, a.s,
                       static_cast<const T*>(a.x), static_cast<const W*>(a.w), a.rstd, static_cast<const W*>(a.dy),
                       static_cast<const T*>(a.ds), a.offset, static_cast<T*>(a.dx), a.dw_part, a.db_part, a.rows,
                       a.cols, 1.0f / (float)a.cols);
  const ColumnSum db{a.db_part, a.db, blocks};
  column_sums<W>({a.dw_part, a.dw, blocks}, MODE == kBias ? &db : nullptr, a.cols, a.s);
  return launched(who);
}

// Workspace: [blocks, cols] dw partials and the same for dbias, each rounded up to 256 bytes.
struct Layout {
  int64_t part, total;
};

template <typename T, typename W, int MODE> Layout layout_for(int64_t rows, int64_t cols) {
  // The aligned plan and the fallback may use different grids: size for the larger.
  const int64_t b1 = bwd_blocks<T, W, MODE>(rows, plan_for(cols, sizeof(T), true, true));
  const int64_t b2 = bwd_blocks<T, W, MODE>(rows, plan_for(cols, sizeof(T), false, true));
  const int64_t blocks = b1 > b2 ? b1 : b2;
  auto up = [](int64_t n) { return (n + 255) / 256 * 256; };
  Layout l;
  l.part = up(blocks * cols * (int64_t)sizeof(float));
  l.total = l.part * (MODE == kBias ? 2 : 1);
  return l;
}

// (x dtype, weight dtype) pairs the kernels implement, in every mode: one
// dtype, or a 16-bit x (with its residual and sum, in the residual-add mode)
// with an fp32 weight.
bool supported_pair(int dtype, int wdtype, int /*mode*/) {
  if (wdtype == dtype) return known_dtype(dtype);
  return wdtype == PK_F32 && (dtype == PK_BF16 || dtype == PK_F16);
}

template <int MODE> Layout layout_of(int64_t rows, int64_t cols, int dtype, int wdtype) {
  if (wdtype != dtype) return dtype == PK_BF16 ? layout_for<bf16, float, MODE>(rows, cols)
                                               : layout_for<f16, float, MODE>(rows, cols);
  switch (dtype) {
    case PK_F32: return layout_for<float, float, MODE>(rows, cols);
    case PK_BF16: return layout_for<bf16, bf16, MODE>(rows, cols);
    default: return layout_for<f16, f16, MODE>(rows, cols);
  }
}

Layout workspace_layout(int64_t rows, int64_t cols, int dtype, int wdtype, int mode) {
  return mode == kBias ? layout_of<kBias>(rows, cols, dtype, wdtype)
                       : mode == kAdd ? layout_of<kAdd>(rows, cols, dtype, wdtype)
                                      : layout_of<kPlain>(rows, cols, dtype, wdtype);
}

// One workspace size serves every backward entry point, mode and weight dtype.
int64_t workspace_bytes(int64_t rows, int64_t cols, int dtype) {
  int64_t n = 0;
  for (int wdtype : {dtype, (int)PK_F32})
    for (int mode : {kPlain, kBias, kAdd}) {
      if (!supported_pair(dtype, wdtype, mode)) continue;
      const int64_t t = workspace_layout(rows, cols, dtype, wdtype, mode).total;
      n = t > n ? t : n;
    }
  return n;
}

template <int MODE> int fwd_dispatch(const FwdArgs& a, int dtype, int wdtype, const char* who) {
  if (wdtype != dtype) return dtype == PK_BF16 ? fwd<bf16, float, MODE>(a, who) : fwd<f16, float, MODE>(a, who);
  switch (dtype) {
    case PK_F32: return fwd<float, float, MODE>(a, who);
    case PK_BF16: return fwd<bf16, bf16, MODE>(a, who);
    default: return fwd<f16, f16, MODE>(a, who);
  }
}

template <int MODE> int bwd_dispatch(const BwdArgs& a, int dtype, int wdtype, const char* who) {
  if (wdtype != dtype) return dtype == PK_BF16 ? bwd<bf16, float, MODE>(a, who) : bwd<f16, float, MODE>(a, who);
  switch (dtype) {
    case PK_F32: return bwd<float, float, MODE>(a, who);
    case PK_BF16: return bwd<bf16, bf16, MODE>(a, who);
    default: return bwd<f16, f16, MODE>(a, who);
  }
}

// Splits the caller's workspace for a backward call of this mode.
int carve(const char* who, void* workspace, int64_t workspace_bytes, int64_t rows, int64_t cols, int dtype,
          int wdtype, int mode, BwdArgs& a) {
  const Layout l = workspace_layout(rows, cols, dtype, wdtype, mode);
  if (workspace_bytes < l.total)
    return fail(PK_ERR_INVALID, "%s: workspace of %lld bytes, need %lld", who, (long long)workspace_bytes,
                (long long)l.total);
  if (!aligned16(workspace)) return fail(PK_ERR_INVALID, "%s: workspace not 16-byte aligned", who);
  char* base = static_cast<char*>(workspace);
  a.dw_part = reinterpret_cast<float*>(base);
  a.db_part = mode == kBias ? reinterpret_cast<float*>(base + l.part) : nullptr;
  return PK_OK;
}

int check_shape(const char* who, int64_t rows, int64_t cols, int dtype, int wdtype = -1, int mode = kPlain) {
  if (rows < 0 || cols < 0) return fail(PK_ERR_INVALID, "%s: negative shape (%lld, %lld)", who, (long long)rows,
                                        (long long)cols);
  if (cols > (int64_t)1 << 30) return fail(PK_ERR_UNSUPPORTED, "%s: %lld columns", who, (long long)cols);
  if (!known_dtype(dtype)) return fail(PK_ERR_UNSUPPORTED, "%s: dtype code %d", who, dtype);
  if (!supported_pair(dtype, wdtype < 0 ? dtype : wdtype, mode))
    return fail(PK_ERR_UNSUPPORTED, "%s: x dtype code %d with weight dtype code %d (one dtype, or a 16-bit x with an "
                "fp32 weight)", who, dtype, wdtype);
  return PK_OK;
}

}  // namespace
}  // namespace pk

// ---------------------------------------------------------------------------
// Fixed scratch for pk_rmsnorm_bwd_noalloc: the dw / dbias partial rows of one
// backward call. Every GPU the library runs on holds its own copy from module
// load until the process ends. Each block writes its whole partial row, so
// nothing needs clearing between calls; two calls that overlap on one GPU (on
// different streams, or from different threads) share the array and race.
static constexpr int64_t kScratchBytes = (int64_t)96 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace pk {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
void* g_scratch_addr[kMaxDevices];  // device address of `scratch` per device, once looked up

// Device address of the current device's scratch array. The array's host-side
// name is only a stand-in for the symbol: its device address is looked up
// once per device with that device current and kept.
int scratch_address(const char* who, void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(PK_ERR_HIP, "%s: no current HIP device", who);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (g_scratch_addr[dev] == nullptr) {
    void* addr = nullptr;
    const hipError_t err = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || addr == nullptr)
      return fail(PK_ERR_HIP, "%s: hipGetSymbolAddress(scratch) on device %d failed: %s", who, dev,
                  hipGetErrorString(err));
    g_scratch_addr[dev] = addr;
  }
  *out = g_scratch_addr[dev];
  return PK_OK;
}

}  // namespace
}  // namespace pk

extern "C" {

int pk_rmsnorm_fwd(const void* x, const void* w, const void* bias, void* y, float* rstd, int64_t rows, int64_t cols,
                   float eps, int dtype, int w_dtype, void* stream) {
  using namespace pk;
  if (int st = check_shape("pk_rmsnorm_fwd", rows, cols, dtype, w_dtype)) return st;
  if (rows == 0) return PK_OK;
  if (cols == 0) return fail(PK_ERR_INVALID, "pk_rmsnorm_fwd: zero-width rows");
  if (!x || !w || !y) return fail(PK_ERR_INVALID, "pk_rmsnorm_fwd: null pointer");
  const FwdArgs a{x, w, bias, nullptr, nullptr, 0.f, y, rstd, rows, (int)cols, eps, static_cast<hipStream_t>(stream)};
  return bias != nullptr ? fwd_dispatch<kBias>(a, dtype, w_dtype, "pk_rmsnorm_fwd")
                         : fwd_dispatch<kPlain>(a, dtype, w_dtype, "pk_rmsnorm_fwd");
}

int64_t pk_rmsnorm_bwd_workspace(int64_t rows, int64_t cols, int dtype) {
  using namespace pk;
  if (rows <= 0 || cols <= 0 || !known_dtype(dtype)) return 0;
  return workspace_bytes(rows, cols, dtype);
}

int pk_rmsnorm_bwd(const void* x, const void* w, const float* rstd, const void* dy, void* dx, void* dw, void* dbias,
                   void* workspace, int64_t workspace_bytes, int64_t rows, int64_t cols, int dtype, int w_dtype,
                   void* stream) {
  using namespace pk;
  const char* who = "pk_rmsnorm_bwd";
  if (int st = check_shape(who, rows, cols, dtype, w_dtype)) return st;
  if (cols == 0) return fail(PK_ERR_INVALID, "pk_rmsnorm_bwd: zero-width rows");
  if (!x || !w || !rstd || !dy || !dx || !dw || !workspace)
    return fail(PK_ERR_INVALID, "pk_rmsnorm_bwd: null pointer");
  if (rows == 0) return fail(PK_ERR_UNSUPPORTED, "pk_rmsnorm_bwd: zero rows (dw is all zeros; fill it host-side)");
  const int mode = dbias != nullptr ? kBias : kPlain;
  BwdArgs a{x, w, dy, nullptr, 0.f, rstd, dx, dw, dbias, nullptr, nullptr, rows, (int)cols,
            static_cast<hipStream_t>(stream)};
  if (int st = carve(who, workspace, workspace_bytes, rows, cols, dtype, w_dtype, mode, a)) return st;
  return mode == kBias ? bwd_dispatch<kBias>(a, dtype, w_dtype, who) : bwd_dispatch<kPlain>(a, dtype, w_dtype, who);
}

int pk_rmsnorm_bwd_noalloc(const void* x, const void* w, const float* rstd, const void* dy, void* dx, void* dw,
                           void* dbias, int64_t rows, int64_t cols, int dtype, int w_dtype, void* stream) {
  using namespace pk;
  const char* who = "pk_rmsnorm_bwd_noalloc";
  if (int st = check_shape(who, rows, cols, dtype, w_dtype)) return st;
  if (cols == 0) return fail(PK_ERR_INVALID, "%s: zero-width rows", who);
  if (rows == 0) return fail(PK_ERR_UNSUPPORTED, "%s: zero rows (dw is all zeros; fill it host-side)", who);
  // The size limit is checked before the pointers, so a caller can probe it
  // with null pointers: a call past the limit then never reaches a launch,
  // even if this check were wrong (the null check below refuses it).
  const int mode = dbias != nullptr ? kBias : kPlain;
  const int64_t need = workspace_layout(rows, cols, dtype, w_dtype, mode).total;
  if (need > kScratchBytes)
    return fail(PK_ERR_UNSUPPORTED, "%s: shape (%lld, %lld) needs %lld bytes of scratch, the fixed array holds %lld",
                who, (long long)rows, (long long)cols, (long long)need, (long long)kScratchBytes);
  if (!x || !w || !rstd || !dy || !dx || !dw) return fail(PK_ERR_INVALID, "%s: null pointer", who);
  void* base = nullptr;
  if (int st = scratch_address(who, &base)) return st;
  BwdArgs a{x, w, dy, nullptr, 0.f, rstd, dx, dw, dbias, nullptr, nullptr, rows, (int)cols,
            static_cast<hipStream_t>(stream)};
  if (int st = carve(who, base, kScratchBytes, rows, cols, dtype, w_dtype, mode, a)) return st;
  return mode == kBias ? bwd_dispatch<kBias>(a, dtype, w_dtype, who) : bwd_dispatch<kPlain>(a, dtype, w_dtype, who);
}

int pk_add_rmsnorm_fwd(const void* x, const void* residual, const void* w, void* y, void* s, float* rstd,
                       int64_t rows, int64_t cols, float eps, float offset, int dtype, int w_dtype, void* stream) {
  using namespace pk;
  const char* who = "pk_add_rmsnorm_fwd";
  if (int st = check_shape(who, rows, cols, dtype, w_dtype, kAdd)) return st;
  if (rows == 0) return PK_OK;
  if (cols == 0) return fail(PK_ERR_INVALID, "pk_add_rmsnorm_fwd: zero-width rows");
  if (!x || !residual || !w || !y || !s) return fail(PK_ERR_INVALID, "pk_add_rmsnorm_fwd: null pointer");
  if (!isfinite(offset)) return fail(PK_ERR_INVALID, "pk_add_rmsnorm_fwd: offset is not finite");
  const FwdArgs a{x, w, nullptr, residual, s, offset, y, rstd, rows, (int)cols, eps, static_cast<hipStream_t>(stream)};
  return fwd_dispatch<kAdd>(a, dtype, w_dtype, who);
}

int pk_add_rmsnorm_bwd(const void* s, const void* w, const float* rstd, const void* dy, const void* ds, void* dx,
                       void* dw, void* workspace, int64_t workspace_bytes, int64_t rows, int64_t cols, float offset,
                       int dtype, int w_dtype, void* stream) {
  using namespace pk;
  const char* who = "pk_add_rmsnorm_bwd";
  if (int st = check_shape(who, rows, cols, dtype, w_dtype, kAdd)) return st;
  if (cols == 0) return fail(PK_ERR_INVALID, "pk_add_rmsnorm_bwd: zero-width rows");
  if (!s || !w || !rstd || !dy || !dx || !dw || !workspace)
    return fail(PK_ERR_INVALID, "pk_add_rmsnorm_bwd: null pointer");
  if (rows == 0) return fail(PK_ERR_UNSUPPORTED, "pk_add_rmsnorm_bwd: zero rows (dw is all zeros; fill it host-side)");
  if (!isfinite(offset)) return fail(PK_ERR_INVALID, "pk_add_rmsnorm_bwd: offset is not finite");
  BwdArgs a{s, w, dy, ds, offset, rstd, dx, dw, nullptr, nullptr, nullptr, rows, (int)cols,
            static_cast<hipStream_t>(stream)};
  if (int st = carve(who, workspace, workspace_bytes, rows, cols, dtype, w_dtype, kAdd, a)) return st;
  return bwd_dispatch<kAdd>(a, dtype, w_dtype, who);
}

}  // extern "C"
