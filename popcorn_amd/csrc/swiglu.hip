// SwiGLU forward / backward: one HBM stream over rows x cols elements.
//
// Each thread moves one 16-byte vector of every operand, loads issued before
// any arithmetic; data is touched once, so loads and stores are
// non-temporal. Small blocks with one vector per thread measured fastest on
// MI355X (forward 64 threads: 0.84 of the 8 TB/s spec at a, b [16384, 14336];
// backward 128 threads), ahead of larger blocks or several vectors per
// thread.
//
// a and b may be rows of a wider tensor (the halves of one gate/up projection):
// each has a row stride, everything else is contiguous. Contiguous operands are
// one row of all the elements, whose ragged end its last thread takes element
// by element. In strided rows the last vector is the one that ends with the
// row: where the width is ragged it overlaps the vector before it and writes
// the same values there. Rows shorter than a vector take the scalar kernels.
#include "api.h"
#include "common.h"

namespace pk {
namespace {

constexpr int kThreads = 256;   // scalar kernels
constexpr int kFwdThreads = 64;  // vector kernels: threads per block
constexpr int kBwdThreads = 128;

// sigmoid(a) in fp32 from the hardware exp2 and reciprocal (each ~1 ulp): the
// stream is HBM-bound only while the per-element VALU work stays this short.
__device__ __forceinline__ float sigmoid_f32(float a) { return __builtin_amdgcn_rcpf(1.0f + __expf(-a)); }

// silu(a) = a * sigmoid(a), torch's a / (1 + exp(-a)) to within ~2 fp32 ulp.
__device__ __forceinline__ float silu_f32(float a) { return a * sigmoid_f32(a); }

// Forward element: torch eager rounds silu's result to T, then the product.
template <typename T> __device__ __forceinline__ T fwd_elem(T a, T b) {
  const float s = round_to<T>(silu_f32(to_f32(a)));
  return from_f32<T>(s * to_f32(b));
}

template <typename T> __device__ __forceinline__ void bwd_elem(T g, T a, T b, T& da, T& db) {
  const float af = to_f32(a), bf = to_f32(b), gf = to_f32(g);
  const float s = sigmoid_f32(af);
  da = from_f32<T>(gf * bf * s * (1.0f + af * (1.0f - s)));
  db = from_f32<T>(gf * af * s);
}

// A thread's vector of rows x cols elements: row r, starting at column c.
struct Rows {
  int64_t cols;
  int64_t as, bs;       // row strides of a and b, elements
  uint32_t nvec;        // vectors per row, the last one ending with the row
  uint32_t mul, pre, shift;  // i / nvec = (((i - h) >> pre) + h) >> shift with h = mulhi(i, mul), for any 32-bit i
};

__device__ __forceinline__ void locate(const Rows& g, uint32_t i, int vec, int64_t& r, int64_t& c) {
  const uint32_t h = __umulhi(i, g.mul);
  const uint32_t q = (((i - h) >> g.pre) + h) >> g.shift;
  r = q;
  c = (int64_t)(i - q * g.nvec) * vec;
  c = c + vec <= g.cols ? c : g.cols - vec;
}

template <typename T, bool ROWS, bool ALIGNED>
__global__ __launch_bounds__(kFwdThreads) void swiglu_fwd_vec(const T* __restrict__ a, const T* __restrict__ b,
                                                              T* __restrict__ y, int64_t nvec, Rows g) {
  constexpr int P = Vec<T>::N;
  const int64_t i = (int64_t)blockIdx.x * kFwdThreads + threadIdx.x;
  if (i >= nvec) return;
  int64_t ao, bo, yo;
  if constexpr (ROWS) {
    int64_t r, c;
    locate(g, (uint32_t)i, P, r, c);
    ao = r * g.as + c;
    bo = r * g.bs + c;
    yo = r * g.cols + c;
  } else {
    ao = bo = yo = i * P;
    if (ao + P > g.cols) {  // the ragged end: the last thread's alone
      for (; ao < g.cols; ++ao) y[ao] = fwd_elem(a[ao], b[ao]);
      return;
    }
  }
  const Vec<T> va = ld16_stream_at<ALIGNED>(a + ao), vb = ld16_stream_at<ALIGNED>(b + bo);
  Vec<T> vy;
#pragma unroll
  for (int j = 0; j < P; ++j) vy.v[j] = fwd_elem(va.v[j], vb.v[j]);
  st16_stream_at<ALIGNED>(y + yo, vy);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void swiglu_fwd_scalar(const T* __restrict__ a, const T* __restrict__ b,
                                                              T* __restrict__ y, int64_t n, Rows g) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
    const int64_t r = i / g.cols, c = i - r * g.cols;
    y[i] = fwd_elem(a[r * g.as + c], b[r * g.bs + c]);
  }
}

template <typename T, bool ROWS, bool ALIGNED>
__global__ __launch_bounds__(kBwdThreads) void swiglu_bwd_vec(const T* __restrict__ dy, const T* __restrict__ a,
                                                              const T* __restrict__ b, T* __restrict__ da,
                                                              T* __restrict__ db, int64_t nvec, Rows g) {
  constexpr int P = Vec<T>::N;
  const int64_t i = (int64_t)blockIdx.x * kBwdThreads + threadIdx.x;
  if (i >= nvec) return;
  int64_t ao, bo, yo;
  if constexpr (ROWS) {
    int64_t r, c;
    locate(g, (uint32_t)i, P, r, c);
    ao = r * g.as + c;
    bo = r * g.bs + c;
    yo = r * g.cols + c;
  } else {
    ao = bo = yo = i * P;
    if (ao + P > g.cols) {  // the ragged end: the last thread's alone
      for (; ao < g.cols; ++ao) bwd_elem(dy[ao], a[ao], b[ao], da[ao], db[ao]);
      return;
    }
  }
  const Vec<T> vg = ld16_stream_at<ALIGNED>(dy + yo);
  const Vec<T> va = ld16_stream_at<ALIGNED>(a + ao), vb = ld16_stream_at<ALIGNED>(b + bo);
  Vec<T> vda, vdb;
#pragma unroll
  for (int j = 0; j < P; ++j) bwd_elem(vg.v[j], va.v[j], vb.v[j], vda.v[j], vdb.v[j]);
  st16_stream_at<ALIGNED>(da + yo, vda);
  st16_stream_at<ALIGNED>(db + yo, vdb);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void swiglu_bwd_scalar(const T* __restrict__ dy, const T* __restrict__ a,
                                                              const T* __restrict__ b, T* __restrict__ da,
                                                              T* __restrict__ db, int64_t n, Rows g) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
    const int64_t r = i / g.cols, c = i - r * g.cols;
    bwd_elem(dy[i], a[r * g.as + c], b[r * g.bs + c], da[i], db[i]);
  }
}

int64_t blocks_for(int64_t work, int64_t per_block) { return (work + per_block - 1) / per_block; }

// The tensors of a call: dy, da, db and y are contiguous [rows, cols].
struct Call {
  const void *dy, *a, *b;
  void *y, *da, *db;
};

// Rows of the layout for the vector kernels: the multiplier of the exact 32-bit
// division by nvec (Granlund and Montgomery's round-up method).
template <int P> Rows rows_of(int64_t cols, int64_t as, int64_t bs) {
  Rows g{cols, as, bs, (uint32_t)((cols + P - 1) / P), 0, 0, 0};
  int l = 0;
  while (l < 32 && ((uint64_t)1 << l) < g.nvec) ++l;  // ceil(log2(nvec))
  g.mul = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - g.nvec)) / g.nvec + 1);
  g.pre = l > 0 ? 1 : 0;
  g.shift = l > 0 ? l - 1 : 0;
  return g;
}

// Launches one slab of rows. Vectors are aligned when every row of every tensor
// starts on 16 bytes and strided rows are whole vectors. Elsewhere they are
// loaded and stored across 16-byte boundaries (bf16 forward, us: contiguous
// [8192, 14336] 103.6, halves of one tensor 105.7 where copying the halves first
// took 277; one operand 2 bytes off 108.9, by element it took the scalar
// kernel; halves of an odd width, [8192, 14335], 128.3).
template <typename T, bool BWD>
void launch_slab(const Call& t, int64_t rows, int64_t cols, int64_t as, int64_t bs, hipStream_t s) {
  constexpr int P = Vec<T>::N;
  constexpr int NTB = BWD ? kBwdThreads : kFwdThreads;
  const T *dy = static_cast<const T*>(t.dy), *a = static_cast<const T*>(t.a), *b = static_cast<const T*>(t.b);
  T *y = static_cast<T*>(t.y), *da = static_cast<T*>(t.da), *db = static_cast<T*>(t.db);
  if (cols < P && rows > 1) {
    const Rows g{cols, as, bs, 0, 0, 0, 0};
    const int64_t n = rows * cols, grid = blocks_for(n, kThreads) < 1024 ? blocks_for(n, kThreads) : 1024;
    if constexpr (BWD)
      hipLaunchKernelGGL(swiglu_bwd_scalar<T>, dim3(grid), dim3(kThreads), 0, s, dy, a, b, da, db, n, g);
    else
      hipLaunchKernelGGL(swiglu_fwd_scalar<T>, dim3(grid), dim3(kThreads), 0, s, a, b, y, n, g);
    return;
  }
  const Rows g = rows_of<P>(cols, as, bs);
  const int64_t per_row = (cols + P - 1) / P, nvec = rows * per_row;
  bool aligned = aligned16(a) && aligned16(b);
  if (rows > 1) aligned = aligned && cols % P == 0 && as % P == 0 && bs % P == 0;
  aligned = aligned && (BWD ? aligned16(dy) && aligned16(da) && aligned16(db) : aligned16(y));
  const dim3 grid((unsigned)blocks_for(nvec, NTB)), block(NTB);
#define PK_SWIGLU(ROWS, ALIGNED)                                                                               \
  if constexpr (BWD)                                                                                           \
    hipLaunchKernelGGL((swiglu_bwd_vec<T, ROWS, ALIGNED>), grid, block, 0, s, dy, a, b, da, db, nvec, g);      \
  else                                                                                                         \
    hipLaunchKernelGGL((swiglu_fwd_vec<T, ROWS, ALIGNED>), grid, block, 0, s, a, b, y, nvec, g);
  if (rows == 1) {
    if (aligned) { PK_SWIGLU(false, true) } else { PK_SWIGLU(false, false) }
  } else {
    if (aligned) { PK_SWIGLU(true, true) } else { PK_SWIGLU(true, false) }
  }
#undef PK_SWIGLU
}

template <typename T, bool BWD>
int run(const char* who, Call t, int64_t rows, int64_t cols, int64_t as, int64_t bs, hipStream_t s) {
  if (rows > 1 && as == cols && bs == cols) {  // contiguous: one row
    cols *= rows;
    rows = 1;
  }
  // slabs of rows whose vectors have 32-bit indexes (one row has 64-bit ones)
  const int64_t per_row = (cols + Vec<T>::N - 1) / Vec<T>::N;
  int64_t most = INT32_MAX / per_row;
  most = rows == 1 || most < 1 ? 1 : most;
  const auto at = [](const void* p, int64_t n) { return const_cast<void*>(static_cast<const void*>(static_cast<const T*>(p) + n)); };
  for (int64_t r = 0; r < rows; r += most) {
    const int64_t n = rows - r < most ? rows - r : most;
    const Call c = BWD ? Call{at(t.dy, r * cols), at(t.a, r * as), at(t.b, r * bs), nullptr, at(t.da, r * cols), at(t.db, r * cols)}
                       : Call{nullptr, at(t.a, r * as), at(t.b, r * bs), at(t.y, r * cols), nullptr, nullptr};
    launch_slab<T, BWD>(c, n, cols, as, bs, s);
  }
  return launched(who);
}

template <bool BWD>
int dispatch(const char* who, const Call& t, int64_t rows, int64_t cols, int64_t as, int64_t bs, int dtype, void* stream) {
  if (rows < 0 || cols < 0)
    return fail(PK_ERR_INVALID, "%s: negative size (%lld, %lld)", who, (long long)rows, (long long)cols);
  if (rows == 0 || cols == 0) return PK_OK;
  if (!t.a || !t.b || (BWD ? !t.dy || !t.da || !t.db : !t.y)) return fail(PK_ERR_INVALID, "%s: null pointer", who);
  if (as < 0 || bs < 0) return fail(PK_ERR_INVALID, "%s: negative row stride", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case PK_F32: return run<float, BWD>(who, t, rows, cols, as, bs, s);
    case PK_BF16: return run<bf16, BWD>(who, t, rows, cols, as, bs, s);
    case PK_F16: return run<f16, BWD>(who, t, rows, cols, as, bs, s);
  }
  return fail(PK_ERR_UNSUPPORTED, "%s: dtype code %d", who, dtype);
}

}  // namespace
}  // namespace pk

extern "C" {

int pk_swiglu_fwd(const void* a, const void* b, void* y, int64_t n, int dtype, void* stream) {
  return pk::dispatch<false>("pk_swiglu_fwd", {nullptr, a, b, y, nullptr, nullptr}, 1, n, 0, 0, dtype, stream);
}

int pk_swiglu_bwd(const void* dy, const void* a, const void* b, void* da, void* db, int64_t n, int dtype,
                  void* stream) {
  return pk::dispatch<true>("pk_swiglu_bwd", {dy, a, b, nullptr, da, db}, 1, n, 0, 0, dtype, stream);
}

int pk_swiglu_rows_fwd(const void* a, const void* b, void* y, int64_t rows, int64_t cols, int64_t a_stride,
                       int64_t b_stride, int dtype, void* stream) {
  return pk::dispatch<false>("pk_swiglu_rows_fwd", {nullptr, a, b, y, nullptr, nullptr}, rows, cols, a_stride, b_stride,
                             dtype, stream);
}

int pk_swiglu_rows_bwd(const void* dy, const void* a, const void* b, void* da, void* db, int64_t rows, int64_t cols,
                       int64_t a_stride, int64_t b_stride, int dtype, void* stream) {
  return pk::dispatch<true>("pk_swiglu_rows_bwd", {dy, a, b, nullptr, da, db}, rows, cols, a_stride, b_stride, dtype,
                            stream);
}

}  // extern "C"
