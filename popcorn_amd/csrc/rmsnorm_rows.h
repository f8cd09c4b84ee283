// The row kernels of RMSNorm and their launches (see rmsnorm.hip), for rows of
// whole, aligned 16-byte packs and for any others of at least one pack.
#pragma once

#include <math.h>

#include "api.h"
#include "colsum.h"
#include "common.h"

namespace pk {

struct Plan {
  bool vec;  // fast path usable
  bool aln;  // every row of every operand is whole, aligned packs
  int ntb;   // threads per block
  int tpr;   // threads per row: 64 or ntb
  int vpt;   // 16-byte packs per thread: 1, 2, 4, 8, 16
};

struct FwdArgs {
  const void *x, *w, *b, *res;
  void* s_out;
  float offset;
  void* y;
  float* rstd;
  int64_t rows;
  int cols;
  float eps;
  hipStream_t s;
};

struct BwdArgs {
  const void *x, *w, *dy, *ds;
  float offset;
  const float* rstd;
  void *dx, *dw, *db;
  float *dw_part, *db_part;
  int64_t rows;
  int cols;
  hipStream_t s;
};

namespace {

constexpr int kThreads = 256;    // fallback kernels and column sums
constexpr int kMaxVpt = 16;

// Sum over the TPR lanes that share a row: TPR = 64 is one wave; TPR = NTB is
// the block, `red` holds one slot per wave and the call is a block barrier.
template <int NTB, int TPR> __device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (TPR == 64) {
    return v;
  } else {
    static_assert(TPR == NTB, "rows span one wave or the whole block");
    constexpr int W = NTB / 64;
    const int wave = threadIdx.x / 64;
    __syncthreads();  // previous readers of `red` are done
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < W; ++i) t += red[i];
    return t;
  }
}

// Pack (16-byte vector) of a row held by slot k of `lane` in the one-shot
// forward. A row of one wave interleaves its packs over the lanes; a row
// spanning the block gives wave w the contiguous packs [w*64*VPT,
// (w+1)*64*VPT), each load of a wave then covering 1 KB in order. With the
// XCD split below, 1.5% faster at 65536 x 8192 bf16 than packs interleaved
// over the whole block; the persistent grid kernel keeps the interleaved
// order, which measured 4% faster there (4096 x 4096 fp32).
template <int NTB, int TPR, int VPT> __device__ __forceinline__ int fwd_pack(int lane, int k) {
  if constexpr (TPR == NTB && NTB > 64) return (lane / 64) * (64 * VPT) + k * 64 + lane % 64;
  else return lane + k * TPR;
}

// Row group of block b in a one-shot launch over `units` groups. Dispatch
// places block b on XCD b % 8; the four even XCDs sweep the first 4*qe groups
// and the four odd XCDs the rest, each front to back (qe = ceil(units / 8),
// grid 8*qe). Returns -1 for the few blocks past the end.
__device__ __forceinline__ int64_t xcd_split_unit(int64_t b, int64_t units) {
  const int64_t qe = (units + 7) / 8;
  const int64_t x = b & 7, local = b >> 3;
  const int64_t u = (x & 1) ? 4 * qe + local * 4 + (x >> 1) : local * 4 + (x >> 1);
  return u < units ? u : -1;
}
inline int64_t xcd_split_grid(int64_t units) { return 8 * ((units + 7) / 8); }

// Where pack v of a row starts, and which of its elements are its own. Rows of
// whole, aligned packs (ALN) are cut every P elements. Any other row of at least
// P elements has its last pack end with the row: the pack's first `skip`
// elements then belong to the pack before it as well, which alone counts them
// in sums; what both of them store there is the same.
template <bool ALN, int P> struct PackAt {
  int start, skip;
  __device__ __forceinline__ PackAt(int v, int nvec, int cols)
      : start(ALN || v < nvec - 1 ? v * P : cols - P), skip(ALN || v < nvec - 1 ? 0 : nvec * P - cols) {}
  __device__ __forceinline__ bool own(int j) const { return ALN || j >= skip; }
};
template <bool ALN, int P> __device__ __forceinline__ int packs_of(int cols) { return ALN ? cols / P : (cols + P - 1) / P; }

// torch: rms = (h * rsqrt(mean(h^2) + eps)).to(T); y = rms * w; y = y + bias.
// Kernel modes: the plain norm, the norm plus bias, and the residual-add form
// (s = x + residual is formed, written out and normalised, with weight + offset).
constexpr int kPlain = 0, kBias = 1, kAdd = 2;

// s = round(x + residual): the sum torch forms at T before normalising it
template <typename T> __device__ __forceinline__ void add_residual(Vec<T>& xv, const Vec<T>& rv) {
#pragma unroll
  for (int j = 0; j < Vec<T>::N; ++j) xv.v[j] = from_f32<T>(to_f32(xv.v[j]) + to_f32(rv.v[j]));
}
// w + offset, rounded to the weight's type like the reference's `weight + offset`
template <typename W, int N> __device__ __forceinline__ Lane<W, N> offset_weight(Lane<W, N> wv, float offset) {
#pragma unroll
  for (int j = 0; j < N; ++j) wv.v[j] = from_f32<W>(to_f32(wv.v[j]) + offset);
  return wv;
}

// torch: n = (h * r).to(T); y = n * w (at W); y = y + bias. With W = T every
// op rounds to T; with W = fp32 only n is rounded.
template <typename T, typename W, bool BIAS> __device__ __forceinline__ W fwd_elem(float xv, float r, float wv, float bv) {
  float y = round_to<T>(xv * r) * wv;
  if constexpr (BIAS) y = round_to<W>(y) + bv;
  return from_f32<W>(y);
}

// One row per TPR lanes, RPB = NTB / TPR rows per block. s_out may be x or res:
// a pack of its own (ALN) is stored once it is loaded, but packs that overlap
// only after the row's reduction, when every lane has the elements it reads.
template <typename T, typename W, int NTB, int TPR, int VPT, int MODE, bool ALN>
__global__ __launch_bounds__(NTB) void rmsnorm_fwd_vec(const T* __restrict__ x, const W* __restrict__ w,
                                                       const W* __restrict__ bias, const T* __restrict__ res,
                                                       T* __restrict__ s_out, float offset, W* __restrict__ y,
                                                       float* __restrict__ rstd, int64_t rows, int cols, float eps,
                                                       float inv_cols) {
  constexpr bool BIAS = MODE == kBias;
  constexpr int P = Vec<T>::N;
  constexpr int RPB = NTB / TPR;
  __shared__ float red[NTB / 64];
  const int lane = threadIdx.x % TPR;
  const int64_t group = xcd_split_unit(blockIdx.x, (rows + RPB - 1) / RPB);
  if (group < 0) return;  // whole block, before any barrier
  const int64_t row = group * RPB + threadIdx.x / TPR;
  const bool live = row < rows;
  const int nvec = packs_of<ALN, P>(cols);
  const T* xr = x + row * cols;

  Vec<T> xv[VPT];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int v = fwd_pack<NTB, TPR, VPT>(lane, k);
    if (live && v < nvec) {
      const PackAt<ALN, P> at(v, nvec, cols);
      xv[k] = ld16_stream_at<ALN>(xr + at.start);
      if constexpr (MODE == kAdd) {
        add_residual(xv[k], ld16_stream_at<ALN>(res + row * cols + at.start));
        if constexpr (ALN) st16_stream_at<ALN>(s_out + row * cols + at.start, xv[k]);
      }
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const float f = at.own(j) ? to_f32(xv[k].v[j]) : 0.f;
        ss += f * f;
      }
    }
  }
  ss = row_sum<NTB, TPR>(ss, red);
  if (!live) return;
  const float r = 1.0f / sqrtf(ss * inv_cols + eps);
  if (rstd != nullptr && lane == 0) rstd[row] = r;

  W* yr = y + row * cols;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int v = fwd_pack<NTB, TPR, VPT>(lane, k);
    if (v < nvec) {
      const PackAt<ALN, P> at(v, nvec, cols);
      if constexpr (MODE == kAdd && !ALN) {
        u32x4 bits = *reinterpret_cast<const u32x4*>(&xv[k]);
        asm volatile("" : "+v"(bits) : "v"(r));  // not before r, for the compiler either
        *reinterpret_cast<u32x4*>(&xv[k]) = bits;
        st16_stream_at<ALN>(s_out + row * cols + at.start, xv[k]);
      }
      Lane<W, P> wv = ld_lane_at<ALN, W, P>(w + at.start);
      if constexpr (MODE == kAdd) wv = offset_weight(wv, offset);
      Lane<W, P> bv;
      if constexpr (BIAS) bv = ld_lane_at<ALN, W, P>(bias + at.start);
      Lane<W, P> out;
#pragma unroll
      for (int j = 0; j < P; ++j)
        out.v[j] = fwd_elem<T, W, BIAS>(to_f32(xv[k].v[j]), r, to_f32(wv.v[j]), BIAS ? to_f32(bv.v[j]) : 0.f);
      st_lane_stream_at<ALN>(yr + at.start, out);
    }
  }
}

// Persistent form of rmsnorm_fwd_vec for short launches: slot s of block b
// takes rows b * RPB + s + k * stride, with w (and bias) in registers and the
// next row's x in flight while the current row is reduced.
template <typename T, typename W, int NTB, int TPR, int VPT, int MODE>
__global__ __launch_bounds__(NTB) void rmsnorm_fwd_grid(const T* __restrict__ x, const W* __restrict__ w,
                                                        const W* __restrict__ bias, const T* __restrict__ res,
                                                        T* __restrict__ s_out, float offset, W* __restrict__ y,
                                                        float* __restrict__ rstd, int64_t rows, int cols, float eps,
                                                        float inv_cols) {
  constexpr bool BIAS = MODE == kBias;
  constexpr int P = Vec<T>::N;
  constexpr int RPB = NTB / TPR;
  __shared__ float red[NTB / 64];
  const int lane = threadIdx.x % TPR;
  const int nvec = cols / P;
  const int64_t stride = (int64_t)gridDim.x * RPB;
  const int64_t first = (int64_t)blockIdx.x * RPB;
  const int64_t row0 = first + threadIdx.x / TPR;
  const int64_t trips = (rows - first + stride - 1) / stride;  // the same for every slot: barriers line up
  Lane<W, P> wv[VPT], bv[VPT];
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int v = lane + k * TPR;
    if (v < nvec) {
      wv[k] = ld_lane<W, P>(w + v * P);
      if constexpr (MODE == kAdd) wv[k] = offset_weight(wv[k], offset);
      if constexpr (BIAS) bv[k] = ld_lane<W, P>(bias + v * P);
    }
  }
  Vec<T> xv[VPT], xn[VPT];
  Vec<T> rv[MODE == kAdd ? VPT : 1], rn[MODE == kAdd ? VPT : 1];
  auto fetch = [&](int64_t row, Vec<T>* xo, Vec<T>* ro) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int v = lane + k * TPR;
      if (row < rows && v < nvec) {
        xo[k] = ld16_stream(x + row * cols + v * P);
        if constexpr (MODE == kAdd) ro[k] = ld16_stream(res + row * cols + v * P);
      }
    }
  };
  fetch(row0, xv, rv);
  for (int64_t t = 0; t < trips; ++t) {
    const int64_t row = row0 + t * stride;
    fetch(row + stride, xn, rn);
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int v = lane + k * TPR;
      if (row < rows && v < nvec) {
        if constexpr (MODE == kAdd) {
          add_residual(xv[k], rv[k]);
          st16_stream(s_out + row * cols + v * P, xv[k]);
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
          const float f = to_f32(xv[k].v[j]);
          ss += f * f;
        }
      }
    }
    ss = row_sum<NTB, TPR>(ss, red);
    if (row < rows) {
      const float r = 1.0f / sqrtf(ss * inv_cols + eps);
      if (rstd != nullptr && lane == 0) rstd[row] = r;
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int v = lane + k * TPR;
        if (v < nvec) {
          Lane<W, P> out;
#pragma unroll
          for (int j = 0; j < P; ++j)
            out.v[j] = fwd_elem<T, W, BIAS>(to_f32(xv[k].v[j]), r, to_f32(wv[k].v[j]), BIAS ? to_f32(bv[k].v[j]) : 0.f);
          st_lane_stream(y + row * cols + v * P, out);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      xv[k] = xn[k];
      if constexpr (MODE == kAdd) rv[k] = rn[k];
    }
  }
}

// ---------------------------------------------------------------------------
// backward

// Adds this lane's VPT*P column values into the block's partial row in LDS
// (slot by slot, so the order is fixed) and lets slot 0 write it out.
template <int NTB, int TPR, int VPT, int P, bool ALN>
__device__ __forceinline__ void flush_partial(float (&acc)[VPT][P], float* lds_row, float* __restrict__ dst,
                                              int nvec, int cols) {
  constexpr int RPB = NTB / TPR;
  const int lane = threadIdx.x % TPR;
  const int slot = threadIdx.x / TPR;
  if constexpr (RPB > 1) {
    for (int s = RPB - 1; s >= 1; --s) {
      if (slot == s) {
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
          const int v = lane + k * TPR;
          if (v < nvec) {
            const PackAt<ALN, P> at(v, nvec, cols);
#pragma unroll
            for (int j = 0; j < P; ++j)
              if (at.own(j)) lds_row[at.start + j] = (s == RPB - 1 ? 0.f : lds_row[at.start + j]) + acc[k][j];
          }
        }
      }
      __syncthreads();
    }
  }
  if (slot == 0) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int v = lane + k * TPR;
      if (v < nvec) {
        const PackAt<ALN, P> at(v, nvec, cols);
#pragma unroll
        for (int j = 0; j < P; j += 4) {
          Lane<float, 4> o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o.v[i] = acc[k][j + i] + (RPB > 1 && at.own(j + i) ? lds_row[at.start + j + i] : 0.f);
          if (ALN || at.skip <= j) {
            st_lane_at<ALN>(dst + at.start + j, o);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (at.own(j + i)) dst[at.start + j + i] = o.v[i];
          }
        }
      }
    }
  }
}

// MODE kAdd: x is the residual sum s, w is used as w + offset, and ds (the
// gradient reaching s from its second use, may be NULL) is added to dx.
template <typename T, typename W, int NTB, int TPR, int VPT, int MODE, bool ALN>
__global__ __launch_bounds__(NTB) void rmsnorm_bwd_vec(const T* __restrict__ x, const W* __restrict__ w,
                                                       const float* __restrict__ rstd, const W* __restrict__ dy,
                                                       const T* __restrict__ ds, float offset, T* __restrict__ dx,
                                                       float* __restrict__ dw_part, float* __restrict__ db_part,
                                                       int64_t rows, int cols, float inv_cols) {
  constexpr bool BIAS = MODE == kBias;
  constexpr bool ADD = MODE == kAdd;
  const bool has_ds = ADD && ds != nullptr;
  constexpr int P = Vec<T>::N;
  constexpr int RPB = NTB / TPR;
  __shared__ float red[NTB / 64];
  extern __shared__ float lds_row[];  // cols floats when RPB > 1
  const int lane = threadIdx.x % TPR;
  const int slot = threadIdx.x / TPR;
  const int nvec = packs_of<ALN, P>(cols);

  float wf[VPT][P], dwa[VPT][P], dba[VPT][P];
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int v = lane + k * TPR;
    Lane<W, P> wv;
    if (v < nvec) wv = ld_lane_at<ALN, W, P>(w + PackAt<ALN, P>(v, nvec, cols).start);
    if constexpr (ADD) wv = offset_weight(wv, offset);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      wf[k][j] = v < nvec ? to_f32(wv.v[j]) : 0.f;
      dwa[k][j] = 0.f;
      dba[k][j] = 0.f;
    }
  }

  // Slot s of block b takes rows b * RPB + s + k * stride; every slot runs
  // the same trip count so block-wide barriers line up.
  const int64_t stride = (int64_t)gridDim.x * RPB;
  const int64_t row0 = (int64_t)blockIdx.x * RPB;
  const int64_t trips = (rows - row0 + stride - 1) / stride;

  Vec<T> xv[VPT], xn[VPT];
  Lane<W, P> gv[VPT], gn[VPT];
  Vec<T> sv[ADD ? VPT : 1], sn[ADD ? VPT : 1];
  auto fetch = [&](int64_t row, Vec<T>* xo, Lane<W, P>* go, Vec<T>* so) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int v = lane + k * TPR;
      if (row < rows && v < nvec) {
        const int64_t at = row * cols + PackAt<ALN, P>(v, nvec, cols).start;
        xo[k] = ld16_stream_at<ALN>(x + at);
        go[k] = ld_lane_stream_at<ALN, W, P>(dy + at);
        if (has_ds) so[k] = ld16_stream_at<ALN>(ds + at);
      }
    }
  };
  fetch(row0 + slot, xv, gv, sv);

  for (int64_t t = 0; t < trips; ++t) {
    const int64_t row = row0 + slot + t * stride;
    const bool live = row < rows;
    fetch(row + stride, xn, gn, sn);  // next row of this slot, in flight during the reduction
    const float r = live ? rstd[row] : 0.f;
    float dot = 0.f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int v = lane + k * TPR;
      if (live && v < nvec) {
        const PackAt<ALN, P> at(v, nvec, cols);
#pragma unroll
        for (int j = 0; j < P; ++j) {
          const float t = to_f32(gv[k].v[j]) * wf[k][j] * (to_f32(xv[k].v[j]) * r);
          dot += at.own(j) ? t : 0.f;
        }
      }
    }
    dot = row_sum<NTB, TPR>(dot, red) * inv_cols;
    if (live) {
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int v = lane + k * TPR;
        if (v < nvec) {
          Vec<T> out;
#pragma unroll
          for (int j = 0; j < P; ++j) {
            const float g = to_f32(gv[k].v[j]);
            const float n = to_f32(xv[k].v[j]) * r;
            float d = r * (g * wf[k][j] - n * dot);
            if constexpr (ADD) d += has_ds ? to_f32(sv[k].v[j]) : 0.f;
            out.v[j] = from_f32<T>(d);
            dwa[k][j] += g * n;
            if constexpr (BIAS) dba[k][j] += g;
          }
          st16_stream_at<ALN>(dx + row * cols + PackAt<ALN, P>(v, nvec, cols).start, out);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      xv[k] = xn[k];
      gv[k] = gn[k];
      if constexpr (ADD) sv[k] = sn[k];
    }
  }

  flush_partial<NTB, TPR, VPT, P, ALN>(dwa, lds_row, dw_part + (int64_t)blockIdx.x * cols, nvec, cols);
  if constexpr (BIAS) {
    if constexpr (RPB > 1) __syncthreads();  // lds_row is reused
    flush_partial<NTB, TPR, VPT, P, ALN>(dba, lds_row, db_part + (int64_t)blockIdx.x * cols, nvec, cols);
  }
}

// ---------------------------------------------------------------------------
// launch planning


inline int pow2_at_least(int64_t n) {
  int p = 1;
  while (p < n) p *= 2;
  return p;
}

// Launch shape for rows of `cols` elements of `esize` bytes: one row per
// wavefront up to 4 packs per lane, wider rows over a block at 4 packs per
// thread (forward) or 2 (backward, which also keeps dw columns in
// registers). Measured on MI355X these beat one-wave rows of 16 packs and
// blocks of 128 / 512 / 1024 threads for 4096-wide fp32 and 8192-wide bf16
// rows.
inline Plan plan_for(int64_t cols, int esize, bool aligned, bool backward) {
  const int P = 16 / esize;
  Plan p{false, aligned && cols % P == 0, kThreads, kThreads, 1};
  if (cols < P) return p;
  const int64_t nvec = (cols + P - 1) / P;
  const int wave_max = 4;
  const int block_vpt = backward ? 2 : 4;
  if (nvec > (int64_t)1024 * kMaxVpt) return p;
  p.vec = true;
  if (nvec <= 64 * wave_max) {  // one wave per row, 4 rows per block
    p.ntb = 256;
    p.tpr = 64;
    p.vpt = pow2_at_least((nvec + 63) / 64);
  } else {  // a block per row
    p.vpt = block_vpt;
    p.ntb = p.tpr = pow2_at_least((nvec + p.vpt - 1) / p.vpt);
    if (p.ntb > 1024) {
      p.ntb = p.tpr = 1024;
      p.vpt = pow2_at_least((nvec + 1023) / 1024);
    }
  }
  return p;
}

// Resident blocks per CU of a kernel at this launch shape (queried once per
// instantiation; each CU of an MI355X is alike).
template <typename K> int resident_per_cu(K kernel, int threads, size_t lds) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, lds) != hipSuccess || n < 1) n = 1;
  return n;
}

template <typename T, typename W, int MODE, bool ALN, int NTB, int TPR, int VPT> int bwd_resident() {
  // dynamic LDS of a 4-rows-per-block shape: one fp32 row of at most 64*4*8 columns
  static const int n = resident_per_cu(rmsnorm_bwd_vec<T, W, NTB, TPR, VPT, MODE, ALN>, NTB,
                                       NTB / TPR > 1 ? (size_t)64 * 4 * 8 * sizeof(float) : 0);
  return n;
}


template <typename T, typename W, int MODE, bool ALN, int NTB, int TPR, int VPT> void launch_fwd_vec(const FwdArgs& a) {
  constexpr int RPB = NTB / TPR;
  const int64_t groups = (a.rows + RPB - 1) / RPB;
  const T *x = static_cast<const T*>(a.x), *res = static_cast<const T*>(a.res);
  const W *w = static_cast<const W*>(a.w), *b = static_cast<const W*>(a.b);
  T* s_out = static_cast<T*>(a.s_out);
  W* y = static_cast<W*>(a.y);
  if constexpr (ALN) {
    // Up to four waves of resident blocks: the persistent grid.
    static const int per_cu = resident_per_cu(rmsnorm_fwd_vec<T, W, NTB, TPR, VPT, MODE, ALN>, NTB, 0);
    static const int per_cu_grid = resident_per_cu(rmsnorm_fwd_grid<T, W, NTB, TPR, VPT, MODE>, NTB, 0);
    if (groups <= (int64_t)4 * cu_count() * per_cu) {
      const int64_t slots = (int64_t)cu_count() * per_cu_grid;
      hipLaunchKernelGGL((rmsnorm_fwd_grid<T, W, NTB, TPR, VPT, MODE>), dim3(groups < slots ? groups : slots), dim3(NTB),
                         0, a.s, x, w, b, res, s_out, a.offset, y, a.rstd, a.rows, a.cols, a.eps, 1.0f / (float)a.cols);
      return;
    }
  }
  hipLaunchKernelGGL((rmsnorm_fwd_vec<T, W, NTB, TPR, VPT, MODE, ALN>), dim3(xcd_split_grid(groups)), dim3(NTB), 0, a.s, x,
                     w, b, res, s_out, a.offset, y, a.rstd, a.rows, a.cols, a.eps, 1.0f / (float)a.cols);
}


template <typename T, typename W, int MODE, bool ALN, int NTB, int TPR, int VPT>
void launch_bwd_vec(const BwdArgs& a, int64_t blocks) {
  constexpr int RPB = NTB / TPR;
  const size_t lds = RPB > 1 ? (size_t)a.cols * sizeof(float) : 0;
  hipLaunchKernelGGL((rmsnorm_bwd_vec<T, W, NTB, TPR, VPT, MODE, ALN>), dim3(blocks), dim3(NTB), lds, a.s,
                     static_cast<const T*>(a.x), static_cast<const W*>(a.w), a.rstd, static_cast<const W*>(a.dy),
                     static_cast<const T*>(a.ds), a.offset, static_cast<T*>(a.dx), a.dw_part, a.db_part, a.rows,
                     a.cols, 1.0f / (float)a.cols);
}

// Every (ntb, tpr, vpt) the planner can return.
#define PK_RMS_FWD_SHAPES(X) X(256, 64, 1) X(256, 64, 2) X(256, 64, 4) X(128, 128, 4) X(256, 256, 4) X(512, 512, 4) \
  X(1024, 1024, 4) X(1024, 1024, 8) X(1024, 1024, 16)
#define PK_RMS_BWD_SHAPES(X) X(256, 64, 1) X(256, 64, 2) X(256, 64, 4) X(256, 256, 2) X(512, 512, 2) \
  X(1024, 1024, 2) X(1024, 1024, 4) X(1024, 1024, 8) X(1024, 1024, 16)

// The forward and the backward at the plan's shape.
template <typename T, typename W, int MODE, bool ALN> void fwd_vec(const FwdArgs& a, const Plan& p) {
#define PK_FWD_CASE(NTB, TPR, VPT) \
  if (p.ntb == NTB && p.tpr == TPR && p.vpt == VPT) return launch_fwd_vec<T, W, MODE, ALN, NTB, TPR, VPT>(a);
  PK_RMS_FWD_SHAPES(PK_FWD_CASE)
#undef PK_FWD_CASE
}

template <typename T, typename W, int MODE, bool ALN> void bwd_vec(const BwdArgs& a, const Plan& p, int64_t blocks) {
#define PK_BWD_CASE(NTB, TPR, VPT) \
  if (p.ntb == NTB && p.tpr == TPR && p.vpt == VPT) return launch_bwd_vec<T, W, MODE, ALN, NTB, TPR, VPT>(a, blocks);
  PK_RMS_BWD_SHAPES(PK_BWD_CASE)
#undef PK_BWD_CASE
}

// Resident blocks per CU of the backward at the plan's shape.
template <typename T, typename W, int MODE, bool ALN> int bwd_vec_resident(const Plan& p) {
#define PK_RES_CASE(NTB, TPR, VPT) \
  if (p.ntb == NTB && p.tpr == TPR && p.vpt == VPT) return bwd_resident<T, W, MODE, ALN, NTB, TPR, VPT>();
  PK_RMS_BWD_SHAPES(PK_RES_CASE)
#undef PK_RES_CASE
  return 1;
}

}  // namespace

// Rows that are not whole, aligned packs (rmsnorm_ragged.hip, a unit of its own for the build's sake).
template <typename T, typename W, int MODE> struct Ragged {
  static void fwd(const FwdArgs& a, const Plan& p);
  static void bwd(const BwdArgs& a, const Plan& p, int64_t blocks);
  static int resident(const Plan& p);
};

}  // namespace pk
