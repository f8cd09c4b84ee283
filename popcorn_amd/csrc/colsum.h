// Deterministic column sums of [parts, cols] fp32 arrays of per-block partial
// rows (weight gradients), in a fixed order so repeated runs give identical bits.
#pragma once

#include "common.h"

namespace pk {
namespace {

// out[c] = sum over p of part[p * cols + c], rounded once to the output's type.
struct ColumnSum {
  const float* part;
  void* out;
  int64_t parts;
};

// A block takes kColCols columns with kColLanes row lanes each: lane l adds rows
// l, l + kColLanes, ... 16 at a time, as a tree, and the lanes are then added as
// trees too, in an order that depends on nothing but `parts`. What bounds it is
// the latency of a lane's chain of loads (the partial rows are in the L2 or the
// MALL), so the lanes are many and the columns few, 16 columns still being whole
// 64-byte pieces of a row: 1280 x 4096 partial rows take 7.5 us, in one launch,
// where a stage per 32 rows and a final one took 5.0 + 3.8 and the gap between
// them, and the two sums of 1280 x 1537 (dw and dbias) 7.5 where four launches took
// 17; 512 x 8192 6.5 (4.9 + 4.6).
constexpr int kColCols = 16;
constexpr int kColLanes = 64;
constexpr int kColThreads = kColCols * kColLanes;
constexpr int kColWaves = kColThreads / 64;

// t[0] + ... + t[N - 1] as a tree (overwrites t)
template <int N> __device__ __forceinline__ float tree_sum(float (&t)[N]) {
#pragma unroll
  for (int w = N / 2; w >= 1; w /= 2)
#pragma unroll
    for (int u = 0; u < w; ++u) t[u] += t[u + w];
  return t[0];
}

// Two sums of one width in one launch (dw and dbias, or the q and the k weight): blockIdx.y picks.
template <typename T>
__global__ __launch_bounds__(kColThreads) void column_sum(ColumnSum first, ColumnSum second, int cols) {
  __shared__ float acc[kColWaves][kColCols];
  const ColumnSum j = blockIdx.y == 0 ? first : second;
  const int cl = threadIdx.x % kColCols, rl = threadIdx.x / kColCols;
  const int c = blockIdx.x * kColCols + cl;
  float s = 0.f;
  if (c < cols) {
    const float* v = j.part + c;
    const int64_t step = (int64_t)kColLanes * cols;
    int64_t p = rl;
    for (; p + 15 * kColLanes < j.parts; p += 16 * kColLanes) {
      float t[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) t[u] = v[p * cols + u * step];
      s += tree_sum(t);
    }
    float t[16];  // the lane's last rows, all in flight together
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = p + u * kColLanes < j.parts ? v[p * cols + u * step] : 0.f;
    s += tree_sum(t);
  }
  // the wave's four row lanes of each column, then the waves
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  if (threadIdx.x % 64 < kColCols) acc[threadIdx.x / 64][cl] = s;
  __syncthreads();
  if (threadIdx.x < kColCols && c < cols) {
    float t[kColWaves];
#pragma unroll
    for (int w = 0; w < kColWaves; ++w) t[w] = acc[w][cl];
    static_cast<T*>(j.out)[c] = from_f32<T>(tree_sum(t));
  }
}

template <typename T>
void column_sums(const ColumnSum& first, const ColumnSum* second, int cols, hipStream_t s) {
  hipLaunchKernelGGL(column_sum<T>, dim3((cols + kColCols - 1) / kColCols, second ? 2 : 1), dim3(kColThreads), 0, s,
                     first, second ? *second : first, cols);
}

}  // namespace
}  // namespace pk
