// The plan of a formed operator and the product of a few of its rows with a vector, shared by the application and by
// the correction equation's CG step.
#pragma once
#include "cc_common.h"

constexpr int FORMED_MATS = 5;   // distinct matrices of one plan
constexpr int FORMED_ROWS = 4;   // rows of a workgroup
struct FormedPlan {
  int n_env, n_mats, has_id, f32;   // f32: the matrices are FP32 (products and sums stay FP64)
  const void* mat[FORMED_MATS];
  double op[FORMED_MATS][4];        // O_g[s'][s], d = 2
  double id[4];                     // coefficient of the identity over the environment legs
};

// Rows row0 .. row0 + 3 of all matrices against x on 512 threads: two waves per row, each every other 64 columns, with
// all their loads (U column steps, U >= n_env / 128) in flight at once; the halves are added in order.
constexpr int FORMED_THREADS = 512;
template <typename T, int NG, int U>
struct FormedRows {
  T v[U][NG];
  __device__ __forceinline__ int row(int row0) const { return row0 + (int)(threadIdx.x >> 7); }
  __device__ __forceinline__ int col(int u) const { return (int)(threadIdx.x & 127) + 128 * u; }
  __device__ __forceinline__ void load(const FormedPlan& f, int row0) {
    const int n = f.n_env, r = row(row0) < n ? row(row0) : n - 1;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = col(u) < n ? col(u) : n - 1;   // clamped; masked in the products
#pragma unroll
      for (int g = 0; g < NG; ++g) v[u][g] = static_cast<const T*>(f.mat[g])[(int64_t)r * n + c];
    }
  }
  // y[row][s'] from x(c, s); red: 16 doubles of LDS.
  template <typename F>
  __device__ __forceinline__ void apply(const FormedPlan& f, int row0, F x, double* red, double* __restrict__ y) {
    const int n = f.n_env, wave = threadIdx.x >> 6;
    // the identity's part, loaded with the rest rather than behind the barrier (160 steps at D = 6: 5.20 -> 5.14 ms)
    const int k = threadIdx.x, r = row0 + (k >> 1), sp1 = k & 1;
    double own = 0.0;
    if (f.has_id && k < 2 * FORMED_ROWS && r < n) own = f.id[2 * sp1] * x(r, 0) + f.id[2 * sp1 + 1] * x(r, 1);
    double acc[NG][2];
#pragma unroll
    for (int g = 0; g < NG; ++g) acc[g][0] = acc[g][1] = 0.0;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (col(u) < n) {
        const double x0 = x(col(u), 0), x1 = x(col(u), 1);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          acc[g][0] += (double)v[u][g] * x0;
          acc[g][1] += (double)v[u][g] * x1;
        }
      }
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
      double a = 0.0;
#pragma unroll
      for (int g = 0; g < NG; ++g) a += f.op[g][2 * sp] * acc[g][0] + f.op[g][2 * sp + 1] * acc[g][1];
      a = cc_wave_sum(a);
      if ((threadIdx.x & 63) == 0) red[wave * 2 + sp] = a;
    }
    __syncthreads();
    if (k < 2 * FORMED_ROWS && r < n) y[2 * r + sp1] = red[(k >> 1) * 4 + sp1] + red[(k >> 1) * 4 + 2 + sp1] + own;
  }
};
