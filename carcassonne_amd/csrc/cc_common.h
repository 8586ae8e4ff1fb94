// Shared definitions for the carcassonne_amd HIP library (gfx950 / CDNA4 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/carcassonne_hip.h"

#define CC_HIP(expr)                                   \
  do {                                                 \
    hipError_t _e = (expr);                            \
    if (_e != hipSuccess) {                            \
      cc_set_last_error(hipGetErrorString(_e));        \
      return CC_ERR_HIP;                               \
    }                                                  \
  } while (0)

#define CC_LAUNCH_CHECK()                              \
  do {                                                 \
    hipError_t _e = hipGetLastError();                 \
    if (_e != hipSuccess) {                            \
      cc_set_last_error(hipGetErrorString(_e));        \
      return CC_ERR_HIP;                               \
    }                                                  \
  } while (0)

void cc_set_last_error(const char* msg);

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

static inline hipStream_t cc_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

static inline unsigned cc_blocks(int64_t n, int threads, unsigned cap = 65535u * 8u) {
  int64_t b = (n + threads - 1) / threads;
  if (b < 1) b = 1;
  if (b > (int64_t)cap) b = cap;
  return (unsigned)b;
}

// Sum of v over the 64 lanes of a wave, the same value in every lane: four shifted adds inside each row of 16 lanes,
// two adds of a row's total to the next rows (data-parallel moves, a few cycles each against an LDS round trip per
// step of a shuffle), lane 63 read out.  The order depends on nothing but the lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ double cc_dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double cc_wave_sum(double v) {
  v = cc_dpp_add<0x111, 0xf>(v);   // row_shr:1
  v = cc_dpp_add<0x112, 0xf>(v);   // row_shr:2
  v = cc_dpp_add<0x114, 0xf>(v);   // row_shr:4
  v = cc_dpp_add<0x118, 0xf>(v);   // row_shr:8: lane 15 of each row holds the row's sum
  v = cc_dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  v = cc_dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3: lane 63 holds the sum
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, 63);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | lo);
}

// Internal (not exported through the C ABI header): operator plans used by the solvers.
int cc_internal_stage3_apply(hipStream_t st, const void* plan, const double* x, double* y);
int64_t cc_internal_stage3_n(const void* plan);
int cc_internal_lp_apply(hipStream_t st, const void* plan, const double* x, double* y);
int64_t cc_internal_lp_n(const void* plan);
int cc_internal_formed_apply(hipStream_t st, const void* plan, const double* x, double* y);
int64_t cc_internal_formed_n(const void* plan);
// C[b][m][j] = sum over k <= j of A[b][m][k] B[k][j] for n x n matrices: B upper triangular (row-major), C row-major,
// A with element strides sAm, sAk.  Half the work of the full product.
int cc_internal_gemm_upper(hipStream_t st, int64_t batch, int64_t n, const double* A, int64_t sAb, int64_t sAm, int64_t sAk,
                           const double* B, int64_t ldb, double* C, int64_t sCb);

// Launch timing (between cc_profile_begin[_sampled] and cc_profile_end, single-threaded use): a kernel
// launch is bracketed by cc_prof_start / cc_prof_stop, which record HIP events on its stream when timing
// is on and the launch is one of the sampled ones of its kind (e0 stays null otherwise).
enum { CC_PROF_FUSED_F64 = 0, CC_PROF_LP = 1, CC_PROF_FORMED = 2, CC_PROF_KINDS = 3 };
int cc_prof_start(hipStream_t st, int kind, hipEvent_t* e0);
int cc_prof_stop(hipStream_t st, int kind, hipEvent_t e0);

// A stage-3 slab channel read in place from a tensor with six index legs: slab[alpha][p'][p] with
// alpha = a0 * na1 + a1, p' = r0 * d1 + r1, p = c0 * d1 + c1 (P = d0 * d1) lives at element offset
// a0 s[0] + a1 s[1] + r0 s[2] + r1 s[3] + c0 s[4] + c1 s[5] of the source.  A contiguous
// (alpha, P, P) array is na1 = d1 = 1, s = {P*P, 0, P, 0, 1, 0}.
struct CCSlabMap {
  int64_t na1, d1;
  int64_t s[6];
};
__host__ __device__ inline int64_t cc_slab_offset(const CCSlabMap& m, int64_t al, int64_t row, int64_t col) {
  const int64_t a0 = al / m.na1, a1 = al - a0 * m.na1;
  const int64_t r0 = row / m.d1, r1 = row - r0 * m.d1, c0 = col / m.d1, c1 = col - c0 * m.d1;
  return a0 * m.s[0] + a1 * m.s[1] + r0 * m.s[2] + r1 * m.s[3] + c0 * m.s[4] + c1 * m.s[5];
}
// Validates the leg sizes (all positive, d0 * d1 = P, na0 * na1 = n_alpha) and non-negative strides.
int cc_slab_map(int64_t na0, int64_t na1, int64_t d0, int64_t d1, const int64_t* strides, CCSlabMap* out);

// Per-alpha gather of one slab into LDS in source order: the four inner legs (r0, r1, c0, c1) sorted by
// stride, largest first, so consecutive threads read consecutive source elements when some leg has
// stride 1.  Element k of the gather has digits k = ((k0 * sz1 + k1) * sz2 + k2) * sz3 + k3; its source
// offset is sum k_i st_i, its slab position row = sum k_i rw_i, col = sum k_i cw_i.
struct CCSlabGather {
  int64_t na1, sa0, sa1;  // alpha = a0 * na1 + a1 at a0 * sa0 + a1 * sa1
  int P;
  int sz[4], rw[4], cw[4];
  int64_t st[4];
};
static inline CCSlabGather cc_slab_gather(const CCSlabMap& m, int64_t d0) {
  CCSlabGather g;
  g.na1 = m.na1;
  g.sa0 = m.s[0];
  g.sa1 = m.s[1];
  g.P = (int)(d0 * m.d1);
  const int size[4] = {(int)d0, (int)m.d1, (int)d0, (int)m.d1};
  const int rw[4] = {(int)m.d1, 1, 0, 0}, cw[4] = {0, 0, (int)m.d1, 1};
  int order[4] = {0, 1, 2, 3};
  for (int i = 1; i < 4; ++i)  // stable insertion sort by stride, descending
    for (int j = i; j > 0 && m.s[2 + order[j]] > m.s[2 + order[j - 1]]; --j) {
      int t = order[j];
      order[j] = order[j - 1];
      order[j - 1] = t;
    }
  for (int i = 0; i < 4; ++i) {
    g.sz[i] = size[order[i]];
    g.st[i] = m.s[2 + order[i]];
    g.rw[i] = rw[order[i]];
    g.cw[i] = cw[order[i]];
  }
  return g;
}
// The same with every leg of extent D (P = D * D) and NTH threads: the index arithmetic divides by
// constants, and each thread issues all its loads before its LDS stores.
template <int D, int NTH>
__device__ inline void cc_slab_load_d(const CCSlabGather& g, const double* __restrict__ src, int64_t al, double* lds, int ld,
                                      double mul) {
  constexpr int n = D * D * D * D, NE = (n + NTH - 1) / NTH;
  const int64_t a0 = al / g.na1, a1 = al - a0 * g.na1;
  const double* base = src + a0 * g.sa0 + a1 * g.sa1;
  double v[NE];
  int at[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = threadIdx.x + NTH * u, ec = e < n ? e : 0;  // clamped: every load in bounds
    const int k3 = ec % D, k2 = (ec / D) % D, k1 = (ec / (D * D)) % D, k0 = ec / (D * D * D);
    v[u] = base[k0 * g.st[0] + k1 * g.st[1] + k2 * g.st[2] + k3 * g.st[3]];
    at[u] = (k0 * g.rw[0] + k1 * g.rw[1] + k2 * g.rw[2] + k3 * g.rw[3]) * ld + k0 * g.cw[0] + k1 * g.cw[1] + k2 * g.cw[2] +
            k3 * g.cw[3];
  }
#pragma unroll
  for (int u = 0; u < NE; ++u)
    if (threadIdx.x + NTH * u < n) lds[at[u]] = v[u] * mul;
}
// A channel given as a weighted sum of tensors with the same legs and strides.
constexpr int CC_SLAB_SOURCES = 8;
struct CCSlabSum {
  int n;
  const double* p[CC_SLAB_SOURCES];
  double c[CC_SLAB_SOURCES];
};
static inline CCSlabSum cc_slab_sum(int n, const double* const* src, const double* coef) {
  CCSlabSum s;
  s.n = n;
  for (int i = 0; i < CC_SLAB_SOURCES; ++i) {
    s.p[i] = src[i < n ? i : 0];
    s.c[i] = i < n ? coef[i] : 0.0;
  }
  return s;
}
// cc_slab_load_d of the sum: lds[row * ld + col] = sum_i c_i src_i, each source's loads in flight together.
template <int D, int NTH>
__device__ inline void cc_slab_load_sum_d(const CCSlabGather& g, const CCSlabSum& src, int64_t al, double* lds, int ld) {
  constexpr int n = D * D * D * D, NE = (n + NTH - 1) / NTH;
  const int64_t a0 = al / g.na1, a1 = al - a0 * g.na1, base = a0 * g.sa0 + a1 * g.sa1;
  double v[NE];
  int at[NE];
  int64_t off[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = threadIdx.x + NTH * u, ec = e < n ? e : 0;  // clamped: every load in bounds
    const int k3 = ec % D, k2 = (ec / D) % D, k1 = (ec / (D * D)) % D, k0 = ec / (D * D * D);
    off[u] = base + k0 * g.st[0] + k1 * g.st[1] + k2 * g.st[2] + k3 * g.st[3];
    at[u] = (k0 * g.rw[0] + k1 * g.rw[1] + k2 * g.rw[2] + k3 * g.rw[3]) * ld + k0 * g.cw[0] + k1 * g.cw[1] + k2 * g.cw[2] +
            k3 * g.cw[3];
    v[u] = src.c[0] * src.p[0][off[u]];
  }
  for (int i = 1; i < src.n; ++i)
#pragma unroll
    for (int u = 0; u < NE; ++u) v[u] += src.c[i] * src.p[i][off[u]];
#pragma unroll
  for (int u = 0; u < NE; ++u)
    if (threadIdx.x + NTH * u < n) lds[at[u]] = v[u];
}
// The same for any leg sizes.
__device__ inline void cc_slab_load_sum(const CCSlabGather& g, const CCSlabSum& src, int64_t al, double* lds, int ld) {
  const int64_t a0 = al / g.na1, a1 = al - a0 * g.na1, base = a0 * g.sa0 + a1 * g.sa1;
  const int n = g.P * g.P;
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    int k = e;
    const int k3 = k % g.sz[3];
    k /= g.sz[3];
    const int k2 = k % g.sz[2];
    k /= g.sz[2];
    const int k1 = k % g.sz[1];
    const int k0 = k / g.sz[1];
    const int64_t off = base + k0 * g.st[0] + k1 * g.st[1] + k2 * g.st[2] + k3 * g.st[3];
    const int row = k0 * g.rw[0] + k1 * g.rw[1] + k2 * g.rw[2] + k3 * g.rw[3];
    const int col = k0 * g.cw[0] + k1 * g.cw[1] + k2 * g.cw[2] + k3 * g.cw[3];
    double v = src.c[0] * src.p[0][off];
    for (int i = 1; i < src.n; ++i) v += src.c[i] * src.p[i][off];
    lds[row * ld + col] = v;
  }
}
// Loads slab alpha into lds[row * ld + col] (row, col < P) with all threads of the block.
__device__ inline void cc_slab_load(const CCSlabGather& g, const double* __restrict__ src, int64_t al, double* lds, int ld,
                                    double mul) {
  const int64_t a0 = al / g.na1, a1 = al - a0 * g.na1;
  const double* base = src + a0 * g.sa0 + a1 * g.sa1;
  const int n = g.P * g.P;
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    int k = e;
    const int k3 = k % g.sz[3];
    k /= g.sz[3];
    const int k2 = k % g.sz[2];
    k /= g.sz[2];
    const int k1 = k % g.sz[1];
    const int k0 = k / g.sz[1];
    const int64_t off = k0 * g.st[0] + k1 * g.st[1] + k2 * g.st[2] + k3 * g.st[3];
    const int row = k0 * g.rw[0] + k1 * g.rw[1] + k2 * g.rw[2] + k3 * g.rw[3];
    const int col = k0 * g.cw[0] + k1 * g.cw[1] + k2 * g.cw[2] + k3 * g.cw[3];
    lds[row * ld + col] = base[off] * mul;
  }
}
