// Lanczos for the lowest eigenpair of the pencil (H, N), N = (L L^T) (x) I_d, on the whitened
// operator W H W^T (W = L^-1 (x) I_d), with full (twice-applied) reorthogonalisation.  All
// vectors and recurrence scalars stay in device memory; the host loop only reads two doubles
// (Ritz value and residual estimate) every `check_every` steps.
#include "cc_formed.h"

#include <cmath>
#include <utility>
#include <vector>

namespace {

// sum_i a[i] b[i] over the 256 threads of a workgroup in a fixed order: each thread loads its DOT_U
// pairs at once (clamped index, masked product), then wave sums, added in wave order.
constexpr int DOT_U = 12;
__device__ inline double block_dot256(int64_t n, const double* __restrict__ a, const double* __restrict__ b, double* red) {
  double acc = 0.0;
  for (int64_t base = threadIdx.x; base < n; base += 256 * DOT_U) {
    double x[DOT_U], y[DOT_U];
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      const int64_t i = base + 256 * u < n ? base + 256 * u : base;
      x[u] = a[i];
      y[u] = b[i];
    }
#pragma unroll
    for (int u = 0; u < DOT_U; ++u)
      if (base + 256 * u < n) acc += x[u] * y[u];
  }
  acc = cc_wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// c[b] = Q_b . w for b < nq; a block b == nq (when launched) gives c[nq] = w . w
__global__ void __launch_bounds__(256) lz_coeff_kernel(int64_t n, const double* __restrict__ Q, const double* __restrict__ w,
                                                       double* __restrict__ c, int nq) {
  __shared__ double red[4];
  const double* q = (int)blockIdx.x == nq ? w : Q + (int64_t)blockIdx.x * n;
  const double t = block_dot256(n, q, w, red);
  if (threadIdx.x == 0) c[blockIdx.x] = t;
}

// w[i] -= sum_j c[j] Q[j][i]   (or z[i] = sum_j c[j] Q[j][i] when `assign`): block = 16 outputs x
// 16 basis slices, slice sums combined in a fixed order.
// sum_j c[j] Q[j][i] over the slice's vectors j = slice, slice + 16, ...: LZ_U loads in flight at a time
constexpr int LZ_U = 5;
__device__ inline double slice_combine(int m, int64_t n, const double* __restrict__ Q, const double* __restrict__ c, int slice,
                                       int64_t i) {
  double acc = 0.0;
  for (int j0 = slice; j0 < m; j0 += 16 * LZ_U) {
    double q[LZ_U], cj[LZ_U];
#pragma unroll
    for (int u = 0; u < LZ_U; ++u) {   // clamped index, masked product
      const int j = j0 + 16 * u < m ? j0 + 16 * u : j0;
      q[u] = Q[(int64_t)j * n + i];
      cj[u] = c[j];
    }
#pragma unroll
    for (int u = 0; u < LZ_U; ++u)
      if (j0 + 16 * u < m) acc += cj[u] * q[u];
  }
  return acc;
}

// w -= Q^T c (assign: w = Q^T c) over the first m basis vectors; record (when given) receives c[m - 1]
__global__ void __launch_bounds__(256) lz_combine_kernel(int m, int64_t n, const double* __restrict__ Q,
                                                         const double* __restrict__ c, double* __restrict__ w, int assign,
                                                         double* __restrict__ record = nullptr) {
  __shared__ double red[16][16];
  if (record != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *record = c[m - 1];
  const int e = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int64_t i = (int64_t)blockIdx.x * 16 + e;
  red[slice][e] = i < n ? slice_combine(m, n, Q, c, slice, i) : 0.0;
  __syncthreads();
  if (slice == 0 && i < n) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[k][e];
    w[i] = assign ? t : w[i] - t;
  }
}

// The second Gram-Schmidt pass and the normalisation in one kernel: q = (w - Q c) / beta with
// beta^2 = w.w - c.c (c[m] holds w.w from lz_coeff_kernel; exact for orthonormal Q, and free of
// cancellation because the second pass's coefficients are at rounding level), beta written by block 0.
__global__ void __launch_bounds__(256) lz_combine_normalize_kernel(int m, int64_t n, const double* __restrict__ Q,
                                                                   const double* __restrict__ c, const double* __restrict__ w,
                                                                   double* __restrict__ q, double* __restrict__ beta) {
  __shared__ double red[16][16];
  const int e = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int64_t i = (int64_t)blockIdx.x * 16 + e;
  __shared__ double sq[4];
  double cc = 0.0;   // c . c over the block
  for (int j = threadIdx.x; j < m; j += 256) cc += c[j] * c[j];
  red[slice][e] = i < n ? slice_combine(m, n, Q, c, slice, i) : 0.0;
  cc = cc_wave_sum(cc);
  if ((threadIdx.x & 63) == 0) sq[threadIdx.x >> 6] = cc;
  __syncthreads();
  const double b2 = c[m] - (((sq[0] + sq[1]) + sq[2]) + sq[3]), b = b2 > 0.0 ? sqrt(b2) : 0.0, inv = b > 0.0 ? 1.0 / b : 0.0;
  if (slice == 0 && i < n) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[k][e];
    q[i] = (w[i] - t) * inv;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *beta = b;
}

// ---- one Gram-Schmidt pass per step, its second one delayed ------------------------------------------------------
// A step multiplies its candidate w as it comes out of the first pass, y = A w, and takes the second pass on w together
// with the first one on y: with c = Q w, d = Q y (over q_0 .. q_{j-1}), b^2 = w.w - c.c and e = (w.y - c.d) / b,
//   q_j = (w - Q^T c) / b,   next w = (y - Q^T d - e q_j) / b,   alpha_j = e / b - c_{j-1},   beta_{j-1} = b.
// (A Q^T c lies in the span that the first pass on y takes out, so it never has to be formed.)  Every vector still gets
// both passes against the vectors as they are, from inner products of its own, but they are three launches per step
// instead of five and read the basis twice instead of four times; a step is all launches: n = 512 (D = 4, chi = 32) 15.7 ->
// 11.5 us, n = 2592 (D = 6, chi = 64) 19.7 -> 15.3 us.

// c[b] = Q_b . w, d[b] = Q_b . y for b < m; block m: w . w and w . y
__global__ void __launch_bounds__(256) lz_coeff2_kernel(int n, int m, const double* __restrict__ Q,
                                                        const double* __restrict__ w, const double* __restrict__ y,
                                                        double* __restrict__ c, double* __restrict__ d) {
  __shared__ double red[2][4];
  const double* q = (int)blockIdx.x == m ? w : Q + (int64_t)blockIdx.x * n;
  double aw = 0.0, ay = 0.0;
  for (int base = threadIdx.x; base < n; base += 256 * DOT_U) {
    double x[DOT_U], u[DOT_U], v[DOT_U];
#pragma unroll
    for (int k = 0; k < DOT_U; ++k) {   // clamped index, masked product
      const int i = base + 256 * k < n ? base + 256 * k : base;
      x[k] = q[i];
      u[k] = w[i];
      v[k] = y[i];
    }
#pragma unroll
    for (int k = 0; k < DOT_U; ++k)
      if (base + 256 * k < n) {
        aw += x[k] * u[k];
        ay += x[k] * v[k];
      }
  }
  aw = cc_wave_sum(aw);
  ay = cc_wave_sum(ay);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = aw;
    red[1][threadIdx.x >> 6] = ay;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    c[blockIdx.x] = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
    d[blockIdx.x] = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
  }
}

// One round of loads for 160 vectors, the last terms' operands among them: with half as many in flight and those read
// behind the barrier a step waits for two more rounds (a solve of 160 steps at
// D = 6, chi = 64 5.29 -> 5.07 ms, at D = 4, chi = 32 2.52 -> 2.40 ms).
constexpr int LZ_STEP_U = 10;
// The step's combinations from c and d (m vectors before this one); w is replaced by the next candidate.  Block = 16
// outputs x 16 basis slices, slice sums combined in a fixed order.
__global__ void __launch_bounds__(256) lz_step_kernel(int m, int n, double* __restrict__ Q, const double* __restrict__ c,
                                                      const double* __restrict__ d, double* __restrict__ w,
                                                      const double* __restrict__ y, double* __restrict__ alpha,
                                                      double* __restrict__ beta) {
  __shared__ double red[2][16][16], sq[2][4];
  const int e = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + e, ic = i < n ? i : n - 1;
  const double wi = w[ic], yi = y[ic], ww = c[m], wy = d[m], last = c[m > 0 ? m - 1 : 0];   // ahead of the barrier
  double cc = 0.0, cd = 0.0;   // c . c and c . d over the block
  for (int j = threadIdx.x; j < m; j += 256) {
    cc += c[j] * c[j];
    cd += c[j] * d[j];
  }
  double ac = 0.0, ad = 0.0;
  for (int j0 = slice; j0 < m; j0 += 16 * LZ_STEP_U) {
    double q[LZ_STEP_U], cj[LZ_STEP_U], dj[LZ_STEP_U];
    const double* p = Q + (int64_t)j0 * n + ic;
#pragma unroll
    for (int u = 0; u < LZ_STEP_U; ++u) {   // clamped index, masked product
      const int j = j0 + 16 * u < m ? j0 + 16 * u : j0;
      q[u] = *p;
      cj[u] = c[j];
      dj[u] = d[j];
      if (j0 + 16 * (u + 1) < m) p += (int64_t)16 * n;
    }
#pragma unroll
    for (int u = 0; u < LZ_STEP_U; ++u)
      if (j0 + 16 * u < m) {
        ac += cj[u] * q[u];
        ad += dj[u] * q[u];
      }
  }
  red[0][slice][e] = ac;
  red[1][slice][e] = ad;
  cc = cc_wave_sum(cc);
  cd = cc_wave_sum(cd);
  if ((threadIdx.x & 63) == 0) {
    sq[0][threadIdx.x >> 6] = cc;
    sq[1][threadIdx.x >> 6] = cd;
  }
  __syncthreads();
  const double b2 = ww - (((sq[0][0] + sq[0][1]) + sq[0][2]) + sq[0][3]);
  const double b = b2 > 0.0 ? sqrt(b2) : 0.0, inv = b > 0.0 ? 1.0 / b : 0.0;
  const double on = (wy - (((sq[1][0] + sq[1][1]) + sq[1][2]) + sq[1][3])) * inv;   // q_j . y
  if (slice == 0 && i < n) {
    double tc = 0.0, td = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      tc += red[0][k][e];
      td += red[1][k][e];
    }
    const double q = (wi - tc) * inv;
    Q[(int64_t)m * n + i] = q;
    w[i] = ((yi - td) - on * q) * inv;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *alpha = on * inv - (m > 0 ? last : 0.0);
    if (m > 0) *beta = b;
  }
}

// beta = |w| without its components c on the m basis vectors (c[m] = w . w)
__global__ void __launch_bounds__(256) lz_beta_kernel(int m, const double* __restrict__ c, double* __restrict__ beta) {
  __shared__ double sq[4];
  double cc = 0.0;
  for (int j = threadIdx.x; j < m; j += 256) cc += c[j] * c[j];
  cc = cc_wave_sum(cc);
  if ((threadIdx.x & 63) == 0) sq[threadIdx.x >> 6] = cc;
  __syncthreads();
  const double b2 = c[m] - (((sq[0] + sq[1]) + sq[2]) + sq[3]);
  if (threadIdx.x == 0) *beta = b2 > 0.0 ? sqrt(b2) : 0.0;
}

// beta = ||w||, q = w / beta (single 1024-thread block, fixed-order tree)
__global__ void __launch_bounds__(1024) lz_normalize_kernel(int64_t n, const double* __restrict__ w, double* __restrict__ q,
                                                            double* __restrict__ beta) {
  __shared__ double red[1024];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) acc += w[i] * w[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  const double b = sqrt(red[0]);
  const double inv = b > 0.0 ? 1.0 / b : 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) q[i] = w[i] * inv;
  if (threadIdx.x == 0 && beta) *beta = b;
}

constexpr int LZ_LDS_M = 640;

// True when T - x I is positive definite, i.e. x lies below the lowest eigenvalue of the tridiagonal
// (a, b): every leading principal minor is positive.  The minors follow p_{i+1} = (a_i - x) p_i -
// b_{i-1}^2 p_{i-1} (one dependent FMA per step, no division); every fourth step both are rescaled by
// the same power of two, which changes no sign.  b2[i] = b[i]^2.
__device__ bool below_spectrum(int m, const double* a, const double* b2, double x) {
  double pm = 1.0, p = a[0] - x;
  bool pd = p > 0.0;
#pragma unroll 8
  for (int i = 1; i < m; ++i) {  // unrolled: the loads of a and b2 run ahead of the recurrence
    const double pn = (a[i] - x) * p - b2[i - 1] * pm;
    pm = p;
    p = pn;
    pd = pd && (p > 0.0);
    if ((i & 3) == 0) {
      int e;
      (void)frexp(p, &e);
      p = ldexp(p, -e);
      pm = ldexp(pm, -e);
    }
  }
  return pd;
}

// Lowest eigenpair of the m x m tridiagonal (a, b): multisection over one wave, then inverse
// iteration (LU with partial pivoting) on lane 0.  out[0] = theta, out[1] = |b[m-1] * s[m-1]|.
__global__ void __launch_bounds__(64) lz_tridiag_kernel(int m, const double* __restrict__ ga, const double* __restrict__ gb,
                                                        double* __restrict__ out, double* __restrict__ s,
                                                        double* __restrict__ scratch, int want_vector) {
  const int lane = threadIdx.x;
  // stage the tridiagonal in LDS (every lane reads all of it in the Sturm sequences)
  __shared__ double lds_ab[3 * LZ_LDS_M];
  const bool in_lds = m <= LZ_LDS_M;
  if (in_lds) {
    for (int i = lane; i < m; i += 64) {
      lds_ab[i] = ga[i];
      lds_ab[LZ_LDS_M + i] = gb[i];
      lds_ab[2 * LZ_LDS_M + i] = gb[i] * gb[i];
    }
    __syncthreads();
  } else {
    for (int i = lane; i < m; i += 64) scratch[i] = gb[i] * gb[i];   // b^2 past the LDS capacity
    __syncthreads();
  }
  const double* a = in_lds ? lds_ab : ga;
  const double* b = in_lds ? lds_ab + LZ_LDS_M : gb;
  const double* b2 = in_lds ? lds_ab + 2 * LZ_LDS_M : scratch;
  double lo = INFINITY, hi = -INFINITY, tnorm = 0.0;
  for (int i = lane; i < m; i += 64) {
    double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < m - 1 ? fabs(b[i]) : 0.0);
    lo = fmin(lo, a[i] - r);
    hi = fmax(hi, a[i] + r);
    tnorm = fmax(tnorm, fabs(a[i]) + r);
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o, 64));
    hi = fmax(hi, __shfl_xor(hi, o, 64));
    tnorm = fmax(tnorm, __shfl_xor(tnorm, o, 64));
  }
  const double eps = 2.220446049250313e-16;
  const double pivmin = fmax(tnorm * 1e-300, 1e-300) + 4.9e-324;
  lo -= 2.0 * eps * tnorm + pivmin;
  hi += 2.0 * eps * tnorm + pivmin;
  // interlacing: the lowest Ritz value never increases with m, so the previous one bounds it
  if (!isnan(out[0])) hi = fmin(hi, out[0] + 4.0 * eps * tnorm + pivmin);
  for (int round = 0; round < 20; ++round) {
    double x = lo + (hi - lo) * (double)(lane + 1) / 65.0;
    unsigned long long mask = __ballot(!below_spectrum(m, a, b2, x));
    if (mask == 0ULL) {
      lo = lo + (hi - lo) * 64.0 / 65.0;
    } else {
      int first = __ffsll((long long)mask) - 1;
      double nhi = lo + (hi - lo) * (double)(first + 1) / 65.0;
      double nlo = first == 0 ? lo : lo + (hi - lo) * (double)first / 65.0;
      lo = nlo;
      hi = nhi;
    }
    if (hi - lo <= 2.0 * eps * fmax(fabs(lo), fabs(hi)) + pivmin) break;
  }
  const double theta = 0.5 * (lo + hi);
  if (!want_vector) {
    if (lane == 0) {
      out[0] = theta;
      out[1] = NAN;
    }
    return;
  }
  // One step of inverse iteration on T - theta I from a fixed start vector: theta is the eigenvalue to
  // a couple of ulps, so one solve already gives the eigenvector.  Lane 0 runs the LU with partial
  // pivoting (the tridiagonal form of LAPACK gttrf) fused with the forward substitution, carrying the
  // running row in registers and storing reciprocal pivots; the back substitution is then a short FMA
  // chain, and the whole wave normalises.  Scratch lives in LDS when it fits, else in global memory.
  __shared__ double lds_scr[4 * LZ_LDS_M];
  double* base = (m <= LZ_LDS_M) ? lds_scr : scratch;
  double* rd = base;            // 1 / pivot of row i
  double* du = base + m;        // first superdiagonal of U
  double* du2 = base + 2 * m;   // second superdiagonal of U (from row swaps)
  double* sv = (m <= LZ_LDS_M) ? base + 3 * m : s;
  __syncthreads();              // every lane is done reading b^2 from the scratch before it is reused
  if (lane == 0) {
    const double tiny = eps * fmax(tnorm, 1e-300);
    auto start = [](int i) { return 1.0 + 0.01 * (double)((i * 7919) % 101) / 101.0; };
    double cd = a[0] - theta, cdu = m > 1 ? b[0] : 0.0, cs = start(0);
#pragma unroll 4
    for (int i = 0; i < m - 1; ++i) {
      const double dn = a[i + 1] - theta, dli = b[i], dun = (i + 1 < m - 1) ? b[i + 1] : 0.0, ns = start(i + 1);
      if (fabs(cd) >= fabs(dli)) {
        if (cd == 0.0) cd = tiny;
        const double f = dli / cd;
        rd[i] = 1.0 / cd;
        du[i] = cdu;
        du2[i] = 0.0;
        sv[i] = cs;
        cd = dn - f * cdu;
        cdu = dun;
        cs = ns - f * cs;
      } else {
        const double f = cd / dli;
        rd[i] = 1.0 / dli;
        du[i] = dn;
        du2[i] = dun;
        sv[i] = ns;
        cd = cdu - f * dn;
        cdu = -f * dun;
        cs = cs - f * ns;
      }
    }
    if (cd == 0.0) cd = tiny;
    rd[m - 1] = 1.0 / cd;
    double x1 = cs * rd[m - 1], x2 = 0.0;
    sv[m - 1] = x1;
#pragma unroll 4
    for (int i = m - 2; i >= 0; --i) {
      const double x = (sv[i] - du[i] * x1 - du2[i] * x2) * rd[i];
      sv[i] = x;
      x2 = x1;
      x1 = x;
    }
  }
  __syncthreads();
  double big = 0.0;
  for (int i = lane; i < m; i += 64) big = fmax(big, fabs(sv[i]));
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  const double ib = big > 0.0 ? 1.0 / big : 1.0;
  double nrm = 0.0;
  for (int i = lane; i < m; i += 64) { const double v = sv[i] * ib; nrm += v * v; }
  for (int o = 32; o > 0; o >>= 1) nrm += __shfl_xor(nrm, o, 64);
  const double sc = ib / sqrt(nrm);
  for (int i = lane; i < m; i += 64) s[i] = sv[i] * sc;
  __syncthreads();
  if (lane == 0) {
    out[0] = theta;
    out[1] = fabs(b[m - 1] * s[m - 1]);
  }
}

__global__ void set_nan_kernel(double* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = NAN;
}

struct Whitening {
  int64_t n_env, d;
  const double *L, *Lt, *W, *Wt;
};

typedef int (*ApplyFn)(hipStream_t, const void*, const double*, double*);

// w = W H W^T q; a formed operator (apply == cc_internal_formed_apply) holds the whitened matrices already
int op_whitened(hipStream_t st, ApplyFn apply, const void* plan, const Whitening& wh, const double* q, double* t1, double* t2,
                double* w) {
  if (apply == cc_internal_formed_apply) return apply(st, plan, q, w);
  int rc = cc_skinny_f64(st, wh.n_env, 2, wh.Wt, (int)wh.d, q, t1);  // t1 = W^T q
  if (rc) return rc;
  rc = apply(st, plan, t1, t2);                                      // t2 = H t1
  if (rc) return rc;
  return cc_skinny_f64(st, wh.n_env, 1, wh.W, (int)wh.d, t2, w);     // w = W t2
}
}  // namespace

extern "C" int cc_lanczos_work_size(int64_t n, int max_iter, int64_t* out) {
  *out = (int64_t)(max_iter + 1) * n + 3 * n + 12 * (int64_t)(max_iter + 2) + 16;
  return CC_OK;
}

static int lanczos_driver(hipStream_t st, ApplyFn apply, const void* plan, int64_t n_env, int64_t d, const double* L,
                          const double* Lt, const double* W, const double* Wt, const double* x0, double tol_residual,
                          double tol_energy, int max_iter, int check_every, double* work, double* x_out,
                          double* host_result);

extern "C" int cc_lanczos_f64(void* stream, const void* plan, int64_t n_env, int64_t d, const double* L, const double* Lt,
                              const double* W, const double* Wt, const double* x0, double tol_residual,
                              double tol_energy, int max_iter, int check_every, double* work, double* x_out,
                              double* host_result /* theta, residual, iterations */) {
  if (!plan || n_env * d <= 0 || max_iter < 1 || check_every < 0) { cc_set_last_error("lanczos: bad arguments"); return CC_ERR_ARG; }
  if (cc_internal_stage3_n(plan) != n_env * d) { cc_set_last_error("lanczos: operator size does not match the whitening"); return CC_ERR_DIM; }
  return lanczos_driver(cc_stream(stream), cc_internal_stage3_apply, plan, n_env, d, L, Lt, W, Wt, x0, tol_residual,
                        tol_energy, max_iter, check_every, work, x_out, host_result);
}

extern "C" int cc_lanczos_lp(void* stream, const void* lp_plan, int64_t n_env, int64_t d, const double* L, const double* Lt,
                             const double* W, const double* Wt, const double* x0, double tol_residual, double tol_energy,
                             int max_iter, int check_every, double* work, double* x_out, double* host_result) {
  if (!lp_plan || n_env * d <= 0 || max_iter < 1 || check_every < 0) { cc_set_last_error("lanczos: bad arguments"); return CC_ERR_ARG; }
  if (cc_internal_lp_n(lp_plan) != n_env * d) { cc_set_last_error("lanczos: operator size does not match the whitening"); return CC_ERR_DIM; }
  return lanczos_driver(cc_stream(stream), cc_internal_lp_apply, lp_plan, n_env, d, L, Lt, W, Wt, x0, tol_residual,
                        tol_energy, max_iter, check_every, work, x_out, host_result);
}

extern "C" int cc_lanczos_formed_f64(void* stream, const void* formed_plan, int64_t n_env, int64_t d, const double* Lt,
                                     const double* Wt, const double* x0, double tol_residual, double tol_energy,
                                     int max_iter, int check_every, double* work, double* x_out, double* host_result) {
  if (!formed_plan || n_env * d <= 0 || max_iter < 1 || check_every < 0) { cc_set_last_error("lanczos: bad arguments"); return CC_ERR_ARG; }
  if (cc_internal_formed_n(formed_plan) != n_env * d) { cc_set_last_error("lanczos: operator size does not match the whitening"); return CC_ERR_DIM; }
  return lanczos_driver(cc_stream(stream), cc_internal_formed_apply, formed_plan, n_env, d, nullptr, Lt, nullptr, Wt, x0,
                        tol_residual, tol_energy, max_iter, check_every, work, x_out, host_result);
}

static int lanczos_driver(hipStream_t st, ApplyFn apply, const void* plan, int64_t n_env, int64_t d, const double* L,
                          const double* Lt, const double* W, const double* Wt, const double* x0, double tol_residual,
                          double tol_energy, int max_iter, int check_every, double* work, double* x_out,
                          double* host_result) {
  const int64_t n = n_env * d;
  Whitening wh{n_env, d, L, Lt, W, Wt};
  double* Q = work;
  double* w = Q + (int64_t)(max_iter + 1) * n;
  double* t1 = w + n;
  double* t2 = t1 + n;
  double* alpha = t2 + n;
  double* beta = alpha + (max_iter + 2);
  double* c = beta + (max_iter + 2);
  double* s = c + (max_iter + 2);
  double* scratch = s + (max_iter + 2);  // 5 * (max_iter + 2)
  double* res = scratch + 5 * (max_iter + 2);
  int rc;

  // q0 = L^T x0 / ||L^T x0||
  rc = cc_skinny_f64(st, n_env, 2, Lt, (int)d, x0, w);
  if (rc) return rc;
  // A low-precision operator takes unit vectors: its FP16 / BF16 inputs would lose a candidate of small norm.
  const bool delayed = apply != cc_internal_lp_apply;
  double* y = Q + (int64_t)max_iter * n;   // delayed: A w (the basis has max_iter vectors there)
  double* dots = s;                        // and the inner products with it (s is made anew by each check)
  lz_normalize_kernel<<<1, 1024, 0, st>>>(n, w, delayed ? t2 : Q, nullptr);
  CC_LAUNCH_CHECK();
  if (delayed) std::swap(w, t2);

  const bool fixed = check_every == 0;  // exactly max_iter steps, no host reads (capturable in a graph)
  set_nan_kernel<<<1, 64, 0, st>>>(res, 2);
  CC_LAUNCH_CHECK();
  double prev_theta = NAN, theta = NAN, resid = NAN;
  int m = 0, checked_m = -1;
  // the Ritz value and vector of T_m and the residual estimate
  auto ritz = [&]() -> int {
    if (delayed) {
      lz_coeff_kernel<<<m + 1, 256, 0, st>>>(n, Q, w, c, m);
      CC_LAUNCH_CHECK();
      lz_beta_kernel<<<1, 256, 0, st>>>(m, c, beta + m - 1);
      CC_LAUNCH_CHECK();
    }
    lz_tridiag_kernel<<<1, 64, 0, st>>>(m, alpha, beta, res, s, scratch, 1);
    CC_LAUNCH_CHECK();
    return CC_OK;
  };
  for (int j = 0; j < max_iter; ++j) {
    double* qj = Q + (int64_t)j * n;
    if (delayed) {
      rc = op_whitened(st, apply, plan, wh, w, t1, t2, y);
      if (rc) return rc;
      lz_coeff2_kernel<<<j + 1, 256, 0, st>>>((int)n, j, Q, w, y, c, dots);
      CC_LAUNCH_CHECK();
      lz_step_kernel<<<(unsigned)((n + 15) / 16), 256, 0, st>>>(j, (int)n, Q, c, dots, w, y, alpha + j, beta + j - 1);
      CC_LAUNCH_CHECK();
    } else {
      rc = op_whitened(st, apply, plan, wh, qj, t1, t2, w);
      if (rc) return rc;
      // full reorthogonalisation, two classical Gram-Schmidt passes against q_0..q_j; the first pass's
      // coefficient on q_j is alpha_j = q_j . A q_j (the three-term recurrence is contained in it)
      lz_coeff_kernel<<<j + 1, 256, 0, st>>>(n, Q, w, c, -1);
      CC_LAUNCH_CHECK();
      lz_combine_kernel<<<(unsigned)((n + 15) / 16), 256, 0, st>>>(j + 1, n, Q, c, w, 0, alpha + j);
      CC_LAUNCH_CHECK();
      // second pass with the normalisation folded in (w . w from one more coefficient block)
      lz_coeff_kernel<<<j + 2, 256, 0, st>>>(n, Q, w, c, j + 1);
      CC_LAUNCH_CHECK();
      lz_combine_normalize_kernel<<<(unsigned)((n + 15) / 16), 256, 0, st>>>(j + 1, n, Q, c, w, Q + (int64_t)(j + 1) * n,
                                                                             beta + j);
      CC_LAUNCH_CHECK();
    }
    m = j + 1;
    if (m == n) break;
    if (!fixed && (m % check_every == 0 || m == max_iter)) {
      // Ritz value, Ritz vector and residual estimate in one pass (one read of two doubles); the
      // residual counts once the value has settled
      if ((rc = ritz())) return rc;
      double h[2];
      CC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, st));
      CC_HIP(hipStreamSynchronize(st));
      theta = h[0];
      resid = h[1];
      checked_m = m;
      const bool settle_check = !std::isnan(prev_theta) && prev_theta - theta <= 1e3 * tol_energy * fabs(theta);
      bool done = m == n || m == max_iter ||
                  (settle_check && (resid <= tol_residual * fabs(theta) ||
                                    (prev_theta - theta <= tol_energy * fabs(theta))));
      prev_theta = theta;
      if (done) break;
    }
  }
  // the final Ritz vector of T_m (already in s when the last check was at this m)
  if (checked_m != m) {
    if ((rc = ritz())) return rc;
    if (!fixed) {
      double h[2];
      CC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, st));
      CC_HIP(hipStreamSynchronize(st));
      theta = h[0];
      resid = h[1];
    }
  }
  // Ritz vector z = Q s, x = W^T z   (N-normalised because ||z|| = 1)
  lz_combine_kernel<<<(unsigned)((n + 15) / 16), 256, 0, st>>>(m, n, Q, s, t2, 1);
  CC_LAUNCH_CHECK();
  rc = cc_skinny_f64(st, n_env, 2, Wt, (int)d, t2, x_out);  // stream-ordered: no wait for it here
  if (rc) return rc;
  if (host_result) {
    host_result[0] = theta;   // NaN in the fixed mode: the Ritz value and residual stay on the device
    host_result[1] = resid;
    host_result[2] = (double)m;
  }
  return CC_OK;
}

// ---------------------------------------------------------------- Jacobi-Davidson pieces
namespace {
// out[j] = sum_i U[j][i] v[i] for j < k  (one block per basis vector, fixed-order tree)
__global__ void __launch_bounds__(256) jd_dots_kernel(int64_t n, const double* __restrict__ U, const double* __restrict__ v,
                                                      double* __restrict__ out, int stride_out) {
  __shared__ double red[4];
  const double t = block_dot256(n, U + (int64_t)blockIdx.x * n, v, red);
  if (threadIdx.x == 0) out[(int64_t)blockIdx.x * stride_out] = t;
}

// y = a*x + b*y with a, b read from device scalars (a = sa[0]*fa, b = sb ? sb[0]*fb : fb)
__global__ void cg_axpby_kernel(int64_t n, const double* __restrict__ sa, double fa, const double* __restrict__ x,
                                const double* __restrict__ sb, double fb, double* __restrict__ y) {
  const double a = (sa ? sa[0] : 1.0) * fa, b = (sb ? sb[0] : 1.0) * fb;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = a * x[i] + (b == 0.0 ? 0.0 : b * y[i]);
}

// ratio[0] = num[0] / den[0] (0 when den == 0)

// lowest eigenpair of the k x k pencil (Hs, Ns), k <= 32, single thread: Cholesky of Ns, cyclic Jacobi
// on L^-1 Hs L^-T, back-transform.  out[0] = value, vec[0..k) N-normalised coefficients.
// Sum of v over the 1024 threads of the workgroup in a fixed order (wave sums, added in wave order);
// every thread gets the result.
__device__ inline double cg_block_sum(double v, double* red) {
  v = cc_wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < 16; ++k) t += red[k];
  return t;
}

// One CG step of the projected correction equation after ap = (W Hlp W^T) p, in one 1024-thread
// workgroup:  ap -= rho p;  ap -= u (u . ap);  alpha = rr / (p . ap);  y += alpha p;  res -= alpha ap;
// rr' = res . res;  p = res + (rr' / rr) p;  rr = rr'.   Fixed-order reductions.
__global__ void __launch_bounds__(1024) cg_step_kernel(int64_t n, const double* __restrict__ rho_dev, const double* __restrict__ u,
                                                       double* __restrict__ ap, double* __restrict__ p,
                                                       double* __restrict__ y, double* __restrict__ res,
                                                       double* __restrict__ rr) {
  __shared__ double red[16];
  const double rho = rho_dev[0];
  double du = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const double a = ap[i] - rho * p[i];
    ap[i] = a;
    du += u[i] * a;
  }
  const double c = cg_block_sum(du, red);
  double pap = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const double a = ap[i] - c * u[i];
    ap[i] = a;
    pap += p[i] * a;
  }
  const double pap_sum = cg_block_sum(pap, red);
  // a converged (zero) residual or search direction ends the iteration with y unchanged, not a NaN
  const double alpha = (pap_sum != 0.0 && rr[0] != 0.0) ? rr[0] / pap_sum : 0.0;
  double rn = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    y[i] += alpha * p[i];
    const double r = res[i] - alpha * ap[i];
    res[i] = r;
    rn += r * r;
  }
  const double rr_new = cg_block_sum(rn, red);
  const double beta = rr[0] != 0.0 ? rr_new / rr[0] : 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) p[i] = res[i] + beta * p[i];
  __syncthreads();
  if (threadIdx.x == 0) rr[0] = rr_new;
}

// The same step with the vectors in registers (n <= 1024 R): one load round, three fixed-order sums,
// one store round (ap is scratch for the next step's operator product and is not written back).
template <int R>
__global__ void __launch_bounds__(1024) cg_step_reg_kernel(int64_t n, const double* __restrict__ rho_dev, const double* __restrict__ u,
                                                           const double* __restrict__ ap, double* __restrict__ p,
                                                           double* __restrict__ y, double* __restrict__ res,
                                                           double* __restrict__ rr) {
  __shared__ double red[16];
  const double rho = rho_dev[0], rr0 = rr[0];
  double a[R], pv[R], uv[R], yv[R], rv[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {  // clamped index: every load in bounds, the values masked in the sums
    const int64_t i = threadIdx.x + 1024 * k, ic = i < n ? i : 0;
    a[k] = ap[ic];
    pv[k] = p[ic];
    uv[k] = u[ic];
    yv[k] = y[ic];
    rv[k] = res[ic];
  }
  double du = 0.0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    a[k] -= rho * pv[k];
    if (threadIdx.x + 1024 * k < n) du += uv[k] * a[k];
  }
  const double c = cg_block_sum(du, red);
  double pap = 0.0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    a[k] -= c * uv[k];
    if (threadIdx.x + 1024 * k < n) pap += pv[k] * a[k];
  }
  const double pap_sum = cg_block_sum(pap, red);
  // a converged (zero) residual or search direction ends the iteration with y unchanged, not a NaN
  const double alpha = (pap_sum != 0.0 && rr0 != 0.0) ? rr0 / pap_sum : 0.0;
  double rn = 0.0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    yv[k] += alpha * pv[k];
    rv[k] -= alpha * a[k];
    if (threadIdx.x + 1024 * k < n) rn += rv[k] * rv[k];
  }
  const double rr_new = cg_block_sum(rn, red);
  const double beta = rr0 != 0.0 ? rr_new / rr0 : 0.0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int64_t i = threadIdx.x + 1024 * k;
    if (i < n) {
      p[i] = rv[k] + beta * pv[k];
      y[i] = yv[k];
      res[i] = rv[k];
    }
  }
  if (threadIdx.x == 0) rr[0] = rr_new;
}

// A CG step and the next product of a formed operator in one launch (n <= 512 V): every workgroup takes the whole
// step in registers -- the vectors come from the cache, and the loads of its matrix rows are in flight meanwhile --
// keeps the new direction in LDS and multiplies its four rows by it.  Workgroup 0 alone writes the vectors, into the
// other set of buffers, because the others may still be reading these.  The same step as cg_step_reg_kernel.  Bound by
// its three sums in a row: 7.8 us at D = 6, against 7.5 us for the step and 6.3 us for the product as two launches.
template <typename T, int NG, int U, int V>
__global__ void __launch_bounds__(FORMED_THREADS) cg_formed_kernel(FormedPlan f, const double* __restrict__ rho_dev,
                                                           const double* __restrict__ u, const double* __restrict__ ap,
                                                           const double* __restrict__ p, const double* __restrict__ res,
                                                           const double* __restrict__ rr, double* __restrict__ y,
                                                           double* __restrict__ ap_out, double* __restrict__ p_out,
                                                           double* __restrict__ res_out, double* __restrict__ rr_out) {
  __shared__ double pn[V * 512];
  __shared__ double red[16];
  const int n = 2 * f.n_env, row0 = blockIdx.x * FORMED_ROWS, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  FormedRows<T, NG, U> rows;
  rows.load(f, row0);
  const double rho = rho_dev[0], rr0 = rr[0];
  double a[V], pv[V], uv[V], rv[V];
#pragma unroll
  for (int k = 0; k < V; ++k) {   // past the end: clamped index, zeroed value (adds nothing to any sum)
    const int i = threadIdx.x + 512 * k, ic = i < n ? i : 0;
    const bool in = i < n;
    a[k] = in ? ap[ic] : 0.0;
    pv[k] = in ? p[ic] : 0.0;
    uv[k] = in ? u[ic] : 0.0;
    rv[k] = in ? res[ic] : 0.0;
  }
  auto block_sum = [&](double v) {   // fixed order: lanes, then waves; every thread gets it
    v = cc_wave_sum(v);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double t = red[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) t += red[w];
    return t;
  };
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    a[k] -= rho * pv[k];
    s += uv[k] * a[k];
  }
  const double c = block_sum(s);
  s = 0.0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    a[k] -= c * uv[k];
    s += pv[k] * a[k];
  }
  const double pap = block_sum(s);
  // a converged (zero) residual or search direction ends the iteration with y unchanged, not a NaN
  const double alpha = (pap != 0.0 && rr0 != 0.0) ? rr0 / pap : 0.0;
  s = 0.0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    rv[k] -= alpha * a[k];
    s += rv[k] * rv[k];
  }
  const double rr1 = block_sum(s), beta = rr0 != 0.0 ? rr1 / rr0 : 0.0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int i = threadIdx.x + 512 * k;
    const double q = rv[k] + beta * pv[k];
    pn[i] = q;
    if (blockIdx.x == 0 && i < n) {
      y[i] += alpha * pv[k];
      res_out[i] = rv[k];
      p_out[i] = q;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) rr_out[0] = rr1;
  __syncthreads();
  rows.apply(f, row0, [&](int col, int sp) { return pn[2 * col + sp]; }, red, ap_out);
}

template <typename T, int NG>
void cg_formed_launch(hipStream_t st, const FormedPlan& f, const double* rho, const double* u, const double* ap, const double* p,
                      const double* res, const double* rr, double* y, double* ap_out, double* p_out, double* res_out,
                      double* rr_out) {
  const unsigned grid = (unsigned)((f.n_env + FORMED_ROWS - 1) / FORMED_ROWS);
  if (f.n_env <= 256) cg_formed_kernel<T, NG, 2, 1><<<grid, FORMED_THREADS, 0, st>>>(f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out);
  else if (f.n_env <= 640) cg_formed_kernel<T, NG, 5, 3><<<grid, FORMED_THREADS, 0, st>>>(f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out);
  else cg_formed_kernel<T, NG, 11, 6><<<grid, FORMED_THREADS, 0, st>>>(f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out);
}

// Whether cg_formed_step serves the plan (FP32 matrices, one to four of them, at most 1408 rows).
bool cg_formed_serves(const FormedPlan& f) { return f.f32 && f.n_mats >= 1 && f.n_mats <= 4 && f.n_env <= 1408; }
int cg_formed_step(hipStream_t st, const FormedPlan& f, const double* rho, const double* u, const double* ap, const double* p,
                   const double* res, const double* rr, double* y, double* ap_out, double* p_out, double* res_out,
                   double* rr_out) {
  switch (f.n_mats) {
    case 1: cg_formed_launch<float, 1>(st, f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out); break;
    case 2: cg_formed_launch<float, 2>(st, f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out); break;
    case 3: cg_formed_launch<float, 3>(st, f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out); break;
    default: cg_formed_launch<float, 4>(st, f, rho, u, ap, p, res, rr, y, ap_out, p_out, res_out, rr_out); break;
  }
  CC_LAUNCH_CHECK();
  return CC_OK;
}

// One wave; the lanes take different rows (Cholesky), columns (the inverse factor), entries (the projected matrix) and
// disjoint rotations: a sweep of the Jacobi iteration is k - 1 rounds (k even; k rounds otherwise) of the circle method,
// each of up to k / 2 rotations, instead of k (k - 1) / 2 one after the other.  Bound by the chain of rounds: 20 us on
// average over a refined solve of eight passes, 33 us with single rotations and the matrices read from memory (k = 8, dense:
// 43 against 99 us; 32: 1.15 against 2.27 ms; 3: 12.0 against 10.6).
__global__ void __launch_bounds__(64) small_geneig_kernel(int k, const double* __restrict__ Hs, const double* __restrict__ Ns,
                                                          double* __restrict__ out, double* __restrict__ vec) {
  // the k x k work matrices live in LDS (no private scratch: concurrent launches on several
  // streams would each need a large scratch allocation)
  __shared__ double Lm[32][33], C[32][33], V[32][33], Li[32][33], hs[32][33], rot[2][16];
  __shared__ int pair[16];
  const int lane = threadIdx.x;
  for (int e = lane; e < k * k; e += 64) {
    const int i = e / k, j = e - i * k;
    Lm[i][j] = Ns[e];     // replaced column by column
    hs[i][j] = Hs[e];
    Li[i][j] = 0.0;
    V[i][j] = (i == j) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int j = 0; j < k; ++j) {
    double s = Lm[j][j];
    for (int c = 0; c < j; ++c) s -= Lm[j][c] * Lm[j][c];
    const double djj = sqrt(fmax(s, 1e-300));
    double t = 0.0;
    if (lane > j && lane < k) {
      t = Lm[lane][j];
      for (int c = 0; c < j; ++c) t -= Lm[lane][c] * Lm[j][c];
      t /= djj;
    }
    __syncthreads();
    if (lane == j) Lm[j][j] = djj;
    if (lane > j && lane < k) Lm[lane][j] = t;
    __syncthreads();
  }
  if (lane < k)
    for (int i = lane; i < k; ++i) {
      double v = (i == lane) ? 1.0 : 0.0;
      for (int t = lane; t < i; ++t) v -= Lm[i][t] * Li[t][lane];
      Li[i][lane] = v / Lm[i][i];
    }
  __syncthreads();
  for (int e = lane; e < k * k; e += 64) {
    const int i = e / k, j = e - i * k;
    double acc = 0.0;
    for (int a = 0; a <= i; ++a)
      for (int b = 0; b <= j; ++b) acc += Li[i][a] * hs[a][b] * Li[j][b];
    C[i][j] = acc;
  }
  __syncthreads();
  const int even = k + (k & 1), rounds = even - 1, pairs = even / 2;
  const int width = k <= 8 ? 8 : k <= 16 ? 16 : 32, l = lane & (width - 1), first = lane / width, stride = 64 / width;
  for (int sweep = 0; sweep < 50; ++sweep) {
    double off = 0.0;     // of the upper triangle, row by row
    if (lane < k)
      for (int j = lane + 1; j < k; ++j) off += C[lane][j] * C[lane][j];
    if (cc_wave_sum(off) < 1e-30) break;
    for (int r = 0; r < rounds; ++r) {
      if (lane < pairs) {
        // the last player stays, the others go round; with k odd the last is none
        const int x = lane ? (r + lane) % rounds : r, y = lane ? (r - lane + rounds) % rounds : even - 1;
        const int p = x < y ? x : y, q = x < y ? y : x;
        const double cpq = q < k ? C[p][q] : 0.0;
        double c = 1.0, sn = 0.0;
        if (cpq != 0.0) {
          const double th = (C[q][q] - C[p][p]) / (2.0 * cpq);
          const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
          c = 1.0 / sqrt(t * t + 1.0);
          sn = t * c;
        }
        rot[0][lane] = c;
        rot[1][lane] = sn;
        pair[lane] = p | (q < k ? q : p) << 8;     // p alone: no rotation
      }
      __syncthreads();
      for (int m = first; m < pairs; m += stride) {
        const int p = pair[m] & 255, q = pair[m] >> 8;
        const double c = rot[0][m], sn = rot[1][m];
        if (l < k && p != q) {
          const double a = C[l][p], b = C[l][q], va = V[l][p], vb = V[l][q];
          C[l][p] = c * a - sn * b;
          C[l][q] = sn * a + c * b;
          V[l][p] = c * va - sn * vb;
          V[l][q] = sn * va + c * vb;
        }
      }
      __syncthreads();
      for (int m = first; m < pairs; m += stride) {
        const int p = pair[m] & 255, q = pair[m] >> 8;
        const double c = rot[0][m], sn = rot[1][m];
        if (l < k && p != q) {
          const double a = C[p][l], b = C[q][l];
          C[p][l] = c * a - sn * b;
          C[q][l] = sn * a + c * b;
        }
      }
      __syncthreads();
    }
  }
  int best = 0;
  for (int i = 1; i < k; ++i)
    if (C[i][i] < C[best][best]) best = i;
  if (lane == 0) out[0] = C[best][best];
  if (lane < k) {  // coefficients = L^-T v
    double acc = 0.0;
    for (int j = lane; j < k; ++j) acc += Li[j][lane] * V[j][best];
    vec[lane] = acc;
  }
}

// out[m][i][j] = sum U_i V_j for V = V0 (m = 0) and V1 (m = 1): one block per entry, the sums of jd_dots_kernel.
__global__ void __launch_bounds__(256) jd_gram_kernel(int64_t n, const double* __restrict__ U, const double* __restrict__ V0,
                                                      const double* __restrict__ V1, double* __restrict__ out) {
  __shared__ double red[4];
  const double* V = blockIdx.z ? V1 : V0;
  const double t = block_dot256(n, U + (int64_t)blockIdx.x * n, V + (int64_t)blockIdx.y * n, red);
  if (threadIdx.x == 0) out[((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * gridDim.y + blockIdx.y] = t;
}

// x = U^T c, r = HU^T c - rho NU^T c, nx = NU^T c over k basis vectors (k <= 32).
__global__ void __launch_bounds__(256) jd_residual_kernel(int k, int64_t n, const double* __restrict__ U,
                                                          const double* __restrict__ HU, const double* __restrict__ NU,
                                                          const double* __restrict__ rho, const double* __restrict__ c,
                                                          double* __restrict__ x, double* __restrict__ r, double* __restrict__ nx) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  double tx = 0.0, th = 0.0, tn = 0.0;
  for (int j = 0; j < k; ++j) {
    const double cj = c[j];
    tx += cj * U[j * n + i];
    th += cj * HU[j * n + i];
    tn += cj * NU[j * n + i];
  }
  x[i] = tx;
  r[i] = th - rho[0] * tn;
  nx[i] = tn;
}
}  // namespace

extern "C" int cc_basis_dots_f64(void* stream, int k, int64_t n, const double* U, const double* v, double* out, int stride_out) {
  if (k <= 0) return CC_OK;
  jd_dots_kernel<<<k, 256, 0, cc_stream(stream)>>>(n, U, v, out, stride_out);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_basis_combine_f64(void* stream, int k, int64_t n, const double* U, const double* c, double* out) {
  lz_combine_kernel<<<(unsigned)((n + 15) / 16), 256, 0, cc_stream(stream)>>>(k, n, U, c, out, 1);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_small_geneig_f64(void* stream, int k, const double* Hs, const double* Ns, double* out, double* vec) {
  if (k < 1 || k > 32) { cc_set_last_error("small_geneig: 1 <= k <= 32"); return CC_ERR_ARG; }
  small_geneig_kernel<<<1, 64, 0, cc_stream(stream)>>>(k, Hs, Ns, out, vec);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_jd_project_f64(void* stream, int k, int64_t n, const double* U, const double* HU, const double* NU,
                                 double* gram, double* value, double* coef, double* x, double* r, double* nx) {
  if (k < 1 || k > 32 || n < 1) { cc_set_last_error("jd project: 1 <= k <= 32"); return CC_ERR_ARG; }
  hipStream_t st = cc_stream(stream);
  jd_gram_kernel<<<dim3((unsigned)k, (unsigned)k, 2), 256, 0, st>>>(n, U, HU, NU, gram);
  CC_LAUNCH_CHECK();
  small_geneig_kernel<<<1, 64, 0, st>>>(k, gram, gram + k * k, value, coef);
  CC_LAUNCH_CHECK();
  jd_residual_kernel<<<cc_blocks(n, 256), 256, 0, st>>>(k, n, U, HU, NU, value, coef, x, r, nx);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_jd_expand_f64(void* stream, int k, int64_t n, double* U, double* t, double* coef) {
  if (k < 1 || k > 32 || n < 1) { cc_set_last_error("jd expand: 1 <= k <= 32"); return CC_ERR_ARG; }
  hipStream_t st = cc_stream(stream);
  for (int pass = 0; pass < 2; ++pass) {
    lz_coeff_kernel<<<k, 256, 0, st>>>(n, U, t, coef, -1);
    CC_LAUNCH_CHECK();
    lz_combine_kernel<<<(unsigned)((n + 15) / 16), 256, 0, st>>>(k, n, U, coef, t, 0);
    CC_LAUNCH_CHECK();
  }
  lz_normalize_kernel<<<1, 1024, 0, st>>>(n, t, U + (int64_t)k * n, nullptr);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_jd_work_size(int64_t n, int64_t* out) {
  *out = 10 * n + 16;
  return CC_OK;
}

// Approximate solution of the projected correction equation
//   (I - u u^T)(W Hlp W^T - rho)(I - u u^T) y = -(I - u u^T) W r,  u = L^T x / |L^T x|,  t = W^T (I - u u^T) y
// by `iters` CG steps on the low-precision operator (all scalars on the device).
static int jd_correction(hipStream_t st, ApplyFn apply, const void* plan, int64_t n_env, int64_t d, const double* Lt,
                         const double* W, const double* Wt, const double* rho_dev, const double* x, const double* r,
                         int iters, double* work, double* t_out) {
  const int64_t n = n_env * d;
  double* u = work;
  double* y = u + n;
  double* res = y + n;
  double* p = res + n;
  double* ap = p + n;
  double* t1 = ap + n;
  double* t2 = t1 + n;
  double* tmp = t2 + n;
  double* sc = tmp + 2 * n;  // scalars: 0 uu, 1 rr, 2 rr_new, 3 pAp, 4 alpha, 5 beta, 6 dot
  const unsigned gb = cc_blocks(n, 256);
  int rc;
  Whitening wh{n_env, d, nullptr, Lt, W, Wt};
  // u = normalized L^T x
  rc = cc_skinny_f64(st, n_env, 2, Lt, (int)d, x, tmp);
  if (rc) return rc;
  lz_normalize_kernel<<<1, 1024, 0, st>>>(n, tmp, u, nullptr);
  CC_LAUNCH_CHECK();
  auto project = [&](double* v) -> int {  // v -= u (u . v)
    rc = cc_dot_f64(st, n, u, v, sc + 6);
    if (rc) return rc;
    cg_axpby_kernel<<<gb, 256, 0, st>>>(n, sc + 6, -1.0, u, nullptr, 1.0, v);
    CC_LAUNCH_CHECK();
    return CC_OK;
  };
  // res = -P W r ; p = res ; y = 0
  rc = cc_skinny_f64(st, n_env, 1, W, (int)d, r, res);
  if (rc) return rc;
  cg_axpby_kernel<<<gb, 256, 0, st>>>(n, nullptr, -1.0, res, nullptr, 0.0, res);
  CC_LAUNCH_CHECK();
  if ((rc = project(res))) return rc;
  rc = cc_fill_f64(st, n, 0.0, y);
  if (rc) return rc;
  cg_axpby_kernel<<<gb, 256, 0, st>>>(n, nullptr, 1.0, res, nullptr, 0.0, p);
  CC_LAUNCH_CHECK();
  rc = cc_dot_f64(st, n, res, res, sc + 1);
  if (rc) return rc;
  const FormedPlan* formed = apply == cc_internal_formed_apply ? static_cast<const FormedPlan*>(plan) : nullptr;
  if (formed && cg_formed_serves(*formed) && iters > 0) {
    // t1, t2 and tmp are free here: the second set of ap, res and p
    double *ap2 = t1, *res2 = t2, *p2 = tmp, *rr = sc + 1, *rr2 = sc + 2;
    if ((rc = apply(st, plan, p, ap))) return rc;
    for (int k = 0; k + 1 < iters; ++k) {
      if ((rc = cg_formed_step(st, *formed, rho_dev, u, ap, p, res, rr, y, ap2, p2, res2, rr2))) return rc;
      double* s;
      s = ap, ap = ap2, ap2 = s;
      s = res, res = res2, res2 = s;
      s = p, p = p2, p2 = s;
      s = rr, rr = rr2, rr2 = s;
    }
    if (n <= 4096) cg_step_reg_kernel<4><<<1, 1024, 0, st>>>(n, rho_dev, u, ap, p, y, res, rr);
    else cg_step_kernel<<<1, 1024, 0, st>>>(n, rho_dev, u, ap, p, y, res, rr);
    CC_LAUNCH_CHECK();
    iters = 0;
  }
  for (int k = 0; k < iters; ++k) {
    // ap = P (W H W^T - rho) p   (p is kept in the projected space)
    rc = op_whitened(st, apply, plan, wh, p, t1, t2, ap);
    if (rc) return rc;
    if (n <= 4096) cg_step_reg_kernel<4><<<1, 1024, 0, st>>>(n, rho_dev, u, ap, p, y, res, sc + 1);
    else cg_step_kernel<<<1, 1024, 0, st>>>(n, rho_dev, u, ap, p, y, res, sc + 1);
    CC_LAUNCH_CHECK();
  }
  if ((rc = project(y))) return rc;
  return cc_skinny_f64(st, n_env, 2, Wt, (int)d, y, t_out);                // t = W^T P y
}

extern "C" int cc_jd_correction_lp(void* stream, const void* lp_plan, int64_t n_env, int64_t d, const double* Lt,
                                   const double* W, const double* Wt, const double* rho_dev, const double* x,
                                   const double* r, int iters, double* work, double* t_out) {
  if (cc_internal_lp_n(lp_plan) != n_env * d) { cc_set_last_error("jd: operator size mismatch"); return CC_ERR_DIM; }
  return jd_correction(cc_stream(stream), cc_internal_lp_apply, lp_plan, n_env, d, Lt, W, Wt, rho_dev, x, r, iters, work, t_out);
}

extern "C" int cc_jd_correction_formed(void* stream, const void* formed_plan, int64_t n_env, int64_t d, const double* Lt,
                                       const double* W, const double* Wt, const double* rho_dev, const double* x,
                                       const double* r, int iters, double* work, double* t_out) {
  if (!formed_plan || cc_internal_formed_n(formed_plan) != n_env * d) { cc_set_last_error("jd: operator size mismatch"); return CC_ERR_DIM; }
  return jd_correction(cc_stream(stream), cc_internal_formed_apply, formed_plan, n_env, d, Lt, W, Wt, rho_dev, x, r, iters, work, t_out);
}

extern "C" int cc_normalize_f64(void* stream, int64_t n, const double* x, double* y) {
  if (n <= 0) return CC_OK;
  lz_normalize_kernel<<<1, 1024, 0, cc_stream(stream)>>>(n, x, y, nullptr);
  CC_LAUNCH_CHECK();
  return CC_OK;
}
