// Dense FP64 linear algebra for the solve: blocked Cholesky, lower-triangular inverse,
// skinny products with the whitening factor, Lanczos reorthogonalisation, and the
// lowest eigenpair of a symmetric tridiagonal matrix.
#include "cc_common.h"

namespace {
constexpr int CB = 64;  // Cholesky block size

// Lane l's value of v (the two 32-bit halves through readlane; l uniform).
__device__ inline double readlane_f64(double v, int l) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u & 0xffffffffull), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

constexpr int CH = 16, NCH = CB / CH;  // broadcast operands are read from LDS in chunks of CH

// r[j] -= s * src(j) for every j > K.  src is read in chunks of CH, one chunk ahead of its FMAs; the
// address of each chunk's loads depends (through an empty asm that takes the FMA results) on the chunk
// two back, so at most two chunks of loaded values are live whatever order the scheduler picks (left to
// itself it issues all 63 loads of a step first and spills).  K is a template parameter so that every
// index into r is a constant and r stays in registers.
template <int K, typename F>
__device__ __forceinline__ void tri_sweep(double (&r)[CB], double s, F src) {
  constexpr int c0 = (K + 1) / CH;
  if constexpr (c0 < NCH) {
    int tok = 0;
    double cur[CH], nxt[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) cur[u] = src(c0 * CH + u);
#pragma unroll
    for (int c = c0; c < NCH; ++c) {
#pragma unroll
      for (int u = 0; u < CH; ++u) nxt[u] = (c + 1 < NCH) ? src((c + 1) * CH + u + tok) : 0.0;
#pragma unroll
      for (int u = 0; u < CH; ++u)
        if (c * CH + u > K) r[c * CH + u] -= s * cur[u];
#pragma unroll
      for (int h = 0; h < CH; h += 8)
        __asm__ volatile("" : "+v"(tok) : "v"(r[c * CH + h + 0]), "v"(r[c * CH + h + 1]), "v"(r[c * CH + h + 2]),
                         "v"(r[c * CH + h + 3]), "v"(r[c * CH + h + 4]), "v"(r[c * CH + h + 5]), "v"(r[c * CH + h + 6]),
                         "v"(r[c * CH + h + 7]));
#pragma unroll
      for (int u = 0; u < CH; ++u) cur[u] = nxt[u];
    }
  }
}

// Cholesky and inverse of a 64 x 64 block in one right-looking sweep, row i of the block held by lane i
// as c[j].  Before step i, c[j] (j > i) holds the mirrored Schur complement S[j][i]; at step i that is
// sqrt(d_i) L[j][i], i.e. -d_i X[j][i] for X = L^-1 (d_i the pivot), and afterwards the forward
// substitution for column i of X applied to y = -d_i x has the same form as the Cholesky update.  So
// every row, whether it still factors (i > K) or already inverts (i < K), does
//   s_i = c[K] / sqrt(d_K),  c[K] = s_i,  c[j] -= s_i s_j  (j > K),
// and row K keeps c[K] = sqrt(d_K) with s_K = 0.  On exit c[j] = L[i][j] (j < i), c[i] = L[i][i] and
// c[j] = -d_i X[j][i] (j > i).  The symmetric updates keep c_i[j] == c_j[i] bit for bit (the same two
// factors meet in each FMA).  A non-positive pivot of a real row records its 1-based index in bad and is
// replaced by 1e-300.
// The block lies in the matrix-core accumulators of four waves, and the sweep goes in panels of 4 columns, the K of one
// MFMA (chol_panels): a panel passes through LDS, every wave factors it for itself, row i in its lane i, and each
// takes the panel's four updates of its accumulators as one product S S^T of the multipliers per 16 columns, the
// next panel's columns first.  One barrier per panel; no update is on the vector units but those inside a panel.
constexpr int PB = 4;
// Steps K .. of the panel at column `first`; the multipliers of step K are left in s[K].
template <int K>
__device__ __forceinline__ void chol_panel_steps(double (&c)[PB], double (&s)[PB], int first, int i, int kb, int& bad) {
  if constexpr (K < PB) {
    const int at = first + K;
    const double pivot = readlane_f64(c[K], at);
    const double d = fmax(pivot, 4.9406564584124654e-324);   // finite whatever the pivot; `bad` says so below
    // 1/sqrt(d): the hardware estimate y (relative error below 2^-22) and one step of third order in e = 1 - d y^2,
    // y + y e (1/2 + 3 e / 8), which leaves e^3 and rounding (within an ulp or so of the rounded quotient);
    // sqrt(d) = d / sqrt(d); far shorter than a correctly rounded square root followed by a division on this step's
    // critical path
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-d * y, y, 1.0);
    const double inv = fma(y * e, fma(0.375, e, 0.5), y);
    const double u = c[K] * inv;
    s[K] = (i == at) ? 0.0 : u;
    c[K] = (i == at) ? d * inv : s[K];
    // this step on the panel's later columns j (row j's multiplier from its lane)
#pragma unroll
    for (int j = K + 1; j < PB; ++j) c[j] -= s[K] * readlane_f64(u, first + j);
    chol_panel_steps<K + 1>(c, s, first, i, kb, bad);
    if (!(pivot > 0.0) && at < kb) bad = at + 1;     // the first of a panel last
  }
}

constexpr int CLD = CB + 2;   // LDS row of a 64 x 64 tile: 16 rows x 2 k of a half wave's MFMA operand hit all 64 banks
typedef double CholTile[CB * CLD];
typedef double CholPanel[CB * PB];
constexpr int CHOL_PANELS = 6;      // in LDS: two in turn that the waves share, one of each wave

// Panel P (columns PB P ..) to LDS
template <int P>
__device__ __forceinline__ void panel_publish(CholPanel* pan, const f64x4 (&acc)[4], int w, int lane) {
  if (((lane & 15) / PB) == P % 4)
#pragma unroll
    for (int r = 0; r < 4; ++r) pan[P & 1][(16 * w + 4 * r + (lane >> 4)) * PB + lane % PB] = acc[P / 4][r];
}

// Panel P, published, and the ones after it; row i's results to s.
template <int P>
__device__ __forceinline__ void chol_panels(f64x4 (&acc)[4], CholTile& s, CholPanel* pan, int w, int lane, int kb, int& bad) {
  if constexpr (P < CB / PB) {
    if (P * PB >= kb) return;
    __syncthreads();
    double c[PB], m[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) c[j] = pan[P & 1][lane * PB + j];
    int failed = 0;
    chol_panel_steps<0>(c, m, P * PB, lane, kb, failed);
    bad = bad ? bad : failed;
    double* own = pan[2 + w];     // read back by this wave alone
#pragma unroll
    for (int j = 0; j < PB; ++j) own[lane * PB + j] = m[j];
    if (w == P % 4)
#pragma unroll
      for (int j = 0; j < PB; ++j) s[lane * CLD + P * PB + j] = c[j];
    if constexpr (P + 1 < CB / PB) {
      const double a = -own[(16 * w + (lane & 15)) * PB + (lane >> 4)];
#pragma unroll
      for (int t = (P + 1) / 4; t < 4; ++t) {
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, own[(16 * t + (lane & 15)) * PB + (lane >> 4)], acc[t], 0, 0, 0);
        if (t == (P + 1) / 4) panel_publish<P + 1>(pan, acc, w, lane);
      }
    }
    chol_panels<P + 1>(acc, s, pan, w, lane, kb, bad);
  }
}

// Factors and inverts a diagonal block of kb rows held in the accumulators of four waves (wave w: row 16 w + 4 r +
// lane / 16, column 16 t + lane % 16 of acc[t][r]; symmetric, anything past kb): L (upper triangle zero) to A, L^-1
// to X, each with its leading dimension; returns the block's first failing pivot in every thread (1-based, 0: none).
// s and pan are scratch.  A dependent chain of 64 pivots.
__device__ __forceinline__ int chol_block(f64x4 (&acc)[4], CholTile& s, CholPanel* pan, int kb, double* __restrict__ A,
                                          int64_t lda, double* __restrict__ X, int64_t ldx) {
  const int i = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (kb < CB) {      // the identity past kb
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * w + 4 * r + (i >> 4), col = 16 * t + (i & 15);
        if (row >= kb || col >= kb) acc[t][r] = row == col ? 1.0 : 0.0;
      }
  }
  int bad = 0;  // first failing pivot, the same in every wave
  panel_publish<0>(pan, acc, w, i);
  chol_panels<0>(acc, s, pan, w, i, kb, bad);
  __syncthreads();
  // X[m][row] = -c_row[m] / d_row below the diagonal, 1 / L[row][row] on it
  const double xd = 1.0 / s[i * CLD + i], rd = -xd * xd;
  double l[16], x[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    l[r] = s[(w + 4 * r) * CLD + i];
    x[r] = s[i * CLD + w + 4 * r];
  }
  A += (int64_t)w * lda + i;
  X += (int64_t)w * ldx + i;
#pragma unroll
  for (int r = 0; r < 16; ++r, A += 4 * lda, X += 4 * ldx) {
    const int m = w + 4 * r;
    if (m < kb && i < kb) {
      *A = (i <= m) ? l[r] : 0.0;
      *X = (m > i) ? x[r] * rd : (m == i ? xd : 0.0);
    }
  }
  return bad;
}

// Tiles in the accumulators of four waves: row 16 w + lane / 16 + 4 r, column 16 t + lane % 16 of acc[t][r].  Every
// access of a thread is one address that advances by four rows, clamped at the edge: a 64-bit product per element costs
// more than the load (33000 cycles for the tiles of a step, 6000 with advancing addresses).
// The 64 x 64 tile at p, rows x cols of it, zero past them.
__device__ __forceinline__ void tile_to_acc(f64x4 (&acc)[4], const double* p, int64_t ld, int rows, int cols, int w, int lane) {
  const int i0 = 16 * w + (lane >> 4), j0 = lane & 15;
  p += (int64_t)(i0 < rows ? i0 : rows - 1) * ld;
  int j[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) j[t] = j0 + 16 * t < cols ? j0 + 16 * t : cols - 1;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t][r] = p[j[t]];
    p += i0 + 4 * (r + 1) < rows ? 4 * ld : 0;
  }
  if (rows < CB || cols < CB) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = (i0 + 4 * r < rows && j0 + 16 * t < cols) ? acc[t][r] : 0.0;
  }
}
// The same for a symmetric tile of kb rows whose lower triangle is read.
__device__ __forceinline__ void tile_to_acc_lower(f64x4 (&acc)[4], const double* p, int64_t ld, int kb, int w, int lane) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * w + 4 * r + (lane >> 4), j = 16 * t + (lane & 15);
      const int row = i > j ? i : j, col = i > j ? j : i;
      acc[t][r] = p[(int64_t)(row < kb ? row : kb - 1) * ld + (col < kb ? col : kb - 1)];
    }
}
__device__ __forceinline__ void tile_write_acc(const f64x4 (&acc)[4], double* p, int64_t ld, int rows, int cols, int w, int lane) {
  const int i0 = 16 * w + (lane >> 4), j0 = lane & 15;
  p += (int64_t)i0 * ld + j0;
#pragma unroll
  for (int r = 0; r < 4; ++r, p += 4 * ld)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (i0 + 4 * r < rows && j0 + 16 * t < cols) p[16 * t] = acc[t][r];
}

// Cholesky and inverse of one diagonal block of at most 64 x 64 rows (lower triangle read): A's block at (k0, k0) is
// replaced by L with its upper triangle zeroed, X receives L^-1, info the first non-positive pivot (1-based, global
// index; `begin`: info is set, else only where no earlier block failed).
__global__ void __launch_bounds__(256) chol_leaf_kernel(int64_t lda, int64_t k0, int kb, double* __restrict__ A,
                                                        double* __restrict__ X, int64_t ldx, int* __restrict__ info, int begin) {
  __shared__ CholTile s;
  __shared__ __attribute__((aligned(16))) CholPanel pan[CHOL_PANELS];
  double* Ak = A + k0 * lda + k0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  f64x4 acc[4];
  tile_to_acc_lower(acc, Ak, lda, kb, w, lane);
  const int bad = chol_block(acc, s, pan, kb, Ak, lda, X, ldx);
  if (threadIdx.x == 0 && (begin || (*info == 0 && bad))) *info = bad ? (int)(k0 + bad) : 0;
}

// A 64 x 64 tile at p in registers (element r of a thread: row tid / 64 + 4 r, column tid % 64; `trans`: the tile's
// transpose), zero past `rows` and `cols` of the tile as stored; then to LDS.
__device__ __forceinline__ void tile_load(double (&v)[16], const double* __restrict__ p, int64_t ld, int rows, int cols, int tid) {
  const int c = tid & 63, r0 = tid >> 6;
  p += (int64_t)(r0 < rows ? r0 : rows - 1) * ld + (c < cols ? c : cols - 1);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    v[r] = *p;
    p += r0 + 4 * (r + 1) < rows ? 4 * ld : 0;
  }
  if (rows < CB || cols < CB) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = (r0 + 4 * r < rows && c < cols) ? v[r] : 0.0;
  }
}
template <bool TRANS>
__device__ __forceinline__ void tile_store(CholTile& s, const double (&v)[16], int tid) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = (tid >> 6) + 4 * r, c = tid & 63;
    s[TRANS ? c * CLD + row : row * CLD + c] = v[r];
  }
}

// acc = S T^T of two tiles in LDS; wave w takes rows 16 w .. 16 w + 15.  LOWER: T is lower triangular, so column tile t
// sums over its first 16 (t + 1) indices only.
template <bool LOWER>
__device__ __forceinline__ void tile_product(f64x4 (&acc)[4], const CholTile& S, const CholTile& T, int w, int lane) {
  const int row = lane & 15, k4 = lane >> 4;
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kk = 0; kk < CB; kk += 4) {
    const double a = S[(16 * w + row) * CLD + kk + k4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (!LOWER || kk < 16 * (t + 1))
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, T[(16 * t + row) * CLD + kk + k4], acc[t], 0, 0, 0);
  }
}
__device__ __forceinline__ void tile_from_acc(CholTile& s, const f64x4 (&acc)[4], int w, int lane) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) s[(16 * w + 4 * r + (lane >> 4)) * CLD + 16 * t + (lane & 15)] = acc[t][r];
}
// s transposed to the 64 x 64 tile at p (rows x cols of it exist)
__device__ __forceinline__ void tile_write_transposed(const CholTile& s, double* __restrict__ p, int64_t ld, int rows, int cols, int tid) {
  const int c = tid & 63;
  double v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = s[c * CLD + (tid >> 6) + 4 * r];
  p += (int64_t)(tid >> 6) * ld + c;
#pragma unroll
  for (int r = 0; r < 16; ++r, p += 4 * ld)
    if (c < cols && (tid >> 6) + 4 * r < rows) *p = v[r];
}

// Step k of A = L L^T with X = L^-1, in blocks of 64, once block k of the diagonal is factored (L_kk, X_kk stored).
// The rows of A are extended by those of the identity, which elimination turns into L^-T:
//   [A; 1] L^-T = [L; L^-T].
// Row blocks M_s of the extended matrix (s > k of A, s <= k of the identity, whose parts so far are held in X's upper
// triangle) and column blocks i > k: M(s, i) -= (M(s, k) X_kk^T) (A(i, k) X_kk^T)^T.  Each workgroup updates one such
// tile and makes both factors itself, so a step is one launch, and the workgroup of the next diagonal block goes on to
// factor it: the chain per step is two tile products and a 64 x 64 factorization.  Finished column blocks go where nothing
// is read any more: L(i, k)^T to A's upper triangle, X(k, j) to X's lower one; chol_finish_kernel moves the former
// into place.
// Latency-bound, 17 us a step: 9 us for the 64 pivots (335 cycles each), 3.2 us for the two products on one CU, 2.5 us
// for the loads (10 us with a 64-bit product per element's address), 1.3 us for the results.  n = 256 / 625 / 1296 /
// 2592 / 4096: 74 / 181 / 380 / 1070 / 2920 us, against 107 / 311 / 757 / 1940 / 4160 us for a recursion with leaves of
// 128 rows on one workgroup (39 us each), four products around each and a copy.  The three products per tile
// instead of one cost nothing while a step's tiles fit the chip (n <= 1400), and less than the recursion's small
// products beyond.
__global__ void __launch_bounds__(256) chol_step_kernel(int64_t n, int k, int blocks, double* __restrict__ A, double* __restrict__ X,
                                                        int* __restrict__ info) {
  __shared__ __attribute__((aligned(16))) CholTile sa;
  __shared__ CholTile sx;
  CholPanel* pan = reinterpret_cast<CholPanel*>(sa);    // sa is free once the next diagonal block is factored
  static_assert(CHOL_PANELS * CB * PB <= CB * CLD, "the panels in one tile");
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // tiles in order: A's lower triangle of the m blocks left (the next diagonal block first), the identity's rows
  // (j <= k) x the m columns, then the finished blocks X(k, j), j < k
  const int m = blocks - 1 - k, lower = m * (m + 1) / 2;
  int b = blockIdx.x, s = 0, i = 0, kind = 0;   // 0: A's rows, 1: the identity's, 2: finished X(k, s)
  if (b < lower) {
    while (b > s) b -= ++s;   // row s, column b <= s
    i = k + 1 + b;
    s += k + 1;
  } else if ((b -= lower) < m * (k + 1)) {
    kind = 1;
    s = b / m;
    i = k + 1 + b % m;
  } else {
    kind = 2;
    s = b - m * (k + 1);
  }
  const int64_t k0 = (int64_t)k * CB, s0 = (int64_t)s * CB, i0 = (int64_t)i * CB;
  auto left = [&](int64_t at) { return (int)(n - at < CB ? n - at : CB); };
  const int kb = left(k0), sb = left(s0), ib = kind == 2 ? 0 : left(i0);
  const bool diagonal = kind == 0 && s == i;
  const double* Xk = X + k0 * n + k0;
  double vx[16], vi[16], vs[16];
  tile_load(vx, Xk, n, kb, kb, tid);
  if (kind != 2) tile_load(vi, A + i0 * n + k0, n, ib, kb, tid);
  if (kind == 0) { if (!diagonal) tile_load(vs, A + s0 * n + k0, n, sb, kb, tid); }
  else if (s != k) tile_load(vs, X + s0 * n + k0, n, sb, kb, tid);
  // the tile itself, as the products leave it (row 16 w + 4 r + lane / 16, column 16 t + lane % 16)
  double* M = (kind == 0 ? A : X) + s0 * n + i0;
  f64x4 out[4];
  const bool fresh = kind == 1 && s == k;      // the identity's row k: nothing there yet
  if (diagonal && k == 0) {
    tile_to_acc_lower(out, M, n, sb, w, lane);    // the caller's; written back with both triangles
  } else if (kind != 2 && !fresh) {
    tile_to_acc(out, M, n, sb, ib, w, lane);
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t) out[t] = (f64x4){0.0, 0.0, 0.0, 0.0};
  }
  tile_store<false>(sx, vx, tid);
  if (kind != 2) tile_store<false>(sa, vi, tid);
  else tile_store<false>(sa, vs, tid);
  __syncthreads();
  f64x4 p[4], q[4];
  tile_product<true>(p, sa, sx, w, lane);      // L(i, k); kind 2: the finished block, X(k, s)^T
  if (kind == 2) {
    __syncthreads();
    tile_from_acc(sa, p, w, lane);
    __syncthreads();
    tile_write_transposed(sa, X + k0 * n + s0, n, kb, sb, tid);
    return;
  }
  if (!diagonal && !fresh) {
    __syncthreads();
    tile_store<false>(sa, vs, tid);
    __syncthreads();
    tile_product<true>(q, sa, sx, w, lane);
  }
  __syncthreads();
  tile_from_acc(sa, p, w, lane);
  if (fresh) tile_store<true>(sx, vx, tid);    // X_kk^T
  else if (!diagonal) tile_from_acc(sx, q, w, lane);
  __syncthreads();
  f64x4 d[4];
  tile_product<false>(d, diagonal ? sa : sx, sa, w, lane);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) out[t][r] -= d[t][r];
  if (diagonal && i == k + 1) {
    __syncthreads();   // sa has been read
    const int bad = chol_block(out, sx, pan, ib, M, n, X + i0 * n + i0, n);
    if (tid == 0 && bad && *info == 0) *info = (int)(i0 + bad);
    return;
  }
  tile_write_acc(out, M, n, sb, ib, w, lane);
  if (fresh) tile_write_transposed(sa, A + k0 * n + i0, n, kb, ib, tid);   // L(i, k)^T
}

// L's blocks below the diagonal from A's upper triangle, whose blocks and X's are then zero.  32 x 32 tiles; those of
// the diagonal 64 x 64 blocks are in place.
__global__ void __launch_bounds__(256) chol_finish_kernel(int64_t n, double* __restrict__ A, double* __restrict__ X) {
  __shared__ double tile[32][33];
  if (blockIdx.x / 2 <= blockIdx.y / 2) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t c = (int64_t)blockIdx.x * 32, r = (int64_t)blockIdx.y * 32;
#pragma unroll
  for (int k = 0; k < 32; k += 8)
    if (c + tx < n) {   // rows r .. r + 31 lie above c, so they exist
      const int64_t at = (r + ty + k) * n + c + tx;
      tile[ty + k][tx] = A[at];
      A[at] = X[at] = 0.0;
    }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 32; k += 8)
    if (c + ty + k < n) A[(c + ty + k) * n + r + tx] = tile[tx][ty + k];
}

// Column sweep of L x = e_j, steps Q..CB-1: x[Q] *= 1/L[Q][Q], then x[m] -= L[m][Q] x[Q] for m > Q.
template <int Q>
__device__ __forceinline__ void inv_steps(double (&x)[CB], const double (*Ls)[CB + 1], const double* rdiag) {
  if constexpr (Q < CB) {
    const double xq = x[Q] * rdiag[Q];
    x[Q] = xq;
    tri_sweep<Q>(x, xq, [&](int m) { return Ls[m][Q]; });
    inv_steps<Q + 1>(x, Ls, rdiag);
  }
}

// Inverse of one lower-triangular diagonal block of at most 64 x 64 on one wave: the block of A at (k0, k0)
// holds L (rows >= kb padded with the identity); lane j solves L x = e_j with L broadcast from LDS and
// writes column j of L^-1 into X at (x0, x0).
__global__ void __launch_bounds__(64) tri_leaf_kernel(int64_t lda, int64_t k0, int kb, const double* __restrict__ A,
                                                      double* __restrict__ X, int64_t ldx, int64_t x0) {
  __shared__ double Ls[CB][CB + 1];
  __shared__ double rdiag[CB];
  const int i = threadIdx.x;
  const int ic = i < kb ? i : 0;  // clamped: every load below is in bounds
  double r[CB];
  const double* arow = A + (k0 + ic) * lda + k0;
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const double v = arow[j < kb ? j : 0];
    r[j] = (i < kb && j <= i) ? v : (i == j ? 1.0 : 0.0);
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) Ls[i][j] = (j <= i) ? r[j] : 0.0;
  __syncthreads();
  rdiag[i] = 1.0 / Ls[i][i];
  __syncthreads();
  double x[CB];
#pragma unroll
  for (int m = 0; m < CB; ++m) x[m] = (m == i) ? 1.0 : 0.0;
  inv_steps<0>(x, Ls, rdiag);
#pragma unroll
  for (int m = 0; m < CB; ++m)  // unrolled: x stays in registers
    if (i < kb && m < kb) X[(x0 + m) * ldx + x0 + i] = x[m];
}

// dst[r][c] = src[r][c] for an rows x cols block with leading dimensions lds / ldd.
__global__ void copy2d_kernel(int64_t rows, int64_t cols, const double* __restrict__ src, int64_t lds,
                              double* __restrict__ dst, int64_t ldd) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < rows * cols; e += (int64_t)gridDim.x * blockDim.x)
    dst[(e / cols) * ldd + e % cols] = src[(e / cols) * lds + e % cols];
}

// Zero the strict upper triangle.
__global__ void zero_upper_kernel(int64_t n, double* __restrict__ A) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += (int64_t)gridDim.x * blockDim.x)
    if (e % n > e / n) A[e] = 0.0;
}

// Y[i][s] = sum_k M[i][k] X[k][s] for k in [kbeg(i), kend(i)) with M row-major n x n,
// tri: 0 full, 1 lower (k <= i), 2 upper (k >= i).  Two waves per output row, each summing one half of
// the row's range (half the serial load rounds of one wave per row); the halves are added in order.
template <int NR>
__global__ void __launch_bounds__(256) skinny_kernel(int64_t n, int tri, const double* __restrict__ M,
                                                     const double* __restrict__ X, double* __restrict__ Y) {
  __shared__ double part[4][NR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = wave & 1;
  const int64_t row = (int64_t)blockIdx.x * 2 + (wave >> 1);
  double acc[NR];
#pragma unroll
  for (int s = 0; s < NR; ++s) acc[s] = 0.0;
  if (row < n) {
    const int64_t rb = (tri == 2) ? row : 0, re = (tri == 1) ? row + 1 : n, mid = rb + (re - rb) / 2;
    const int64_t kb = half ? mid : rb, ke = half ? re : mid;
    const double* mr = M + row * n;
    int64_t k = kb + lane;
    for (; k + 192 < ke; k += 256) {  // four independent row loads in flight per lane
      const double m0 = mr[k], m1 = mr[k + 64], m2 = mr[k + 128], m3 = mr[k + 192];
#pragma unroll
      for (int s = 0; s < NR; ++s)
        acc[s] += m0 * X[k * NR + s] + m1 * X[(k + 64) * NR + s] + m2 * X[(k + 128) * NR + s] + m3 * X[(k + 192) * NR + s];
    }
    for (; k < ke; k += 64) {
      const double m = mr[k];
#pragma unroll
      for (int s = 0; s < NR; ++s) acc[s] += m * X[k * NR + s];
    }
  }
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    double v = acc[s];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    acc[s] = v;
  }
  if (lane == 0) {
#pragma unroll
    for (int s = 0; s < NR; ++s) part[wave][s] = acc[s];
  }
  __syncthreads();
  if (lane == 0 && half == 0 && row < n) {
#pragma unroll
    for (int s = 0; s < NR; ++s) Y[row * NR + s] = part[wave][s] + part[wave + 1][s];
  }
}

// B = A^T for n x n row-major matrices: one 32 x 32 tile per workgroup (32 x 8 threads), read and written
// along rows through an LDS tile padded to 33 columns.
__global__ void __launch_bounds__(256) transpose_kernel(int64_t n, const double* __restrict__ A, double* __restrict__ B) {
  __shared__ double tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
#pragma unroll
  for (int k = 0; k < 32; k += 8) {
    const int64_t r = r0 + ty + k, c = c0 + tx;
    if (r < n && c < n) tile[ty + k][tx] = A[r * n + c];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 32; k += 8) {
    const int64_t r = c0 + ty + k, c = r0 + tx;   // B[r][c] = A[c][r]
    if (r < n && c < n) B[r * n + c] = tile[tx][ty + k];
  }
}

// Split of a diagonal range of sz > CB rows at a block boundary near its middle.
inline int64_t split_rows(int64_t sz) { return ((sz + CB - 1) / CB / 2) * CB; }

// Recursive inverse of the lower-triangular range [off, off + sz) of L: X11, X22 recursively, then
// X21 = -X22 (L21 X11); leaves are tri_leaf_kernel.
int trtri_rec(void* stream, int64_t n, int64_t off, int64_t sz, const double* L, double* X, double* tmp) {
  hipStream_t st = cc_stream(stream);
  if (sz <= CB) {
    tri_leaf_kernel<<<1, 64, 0, st>>>(n, off, (int)sz, L, X, n, off);
    CC_LAUNCH_CHECK();
    return CC_OK;
  }
  const int64_t n1 = split_rows(sz), n2 = sz - n1;
  int rc = trtri_rec(stream, n, off, n1, L, X, tmp);
  if (rc) return rc;
  rc = trtri_rec(stream, n, off + n1, n2, L, X, tmp);
  if (rc) return rc;
  const double* L21 = L + (off + n1) * n + off;
  const double* X11 = X + off * n + off;
  double* X21 = X + (off + n1) * n + off;
  rc = cc_gemm_f64(stream, 1, n2, n1, n1, 1.0, L21, 0, n, 1, X11, 0, n, 1, 0.0, tmp, 0, n1, 1);
  if (rc) return rc;
  return cc_gemm_f64(stream, 1, n2, n1, n2, -1.0, X21 + n1, 0, n, 1, tmp, 0, n1, 1, 0.0, X21, 0, n, 1);
}
}  // namespace

extern "C" int cc_linalg_work_size(int64_t n, int64_t* out) {
  const int64_t blocked = (int64_t)CB * CB + (int64_t)CB * n, recursive = n * n / 4 + 1;
  *out = blocked > recursive ? blocked : recursive;
  return CC_OK;
}

// Right-looking blocked Cholesky: diagonal block factored and inverted by chol_leaf_kernel, the panel as a GEMM
// against that inverse, the trailing update as a GEMM.
extern "C" int cc_cholesky_f64(void* stream, int64_t n, double* A, int* info_dev, double* work) {
  if (n <= 0) { cc_set_last_error("cholesky: n must be positive"); return CC_ERR_ARG; }
  hipStream_t st = cc_stream(stream);
  double* dinv = work;
  double* tmp = work + CB * CB;
  for (int64_t k0 = 0; k0 < n; k0 += CB) {
    int kb = (int)((n - k0) < CB ? (n - k0) : CB);
    chol_leaf_kernel<<<1, 256, 0, st>>>(n, k0, kb, A, dinv, kb, info_dev, k0 == 0);
    CC_LAUNCH_CHECK();
    int64_t rest = n - k0 - kb;
    if (rest > 0) {
      double* Pn = A + (k0 + kb) * n + k0;
      // tmp = A_panel * Linv_kk^T ; A_panel = tmp
      int rc = cc_gemm_f64(stream, 1, rest, kb, kb, 1.0, Pn, 0, n, 1, dinv, 0, 1, kb, 0.0, tmp, 0, kb, 1);
      if (rc) return rc;
      copy2d_kernel<<<cc_blocks(rest * kb, 256), 256, 0, st>>>(rest, kb, tmp, kb, Pn, n);
      CC_LAUNCH_CHECK();
      double* T = A + (k0 + kb) * n + (k0 + kb);
      rc = cc_gemm_f64(stream, 1, rest, rest, kb, -1.0, Pn, 0, n, 1, Pn, 0, 1, n, 1.0, T, 0, n, 1);
      if (rc) return rc;
    }
  }
  zero_upper_kernel<<<cc_blocks(n * n, 256), 256, 0, st>>>(n, A);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

// A = L L^T in place (upper zeroed) and X = L^-1 (upper zero) in one pass over the block columns (chol_step_kernel).
extern "C" int cc_cholesky_inverse_f64(void* stream, int64_t n, double* A, double* X, int* info_dev, double* work) {
  (void)work;
  if (n <= 0) { cc_set_last_error("cholesky_inverse: n must be positive"); return CC_ERR_ARG; }
  const int64_t blocks = (n + CB - 1) / CB;
  if (blocks > 32767) { cc_set_last_error("cholesky_inverse: matrix too large"); return CC_ERR_UNSUPPORTED; }
  hipStream_t st = cc_stream(stream);
  chol_leaf_kernel<<<1, 256, 0, st>>>(n, 0, (int)(n < CB ? n : CB), A, X, n, info_dev, 1);
  CC_LAUNCH_CHECK();
  if (blocks == 1) return CC_OK;
  for (int k = 0; k < (int)blocks; ++k) {
    const int64_t m = blocks - 1 - k, tiles = m * (m + 1) / 2 + m * (k + 1) + k;
    chol_step_kernel<<<(unsigned)tiles, 256, 0, st>>>(n, k, (int)blocks, A, X, info_dev);
    CC_LAUNCH_CHECK();
  }
  const unsigned t32 = (unsigned)((n + 31) / 32);
  chol_finish_kernel<<<dim3(t32, t32), 256, 0, st>>>(n, A, X);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

// X = L^-1 for lower-triangular L, recursively (leaves on one wave each, GEMMs for the off-diagonal blocks).
extern "C" int cc_trtri_lower_f64(void* stream, int64_t n, const double* L, double* X, double* work) {
  if (n <= 0) { cc_set_last_error("trtri: n must be positive"); return CC_ERR_ARG; }
  int rc = cc_fill_f64(stream, n * n, 0.0, X);
  if (rc) return rc;
  return trtri_rec(stream, n, 0, n, L, X, work);
}

extern "C" int cc_transpose_f64(void* stream, int64_t n, const double* A, double* B) {
  if (n <= 0) return CC_OK;
  const int64_t tiles = (n + 31) / 32;
  if (tiles > 65535) { cc_set_last_error("transpose: n too large for one launch"); return CC_ERR_UNSUPPORTED; }
  transpose_kernel<<<dim3((unsigned)tiles, (unsigned)tiles), 256, 0, cc_stream(stream)>>>(n, A, B);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_skinny_f64(void* stream, int64_t n, int tri, const double* M, int nrhs, const double* X, double* Y) {
  if (n <= 0) return CC_OK;
  unsigned g = (unsigned)((n + 1) / 2);
  hipStream_t st = cc_stream(stream);
  switch (nrhs) {
    case 1: skinny_kernel<1><<<g, 256, 0, st>>>(n, tri, M, X, Y); break;
    case 2: skinny_kernel<2><<<g, 256, 0, st>>>(n, tri, M, X, Y); break;
    case 3: skinny_kernel<3><<<g, 256, 0, st>>>(n, tri, M, X, Y); break;
    case 4: skinny_kernel<4><<<g, 256, 0, st>>>(n, tri, M, X, Y); break;
    default: cc_set_last_error("skinny: nrhs must be 1..4"); return CC_ERR_UNSUPPORTED;
  }
  CC_LAUNCH_CHECK();
  return CC_OK;
}

// ---- relaxOver's restart (one native call; the scalars stay on the device) ---------------------------------------
namespace {
constexpr int RELAX_MAX_K = 16;
struct RelaxCoef {
  double c[RELAX_MAX_K];
};
// x . y on the whole workgroup, summed as cc_dot_f64 sums it
__device__ double block_dot(int64_t n, const double* x, const double* y, double* red) {
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) acc += x[i] * y[i];
  __syncthreads();
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  return red[0];
}
// v = sum_j c[j] basis[j], scaled to unit norm, into basis[0]
__global__ void __launch_bounds__(1024) relax_combine_kernel(int64_t n, int count, const RelaxCoef coef, double* basis,
                                                             double* tmp, double* out) {
  __shared__ double red[1024];
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    double v = 0.0;
    for (int j = 0; j < count; ++j) v += coef.c[j] * basis[j * n + i];
    tmp[i] = v;
  }
  __syncthreads();
  const double s = 1.0 / sqrt(block_dot(n, tmp, tmp, red));
  for (int64_t i = threadIdx.x; i < n; i += 1024) basis[i] = s * tmp[i];
  if (threadIdx.x == 0) out[0] = 0.0;   // vectors of the basis, once it has ended
}
// basis[m] = mbasis[m - 1] orthogonalized against basis[0..m-1] (the coefficients first, then the subtractions), scaled;
// zero, and out[0] = m, where nothing is left of it
__global__ void __launch_bounds__(1024) relax_extend_kernel(int64_t n, int m, double* basis, const double* mbasis,
                                                            double* out) {
  __shared__ double red[1024];
  double* w = basis + m * n;
  const double* y = mbasis + (m - 1) * n;
  double c[RELAX_MAX_K];
#pragma unroll
  for (int j = 0; j < RELAX_MAX_K; ++j)
    if (j < m) c[j] = block_dot(n, basis + j * n, y, red);
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    double v = y[i];
#pragma unroll
    for (int j = 0; j < RELAX_MAX_K; ++j)
      if (j < m) v += -c[j] * basis[j * n + i];
    w[i] = v;
  }
  __syncthreads();
  const double nn = block_dot(n, w, w, red), norm = sqrt(nn > 0.0 ? nn : 0.0);
  const bool ended = norm <= 1e-14 || out[0] > 0.0;   // a vector after the basis has ended stays zero
  const double s = 1.0 / norm;
  __syncthreads();
  for (int64_t i = threadIdx.x; i < n; i += 1024) w[i] = ended ? 0.0 : s * w[i];
  if (threadIdx.x == 0 && ended && !(out[0] > 0.0)) out[0] = m;
}
// out[1 + i k + j] = basis[i] . mbasis[j]; the number of vectors where the basis did not end before
__global__ void __launch_bounds__(1024) relax_products_kernel(int64_t n, int k, const double* basis, const double* mbasis,
                                                              double* out) {
  __shared__ double red[1024];
  const int i = blockIdx.x / k, j = blockIdx.x % k;
  const double v = block_dot(n, basis + i * n, mbasis + j * n, red);
  if (threadIdx.x == 0) {
    out[1 + blockIdx.x] = v;
    if (blockIdx.x == 0 && !(out[0] > 0.0)) out[0] = k;
  }
}
}  // namespace

// A restart is a chain of small matrix-vector products and reductions; what it costs is launches and, with a host that
// reads every scalar, a synchronization per scalar: at n = 32, k = 3 (9 products, 21 dots) 0.50 ms from Python and
// 0.06 ms here.
extern "C" int cc_relax_krylov_f64(void* stream, int64_t n, int k, const double* H, const double* W, const double* Wt,
                                   int count, const double* coef, int last, double* basis, double* mbasis, double* tmp,
                                   double* out) {
  if (n < 1 || k < 1 || k > RELAX_MAX_K || count < 1 || count > k) { cc_set_last_error("relax: bad sizes"); return CC_ERR_ARG; }
  hipStream_t st = cc_stream(stream);
  RelaxCoef c = {};
  for (int j = 0; j < count; ++j) c.c[j] = coef[j];
  relax_combine_kernel<<<1, 1024, 0, st>>>(n, count, c, basis, tmp, out);
  CC_LAUNCH_CHECK();
  for (int i = 0; i < (last ? 1 : k); ++i) {
    const double* x = basis + i * n;
    double* y = mbasis + i * n;
    int rc;
    if (!W) {
      rc = cc_skinny_f64(stream, n, 0, H, 1, x, y);
    } else {
      rc = cc_skinny_f64(stream, n, 0, H, 1, x, tmp);
      if (!rc && Wt) rc = cc_skinny_f64(stream, n, 1, W, 1, tmp, tmp + n);
      if (!rc) rc = Wt ? cc_skinny_f64(stream, n, 2, Wt, 1, tmp + n, y) : cc_skinny_f64(stream, n, 0, W, 1, tmp, y);
    }
    if (rc) return rc;
    if (!last && i + 1 < k) {
      relax_extend_kernel<<<1, 1024, 0, st>>>(n, i + 1, basis, mbasis, out);
      CC_LAUNCH_CHECK();
    }
  }
  const int rows = last ? 1 : k;
  relax_products_kernel<<<(unsigned)(rows * rows), 1024, 0, st>>>(n, rows, basis, mbasis, out);
  CC_LAUNCH_CHECK();
  return CC_OK;
}
