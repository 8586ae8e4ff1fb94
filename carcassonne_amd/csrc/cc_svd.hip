// Thin SVD by one-sided Jacobi (Hestenes) with the round-robin parallel ordering:
// one 1024-thread workgroup per matrix, one wave per disjoint column pair per round.
// The columns of A and V live in LDS when (m + n) n <= 8192 doubles (64 KiB, every Gram matrix of a
// bond up to 64 and the small normalizations), otherwise in global memory (`work`), so m is unbounded;
// n <= 256.  Both placements do the same arithmetic in the same order.
#include "cc_common.h"

namespace {
constexpr int SVD_THREADS = 1024;
constexpr int SVD_MAX_N = 256;
constexpr double SVD_ZERO = 0x1p-960;  // singular values below this count as zero (W / s loses precision)

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int SVD_LDS_DOUBLES = 8192;

// Player at position e (0 <= e < np) of round r of the round-robin tournament: position 0 keeps player 0,
// the others rotate by one position per round (after np - 1 rounds every pair has met once).
__device__ inline int tournament_player(int e, int r, int np) {
  if (e == 0) return 0;
  const int k = np - 1;
  return 1 + ((e - 1 - r) % k + k) % k;
}

template <bool IN_LDS>
__global__ void __launch_bounds__(SVD_THREADS) svd_jacobi_kernel(int64_t m, int n, const double* __restrict__ A,
                                                                 double* __restrict__ U, double* __restrict__ S,
                                                                 double* __restrict__ Vt, double* __restrict__ work) {
  const int64_t b = blockIdx.x;
  A += b * m * n;
  U += b * m * n;
  S += b * n;
  Vt += b * n * n;
  __shared__ double cols[IN_LDS ? SVD_LDS_DOUBLES : 1];
  double* W = IN_LDS ? cols : work + b * (m * n + (int64_t)n * n);  // W[j][i] = column j of A (n x m)
  double* V = W + m * n;                                             // V[j][k] = column j of V (n x n)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = SVD_THREADS / 64;
  __shared__ int rotated;
  __shared__ double snorm[SVD_MAX_N];
  __shared__ int perm[SVD_MAX_N];

  for (int64_t e = tid; e < m * n; e += SVD_THREADS) {
    int64_t i = e / n;
    int j = (int)(e % n);
    W[(int64_t)j * m + i] = A[e];
  }
  for (int e = tid; e < n * n; e += SVD_THREADS) V[e] = (e / n == e % n) ? 1.0 : 0.0;
  const int np = (n + 1) & ~1;  // even count; index n (when odd) is a dummy
  __syncthreads();

  for (int sweep = 0; sweep < 60; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      for (int pr = wave; pr < np / 2; pr += nwaves) {
        int p = tournament_player(pr, round, np), q = tournament_player(np - 1 - pr, round, np);
        if (p >= n || q >= n) continue;
        if (p > q) { int t = p; p = q; q = t; }
        double* wp = W + (int64_t)p * m;
        double* wq = W + (int64_t)q * m;
        double al = 0.0, be = 0.0, ga = 0.0;
        for (int64_t i = lane; i < m; i += 64) {
          double x = wp[i], y = wq[i];
          al += x * x;
          be += y * y;
          ga += x * y;
        }
        al = wave_sum(al);
        be = wave_sum(be);
        ga = wave_sum(ga);
        if (ga != 0.0 && fabs(ga) > 1e-15 * sqrt(al * be)) {
          double zeta = (be - al) / (2.0 * ga);
          double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
          double c = 1.0 / sqrt(1.0 + t * t), s = c * t;
          for (int64_t i = lane; i < m; i += 64) {
            double x = wp[i], y = wq[i];
            wp[i] = c * x - s * y;
            wq[i] = s * x + c * y;
          }
          double* vp = V + (int64_t)p * n;
          double* vq = V + (int64_t)q * n;
          for (int k = lane; k < n; k += 64) {
            double x = vp[k], y = vq[k];
            vp[k] = c * x - s * y;
            vq[k] = s * x + c * y;
          }
          if (lane == 0) rotated = 1;
        }
      }
      __syncthreads();
    }
    if (!rotated) break;
  }

  // singular values = column norms, sorted descending (stable by index)
  for (int j = wave; j < n; j += nwaves) {
    double s2 = 0.0;
    for (int64_t i = lane; i < m; i += 64) { double x = W[(int64_t)j * m + i]; s2 += x * x; }
    s2 = wave_sum(s2);
    if (lane == 0) snorm[j] = sqrt(s2);
  }
  __syncthreads();
  for (int j = tid; j < n; j += SVD_THREADS) {
    int r = 0;
    for (int k = 0; k < n; ++k) r += (snorm[k] > snorm[j]) || (snorm[k] == snorm[j] && k < j);
    perm[r] = j;
  }
  __syncthreads();
  for (int r = tid; r < n; r += SVD_THREADS) S[r] = snorm[perm[r]];
  for (int64_t e = tid; e < m * n; e += SVD_THREADS) {
    int64_t i = e / n;
    int r = (int)(e % n);
    int j = perm[r];
    double s = snorm[j];
    U[e] = s >= SVD_ZERO ? W[(int64_t)j * m + i] / s : 0.0;
  }
  for (int e = tid; e < n * n; e += SVD_THREADS) {
    int r = e / n, k = e % n;
    Vt[e] = V[(int64_t)perm[r] * n + k];
  }

  // Columns of zero singular value carry no direction of A; give them an orthonormal completion so U
  // always has orthonormal columns (LAPACK's thin U does, and polar factors U Vt must be isometries).
  // Column r takes the unit vector e_k least covered by the accepted columns (smallest row norm, lowest
  // k on ties, so |P_perp e_k|^2 >= (m - r) / m), orthogonalised twice and normalised.
  __shared__ int first_zero;
  __shared__ double coef[SVD_MAX_N];
  __shared__ double red_v[SVD_THREADS / 64];
  __shared__ int64_t red_i[SVD_THREADS / 64];
  if (tid == 0) {
    int f = n;
    while (f > 0 && !(snorm[perm[f - 1]] >= SVD_ZERO)) --f;
    first_zero = f;
  }
  __syncthreads();
  if (first_zero == n) return;
  double* rn = W;  // m row norms of U's accepted columns (W is no longer needed)
  for (int64_t i = tid; i < m; i += SVD_THREADS) {
    double a = 0.0;
    for (int c = 0; c < first_zero; ++c) { double u = U[i * n + c]; a += u * u; }
    rn[i] = a;
  }
  __syncthreads();
  for (int r = first_zero; r < n; ++r) {
    // k = argmin over rows of rn (lowest index on ties)
    double bv = INFINITY;
    int64_t bi = m;
    for (int64_t i = tid; i < m; i += SVD_THREADS)
      if (rn[i] < bv) { bv = rn[i]; bi = i; }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      double ov = __shfl_xor(bv, o, 64);
      int64_t oi = __shfl_xor(bi, o, 64);
      if (ov < bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (lane == 0) { red_v[wave] = bv; red_i[wave] = bi; }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < nwaves; ++w)
        if (red_v[w] < red_v[0] || (red_v[w] == red_v[0] && red_i[w] < red_i[0])) { red_v[0] = red_v[w]; red_i[0] = red_i[w]; }
    }
    __syncthreads();
    const int64_t k = red_i[0] < m ? red_i[0] : 0;  // NaN row norms leave no candidate
    for (int c = tid; c < r; c += SVD_THREADS) coef[c] = U[k * n + c];
    __syncthreads();
    for (int64_t i = tid; i < m; i += SVD_THREADS) {
      double v = (i == k) ? 1.0 : 0.0;
      for (int c = 0; c < r; ++c) v -= U[i * n + c] * coef[c];
      U[i * n + r] = v;
    }
    __syncthreads();
    // second Gram-Schmidt pass: coef[c] = <U_c, v>, one wave per column
    for (int c = wave; c < r; c += nwaves) {
      double d = 0.0;
      for (int64_t i = lane; i < m; i += 64) d += U[i * n + c] * U[i * n + r];
      d = wave_sum(d);
      if (lane == 0) coef[c] = d;
    }
    __syncthreads();
    double nn = 0.0;
    for (int64_t i = tid; i < m; i += SVD_THREADS) {
      double v = U[i * n + r];
      for (int c = 0; c < r; ++c) v -= U[i * n + c] * coef[c];
      U[i * n + r] = v;
      nn += v * v;
    }
    nn = wave_sum(nn);
    if (lane == 0) red_v[wave] = nn;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int w = 0; w < nwaves; ++w) t += red_v[w];
      red_v[0] = 1.0 / sqrt(t);
    }
    __syncthreads();
    const double sc = red_v[0];
    for (int64_t i = tid; i < m; i += SVD_THREADS) {
      double v = U[i * n + r] * sc;
      U[i * n + r] = v;
      rn[i] += v * v;
    }
    __syncthreads();
  }
}
// Eigen-decomposition of a symmetric n x n matrix (n <= 64) by the parallel cyclic Jacobi method on one workgroup.  The
// odd-even ordering: rounds alternate between the position pairs (2k, 2k + 1) and (2k + 1, 2k + 2), and a pair swaps
// places as it rotates (G -> J^T G J, V -> V J), so that after np rounds every two columns have met once and the order is
// reversed.  A pair is rotated while |g_pq| > 1e-15 sqrt(|g_pp g_qq|) and |g_pq| > 1e-15 tr|G| (off-diagonal entries
// below the second bound move the eigenvalues by less than the rounding of G itself, and rotating them would not
// terminate for rank-deficient G), otherwise it only swaps.  Outputs: lam descending and Vt[r][i] = component i of
// eigenvector r.
//
// Bound by the chain of a round (read, angle, rotate, write, barrier), 64 of them per sweep, so everything in it is
// short: one barrier per round; the angle from two reciprocal square roots; the matrix in position coordinates, where
// addresses are fixed per thread and parity and free of bank conflicts, its upper half only.  Waves 0 to 3 (one per
// SIMD) hold G: each computes all angles itself and rotates the 2 x 2 blocks between pair k and pairs k + d; what a
// round reads and what it writes of the diagonal and of the pairs' own entries are different cells.  Waves 4 to 7
// keep V in registers, a row's columns 2k, 2k + 1 in lane k, one round behind.  n = 64, ten sweeps: 309 us (0.48 us a round,
// half of it the LDS reads, the rotation and the barrier), against 733 us for the round-robin order with two barriers,
// three divides and two square roots per round and V in LDS; n = 21: 75 us for 150.
constexpr int SYM_THREADS = 512;
constexpr int SYM_MAX_N = 64;
constexpr int SYM_HALF = SYM_MAX_N / 2;
// LDS cells (doubles): G, then the pairs' entries as the next round of their parity reads them (GP) and as the last one
// left them (GA), then cells for lanes without a block
constexpr int SYM_G = (SYM_HALF + 1) * SYM_MAX_N, SYM_GP = SYM_G, SYM_GA = SYM_GP + 2 * SYM_HALF,
              SYM_IDLE = SYM_GA + 2 * SYM_HALF, SYM_CELLS = SYM_IDLE + 64;

// cell of entry (i, j), i != j mod np: by circular distance and row, rows of one parity next to each other
__device__ inline int sym_cell(int i, int j, int np) {
  const int h = np / 2;
  i %= np;
  j %= np;
  int d = j - i + (j < i ? np : 0);
  if (d > h || (d == h && i >= h)) {
    i = j;
    d = np - d;
  }
  return (2 * d + (i & 1)) * SYM_HALF + (i >> 1);
}

// 1 / sqrt(x), x > 0 normal: the hardware's estimate (24 bits) and one step of third order
__device__ inline double sym_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x), e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// lane l takes `v` of lane l + 1; the last lane zero
__device__ inline double sym_from_next(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// lane l takes `v` of lane l - 1; lane 0 keeps `old`
__device__ inline double sym_from_previous(double old, double v) {
  const long long b = __double_as_longlong(v), o = __double_as_longlong(old);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

struct SymLds {
  double g[SYM_CELLS];
  double dg[2][SYM_MAX_N];                     // diagonal, read by rounds of one parity, written by the other's
  double rc[2][SYM_HALF], rs[2][SYM_HALF];     // rotations of the last two rounds
  int rank[SYM_MAX_N];
  int again;
};

// one thread's part of G
struct SymBlocks {
  int k, h, np;
  double floor_abs;
  int partner[2];
  int cell[2][2][4];      // [parity][block][entry]
  int next_pair[2];       // where entry 2 of block 0 goes when it is a pair's entry of the next round, else its cell
};

// Pair k of a round of parity O: positions 2k + O and 2k + 1 + O mod np.  New values (x the first's, y the second's):
// s x + c y and c x - s y.  In odd rounds the last pair (position np - 1 and 0) stays as it is: c = 0, s = 1, + s y.
template <int O>
__device__ inline bool sym_round(SymLds& L, const SymBlocks& B, bool writer) {
  const int k = B.k, P = 2 * k + O, Q = (O && k == B.h - 1) ? 0 : P + 1;
  const bool still = k >= B.h || (O && k == B.h - 1);
  const int Pc = k < B.h ? P : 0, Qc = k < B.h ? Q : 0;
  const double a = L.dg[O][Pc], bb = L.dg[O][Qc], g = L.g[SYM_GP + O * SYM_HALF + k];
  __builtin_amdgcn_sched_barrier(0);   // the angle's operands first
  double x[2][4];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) x[b][e] = L.g[B.cell[O][b][e]];
  __builtin_amdgcn_sched_barrier(0);
  const double gg = g * g;
  const bool on = !still & (fabs(g) > B.floor_abs) & (gg > 1e-30 * fabs(a * bb));
  const double d = bb - a;
  const double r = sym_rsqrt(__builtin_fma(4.0, gg, d * d));
  const double c2 = __builtin_fma(0.5 * fabs(d), r, 0.5), q = sym_rsqrt(c2);
  const double sr = (d >= 0.0 ? g : -g) * r * q;
  const double c = on ? c2 * q : (still ? 0.0 : 1.0), s = on ? sr : (still ? 1.0 : 0.0);
  double c1[2], s1[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    c1[b] = __shfl(c, B.partner[b], 64);
    s1[b] = __shfl(s, B.partner[b], 64);
  }
  const double sq = (O && k == B.h - 1) ? s : -s;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const double q1 = (O && B.partner[b] == B.h - 1) ? s1[b] : -s1[b];
    const double y00 = s * x[b][0] + c * x[b][2], y01 = s * x[b][1] + c * x[b][3];
    const double y10 = c * x[b][0] + sq * x[b][2], y11 = c * x[b][1] + sq * x[b][3];
    L.g[B.cell[O][b][0]] = s1[b] * y00 + c1[b] * y01;
    L.g[B.cell[O][b][1]] = c1[b] * y00 + q1 * y01;
    L.g[b ? B.cell[O][b][2] : B.next_pair[O]] = s1[b] * y10 + c1[b] * y11;
    L.g[B.cell[O][b][3]] = c1[b] * y10 + q1 * y11;
  }
  if (writer) {
    const double tg = on ? sr * q * g : 0.0;
    L.rc[O][k] = c;
    L.rs[O][k] = s;
    if (k < B.h) {
      L.dg[1 - O][P] = still ? a : bb + tg;
      L.dg[1 - O][Q] = still ? bb : a - tg;
      L.g[SYM_GA + O * SYM_HALF + k] = on ? 0.0 : g;
    }
  }
  return on;
}

// V through the rotations of a round of parity O: x0, x1 = columns 2k, 2k + 1 of eight rows, two rows per wave step in
// the half waves.  In odd rounds a lane borrows column 2k + 2 from the next lane and hands it back; where the next lane
// is not the next pair (the last pair, idle lanes) it goes back as it came (c = 0, s = 1, + s y).
template <int O>
__device__ inline void sym_vectors(const SymLds& L, int k, int h, double (&x0)[8], double (&x1)[8]) {
  const double c = L.rc[O][k], s = L.rs[O][k], sq = (O && k >= h - 1) ? s : -s;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    if (O == 0) {
      const double a = s * x0[u] + c * x1[u], b = c * x0[u] + sq * x1[u];
      x0[u] = a;
      x1[u] = b;
    } else {
      const double y = sym_from_next(x0[u]);   // column 2k + 2
      const double a = s * x1[u] + c * y, b = c * x1[u] + sq * y;
      x1[u] = a;
      x0[u] = sym_from_previous(x0[u], b);
    }
  }
}

__global__ void __launch_bounds__(SYM_THREADS) sym_jacobi_kernel(int n, const double* __restrict__ A,
                                                                 double* __restrict__ lam, double* __restrict__ Vt) {
  __shared__ SymLds L;
  const int np = n > 5 ? (n + 1) & ~1 : 6, h = np / 2;   // positions past n hold zeros; at least three pairs
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, k = lane & 31;
  const double tr = cc_wave_sum(lane < n ? fabs(A[lane * n + lane]) : 0.0);
  const int ex = tr > 0.0 && tr < INFINITY ? ilogb(tr) : 0;   // scaled by 2^-ex: the trace is in [1, 2)
  for (int e = tid; e < np * np; e += SYM_THREADS) {
    const int i = e / np, j = e % np;
    const double v = i < n && j < n ? ldexp(A[i * n + j], -ex) : 0.0;
    if (i == j) L.dg[0][i] = v;
    else if (i < j) L.g[sym_cell(i, j, np)] = v;
    if (j == i + 1) L.g[(i & 1 ? SYM_GA : SYM_GP) + (i & 1) * SYM_HALF + (i >> 1)] = v;
    if (i == 0 && j == np - 1) L.g[SYM_GA + SYM_HALF + h - 1] = v;
  }
  if (tid < 64) L.g[SYM_IDLE + tid] = 0.0;
  SymBlocks B;
  double x0[8], x1[8];
  const bool vectors = wave >= 4;
  if (!vectors) {
    __builtin_amdgcn_s_setprio(2);   // the chain; V has time to spare
    B.k = k;
    B.h = h;
    B.np = np;
    B.floor_abs = 1e-15 * ldexp(tr, -ex);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int d = 2 * wave + (lane >> 5) + 1 + 8 * b;
      const bool active = k < h && (2 * d < h || (2 * d == h && k < h / 2));
      B.partner[b] = active ? (k + d) % h : 0;
#pragma unroll
      for (int O = 0; O < 2; ++O)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          B.cell[O][b][e] = active ? sym_cell(2 * k + O + (e >> 1), 2 * (k + d) + O + (e & 1), np) : SYM_IDLE + lane;
    }
    // between a pair's second and the next pair's first position lies a pair of the other parity
#pragma unroll
    for (int O = 0; O < 2; ++O) {
      B.next_pair[O] = B.cell[O][0][2];
      if (wave == 0 && lane < 32 && k < h) {
        const int pair = O ? (k + 1) % h : k;
        B.next_pair[O] = SYM_GP + (1 - O) * SYM_HALF + pair;
        B.cell[O][0][2] = SYM_GA + (1 - O) * SYM_HALF + pair;
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = 2 * (wave - 4) + (lane >> 5) + 8 * u;
      x0[u] = 2 * k == i && i < np ? 1.0 : 0.0;
      x1[u] = 2 * k + 1 == i && i < np ? 1.0 : 0.0;
    }
  }
  __syncthreads();
  int sweeps = 0;
  for (;;) {
    bool on = false;
    for (int t = 0; t < np; t += 2) {
      if (!vectors) on |= sym_round<0>(L, B, wave == 0 && lane < 32);
      else if (sweeps + t > 0) sym_vectors<1>(L, k, h, x0, x1);
      __syncthreads();
      if (!vectors) on |= sym_round<1>(L, B, wave == 0 && lane < 32);
      else sym_vectors<0>(L, k, h, x0, x1);
      __syncthreads();
    }
    ++sweeps;
    const bool any = __any(on);
    if (tid == 0) L.again = any;
    __syncthreads();
    if (!L.again || sweeps == 60) break;
  }
  if (vectors) sym_vectors<1>(L, k, h, x0, x1);
  if (tid < np) {
    const bool back = sweeps & 1;
    const double dj = L.dg[0][tid];
    int r = 0;
    for (int i = 0; i < np; ++i) {
      const double di = L.dg[0][i];
      if ((back ? np - 1 - i : i) < n) r += (di > dj) || (di == dj && i < tid);
    }
    const bool real = (back ? np - 1 - tid : tid) < n;
    L.rank[tid] = real ? r : -1;
    if (real && r < n) lam[r] = ldexp(dj, ex);
  }
  __syncthreads();
  if (vectors && k < h) {
    const int r0 = L.rank[2 * k], r1 = L.rank[2 * k + 1];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = 2 * (wave - 4) + (lane >> 5) + 8 * u;
      if (i < n) {
        if (r0 >= 0) Vt[(int64_t)r0 * n + i] = x0[u];
        if (r1 >= 0) Vt[(int64_t)r1 * n + i] = x1[u];
      }
    }
  }
}

void launch_svd(hipStream_t st, unsigned batch, int64_t m, int n, const double* A, double* U, double* S, double* Vt,
                double* work) {
  if ((m + n) * n <= SVD_LDS_DOUBLES)
    svd_jacobi_kernel<true><<<batch, SVD_THREADS, 0, st>>>(m, n, A, U, S, Vt, work);
  else
    svd_jacobi_kernel<false><<<batch, SVD_THREADS, 0, st>>>(m, n, A, U, S, Vt, work);
}
}  // namespace

extern "C" int cc_svd_work_size(int64_t batch, int64_t m, int64_t n, int64_t* out) {
  *out = batch * (m * n + n * n);
  return CC_OK;
}

extern "C" int cc_svd_f64(void* stream, int64_t batch, int64_t m, int64_t n, const double* A, double* U, double* S,
                          double* Vt, double* work) {
  if (batch < 0 || m < 0 || n < 0) { cc_set_last_error("cc_svd_f64: negative size"); return CC_ERR_ARG; }
  if (n > SVD_MAX_N) { cc_set_last_error("cc_svd_f64: more than 256 columns"); return CC_ERR_UNSUPPORTED; }
  if (m < n) { cc_set_last_error("cc_svd_f64: needs m >= n"); return CC_ERR_ARG; }
  if (batch == 0 || n == 0) return CC_OK;
  launch_svd(cc_stream(stream), (unsigned)batch, m, (int)n, A, U, S, Vt, work);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

// ---- truncation basis of a fused environment bond -----------------------------------------------------
namespace {
// Cs[(x, a, b)][j] = (C[(x, a, b)][j] + C[(x, b, a)][j]) / 2: the part of the bond matricization that is
// symmetric under the ket <-> bra exchange of the absorbed center legs (a, b).
__global__ void fused_symmetrize_kernel(int64_t nx, int64_t na, int64_t far, const double* __restrict__ C,
                                        double* __restrict__ Cs) {
  const int64_t total = nx * na * na * far;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = i % far, r = i / far, b = r % na, a = (r / na) % na, x = r / (na * na);
    Cs[i] = 0.5 * (C[i] + C[((x * na + b) * na + a) * far + j]);
  }
}
// One workgroup per column j of U (m x n row-major): the column is negated when its entry of largest
// magnitude (the first such row) is negative, so that SVD bases computed by different routines agree.
__global__ void sign_normalize_columns_kernel(int64_t m, int64_t n, double* __restrict__ U) {
  __shared__ double best_v[256];
  __shared__ int64_t best_i[256];
  const int64_t j = blockIdx.x;
  double bv = -1.0;
  int64_t bi = m;
  for (int64_t i = threadIdx.x; i < m; i += blockDim.x) {
    const double a = fabs(U[i * n + j]);
    if (a > bv) { bv = a; bi = i; }
  }
  best_v[threadIdx.x] = bv;
  best_i[threadIdx.x] = bi;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      const double v2 = best_v[threadIdx.x + o];
      const int64_t i2 = best_i[threadIdx.x + o];
      if (v2 > best_v[threadIdx.x] || (v2 == best_v[threadIdx.x] && i2 < best_i[threadIdx.x])) {
        best_v[threadIdx.x] = v2;
        best_i[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  const int64_t ib = best_i[0];
  if (ib < m && U[ib * n + j] < 0.0)
    for (int64_t i = threadIdx.x; i < m; i += blockDim.x) U[i * n + j] = -U[i * n + j];
}
}  // namespace

extern "C" int cc_sign_normalize_columns_f64(void* stream, int64_t m, int64_t n, double* U) {
  if (m < 0 || n < 0) { cc_set_last_error("sign normalize: negative size"); return CC_ERR_ARG; }
  if (m == 0 || n == 0) return CC_OK;
  sign_normalize_columns_kernel<<<(unsigned)n, 256, 0, cc_stream(stream)>>>(m, n, U);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

namespace {
// W[i][j] = V[i][j] / s_j with V = Vt^T and s_j = sqrt(lambda_j) the singular values of the matrix whose Gram
// eigenvalues lambda (descending) and vectors Vt came from the SVD of the Gram matrix; columns whose s_j is at
// most 1e-7 s_0 (below what the Gram matrix resolves) are zero.  S_out receives every s_j.
__global__ void fused_gram_scale_kernel(int64_t far, int64_t k, const double* __restrict__ lam, const double* __restrict__ Vt,
                                        double* __restrict__ W, double* __restrict__ S_out) {
  const double s0 = sqrt(fmax(lam[0], 0.0));
  for (int64_t e = threadIdx.x; e < far * k; e += blockDim.x) {
    const int64_t i = e / k, j = e % k;
    const double sj = sqrt(fmax(lam[j], 0.0));
    W[e] = (sj > 1e-7 * s0 && sj > 0.0) ? Vt[j * far + i] / sj : 0.0;
  }
  for (int64_t j = threadIdx.x; j < far; j += blockDim.x) S_out[j] = sqrt(fmax(lam[j], 0.0));
}
}  // namespace

// The Gram product G = Cs^T Cs has a far x far output and a sum over m: for m >= 2048 (and far <= 128) it
// is cut into fused_gram_slices(m) slices summed by one batched product, and the slices are added in
// order by a second product with a vector of ones (a single product would occupy a handful of
// workgroups for the whole sum).
inline int64_t fused_gram_slices(int64_t m, int64_t far) { return (m >= 2048 && far <= 128) ? (m / 64 < 64 ? m / 64 : 64) : 1; }

extern "C" int cc_fused_truncation_work_size(int64_t nx, int64_t na, int64_t far, int64_t* out) {
  const int64_t m = nx * na * na;
  int64_t svd = 0;
  cc_svd_work_size(1, far, far, &svd);
  const int64_t S = fused_gram_slices(m, far);
  *out = svd + m * far + 4 * far * far + far + (S > 1 ? (S + 1) * far * far + (S + 1) : 0);
  return CC_OK;
}

// The leading left singular vectors of the symmetrized C (m x far, m >= far) from its Gram matrix:
// G = Cs^T Cs = V diag(lambda) V^T (two-sided Jacobi on the far x far G for far <= 64, else one-sided Jacobi),
// U = Cs V diag(1/sqrt(lambda)).
extern "C" int cc_fused_truncation_f64(void* stream, int64_t nx, int64_t na, int64_t far, int64_t new_dim,
                                       const double* C, double* U_out, double* S_out, double* work) {
  const int64_t m = nx * na * na;
  if (nx < 1 || na < 1 || far < 1 || new_dim < 1) { cc_set_last_error("fused truncation: bad sizes"); return CC_ERR_ARG; }
  if (far > SVD_MAX_N) { cc_set_last_error("fused truncation: far bond above 256"); return CC_ERR_UNSUPPORTED; }
  if (m < far) { cc_set_last_error("fused truncation: the fused bond must be at least the far bond"); return CC_ERR_ARG; }
  if (new_dim > far) { cc_set_last_error("fused truncation: new dimension above the rank bound (the far bond)"); return CC_ERR_ARG; }
  hipStream_t st = cc_stream(stream);
  int64_t svd_work = 0;
  cc_svd_work_size(1, far, far, &svd_work);
  double* Cs = work + svd_work;
  double* G = Cs + m * far;
  double* Ug = G + far * far;
  double* Vt = Ug + far * far;
  double* W = Vt + far * far;
  double* lam = W + far * far;
  const unsigned blocks = (unsigned)((m * far + 255) / 256 < 65535 ? (m * far + 255) / 256 : 65535);
  fused_symmetrize_kernel<<<blocks, 256, 0, st>>>(nx, na, far, C, Cs);
  CC_LAUNCH_CHECK();
  int rc;
  const int64_t S = fused_gram_slices(m, far);
  if (S > 1) {
    double* parts = lam + far;                       // (S + 1) slices of far x far
    double* ones = parts + (S + 1) * far * far;      // S + 1 ones
    const int64_t kc = m / S, rest = m - S * kc, np = S + (rest ? 1 : 0);
    rc = cc_gemm_f64(stream, S, far, far, kc, 1.0, Cs, kc * far, 1, far, Cs, kc * far, far, 1, 0.0, parts, far * far, far, 1);
    if (rc) return rc;
    if (rest) {
      rc = cc_gemm_f64(stream, 1, far, far, rest, 1.0, Cs + S * kc * far, 0, 1, far, Cs + S * kc * far, 0, far, 1, 0.0,
                       parts + S * far * far, 0, far, 1);
      if (rc) return rc;
    }
    rc = cc_fill_f64(stream, np, 1.0, ones);
    if (rc) return rc;
    rc = cc_gemm_f64(stream, 1, 1, far * far, np, 1.0, ones, 0, np, 1, parts, 0, far * far, 1, 0.0, G, 0, far * far, 1);
  } else {
    rc = cc_gemm_f64(stream, 1, far, far, m, 1.0, Cs, 0, 1, far, Cs, 0, far, 1, 0.0, G, 0, far, 1);
  }
  if (rc) return rc;
  if (far <= SYM_MAX_N)
    sym_jacobi_kernel<<<1, SYM_THREADS, 0, st>>>((int)far, G, lam, Vt);
  else
    launch_svd(st, 1, far, (int)far, G, Ug, lam, Vt, work);
  CC_LAUNCH_CHECK();
  fused_gram_scale_kernel<<<1, 256, 0, st>>>(far, new_dim, lam, Vt, W, S_out);
  CC_LAUNCH_CHECK();
  rc = cc_gemm_f64(stream, 1, m, new_dim, far, 1.0, Cs, 0, far, 1, W, 0, new_dim, 1, 0.0, U_out, 0, new_dim, 1);
  if (rc) return rc;
  return cc_sign_normalize_columns_f64(stream, m, new_dim, U_out);
}
