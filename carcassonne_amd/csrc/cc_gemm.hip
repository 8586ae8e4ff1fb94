// FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4f64) with arbitrary element
// strides, batched over grid.z.  A 256-thread workgroup computes a T x T tile (T = 64 or 32)
// in K steps of 16 (T = 64) or 32; the four waves own (T/2) x (T/2) sub-tiles, i.e. 2x2 MFMA tiles
// (T = 64) or one MFMA tile (T = 32, for grids that would leave most CUs idle with 64-wide tiles).
// Bound by the FP64 matrix cores on large products.  What costs there is anything that makes a wave wait
// inside a K step: operands are loaded one step ahead into registers through addresses that only advance
// (no index arithmetic, no edge masks in the loop), go through two LDS buffers with one barrier per step,
// and the LDS layouts have no bank conflicts.  4096^3: 2.56 -> 2.15 ms (53.8 -> 63.8 TFLOP/s, 82 % of the
// FP64 matrix rate) against single-buffered steps of 32 with masked loads; 1296 x 1296 x 4096: 344 -> 285 us.
// Operand fragments (probed on gfx950):
//   A[i][k] in lane i + 16k, B[k][j] in lane j + 16k, D[i][j] in lane j + 16(i%4), reg i/4.
#include "cc_common.h"

namespace {
struct GemmArgs {
  int64_t M, N, K;
  double alpha, beta;
  const double* A; int64_t sAb, sAm, sAk;
  const double* B; int64_t sBb, sBk, sBn;
  double* C; int64_t sCb, sCm, sCn;
  int64_t batch0;
  // > 0: B is upper triangular (columns up to n0 + T - 1 of C take k < n0 + T only); tiles per dimension, one-dimensional grid
  unsigned upper, batches;
};

// The operand tile of one K step (T rows or columns x BK) in LDS, in the order its loader writes without
// conflicts and the MFMA fragments (16 consecutive rows at four consecutive k) read without conflicts:
//   K_FAST (consecutive threads along k)     [row][BK + 2]: 16 rows x 2 k of a half wave hit all 64 banks
//   else   (consecutive threads along rows)  [k][T + 16]: 2 k x 16 rows of a half wave hit all 64 banks
template <int T, int BK, bool K_FAST>
struct Tile {
  static constexpr int SIZE = K_FAST ? T * (BK + 2) : BK * (T + 16);
  static constexpr int NL = T * BK / 256;  // elements per thread and K step
  static __device__ __forceinline__ int at(int i, int k) { return K_FAST ? i * (BK + 2) + k : k * (T + 16) + i; }
  // element r of thread tid
  static __device__ __forceinline__ int row(int tid, int r) { return K_FAST ? tid / BK + (256 / BK) * r : tid % T; }
  static __device__ __forceinline__ int kk(int tid, int r) { return K_FAST ? tid % BK : tid / T + (256 / T) * r; }
};

// Loader layouts: which index runs across consecutive threads.
template <int T, bool A_K_FAST, bool B_N_FAST>
__global__ void __launch_bounds__(256) gemm_f64_kernel(GemmArgs g) {
  constexpr int BK = T == 64 ? 16 : 32;   // a K step of either tile: 16 MFMAs per wave or 8
  typedef Tile<T, BK, A_K_FAST> TA;
  typedef Tile<T, BK, !B_N_FAST> TB;
  constexpr int TM = T / 32;           // 16-wide MFMA tiles per wave and dimension
  constexpr int NL = TA::NL;
  __shared__ double As[2][TA::SIZE];
  __shared__ double Bs[2][TB::SIZE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  int64_t bz = g.batch0 + blockIdx.z, m0 = (int64_t)blockIdx.y * T, n0 = (int64_t)blockIdx.x * T;
  if (g.upper) {
    // Tiles of the last columns have the longest sums.  They are dealt out to 256 CUs from the longest down and back
    // again, so that the tiles a CU holds at once add up to the same everywhere; in the order of a plain grid some CUs had
    // two thirds more than the mean.  Both products of one / two / four matrices of 1296 rows: 178 / 274 / 515 -> 149 /
    // 233 / 423 us.
    const unsigned t = g.upper, per_col = t * g.batches, at = blockIdx.x % 256, round = blockIdx.x - at;
    const unsigned width = gridDim.x - round < 256 ? gridDim.x - round : 256;
    const unsigned rank = round + (round / 256 % 2 ? width - 1 - at : at);
    bz = rank % per_col / t;
    m0 = (int64_t)(rank % t) * T;
    n0 = (int64_t)(t - 1 - rank / per_col) * T;
  }
  double* C = g.C + bz * g.sCb;
  const int64_t K = g.upper && n0 + T < g.K ? n0 + T : g.K;

  f64x4 acc[TM][TM];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = (f64x4){0.0, 0.0, 0.0, 0.0};

  // One address per element, advanced by a K step; rows past the edge read the last row (their results are
  // not written), so only the last K step needs a mask.
  const double *pa[NL], *pb[NL];
#pragma unroll
  for (int r = 0; r < NL; ++r) {
    const int64_t gi = m0 + TA::row(tid, r), gj = n0 + TB::row(tid, r);
    pa[r] = g.A + bz * g.sAb + (gi < g.M ? gi : g.M - 1) * g.sAm + TA::kk(tid, r) * g.sAk;
    pb[r] = g.B + bz * g.sBb + (gj < g.N ? gj : g.N - 1) * g.sBn + TB::kk(tid, r) * g.sBk;
  }
  const int64_t da = BK * g.sAk, db = BK * g.sBk;
  double ra[NL], rb[NL];
  auto load = [&]() {
#pragma unroll
    for (int r = 0; r < NL; ++r) {
      ra[r] = *pa[r];
      rb[r] = *pb[r];
      pa[r] += da;
      pb[r] += db;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < NL; ++r) {
      As[buf][TA::at(TA::row(tid, r), TA::kk(tid, r))] = ra[r];
      Bs[buf][TB::at(TB::row(tid, r), TB::kk(tid, r))] = rb[r];
    }
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      double af[TM], bf[TM];
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        af[t] = As[buf][TA::at(wr * (T / 2) + t * 16 + (lane & 15), kk + (lane >> 4))];
        bf[t] = Bs[buf][TB::at(wc * (T / 2) + t * 16 + (lane & 15), kk + (lane >> 4))];
      }
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
  };

  // Two LDS buffers and one barrier per K step: the next step's loads are in flight during a step's products,
  // and a buffer is written again only after every wave passed the barrier of the step in between.
  const int full = (int)(K / BK), rest = (int)(K % BK);
  if (full > 0) load();
  for (int s = 0; s < full; ++s) {
    store(s & 1);
    __syncthreads();
    if (s + 1 < full) load();
    compute(s & 1);
  }
  if (rest > 0) {
#pragma unroll
    for (int r = 0; r < NL; ++r) {
      ra[r] = TA::kk(tid, r) < rest ? *pa[r] : 0.0;
      rb[r] = TB::kk(tid, r) < rest ? *pb[r] : 0.0;
    }
    store(full & 1);
    __syncthreads();
    compute(full & 1);
  }

#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int64_t gi = m0 + wr * (T / 2) + a * 16 + 4 * r + (lane >> 4);
        int64_t gj = n0 + wc * (T / 2) + b * 16 + (lane & 15);
        if (gi < g.M && gj < g.N) {
          double* p = C + gi * g.sCm + gj * g.sCn;
          double v = g.alpha * acc[a][b][r];
          *p = (g.beta == 0.0) ? v : v + g.beta * (*p);
        }
      }
}

template <int T>
void launch_gemm(const GemmArgs& g, dim3 grid, bool a_k_fast, bool b_n_fast, hipStream_t st) {
  if (a_k_fast && b_n_fast) gemm_f64_kernel<T, true, true><<<grid, 256, 0, st>>>(g);
  else if (a_k_fast) gemm_f64_kernel<T, true, false><<<grid, 256, 0, st>>>(g);
  else if (b_n_fast) gemm_f64_kernel<T, false, true><<<grid, 256, 0, st>>>(g);
  else gemm_f64_kernel<T, false, false><<<grid, 256, 0, st>>>(g);
}
}  // namespace

extern "C" int cc_gemm_f64(void* stream, int64_t batch, int64_t M, int64_t N, int64_t K, double alpha,
                           const double* A, int64_t sAb, int64_t sAm, int64_t sAk,
                           const double* B, int64_t sBb, int64_t sBk, int64_t sBn, double beta,
                           double* C, int64_t sCb, int64_t sCm, int64_t sCn) {
  if (batch < 0 || M < 0 || N < 0 || K < 0) { cc_set_last_error("cc_gemm_f64: negative size"); return CC_ERR_ARG; }
  if (batch == 0 || M == 0 || N == 0) return CC_OK;
  GemmArgs g{M, N, K, alpha, beta, A, sAb, sAm, sAk, B, sBb, sBk, sBn, C, sCb, sCm, sCn, 0, 0, 0};
  // 64-wide tiles unless that grid would leave most of the 256 CUs idle
  const int64_t tiles64 = ((N + 63) / 64) * ((M + 63) / 64) * batch;
  const int T = tiles64 < 160 ? 32 : 64;
  int64_t gx = (N + T - 1) / T, gy = (M + T - 1) / T;
  if (gx > 2147483647LL || gy > 65535) { cc_set_last_error("cc_gemm_f64: matrix too large for one launch"); return CC_ERR_UNSUPPORTED; }
  bool a_k_fast = (sAk == 1) || (sAm != 1 && (sAk < sAm));
  bool b_n_fast = (sBn == 1) || (sBk != 1 && (sBn < sBk));
  hipStream_t st = cc_stream(stream);
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
    g.batch0 = b0;
    dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)nb);
    if (T == 32) launch_gemm<32>(g, grid, a_k_fast, b_n_fast, st);
    else launch_gemm<64>(g, grid, a_k_fast, b_n_fast, st);
    CC_LAUNCH_CHECK();
  }
  return CC_OK;
}

int cc_internal_gemm_upper(hipStream_t st, int64_t batch, int64_t n, const double* A, int64_t sAb, int64_t sAm, int64_t sAk,
                           const double* B, int64_t ldb, double* C, int64_t sCb) {
  GemmArgs g{n, n, n, 1.0, 0.0, A, sAb, sAm, sAk, B, 0, ldb, 1, C, sCb, n, 1, 0, 0, (unsigned)batch};
  const int64_t tiles64 = ((n + 63) / 64) * ((n + 63) / 64) * batch;
  const int T = tiles64 < 160 ? 32 : 64;
  const int64_t t = (n + T - 1) / T;
  if (batch > 65535 || t * t > 2147483647LL / batch) { cc_set_last_error("gemm: matrix too large for one launch"); return CC_ERR_UNSUPPORTED; }
  g.upper = (unsigned)t;
  const dim3 grid((unsigned)(t * t * batch));
  if (T == 32) launch_gemm<32>(g, grid, sAk == 1, true, st);
  else launch_gemm<64>(g, grid, sAk == 1, true, st);
  CC_LAUNCH_CHECK();
  return CC_OK;
}
