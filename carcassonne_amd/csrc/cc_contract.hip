// FP64 tensor contractions on matrix cores with the legs read and written where they lie:
//   C_o[m, n] = sum over o's terms t and over k of A_t[m, k] B_t[k, n]
// where m, n and k are groups of legs with strides of their own in each tensor (all A alike, all B, all C).  Every
// output of a call goes into one launch, and the terms of one output are one long sum.
//
// What it replaces is a permutation of each operand (a pass over memory and a launch), a product, and an addition per
// term.  The tile kernel is that of cc_gemm.hip (operands one K step ahead in registers, two LDS buffers, one barrier
// per step, conflict-free layouts) with offset tables for addresses: those of the tile's rows and columns and of up to
// CT_KT values of k are made once in LDS, so a step costs one table read per element whatever the legs are.
// Bound by the FP64 matrix cores on large products; the tile's width follows N (16 to 80 columns on 128 rows, else
// 64 x 64), so that a leg pair of 36 is not multiplied as 64; grids that would leave CUs idle take 32 x 32 tiles, and
// long sums there are split over workgroups and added in order.
#include "cc_common.h"

#include <algorithm>
#include <utility>

namespace {
constexpr int CT_RANK = 12;      // legs per group
constexpr int CT_OUT = 16;       // outputs and terms per launch
constexpr int CT_TERMS = 32;
constexpr int CT_KT = 1024;      // offsets of k in LDS at a time

struct Leg {
  int64_t n, s[2];               // extent and its strides in the two tensors that have it
};
struct Legs {
  int count;
  Leg l[CT_RANK];
};
struct LegGroup {
  int rank;
  uint32_t n[CT_RANK], magic[CT_RANK], shift[CT_RANK];
  int s[2][CT_RANK];
};
struct ContractArgs {
  int M, N, K, tiles_n, splits;
  LegGroup m, n, k;              // strides in (A, C), (B, C), (A, B)
  int first[CT_OUT + 1];         // terms of output o: first[o] .. first[o + 1]
  const double *A[CT_TERMS], *B[CT_TERMS];
  double* C[CT_OUT];
  double* work;                  // splits > 1: splits partial results per output, M x N each
};

// Index i split into the group's legs, divisions by the invariant extents as a multiply-high and shifts (Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994).
__device__ __forceinline__ void leg_offsets(const LegGroup& g, uint32_t i, int& a, int& b) {
  a = b = 0;
  for (int l = g.rank - 1; l >= 0; --l) {
    const uint32_t t = __umulhi(g.magic[l], i), q = g.n[l] == 1 ? i : (t + ((i - t) >> 1)) >> (g.shift[l] - 1);
    const int r = (int)(i - q * g.n[l]);
    a += r * g.s[0][l];
    b += r * g.s[1][l];
    i = q;
  }
}

// WM x WN waves of TM x TN MFMA tiles
template <int WM, int WN, int TM, int TN, int BK, bool A_K_FAST>
__global__ void __launch_bounds__(256) contract_kernel(const ContractArgs g) {
  constexpr int R = 16 * WM * TM, W = 16 * WN * TN, NA = R * BK / 256, NB = W * BK / 256;
  constexpr int LA = A_K_FAST ? BK + 2 : R + 16, SA = A_K_FAST ? R * LA : BK * LA, LB = W % 32 ? W : W + 16;
  static_assert(WM * WN == 4 && R * BK % 256 == 0 && W * BK % 256 == 0 && CT_KT % BK == 0, "tile shape");
  __shared__ double As[2][SA];
  __shared__ double Bs[2][BK * LB];
  __shared__ int ka[CT_KT], kb[CT_KT], row_a[R], row_c[R], col_b[W], col_c[W];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WN * TM * 16, wc = wave % WN * TN * 16;
  const int m0 = (int)(blockIdx.x / (unsigned)g.tiles_n) * R, n0 = (int)(blockIdx.x % (unsigned)g.tiles_n) * W;
  const int o = (int)blockIdx.z / g.splits, split = (int)blockIdx.z % g.splits;

  // rows and columns past the edge read the last one; their results are not written
  for (int i = tid; i < R + W; i += 256) {
    int a, b;
    if (i < R) {
      leg_offsets(g.m, (uint32_t)(m0 + i < g.M ? m0 + i : g.M - 1), a, b);
      row_a[i] = a;
      row_c[i] = b;
    } else {
      const int j = i - R;
      leg_offsets(g.n, (uint32_t)(n0 + j < g.N ? n0 + j : g.N - 1), a, b);
      col_b[j] = a;
      col_c[j] = b;
    }
  }
  auto table = [&](int base) {
    for (int i = tid; i < CT_KT; i += 256) {
      if (base + i >= g.K + BK) break;
      int a = 0, b = 0;
      if (base + i < g.K) leg_offsets(g.k, (uint32_t)(base + i), a, b);
      ka[i] = a;
      kb[i] = b;
    }
  };

  // steps of BK within one term; the terms of the output follow each other
  const int per_term = (g.K + BK - 1) / BK, all = (g.first[o + 1] - g.first[o]) * per_term;
  const int s0 = (int)((int64_t)all * split / g.splits), s1 = (int)((int64_t)all * (split + 1) / g.splits);
  int term = g.first[o] + s0 / per_term, k0 = s0 % per_term * BK, base = k0 / CT_KT * CT_KT;
  table(base);
  __syncthreads();

  int ra_off[NA], rb_off[NB], ra_k[NA], rb_k[NB];
#pragma unroll
  for (int r = 0; r < NA; ++r) {
    const int e = tid + 256 * r;
    ra_k[r] = A_K_FAST ? e % BK : e / R;
    ra_off[r] = row_a[A_K_FAST ? e / BK : e % R];
  }
#pragma unroll
  for (int r = 0; r < NB; ++r) {
    const int e = tid + 256 * r;
    rb_k[r] = e / W;
    rb_off[r] = col_b[e % W];
  }
  double ra[NA], rb[NB];
  auto load = [&]() {
    if (k0 >= base + CT_KT || k0 < base) {   // uniform; only where K > CT_KT
      __syncthreads();
      base = k0 / CT_KT * CT_KT;
      table(base);
      __syncthreads();
    }
    const double* A = g.A[term];
    const double* B = g.B[term];
    const int at = k0 - base;
#pragma unroll
    for (int r = 0; r < NA; ++r) ra[r] = A[(int64_t)ra_off[r] + ka[at + ra_k[r]]];
#pragma unroll
    for (int r = 0; r < NB; ++r) rb[r] = B[(int64_t)rb_off[r] + kb[at + rb_k[r]]];
    if (k0 + BK > g.K) {
#pragma unroll
      for (int r = 0; r < NA; ++r)
        if (k0 + ra_k[r] >= g.K) ra[r] = 0.0;
#pragma unroll
      for (int r = 0; r < NB; ++r)
        if (k0 + rb_k[r] >= g.K) rb[r] = 0.0;
    }
    k0 += BK;
    if (k0 >= g.K) {
      k0 = 0;
      ++term;
    }
  };
  f64x4 acc[TM][TN], sum[TM][TN];   // of the term at hand, of the finished ones
  auto clear = [&](f64x4 (&v)[TM][TN]) {
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) v[a][b] = (f64x4){0.0, 0.0, 0.0, 0.0};
  };
  clear(acc);
  clear(sum);
  int left = per_term - s0 % per_term;   // steps of the term at hand
  bool single = true;
  if (s0 < s1) load();
  for (int s = s0; s < s1; ++s) {
    double* as = As[(s - s0) & 1];
    double* bs = Bs[(s - s0) & 1];
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int e = tid + 256 * r;
      as[A_K_FAST ? e / BK * LA + e % BK : e / R * LA + e % R] = ra[r];
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int e = tid + 256 * r;
      bs[e / W * LB + e % W] = rb[r];
    }
    __syncthreads();
    if (s + 1 < s1) load();
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      double af[TM], bf[TN];
      const int k = kk + (lane >> 4);
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        const int i = wr + 16 * t + (lane & 15);
        af[t] = as[A_K_FAST ? i * LA + k : k * LA + i];
      }
#pragma unroll
      for (int t = 0; t < TN; ++t) bf[t] = bs[k * LB + wc + 16 * t + (lane & 15)];
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    if (--left == 0 && s + 1 < s1) {   // the next term
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) sum[a][b] = single ? acc[a][b] : sum[a][b] + acc[a][b];
      clear(acc);
      left = per_term;
      single = false;
    }
  }
  if (!single) {
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) acc[a][b] = sum[a][b] + acc[a][b];
  }

  double* C = g.splits > 1 ? g.work + (int64_t)blockIdx.z * g.M * g.N : g.C[o];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = wr + 16 * a + 4 * r + (lane >> 4), j = wc + 16 * b + (lane & 15);
        if (m0 + i < g.M && n0 + j < g.N)
          C[g.splits > 1 ? (int64_t)(m0 + i) * g.N + n0 + j : (int64_t)row_c[i] + col_c[j]] = acc[a][b][r];
      }
}

// The partial results of split sums, added in order.
__global__ void __launch_bounds__(256) contract_reduce_kernel(const ContractArgs g) {
  const int64_t mn = (int64_t)g.M * g.N, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= mn) return;
  const double* p = g.work + (int64_t)blockIdx.y * g.splits * mn + e;
  double v = 0.0;
  for (int s = 0; s < g.splits; ++s) v += p[s * mn];
  int a, rc, cc;
  leg_offsets(g.m, (uint32_t)(e / g.N), a, rc);
  leg_offsets(g.n, (uint32_t)(e % g.N), a, cc);
  g.C[blockIdx.y][(int64_t)rc + cc] = v;
}

// Legs in the order given by stride `by` (largest first; by < 0: as they are), unit legs dropped, neighbours merged where
// both tensors allow.
int arrange(Legs& v, int by, LegGroup& g, int64_t& total) {
  for (int i = 1; i < v.count && by >= 0; ++i)
    for (int j = i; j > 0 && v.l[j - 1].s[by] < v.l[j].s[by]; --j) std::swap(v.l[j - 1], v.l[j]);
  int n = 0;
  total = 1;
  for (int i = 0; i < v.count; ++i) {
    const Leg l = v.l[i];
    if (l.n > 2147483647LL / total) return CC_ERR_UNSUPPORTED;
    total *= l.n;
    if (l.n == 1) continue;
    if (l.s[0] < 0 || l.s[0] > 2147483647LL || l.s[1] < 0 || l.s[1] > 2147483647LL) return CC_ERR_UNSUPPORTED;
    if (n && v.l[n - 1].s[0] == l.n * l.s[0] && v.l[n - 1].s[1] == l.n * l.s[1])
      v.l[n - 1] = {v.l[n - 1].n * l.n, {l.s[0], l.s[1]}};
    else
      v.l[n++] = l;
  }
  g.rank = n;
  for (int i = 0; i < n; ++i) {
    const uint64_t e = (uint64_t)v.l[i].n;
    const uint32_t l = (uint32_t)(64 - __builtin_clzll(e - 1));
    g.n[i] = (uint32_t)e;
    g.shift[i] = l;
    g.magic[i] = (uint32_t)((((1ull << l) - e) << 32) / e + 1);
    for (int t = 0; t < 2; ++t) g.s[t][i] = (int)v.l[i].s[t];
  }
  return CC_OK;
}

int64_t least(const Legs& v, int t) {
  int64_t least = INT64_MAX;
  for (int i = 0; i < v.count; ++i)
    if (v.l[i].n > 1) least = std::min(least, v.l[i].s[t]);
  return least;
}

int64_t reach(const LegGroup& g, int t) {
  int64_t v = 0;
  for (int i = 0; i < g.rank; ++i) v += ((int64_t)g.n[i] - 1) * g.s[t][i];
  return v;
}

struct Shape {
  bool a_k_fast, swapped;
  int tall;        // columns / 16 of a 128-row tile, 0: square
  int T;           // of a square tile
  int splits;      // for an output of one term
};

// The order of the legs and the tile of a contraction (`legs`: extent and two strides each, rm + rn + rk of them).
int plan(int rm, int rn, int rk, const int64_t* legs, int n_out, const int* terms, ContractArgs& g, Shape& sh) {
  if (rm < 0 || rn < 0 || rk < 0 || n_out < 1) { cc_set_last_error("contract: bad sizes"); return CC_ERR_ARG; }
  Legs v[3];
  const int ranks[3] = {rm, rn, rk};
  for (int q = 0, at = 0; q < 3; ++q) {
    if (ranks[q] > CT_RANK) { cc_set_last_error("contract: more than 12 legs in a group"); return CC_ERR_UNSUPPORTED; }
    v[q].count = ranks[q];
    for (int i = 0; i < ranks[q]; ++i, at += 3) {
      if (legs[at] < 1) { cc_set_last_error("contract: empty leg"); return CC_ERR_ARG; }
      v[q].l[i] = {legs[at], {legs[at + 1], legs[at + 2]}};
    }
  }
  // C is written along its columns: its fastest leg belongs to B's side
  sh.swapped = least(v[0], 1) < least(v[1], 1);
  if (sh.swapped) {
    std::swap(v[0], v[1]);
    for (int i = 0; i < rk; ++i) std::swap(v[2].l[i].s[0], v[2].l[i].s[1]);
  }
  // sums run over k in the caller's order of its legs
  int64_t fastest = INT64_MAX;
  for (int i = 0; i < rk; ++i)
    if (v[2].l[i].n > 1) fastest = v[2].l[i].s[0];
  sh.a_k_fast = fastest < least(v[0], 0);
  int64_t M, N, K;
  int rc = arrange(v[0], 0, g.m, M);
  if (!rc) rc = arrange(v[1], 1, g.n, N);
  if (!rc) rc = arrange(v[2], -1, g.k, K);
  if (rc || reach(g.m, 0) + reach(g.k, 0) > 2147483647LL || reach(g.n, 0) + reach(g.k, 1) > 2147483647LL ||
      reach(g.m, 1) + reach(g.n, 1) > 2147483647LL || K > 2147483647LL - 64) {
    cc_set_last_error("contract: legs beyond 32-bit offsets");
    return CC_ERR_UNSUPPORTED;
  }
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  // 128 rows and as many columns as N needs where N is narrow and the grid is still large: five outputs of 147456 x 36
  // with K = 72 take 244 us against 290 us on 64 x 64 tiles, x 25 with K = 50 (102400 rows) 124 against 171, x 16 with
  // K = 32 (65536 rows) 35 against 62.  32 x 32 tiles and split sums where fewer than 160 tiles of 64 x 64 would be left
  // for 256 CUs (the line of the plain product).
  const int64_t tall = (M + 127) / 128 * n_out, square = (M + 63) / 64 * ((N + 63) / 64) * n_out;
  sh.tall = N <= 80 && tall >= 160 ? (int)((N + 15) / 16) : 0;
  sh.T = square >= 160 ? 64 : 32;
  // long sums: three workgroups per CU where that leaves each at least eight steps of 16 (64 x 64 tiles: five outputs of
  // 64 x 2304 with K = 2304 take 144 us whole and 94 us split), one per CU and four steps of 32 for the small tiles
  sh.splits = 1;
  if (!sh.tall) {
    const int T = sh.T;
    const int64_t tiles = (M + T - 1) / T * ((N + T - 1) / T) * n_out;
    int most = 0;
    for (int o = 0; o < n_out; ++o) most = std::max(most, terms[o]);
    const int64_t steps = T == 64 ? (K + 15) / 16 * most : (K + 31) / 32 * most;
    sh.splits = (int)std::max<int64_t>(1, T == 64 ? std::min(steps / 8, 768 / tiles) : std::min(steps / 4, 256 / tiles));
  }
  return CC_OK;
}

template <bool A_K_FAST>
void launch(const Shape& sh, const ContractArgs& g, dim3 grid, hipStream_t st) {
  switch (sh.tall) {
    case 1: contract_kernel<4, 1, 2, 1, 16, A_K_FAST><<<grid, 256, 0, st>>>(g); break;
    case 2: contract_kernel<4, 1, 2, 2, 16, A_K_FAST><<<grid, 256, 0, st>>>(g); break;
    case 3: contract_kernel<4, 1, 2, 3, 16, A_K_FAST><<<grid, 256, 0, st>>>(g); break;
    case 4: contract_kernel<4, 1, 2, 4, 16, A_K_FAST><<<grid, 256, 0, st>>>(g); break;
    case 5: contract_kernel<4, 1, 2, 5, 16, A_K_FAST><<<grid, 256, 0, st>>>(g); break;
    default:
      if (sh.T == 64) contract_kernel<2, 2, 2, 2, 16, A_K_FAST><<<grid, 256, 0, st>>>(g);
      else contract_kernel<2, 2, 1, 1, 32, A_K_FAST><<<grid, 256, 0, st>>>(g);
  }
}
}  // namespace

extern "C" int cc_contract_work_size(int rm, int rn, int rk, const int64_t* legs, int n_out, const int* terms, int64_t* out) {
  ContractArgs g;
  Shape sh;
  const int rc = plan(rm, rn, rk, legs, n_out, terms, g, sh);
  if (rc) return rc;
  *out = sh.splits > 1 ? (int64_t)sh.splits * std::min(n_out, CT_OUT) * g.M * g.N : 0;
  return CC_OK;
}

extern "C" int cc_contract_f64(void* stream, int rm, int rn, int rk, const int64_t* legs, int n_out, const int* terms,
                               const double* const* A, const double* const* B, double* const* C, double* work) {
  ContractArgs g = {};
  Shape sh;
  const int rc = plan(rm, rn, rk, legs, n_out, terms, g, sh);
  if (rc) return rc;
  hipStream_t st = cc_stream(stream);
  if (sh.swapped) std::swap(A, B);
  g.splits = work ? sh.splits : 1;
  g.work = work;
  const int R = sh.tall ? 128 : sh.T, W = sh.tall ? 16 * sh.tall : sh.T;
  g.tiles_n = (g.N + W - 1) / W;
  const int64_t tiles = (int64_t)((g.M + R - 1) / R) * g.tiles_n;
  if (tiles > 2147483647LL) { cc_set_last_error("contract: too large for one launch"); return CC_ERR_UNSUPPORTED; }
  for (int o = 0, at = 0; o < n_out;) {
    int n = 0, t = 0;
    for (; n < CT_OUT && o + n < n_out; ++n) {
      const int more = terms[o + n];
      if (more < 1 || more > CT_TERMS) { cc_set_last_error("contract: 1 to 32 terms per output"); return CC_ERR_ARG; }
      if (t + more > CT_TERMS) break;
      g.first[n] = t;
      g.C[n] = C[o + n];
      for (int i = 0; i < more; ++i) {
        g.A[t + i] = A[at + t + i];
        g.B[t + i] = B[at + t + i];
      }
      t += more;
    }
    g.first[n] = t;
    const dim3 grid((unsigned)tiles, 1, (unsigned)(n * g.splits));
    if (sh.a_k_fast) launch<true>(sh, g, grid, st);
    else launch<false>(sh, g, grid, st);
    CC_LAUNCH_CHECK();
    if (g.splits > 1) {
      const int64_t mn = (int64_t)g.M * g.N;
      contract_reduce_kernel<<<dim3((unsigned)((mn + 255) / 256), (unsigned)n), 256, 0, st>>>(g);
      CC_LAUNCH_CHECK();
    }
    o += n;
    at += t;
  }
  return CC_OK;
}
