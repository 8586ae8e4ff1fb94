// The stage-3 operator formed once as dense matrices over the environment legs, for solves that apply it many
// times (the reference's own cost rule, Multiplier.isCheaperToFormMatrix, utils.py:203-206; the matrices are those
// of formDenseStage3_formMatrix, tensors/_2d/dense.py:176-203, before the site operator is attached):
//
//   H = sum_g O_g (x) G_g,   G_g[(p'q')][(pq)] = sum over the products (A, B) of group g of
//                                                sum_alpha A[alpha][p'][p] B[alpha][q'][q]
//
// with one group per distinct site operator.  A matvec through the slabs costs 8 n_alpha P^3 FLOP per product and
// re-reads every slab; a formed matrix costs 2 n_alpha P^4 once, P / 4 matvecs' worth, and is then P^4 doubles.
#include "cc_formed.h"

namespace {
constexpr int FORM_MAX = 16;      // products (and distinct matrices) per call

// ---- slab channels joined (and summed) into (alpha, P, P) arrays ------------------------------------------------
// out[alpha][row][col] = sum_i c_i src_i[slab map]: a gather in source order into LDS (coalesced reads), written
// row-major.  HBM-bound: (n_src + 1) passes over a channel.
template <int D>
__global__ void __launch_bounds__(256) slab_join_kernel_d(int64_t n_alpha, CCSlabGather g, CCSlabSum src, double* __restrict__ out) {
  constexpr int n = D * D * D * D;
  __shared__ double s[n];
  for (int64_t al = blockIdx.x; al < n_alpha; al += gridDim.x) {
    cc_slab_load_sum_d<D, 256>(g, src, al, s, D * D);
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += 256) out[al * n + e] = s[e];
    __syncthreads();
  }
}

// The same for any leg sizes.
__global__ void __launch_bounds__(256) slab_join_kernel(int64_t n_alpha, int64_t P, CCSlabMap map, CCSlabSum src,
                                                        double* __restrict__ out) {
  const int64_t PP = P * P, n = n_alpha * PP;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int64_t al = e / PP, x = e - al * PP, off = cc_slab_offset(map, al, x / P, x % P);
    double v = src.c[0] * src.p[0][off];
    for (int i = 1; i < src.n; ++i) v += src.c[i] * src.p[i][off];
    out[e] = v;
  }
}

// ---- the formation product --------------------------------------------------------------------------------------
struct FormArgs {
  int n_groups, split;
  int begin[FORM_MAX + 1];                 // products of group g: [begin[g], begin[g + 1])
  const double *A[FORM_MAX], *B[FORM_MAX];
  int64_t n_alpha;
  int P, Q, tm, tn;
};

constexpr int FT = 64, FK = 16, FLD = FT + 16;  // tile, K step, LDS row (2 k x 16 rows of a half wave: 64 banks)

// Row-major index of element (row = p'P + p, col = q'Q + q) in the (p'q') x (pq) matrix.
__device__ __forceinline__ int64_t form_at(int row, int col, int P, int Q) {
  const int pp = row / P, p = row - pp * P, qq = col / Q, q = col - qq * Q;
  return ((int64_t)pp * Q + qq) * ((int64_t)P * Q) + (int64_t)p * Q + q;
}

// One 64 x 64 tile of one group's product over a part of its K range (the products' alpha ranges in a row), the
// same double-buffered loop as cc_gemm_f64.  A product of D = 6 has 441 tiles for 256 CUs that hold three
// workgroups each, so a group's K range is cut into `split` parts (summed in order by form_reduce_kernel) until the
// last wave of workgroups weighs little, and parts go to XCDs in turn: every workgroup of a part runs on the same
// XCD, whose L2 then reads that part of the slabs alone.
__global__ void __launch_bounds__(256) form_kernel(FormArgs f, double* __restrict__ out) {
  __shared__ double As[2][FK * FLD];
  __shared__ double Bs[2][FK * FLD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;
  const int tiles = f.tm * f.tn, units = f.n_groups * f.split, b = blockIdx.x;
  const int unit = units % 8 == 0 ? (b & 7) + 8 * ((b >> 3) / tiles) : b / tiles;
  const int tile = units % 8 == 0 ? (b >> 3) % tiles : b % tiles;
  const int g = unit / f.split, part = unit - g * f.split;
  const int PP = f.P * f.P, QQ = f.Q * f.Q;
  const int m0 = (tile / f.tn) * FT, n0 = (tile % f.tn) * FT;
  const int spp = (int)((f.n_alpha + FK - 1) / FK);  // K steps per product
  const int64_t S = (int64_t)(f.begin[g + 1] - f.begin[g]) * spp;
  const int64_t s0 = S * part / f.split, s1 = S * (part + 1) / f.split;

  f64x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[a][c] = (f64x4){0.0, 0.0, 0.0, 0.0};

  // element r of this thread: row tid % 64 of the tile (clamped at the edge; such results are not written), k = tid / 64 + 4 r
  const int col = tid & 63, k4 = tid >> 6;
  const int ra0 = m0 + col < PP ? m0 + col : PP - 1, rb0 = n0 + col < QQ ? n0 + col : QQ - 1;
  int prod = f.begin[g] + (int)(s0 / spp), ks = (int)(s0 % spp);
  const double *pa = f.A[prod < FORM_MAX ? prod : 0] + ((int64_t)ks * FK + k4) * PP + ra0;
  const double *pb = f.B[prod < FORM_MAX ? prod : 0] + ((int64_t)ks * FK + k4) * QQ + rb0;
  double ra[4], rb[4];
  auto load = [&]() {   // the K step at (prod, ks), then on to the next one
    const int64_t left = f.n_alpha - (int64_t)ks * FK;
    if (left >= FK) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ra[r] = pa[(int64_t)4 * r * PP];
        rb[r] = pb[(int64_t)4 * r * QQ];
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ra[r] = k4 + 4 * r < left ? pa[(int64_t)4 * r * PP] : 0.0;
        rb[r] = k4 + 4 * r < left ? pb[(int64_t)4 * r * QQ] : 0.0;
      }
    }
    pa += (int64_t)FK * PP;
    pb += (int64_t)FK * QQ;
    if (++ks == spp) {
      ks = 0;
      if (++prod < f.begin[g + 1]) {
        pa = f.A[prod] + (int64_t)k4 * PP + ra0;
        pb = f.B[prod] + (int64_t)k4 * QQ + rb0;
      }
    }
  };
  if (s0 < s1) load();
  for (int64_t s = s0; s < s1; ++s) {
    const int buf = (int)(s & 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      As[buf][(k4 + 4 * r) * FLD + col] = ra[r];
      Bs[buf][(k4 + 4 * r) * FLD + col] = rb[r];
    }
    __syncthreads();
    if (s + 1 < s1) load();
#pragma unroll
    for (int kk = 0; kk < FK; kk += 4) {
      double af[2], bf[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        af[t] = As[buf][(kk + (lane >> 4)) * FLD + wr * 32 + t * 16 + (lane & 15)];
        bf[t] = Bs[buf][(kk + (lane >> 4)) * FLD + wc * 32 + t * 16 + (lane & 15)];
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[c], acc[a][c], 0, 0, 0);
    }
  }
  double* o = out + (int64_t)unit * PP * QQ;   // split > 1: the part's own array; split = 1: the matrix itself
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = m0 + wr * 32 + a * 16 + 4 * r + (lane >> 4), gj = n0 + wc * 32 + c * 16 + (lane & 15);
        if (gi < PP && gj < QQ) o[f.split > 1 ? (int64_t)gi * QQ + gj : form_at(gi, gj, f.P, f.Q)] = acc[a][c][r];
      }
}

// out[g][(p'q')][(pq)] = sum of the group's parts, in order.
__global__ void __launch_bounds__(256) form_reduce_kernel(int split, int P, int Q, const double* __restrict__ parts,
                                                          double* __restrict__ out) {
  const int64_t nn = (int64_t)P * P * Q * Q;
  const double* src = parts + (int64_t)blockIdx.y * split * nn;
  double* dst = out + (int64_t)blockIdx.y * nn;
  const int row = blockIdx.x;                   // (p', q')
  const int pp = row / Q, qq = row - pp * Q;
  for (int e = threadIdx.x; e < P * Q; e += 256) {
    const int p = e / Q, q = e - p * Q;
    const int64_t at = ((int64_t)pp * P + p) * ((int64_t)Q * Q) + (int64_t)qq * Q + q;
    double t = src[at];
    for (int k = 1; k < split; ++k) t += src[k * nn + at];
    dst[(int64_t)row * (P * Q) + e] = t;
  }
}

// Parts of a group's K range: enough workgroups for several waves of the chip (256 CUs x 3), each with at least
// FORM_MIN_STEPS K steps, a multiple of 8 parts in all so that each stays on one XCD.  The sums of parts are also the more
// accurate ones: N at D = 2, chi = 50 is 1.3e-16 off sums in 80 bits, 1.3e-15 as one running sum per entry.
constexpr int FORM_MIN_STEPS = 8;
int form_split(int n_groups, int max_products, int64_t n_alpha, int64_t P, int64_t Q) {
  const int64_t tiles = ((P * P + FT - 1) / FT) * ((Q * Q + FT - 1) / FT);
  const int64_t steps = (int64_t)max_products * ((n_alpha + FK - 1) / FK);
  int split = 1;
  while (tiles * n_groups * split < 4 * 768 && steps / (2 * split) >= FORM_MIN_STEPS && split < 64) split *= 2;
  return split;
}

// ---- application ------------------------------------------------------------------------------------------------
// y[e][s'] = sum_g sum_s O_g[s'][s] sum_f M_g[e][f] x[f][s]  (+ sum_s id[s'][s] x[e][s]): four rows per workgroup, two
// waves per row, every load of a row in flight at once.  Bound by that one round of loads
// and by the launch at these sizes: 7.0 us for two FP64 matrices at D = 6 (27 MB, 3.9 TB/s; one wave per row with the
// columns in three rounds 8.0 us, four rows' columns split over four waves 8.2 us), 3.9 us at D = 4 (1 MB).
template <typename T, int NG, int U>
__global__ void __launch_bounds__(FORMED_THREADS) formed_apply_kernel(FormedPlan f, const double* __restrict__ x,
                                                                     double* __restrict__ y) {
  __shared__ double red[16];
  const int row0 = blockIdx.x * FORMED_ROWS;
  FormedRows<T, NG, U> rows;
  rows.load(f, row0);
  rows.apply(f, row0, [&](int c, int s) { return x[2 * c + s]; }, red, y);
}

// The same for matrices of more than 11 x 128 columns: one wave per row.
template <typename T, int NG>
__global__ void __launch_bounds__(256) formed_apply_any_kernel(FormedPlan f, const double* __restrict__ x, double* __restrict__ y) {
  const int lane = threadIdx.x & 63, n = f.n_env, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= n) return;
  double acc[NG][2];
#pragma unroll
  for (int g = 0; g < NG; ++g) acc[g][0] = acc[g][1] = 0.0;
  for (int c = lane; c < n; c += 64) {
    const double x0 = x[2 * c], x1 = x[2 * c + 1];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const double m = (double)static_cast<const T*>(f.mat[g])[(int64_t)row * n + c];
      acc[g][0] += m * x0;
      acc[g][1] += m * x1;
    }
  }
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int s = 0; s < 2; ++s) acc[g][s] = cc_wave_sum(acc[g][s]);
  if (lane < 2) {
    double t = 0.0;
#pragma unroll
    for (int g = 0; g < NG; ++g) t += f.op[g][lane * 2] * acc[g][0] + f.op[g][lane * 2 + 1] * acc[g][1];
    if (f.has_id) t += f.id[lane * 2] * x[row * 2] + f.id[lane * 2 + 1] * x[row * 2 + 1];
    y[row * 2 + lane] = t;
  }
}

// No matrices: the operator is id (x) 1.
__global__ void formed_identity_kernel(FormedPlan f, const double* __restrict__ x, double* __restrict__ y) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < 2 * f.n_env) y[i] = f.id[(i & 1) * 2] * x[i & ~1] + f.id[(i & 1) * 2 + 1] * x[i | 1];
}

template <typename T, int NG>
void formed_launch_mats(hipStream_t st, const FormedPlan& f, const double* x, double* y) {
  const unsigned grid = (unsigned)((f.n_env + FORMED_ROWS - 1) / FORMED_ROWS);
  if (f.n_env <= 256) formed_apply_kernel<T, NG, 2><<<grid, FORMED_THREADS, 0, st>>>(f, x, y);
  else if (f.n_env <= 640) formed_apply_kernel<T, NG, 5><<<grid, FORMED_THREADS, 0, st>>>(f, x, y);
  else if (f.n_env <= 1408) formed_apply_kernel<T, NG, 11><<<grid, FORMED_THREADS, 0, st>>>(f, x, y);
  else formed_apply_any_kernel<T, NG><<<(unsigned)((f.n_env + 3) / 4), 256, 0, st>>>(f, x, y);
}
template <typename T>
int formed_launch(hipStream_t st, const FormedPlan& f, const double* x, double* y) {
  switch (f.n_mats) {
    case 0: formed_identity_kernel<<<(unsigned)((2 * f.n_env + 255) / 256), 256, 0, st>>>(f, x, y); break;
    case 1: formed_launch_mats<T, 1>(st, f, x, y); break;
    case 2: formed_launch_mats<T, 2>(st, f, x, y); break;
    case 3: formed_launch_mats<T, 3>(st, f, x, y); break;
    case 4: formed_launch_mats<T, 4>(st, f, x, y); break;
    default: formed_launch_mats<T, 5>(st, f, x, y); break;
  }
  CC_LAUNCH_CHECK();
  return CC_OK;
}
int formed_apply(hipStream_t st, const FormedPlan& f, const double* x, double* y) {
  hipEvent_t e0 = nullptr;
  int rc = cc_prof_start(st, CC_PROF_FORMED, &e0);
  if (rc) return rc;
  rc = f.f32 ? formed_launch<float>(st, f, x, y) : formed_launch<double>(st, f, x, y);
  return rc ? rc : cc_prof_stop(st, CC_PROF_FORMED, e0);
}
}  // namespace

int cc_internal_formed_apply(hipStream_t st, const void* plan, const double* x, double* y) {
  return formed_apply(st, *static_cast<const FormedPlan*>(plan), x, y);
}
int64_t cc_internal_formed_n(const void* plan) { return 2 * (int64_t) static_cast<const FormedPlan*>(plan)->n_env; }

extern "C" int cc_slab_join_f64(void* stream, int n_src, const double* const* src, const double* host_coef, int64_t na0,
                                int64_t na1, int64_t d0, int64_t d1, const int64_t* strides, double* out) {
  CCSlabMap map;
  int rc = cc_slab_map(na0, na1, d0, d1, strides, &map);
  if (rc) return rc;
  if (n_src < 1 || n_src > CC_SLAB_SOURCES) { cc_set_last_error("slab join: 1 to 8 sources"); return CC_ERR_ARG; }
  const CCSlabSum s = cc_slab_sum(n_src, src, host_coef);
  const int64_t n_alpha = na0 * na1, P = d0 * d1;
  const CCSlabGather g = cc_slab_gather(map, d0);
  const unsigned grid = (unsigned)(n_alpha < 16384 ? n_alpha : 16384);
  hipStream_t st = cc_stream(stream);
  if (d0 == d1 && d0 >= 2 && d0 <= 6) {
    switch (d0) {
      case 2: slab_join_kernel_d<2><<<grid, 256, 0, st>>>(n_alpha, g, s, out); break;
      case 3: slab_join_kernel_d<3><<<grid, 256, 0, st>>>(n_alpha, g, s, out); break;
      case 4: slab_join_kernel_d<4><<<grid, 256, 0, st>>>(n_alpha, g, s, out); break;
      case 5: slab_join_kernel_d<5><<<grid, 256, 0, st>>>(n_alpha, g, s, out); break;
      default: slab_join_kernel_d<6><<<grid, 256, 0, st>>>(n_alpha, g, s, out); break;
    }
  } else {
    slab_join_kernel<<<cc_blocks(n_alpha * P * P, 256), 256, 0, st>>>(n_alpha, P, map, s, out);
  }
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_form_work_size(int n_groups, int max_products, int64_t n_alpha, int64_t P, int64_t Q, int64_t* out) {
  if (n_groups < 1 || max_products < 1 || n_alpha < 1 || P < 1 || Q < 1) { cc_set_last_error("form: bad sizes"); return CC_ERR_ARG; }
  const int split = form_split(n_groups, max_products, n_alpha, P, Q);
  *out = split > 1 ? (int64_t)n_groups * split * P * P * Q * Q : 1;
  return CC_OK;
}

extern "C" int cc_form_f64(void* stream, int n_groups, const int* group_begin, const double* const* A, const double* const* B,
                           int64_t n_alpha, int64_t P, int64_t Q, double* out, double* work) {
  if (n_groups < 1 || n_groups > FORM_MAX || n_alpha < 1 || P < 1 || Q < 1 || P > 4096 || Q > 4096) {
    cc_set_last_error("form: bad sizes");
    return CC_ERR_ARG;
  }
  FormArgs f;
  int most = 0;
  f.n_groups = n_groups;
  for (int g = 0; g <= n_groups; ++g) {
    f.begin[g] = group_begin[g];
    if (group_begin[g] < 0 || group_begin[g] > FORM_MAX || (g > 0 && group_begin[g] <= group_begin[g - 1])) {
      cc_set_last_error("form: every group needs products, 16 in all at most");
      return CC_ERR_ARG;
    }
    if (g > 0 && group_begin[g] - group_begin[g - 1] > most) most = group_begin[g] - group_begin[g - 1];
  }
  for (int i = 0; i < FORM_MAX; ++i) {
    f.A[i] = A[i < group_begin[n_groups] ? i : 0];
    f.B[i] = B[i < group_begin[n_groups] ? i : 0];
  }
  f.n_alpha = n_alpha;
  f.P = (int)P;
  f.Q = (int)Q;
  f.tm = (int)((P * P + FT - 1) / FT);
  f.tn = (int)((Q * Q + FT - 1) / FT);
  f.split = form_split(n_groups, most, n_alpha, P, Q);
  hipStream_t st = cc_stream(stream);
  form_kernel<<<(unsigned)((int64_t)f.tm * f.tn * n_groups * f.split), 256, 0, st>>>(f, f.split > 1 ? work : out);
  CC_LAUNCH_CHECK();
  if (f.split > 1) {
    form_reduce_kernel<<<dim3((unsigned)(P * Q), (unsigned)n_groups), 256, 0, st>>>(f.split, f.P, f.Q, work, out);
    CC_LAUNCH_CHECK();
  }
  return CC_OK;
}

extern "C" int cc_whiten_f64(void* stream, int64_t n, int n_mats, const double* G, const double* Wt, double* K, double* work) {
  if (n < 1 || n_mats < 1) { cc_set_last_error("whiten: bad sizes"); return CC_ERR_ARG; }
  // work[c][i] = sum_{k <= i} G[k][c] W[i][k], then K[i][j] = sum_{c <= j} work[c][i] W[j][c]: both products with the
  // sum index slow in both operands, cut off at the diagonal of W
  int rc = cc_internal_gemm_upper(cc_stream(stream), n_mats, n, G, n * n, 1, n, Wt, n, work, n * n);
  if (rc) return rc;
  return cc_internal_gemm_upper(cc_stream(stream), n_mats, n, work, n * n, 1, n, Wt, n, K, n * n);
}

static int formed_plan_create(void** out, int64_t n_env, int64_t d, int n_mats, const void* const* mats, int f32,
                              const double* host_ops, const double* host_id) {
  *out = nullptr;
  if (d != 2 || n_env < 1 || n_env > 1 << 20 || n_mats < 0 || n_mats > FORMED_MATS || (n_mats == 0 && !host_id)) {
    cc_set_last_error("formed operator: d = 2 and at most 5 matrices");
    return CC_ERR_UNSUPPORTED;
  }
  FormedPlan* f = new FormedPlan();
  f->n_env = (int)n_env;
  f->n_mats = n_mats;
  f->has_id = host_id != nullptr;
  f->f32 = f32;
  for (int g = 0; g < n_mats; ++g) {
    f->mat[g] = mats[g];
    for (int e = 0; e < 4; ++e) f->op[g][e] = host_ops[4 * g + e];
  }
  for (int e = 0; e < 4; ++e) f->id[e] = host_id ? host_id[e] : 0.0;
  *out = f;
  return CC_OK;
}

extern "C" int cc_formed_plan_create(void** out, int64_t n_env, int64_t d, int n_mats, const double* const* mats,
                                     const double* host_ops, const double* host_id) {
  return formed_plan_create(out, n_env, d, n_mats, reinterpret_cast<const void* const*>(mats), 0, host_ops, host_id);
}

extern "C" int cc_formed_plan_create_f32(void** out, int64_t n_env, int64_t d, int n_mats, const float* const* mats,
                                         const double* host_ops, const double* host_id) {
  return formed_plan_create(out, n_env, d, n_mats, reinterpret_cast<const void* const*>(mats), 1, host_ops, host_id);
}

extern "C" int cc_formed_plan_apply(void* stream, const void* plan, const double* x, double* y) {
  if (!plan) { cc_set_last_error("null plan"); return CC_ERR_ARG; }
  return formed_apply(cc_stream(stream), *static_cast<const FormedPlan*>(plan), x, y);
}

extern "C" int cc_formed_plan_destroy(void* plan) {
  delete static_cast<FormedPlan*>(plan);
  return CC_OK;
}
