// Learned warm start: a 3-layer MLP proposing the eigensolver's start vector, with its own training.
//
//   x (K0) -> h1 = relu(W1 x + b1) (H) -> h2 = relu(W2 h1 + b2) (H) -> y = W3 h2 + b3 (NO)
//
// Parameters live in one FP32 master buffer laid out [W1 (H x K0), b1 (H), W2 (H x H), b2 (H), W3 (NO x H),
// b3 (NO)] (weights row-major out x in) with an FP16 mirror.  The forward pass multiplies FP16 activations
// by FP16 weights on matrix cores (v_mfma_f32_16x16x16f16, FP32 accumulation) and keeps each hidden layer
// in FP32 and as the FP16 copy the next layer reads.  The backward pass is FP32 (FP32 matrix-core products
// over the same FP16 values the forward used), the loss is the sign-free misalignment 1 - (y.v)^2 / (|y|^2 |v|^2)
// with the converged state v, and Adam updates the FP32 master and refreshes the FP16 mirror.  All sums
// run in a fixed order.
#include "cc_common.h"

namespace {
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

struct MlpDims {
  int64_t K0, H, NO;
  int64_t w1, b1, w2, b2, w3, b3, total;
};
MlpDims mlp_dims(int64_t K0, int64_t H, int64_t NO) {
  MlpDims d;
  d.K0 = K0;
  d.H = H;
  d.NO = NO;
  d.w1 = 0;
  d.b1 = d.w1 + H * K0;
  d.w2 = d.b1 + H;
  d.b2 = d.w2 + H * H;
  d.w3 = d.b2 + H;
  d.b3 = d.w3 + NO * H;
  d.total = d.b3 + NO;
  return d;
}

// element-aligned vectors: the pointers are a caller's
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 h8u __attribute__((ext_vector_type(8), aligned(2)));

// Both products of this file: 32 x 32 outputs per workgroup, one 16 x 16 MFMA tile per wave, K in chunks through LDS.
// Their operands are small (half a megabyte per layer), so what counts is the wait for the first loads and the chain of
// a tile's matrix instructions: tiles small enough to reach every CU, MLP_AHEAD chunks of loads in flight.  Every sum
// runs over k in order (v_mfma_f32_16x16x4f32 rounds once per term, like an FMA chain), so results do not depend on
// the tiling.
constexpr int MLP_AHEAD = 4;

// Y[i][j] = act(sum_k X[i][k] W[j][k] + b[j]), X (M x K) and W (N x K) FP16 row-major, K % 16 == 0, N % 32 == 0; writes Y
// (FP32) and, if Yh, its FP16 copy.  At 256 rows, 512 x 512: 6.5 us; with 64 x 64 tiles (32 workgroups) and 16 k per
// step 12.7 us.  LDS rows of 136: a fragment read touches every bank once.
// Operand fragments: A[i][k] in lane i + 16(k/4), element k%4; B[k][j] in lane j + 16(k/4), element k%4;
// D[i][j] in lane j + 16(i/4), register i%4.
constexpr int MLP_FC = 128, MLP_FLD = MLP_FC + 8;
__global__ void __launch_bounds__(256) mlp_linear_kernel(int64_t M, int64_t N, int64_t K, const _Float16* __restrict__ X,
                                                         const _Float16* __restrict__ W, const float* __restrict__ b,
                                                         int relu, float* __restrict__ Y, _Float16* __restrict__ Yh) {
  __shared__ __attribute__((aligned(16))) _Float16 Xs[2][32 * MLP_FLD];
  __shared__ __attribute__((aligned(16))) _Float16 Ws[2][32 * MLP_FLD];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l = lane & 15, g = lane >> 4;
  const int row = t >> 3, kt = 16 * (t & 7), at = row * MLP_FLD + kt;
  const int x_from = (16 * (wave >> 1) + l) * MLP_FLD + 4 * g, w_from = (16 * (wave & 1) + l) * MLP_FLD + 4 * g;
  const int64_t chunks = (K + MLP_FC - 1) / MLP_FC, j = (int64_t)blockIdx.x * 32 + 16 * (wave & 1) + l;
  const _Float16* wp = W + ((int64_t)blockIdx.x * 32 + row) * K + kt;
  for (int64_t i0 = (int64_t)blockIdx.y * 32; i0 < M; i0 += (int64_t)gridDim.y * 32) {
    const _Float16* xp = X + (i0 + row) * K + kt;
    const bool in = i0 + row < M;
    h8u xr[MLP_AHEAD][2], wr[MLP_AHEAD][2];
    auto load = [&](h8u (&x)[2], h8u (&w)[2], int64_t c) {
      x[0] = x[1] = w[0] = w[1] = (h8u){0, 0, 0, 0, 0, 0, 0, 0};
      if (c * MLP_FC + kt < K) {
        w[0] = *reinterpret_cast<const h8u*>(wp + c * MLP_FC);
        w[1] = *reinterpret_cast<const h8u*>(wp + c * MLP_FC + 8);
        if (in) {
          x[0] = *reinterpret_cast<const h8u*>(xp + c * MLP_FC);
          x[1] = *reinterpret_cast<const h8u*>(xp + c * MLP_FC + 8);
        }
      }
    };
#pragma unroll
    for (int q = 0; q < MLP_AHEAD; ++q) load(xr[q], wr[q], q);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int64_t c0 = 0; c0 < chunks; c0 += MLP_AHEAD) {
#pragma unroll
      for (int q = 0; q < MLP_AHEAD; ++q) {
        const int64_t c = c0 + q;
        if (c >= chunks) break;
        _Float16* xs = Xs[q & 1];
        _Float16* ws = Ws[q & 1];
        *reinterpret_cast<h8u*>(xs + at) = xr[q][0];
        *reinterpret_cast<h8u*>(xs + at + 8) = xr[q][1];
        *reinterpret_cast<h8u*>(ws + at) = wr[q][0];
        *reinterpret_cast<h8u*>(ws + at + 8) = wr[q][1];
        __syncthreads();
        load(xr[q], wr[q], c + MLP_AHEAD);
#pragma unroll
        for (int s = 0; s < MLP_FC / 16; ++s)
          if (c * MLP_FC + 16 * s < K)
            acc = __builtin_amdgcn_mfma_f32_16x16x16f16(*reinterpret_cast<const h4*>(xs + x_from + 16 * s),
                                                        *reinterpret_cast<const h4*>(ws + w_from + 16 * s), acc, 0, 0, 0);
      }
    }
    __syncthreads();   // the next rows are written where these were read
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = i0 + 16 * (wave >> 1) + 4 * g + r;
      if (i < M) {
        float v = acc[r] + b[j];
        if (relu) v = v > 0.f ? v : 0.f;
        Y[i * N + j] = v;
        if (Yh) Yh[i * N + j] = (_Float16)v;
      }
    }
  }
}

// One product of the backward pass: C[i][j] = sum_k A(i, k) B[k][j], A FP32, B FP16 row-major with N columns, C
// row-major.  A is stored M x K (`rows`: the gradient passed on, K % 64 == 0, any M; C is zeroed where mask[i][j] <= 0,
// the activation the ReLU left) or K x M (a weight gradient, M % 64 == 0, any K; `rowsum` also receives sum_k A(i, k)).
struct MlpJob {
  int64_t M, N, K;
  const float* A;
  bool rows;
  const _Float16* B;
  float* C;
  const float* mask;
  float* rowsum;
};
struct MlpJobs {
  MlpJob job[2];
  int64_t tiles0, tiles;   // tiles of the first product, of all
};

// Up to two products in one launch (a layer's weight gradient and the gradient passed on share their operand), FP32 on
// v_mfma_f32_16x16x4f32; bias sums are a product with ones.  LDS rows: A stored M x K keeps k contiguous (stride 68), A
// stored K x M and B keep i and j contiguous (stride 48); both reads then touch every bank once.  At 256 samples, widths
// 272-512-512-512, a whole backward pass takes 29 us (6 to 14 us per launch); as FMA tiles on 64 to 128 workgroups (64 us a
// product), with the bias sums as one thread per column (36 us) and the masks as kernels of their own, 443 us; 8192 samples, a whole training step: 0.47 ms for 10.8.
constexpr int MLP_KC = 64, MLP_LDR = MLP_KC + 4, MLP_LDK = 48;

// One tile.  SUMS: also the row sums of A (the waves of the first columns, where they are asked for).
template <bool ROWS, bool SUMS>
__device__ inline void mlp_grad_tile(const MlpJob& jb, int64_t i0, int64_t j0, float (&As)[2][MLP_KC * MLP_LDK],
                                     float (&Bs)[2][MLP_KC * MLP_LDK]) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l = lane & 15, g = lane >> 4;
  const int wi = 16 * (wave >> 1), wj = 16 * (wave & 1);
  const int a_at = ROWS ? (t >> 3) * MLP_LDR + 8 * (t & 7) : (t >> 2) * MLP_LDK + 8 * (t & 3);
  const int b_at = (t >> 2) * MLP_LDK + 8 * (t & 3);
  const int a_from = ROWS ? (wi + l) * MLP_LDR + g : g * MLP_LDK + wi + l;
  constexpr int a_step = ROWS ? 4 : 4 * MLP_LDK;
  const int b_from = g * MLP_LDK + wj + l;
  // this thread's share of a chunk: eight values of A, eight columns of B's row t / 4; out of range: zero
  const int64_t K = jb.K, kb = t >> 2, N = jb.N, j8 = j0 + 8 * (t & 3), ia = ROWS ? i0 + (t >> 3) : i0 + 8 * (t & 3);
  const float* pa = ROWS ? jb.A + ia * K + 8 * (t & 7) : jb.A + kb * jb.M + ia;
  const int64_t a_next = ROWS ? MLP_KC : MLP_KC * jb.M, b_next = MLP_KC * N;
  const _Float16* pb = jb.B + kb * N + j8;
  const int64_t ka = ROWS ? (ia < jb.M ? 0 : K) : kb, kj = j8 < N ? kb : K;   // the first k this thread loads
  f4u a[MLP_AHEAD][2];
  h8u b[MLP_AHEAD];
  int64_t k0 = 0;   // of the next chunk to load
  auto load = [&](f4u (&x)[2], h8u& y) {
    x[0] = x[1] = (f4u){0.f, 0.f, 0.f, 0.f};
    y = (h8u){0, 0, 0, 0, 0, 0, 0, 0};
    if (k0 + ka < K) {
      x[0] = *reinterpret_cast<const f4u*>(pa);
      x[1] = *reinterpret_cast<const f4u*>(pa + 4);
    }
    if (k0 + kj < K) y = *reinterpret_cast<const h8u*>(pb);
    pa += a_next;
    pb += b_next;
    k0 += MLP_KC;
  };
#pragma unroll
  for (int q = 0; q < MLP_AHEAD; ++q) load(a[q], b[q]);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, sum = {0.f, 0.f, 0.f, 0.f};
  const int chunks = (int)((K + MLP_KC - 1) / MLP_KC);
  for (int c = 0; c < chunks; c += MLP_AHEAD) {
#pragma unroll
    for (int q = 0; q < MLP_AHEAD; ++q) {
      if (c + q >= chunks) break;
      float* as = As[q & 1];
      float* bs = Bs[q & 1];
      *reinterpret_cast<f32x4*>(as + a_at) = a[q][0];
      *reinterpret_cast<f32x4*>(as + a_at + 4) = a[q][1];
      *reinterpret_cast<f32x4*>(bs + b_at) = (f32x4){(float)b[q][0], (float)b[q][1], (float)b[q][2], (float)b[q][3]};
      *reinterpret_cast<f32x4*>(bs + b_at + 4) = (f32x4){(float)b[q][4], (float)b[q][5], (float)b[q][6], (float)b[q][7]};
      __syncthreads();
      load(a[q], b[q]);
#pragma unroll
      for (int s = 0; s < MLP_KC / 4; ++s) {
        const float x = as[a_from + s * a_step], y = bs[b_from + s * 4 * MLP_LDK];
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc, 0, 0, 0);
        if (SUMS) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x, 1.f, sum, 0, 0, 0);
      }
    }
  }
  const int64_t j = j0 + wj + l;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t i = i0 + wi + 4 * g + r;
    if (i < jb.M && j < N) {
      float v = acc[r];
      if (ROWS && !(jb.mask[i * N + j] > 0.f)) v = 0.f;
      jb.C[i * N + j] = v;
    }
    if (SUMS && wj == 0 && l == 0) jb.rowsum[i] = sum[r];   // M % 64 == 0
  }
}

__global__ void __launch_bounds__(256) mlp_grad_kernel(const MlpJobs jobs) {
  __shared__ __attribute__((aligned(16))) float As[2][MLP_KC * MLP_LDK];
  __shared__ __attribute__((aligned(16))) float Bs[2][MLP_KC * MLP_LDK];
  static_assert(32 * MLP_LDR <= MLP_KC * MLP_LDK, "both layouts of A fit");
  for (int64_t u = blockIdx.x; u < jobs.tiles; u += gridDim.x) {
    const MlpJob jb = u >= jobs.tiles0 ? jobs.job[1] : jobs.job[0];
    const int64_t tile = u >= jobs.tiles0 ? u - jobs.tiles0 : u, tiles_n = (jb.N + 31) / 32;
    const int64_t i0 = tile / tiles_n * 32, j0 = tile % tiles_n * 32;
    if (jb.rows) mlp_grad_tile<true, false>(jb, i0, j0, As, Bs);
    else if (j0 == 0) mlp_grad_tile<false, true>(jb, i0, j0, As, Bs);
    else mlp_grad_tile<false, false>(jb, i0, j0, As, Bs);
    __syncthreads();   // the next tile writes where this one's last chunks were read
  }
}

// Per sample b (one 256-thread workgroup): loss[b] = 1 - (y.v)^2 / (|y|^2 |v|^2) and
// dY[b] = scale * d loss / d y = scale * (2 (y.v)^2 / (|y|^4 |v|^2) y - 2 (y.v) / (|y|^2 |v|^2) v).
__global__ void __launch_bounds__(256) mlp_loss_kernel(int64_t NO, const float* __restrict__ Y, const float* __restrict__ V,
                                                       float scale, float* __restrict__ loss, float* __restrict__ dY) {
  __shared__ float red[3][4];
  const int64_t b = blockIdx.x;
  const float* y = Y + b * NO;
  const float* v = V + b * NO;
  float yy = 0.f, vv = 0.f, yv = 0.f;
  for (int64_t i = threadIdx.x; i < NO; i += 256) {
    yy += y[i] * y[i];
    vv += v[i] * v[i];
    yv += y[i] * v[i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    yy += __shfl_xor(yy, o, 64);
    vv += __shfl_xor(vv, o, 64);
    yv += __shfl_xor(yv, o, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wave] = yy;
    red[1][wave] = vv;
    red[2][wave] = yv;
  }
  __syncthreads();
  yy = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
  vv = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
  yv = ((red[2][0] + red[2][1]) + red[2][2]) + red[2][3];
  const float yyc = fmaxf(yy, 1e-30f), vvc = fmaxf(vv, 1e-30f);
  const float cy = scale * 2.f * yv * yv / (yyc * yyc * vvc), cv = -scale * 2.f * yv / (yyc * vvc);
  for (int64_t i = threadIdx.x; i < NO; i += 256) dY[b * NO + i] = cy * y[i] + cv * v[i];
  if (threadIdx.x == 0) loss[b] = 1.f - yv * yv / (yyc * vvc);
}

// Adam on the FP32 master parameters with bias correction; refreshes the FP16 mirror.
__global__ void mlp_adam_kernel(int64_t n, float* __restrict__ P, const float* __restrict__ G, float* __restrict__ Mv,
                                float* __restrict__ Vv, _Float16* __restrict__ P16, float lr, float b1, float b2, float eps,
                                float c1, float c2) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const float g = G[e];
    const float m = b1 * Mv[e] + (1.f - b1) * g, v = b2 * Vv[e] + (1.f - b2) * g * g;
    Mv[e] = m;
    Vv[e] = v;
    const float p = P[e] - lr * (m / c1) / (sqrtf(v / c2) + eps);
    P[e] = p;
    P16[e] = (_Float16)p;
  }
}

// One feature row: each of the n_spec spectra (k singular values, descending) divided by its largest value,
// then h, zero padding to K0; FP16.
__global__ void mlp_features_kernel(int n_spec, int k, const double* __restrict__ S, double h, int64_t K0,
                                    _Float16* __restrict__ out) {
  for (int64_t e = threadIdx.x; e < K0; e += blockDim.x) {
    float v = 0.f;
    if (e < (int64_t)n_spec * k) {
      const int sp = (int)(e / k);
      const double top = S[(int64_t)sp * k];
      v = top > 0.0 ? (float)(S[e] / top) : 0.f;
    } else if (e == (int64_t)n_spec * k) {
      v = (float)h;
    }
    out[e] = (_Float16)v;
  }
}

int mlp_grad(hipStream_t st, const MlpJob& first, const MlpJob* second) {
  MlpJobs jobs = {};
  jobs.job[0] = first;
  jobs.tiles0 = jobs.tiles = (first.M + 31) / 32 * ((first.N + 31) / 32);
  if (second) {
    jobs.job[1] = *second;
    jobs.tiles += (second->M + 31) / 32 * ((second->N + 31) / 32);
  }
  mlp_grad_kernel<<<(unsigned)(jobs.tiles < 65536 ? jobs.tiles : 65536), 256, 0, st>>>(jobs);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

int check_dims(int64_t B, int64_t K0, int64_t H, int64_t NO) {
  if (B < 1 || K0 < 16 || K0 % 16 || H < 64 || H % 64 || NO < 64 || NO % 64) {
    cc_set_last_error("mlp: need batch >= 1, K0 % 16 == 0, H and NO multiples of 64");
    return CC_ERR_DIM;
  }
  return CC_OK;
}
}  // namespace

extern "C" int cc_mlp_param_count(int64_t K0, int64_t H, int64_t NO, int64_t* out) {
  *out = mlp_dims(K0, H, NO).total;
  return CC_OK;
}

extern "C" int cc_mlp_features(void* stream, int n_spec, int k, const double* S, double h, int64_t K0, void* out16) {
  if (n_spec < 1 || k < 1 || (int64_t)n_spec * k + 1 > K0) {
    cc_set_last_error("mlp features: K0 must hold n_spec * k + 1 values");
    return CC_ERR_DIM;
  }
  mlp_features_kernel<<<1, 256, 0, cc_stream(stream)>>>(n_spec, k, S, h, K0, static_cast<_Float16*>(out16));
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_mlp_forward(void* stream, int64_t B, int64_t K0, int64_t H, int64_t NO, const void* P16, const float* P32,
                              const void* X16, void* A16, float* A32, float* Y) {
  int rc = check_dims(B, K0, H, NO);
  if (rc) return rc;
  hipStream_t st = cc_stream(stream);
  const MlpDims d = mlp_dims(K0, H, NO);
  const _Float16* p = static_cast<const _Float16*>(P16);
  _Float16* h1h = static_cast<_Float16*>(A16);
  _Float16* h2h = h1h + B * H;
  float* h1 = A32;
  float* h2 = A32 + B * H;
  const unsigned gy = (unsigned)(B < 32 * 65535LL ? (B + 31) / 32 : 65535);
  mlp_linear_kernel<<<dim3((unsigned)(H / 32), gy), 256, 0, st>>>(B, H, K0, static_cast<const _Float16*>(X16), p + d.w1,
                                                                  P32 + d.b1, 1, h1, h1h);
  CC_LAUNCH_CHECK();
  mlp_linear_kernel<<<dim3((unsigned)(H / 32), gy), 256, 0, st>>>(B, H, H, h1h, p + d.w2, P32 + d.b2, 1, h2, h2h);
  CC_LAUNCH_CHECK();
  mlp_linear_kernel<<<dim3((unsigned)(NO / 32), gy), 256, 0, st>>>(B, NO, H, h2h, p + d.w3, P32 + d.b3, 0, Y, nullptr);
  CC_LAUNCH_CHECK();
  return CC_OK;
}

extern "C" int cc_mlp_work_size(int64_t B, int64_t H, int64_t NO, int64_t* out) {
  *out = B * NO + 2 * B * H;  // floats: dY, dZ2, dZ1
  return CC_OK;
}

extern "C" int cc_mlp_backward(void* stream, int64_t B, int64_t K0, int64_t H, int64_t NO, const void* P16,
                               const void* X16, const void* A16, const float* A32, const float* Y, const float* target,
                               float* loss, float* G, float* work) {
  int rc = check_dims(B, K0, H, NO);
  if (rc) return rc;
  hipStream_t st = cc_stream(stream);
  const MlpDims d = mlp_dims(K0, H, NO);
  const _Float16* p = static_cast<const _Float16*>(P16);
  const _Float16* x = static_cast<const _Float16*>(X16);
  const _Float16* h1h = static_cast<const _Float16*>(A16);
  const _Float16* h2h = h1h + B * H;
  const float* h1 = A32;
  const float* h2 = A32 + B * H;
  float* dY = work;
  float* dZ2 = dY + B * NO;
  float* dZ1 = dZ2 + B * H;
  mlp_loss_kernel<<<(unsigned)B, 256, 0, st>>>(NO, Y, target, 1.f / (float)B, loss, dY);
  CC_LAUNCH_CHECK();
  // per layer: dW = dZ^T h with its bias sums, and the gradient passed on, dZ W where the activation is positive
  const MlpJob w3 = {NO, H, B, dY, false, h2h, G + d.w3, nullptr, G + d.b3};
  const MlpJob z2 = {B, H, NO, dY, true, p + d.w3, dZ2, h2, nullptr};
  if ((rc = mlp_grad(st, w3, &z2))) return rc;
  const MlpJob w2 = {H, H, B, dZ2, false, h1h, G + d.w2, nullptr, G + d.b2};
  const MlpJob z1 = {B, H, H, dZ2, true, p + d.w2, dZ1, h1, nullptr};
  if ((rc = mlp_grad(st, w2, &z1))) return rc;
  const MlpJob w1 = {H, K0, B, dZ1, false, x, G + d.w1, nullptr, G + d.b1};
  return mlp_grad(st, w1, nullptr);
}

extern "C" int cc_mlp_adam(void* stream, int64_t n, float* P32, const float* G, float* M, float* V, void* P16, double lr,
                           double beta1, double beta2, double eps, int64_t step) {
  if (step < 1) { cc_set_last_error("mlp adam: step counts from 1"); return CC_ERR_ARG; }
  const float c1 = (float)(1.0 - pow(beta1, (double)step)), c2 = (float)(1.0 - pow(beta2, (double)step));
  mlp_adam_kernel<<<cc_blocks(n, 256), 256, 0, cc_stream(stream)>>>(n, P32, G, M, V, static_cast<_Float16*>(P16),
                                                                    (float)lr, (float)beta1, (float)beta2, (float)eps, c1, c2);
  CC_LAUNCH_CHECK();
  return CC_OK;
}
