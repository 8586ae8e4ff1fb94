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

// Y[i][j] = act(sum_k X[i][k] W[j][k] + b[j]): one 16 x 16 MFMA tile per wave, 32 x 32 outputs per workgroup, the
// operands loaded straight from memory in fragment order, MLP_AHEAD K steps at a time.  X (M x K) and W (N x K) are FP16
// row-major, K % 16 == 0, N % 32 == 0; rows past M read the last row and are not written.  Writes Y (FP32) and, if Yh,
// its FP16 copy.  Bound by load latency (a layer's weights are 0.5 MB): at 256 rows, 512 x 512, 12.7 us with 64 x 64
// tiles through LDS (32 workgroups), 9.3 us here.  The sums run over K in order, so results do not depend on the tiling.
// Operand fragments: A[i][k] in lane i + 16(k/4), element k%4; B[k][j] in lane j + 16(k/4), element k%4;
// D[i][j] in lane j + 16(i/4), register i%4.
constexpr int MLP_AHEAD = 8;
__global__ void __launch_bounds__(256) mlp_linear_kernel(int64_t M, int64_t N, int64_t K, const _Float16* __restrict__ X,
                                                         const _Float16* __restrict__ W, const float* __restrict__ b,
                                                         int relu, float* __restrict__ Y, _Float16* __restrict__ Yh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t j = (int64_t)blockIdx.x * 32 + 16 * (wave & 1) + (lane & 15);
  const h4* wp = reinterpret_cast<const h4*>(W + j * K) + (lane >> 4);
  const int steps = (int)(K / 16);
  for (int64_t i0 = (int64_t)blockIdx.y * 32 + 16 * (wave >> 1); i0 < M; i0 += (int64_t)gridDim.y * 32) {
    const int64_t xi = i0 + (lane & 15) < M ? i0 + (lane & 15) : M - 1;
    const h4* xp = reinterpret_cast<const h4*>(X + xi * K) + (lane >> 4);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += MLP_AHEAD) {
      h4 xa[MLP_AHEAD], wb[MLP_AHEAD];
#pragma unroll
      for (int u = 0; u < MLP_AHEAD; ++u) {
        const int s = s0 + u < steps ? s0 + u : steps - 1;   // clamped; skipped below
        xa[u] = xp[4 * s];
        wb[u] = wp[4 * s];
      }
#pragma unroll
      for (int u = 0; u < MLP_AHEAD; ++u)
        if (s0 + u < steps) acc = __builtin_amdgcn_mfma_f32_16x16x16f16(xa[u], wb[u], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = i0 + 4 * (lane >> 4) + r;
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
// row-major.  A is stored M x K (`rows`: the gradient passed on, K % 64 == 0, any M) or K x M (a weight gradient,
// M % 64 == 0, any K).  `mask`: C is zeroed where mask[i][j] <= 0 (the activation the ReLU left).  `rowsum`: also
// receives sum_k A(i, k).
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

// element-aligned vectors: the pointers are a caller's
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef _Float16 h2u __attribute__((ext_vector_type(2), aligned(2)));

// One wave's part of a tile, K chunks c0 .. c1 of 16 each.  Chunk c is summed in the order k = 16 c + 4 g + u for lane
// group g at step u, so that a lane's four steps are neighbours in memory; rows and columns alternate between the two
// 16-wide tiles of a pair (2 (lane % 16) + t), so that one load feeds both.  MLP_CHUNKS chunks are loaded together.
// Rows past M and columns past N read the last ones and are not written; steps past K count as zero.
constexpr int MLP_CHUNKS = 4;
template <bool ROWS>
__device__ inline void mlp_grad_wave(const MlpJob& jb, int64_t i0, int64_t j0, int64_t c0, int64_t c1, int l, int g,
                                     f32x4 (&acc)[2][2], float (&rs)[2]) {
  const int64_t M = jb.M, N = jb.N, K = jb.K;
  const float* __restrict__ A = jb.A;
  const _Float16* __restrict__ B = jb.B + (j0 + 2 * l < N ? j0 + 2 * l : N - 2);   // N is even
  const int64_t r0 = i0 + 2 * l < M ? i0 + 2 * l : M - 1, r1 = i0 + 2 * l + 1 < M ? i0 + 2 * l + 1 : M - 1;
  for (int64_t c = c0; c < c1; c += MLP_CHUNKS) {
    float av[MLP_CHUNKS][2][4];
    h2u bv[MLP_CHUNKS][4];
#pragma unroll
    for (int q = 0; q < MLP_CHUNKS; ++q) {
      const int64_t k0 = 16 * (c + q < c1 ? c + q : c1 - 1) + 4 * g;
      if (ROWS) {
        const f4u x0 = *reinterpret_cast<const f4u*>(A + r0 * K + k0), x1 = *reinterpret_cast<const f4u*>(A + r1 * K + k0);
#pragma unroll
        for (int u = 0; u < 4; ++u) { av[q][0][u] = x0[u]; av[q][1][u] = x1[u]; }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t k = ROWS || k0 + u < K ? k0 + u : K - 1;
        bv[q][u] = *reinterpret_cast<const h2u*>(B + k * N);
        if (!ROWS) {
          const f2u x = *reinterpret_cast<const f2u*>(A + k * M + r0);
          av[q][0][u] = x[0];
          av[q][1][u] = x[1];
          if (k0 + u >= K) {
            av[q][0][u] = av[q][1][u] = 0.f;
            bv[q][u] = (h2u){0, 0};
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < MLP_CHUNKS; ++q) {
      if (c + q >= c1) break;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          rs[a] += av[q][a][u];
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[q][a][u], (float)bv[q][u][b], acc[a][b], 0, 0, 0);
        }
    }
  }
}

// Up to two products in one launch (a layer's weight gradient and the gradient passed on share their operand).  32 x 32
// outputs per workgroup on v_mfma_f32_16x16x4f32; the four waves take a quarter of K each, straight from memory, and
// are added in order through LDS, so that a product of 256 x 512 x 512 fills the chip and a wave's K loop is short.
// FP32 throughout; bound by load latency.  At 256 samples, widths 272-512-512-512, a whole backward pass takes 39 us (each
// launch 11.7 us); as FMA tiles on 64 to 128 workgroups (64 us a product), with the bias sums as one thread per column
// (36 us) and the masks as kernels of their own, it took 443 us; at 8192 samples a whole training step 1.01 ms for 10.8.
__global__ void __launch_bounds__(256) mlp_grad_kernel(const MlpJobs jobs) {
  __shared__ float part[4][32][33];
  __shared__ float rows[4][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 15, g = lane >> 4;
  for (int64_t t = blockIdx.x; t < jobs.tiles; t += gridDim.x) {
    const MlpJob& jb = jobs.job[t >= jobs.tiles0];
    const int64_t tile = t >= jobs.tiles0 ? t - jobs.tiles0 : t, tiles_n = (jb.N + 31) / 32, tn = tile % tiles_n;
    const int64_t i0 = tile / tiles_n * 32, j0 = tn * 32;
    const int64_t chunks = (jb.K + 15) / 16, c0 = chunks * wave / 4, c1 = chunks * (wave + 1) / 4;
    f32x4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float rs[2] = {0.f, 0.f};
    if (jb.rows) mlp_grad_wave<true>(jb, i0, j0, c0, c1, l, g, acc, rs);
    else mlp_grad_wave<false>(jb, i0, j0, c0, c1, l, g, acc, rs);
    __syncthreads();   // the previous tile's sums are read
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][2 * (4 * g + r) + a][2 * l + b] = acc[a][b][r];
      rs[a] += __shfl_xor(rs[a], 16, 64);
      rs[a] += __shfl_xor(rs[a], 32, 64);
      if (g == 0) rows[wave][2 * l + a] = rs[a];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * 32; e += 256) {
      const int i = e >> 5, j = e & 31;
      const int64_t gi = i0 + i, gj = j0 + j;
      if (gi < jb.M && gj < jb.N) {
        float v = ((part[0][i][j] + part[1][i][j]) + part[2][i][j]) + part[3][i][j];
        if (jb.mask && !(jb.mask[gi * jb.N + gj] > 0.f)) v = 0.f;
        jb.C[gi * jb.N + gj] = v;
      }
    }
    if (jb.rowsum && tn == 0 && threadIdx.x < 32)   // M % 64 == 0 where it is asked for
      jb.rowsum[i0 + threadIdx.x] =
          ((rows[0][threadIdx.x] + rows[1][threadIdx.x]) + rows[2][threadIdx.x]) + rows[3][threadIdx.x];
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
