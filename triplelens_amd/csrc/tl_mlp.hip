// Kernels of the surrogate network (tl_mlp.h).
//
// The products use v_mfma_f32_16x16x16_bf16.  Its operands, per lane l of the
// wavefront: A row (l % 16) with k = 4 (l / 16) + j, B column (l % 16) with the
// same k, j = 0..3; the accumulator holds column (l % 16), rows 4 (l / 16) + j.
// A sum over K is a chain of these products in k order.
//
// The network is small (200k parameters; a batch of 1024 rows is 1.2 GFLOP of
// training), so what bounds it is the number of launches and the latency of
// each layer, not the matrix cores.  A row's activations and gradients depend
// on other rows only through the weight gradients: one workgroup carries 16
// rows through all layers forward and back with the activations in LDS, and
// a second launch forms every layer's weight gradient and takes the Adam step
// with it.  Measured, against a launch per layer and product (with 2-byte
// loads) and per pass over the parameters: the kernels of a training step of
// 1024 rows 533 -> 41 us in 2 launches instead of 25, those of an inference of
// 4096 rows 160 -> 14.5 us in one.
#include <hip/hip_runtime.h>
#include <math.h>

#include "tl_mlp.h"

namespace tl {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr size_t mlp_w(int l) {
  size_t off = 0;
  for (int k = 0; k < l; k++) off += (size_t)mlp_K(k) * mlp_N(k) + mlp_N(k);
  return off;
}
constexpr size_t mlp_b(int l) { return mlp_w(l) + (size_t)mlp_K(l) * mlp_N(l); }
constexpr size_t kMlpTotal = mlp_b(kMlpLayers - 1) + mlp_N(kMlpLayers - 1);

MlpLayout mlp_layout() {
  MlpLayout L;
  for (int l = 0; l < kMlpLayers; l++) {
    L.K[l] = mlp_K(l);
    L.N[l] = mlp_N(l);
    L.w[l] = mlp_w(l);
    L.b[l] = mlp_b(l);
  }
  L.total = kMlpTotal;
  return L;
}

__device__ __forceinline__ uint16_t f2bf(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((unsigned)h << 16); }

// GELU(z) and its derivative, e = erf(z / sqrt 2)
__device__ __forceinline__ float gelu_erf(float z) { return erff(z * 0.70710678118654752f); }
__device__ __forceinline__ float gelu(float z, float e) { return 0.5f * z * (1.0f + e); }
__device__ __forceinline__ float gelu_d(float z, float e) {
  return 0.5f * (1.0f + e) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// The orders of the operands in memory.  A product of length K reads, per lane,
// the fragments of its steps: with K = 256 two steps' (16 bytes) at once, so
// that a wavefront's load is 1 KB in a row.  Measured against row-major copies
// (8-byte loads from 16 rows) with 1024 rows: row kernel 58.7 -> 22.0 us, weight
// gradients 36.3 -> 19.5 us.
//   frag_at: element k of column c of a weight operand.
//   part_at: element (row r of the batch, column c) of a layer's input or
//   gradient, a fragment of the weight gradients' products over the rows.
__host__ __device__ __forceinline__ size_t frag_at(int K, int c, int k) {
  const int lane = (c & 15) + 16 * ((k & 15) >> 2);
  if (K == 16) return ((size_t)(c >> 4) * 64 + lane) * 4 + (k & 3);
  return (((size_t)(c >> 4) * (K / 32) + (k >> 5)) * 64 + lane) * 8 + ((k >> 4) & 1) * 4 + (k & 3);
}
__host__ __device__ __forceinline__ size_t part_at(int rows, int r, int c) {
  const int lane = (c & 15) + 16 * ((r & 15) >> 2);
  return ((size_t)(c >> 4) * (rows >> 4) + (r >> 4)) * 256 + lane * 4 + (r & 3);
}

// Four consecutive elements of a fragment.
__device__ __forceinline__ void store4(uint16_t* p, const uint16_t (&v)[4]) {
  *reinterpret_cast<bf16x4*>(p) = bf16x4{(short)v[0], (short)v[1], (short)v[2], (short)v[3]};
}

// ---- rows: forward (and backward) ------------------------------------------
constexpr int kRowWaves = 16;        // wavefront w owns columns 16 w .. 16 w + 15
constexpr int kLdAct = 256 + 8;      // LDS row of activations: rows start 4 banks apart

// The B operand of column tile `tile`, the whole K range.
template <int K>
struct BFrag {
  bf16x4 v[K / 16];
};
template <int K>
__device__ __forceinline__ BFrag<K> load_b(const uint16_t* src, int tile, int ln) {
  BFrag<K> f;
  if (K == 16) {
    f.v[0] = *reinterpret_cast<const bf16x4*>(src + ((size_t)tile * 64 + ln) * 4);
  } else {
#pragma unroll
    for (int s = 0; s < K / 32; s++) {
      const bf16x8 t =
          *reinterpret_cast<const bf16x8*>(src + (((size_t)tile * (K / 32) + s) * 64 + ln) * 8);
      f.v[2 * s] = __builtin_shufflevector(t, t, 0, 1, 2, 3);
      f.v[2 * s + 1] = __builtin_shufflevector(t, t, 4, 5, 6, 7);
    }
  }
  return f;
}
template <int K>
__device__ __forceinline__ f32x4 row_product(const uint16_t* act, int lr, int lk,
                                             const BFrag<K>& b) {
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < K / 16; s++)
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
        *reinterpret_cast<const bf16x4*>(act + (size_t)lr * kLdAct + 16 * s + lk), b.v[s], acc, 0,
        0, 0);
  return acc;
}

struct RowArgs {
  MlpWeights w;
  const float* x;
  int n;        // rows
  float* out;   // inference: n x 2
  MlpTrainRows t;
};

// One workgroup carries 16 rows through the network.  A layer's weights are
// loaded before the barrier that ends the layer before it.
template <bool TRAIN>
__global__ void __launch_bounds__(64 * kRowWaves) mlp_rows_kernel(RowArgs a) {
  __shared__ __align__(16) uint16_t act[2][kMlpTile][kLdAct];
  __shared__ float outv[kMlpTile][kMlpOutPad];
  const int tid = threadIdx.x, ln = tid & 63, w = tid >> 6;
  const int lr = ln & 15, lk = (ln >> 4) * 4;
  const int row0 = blockIdx.x * kMlpTile, col = 16 * w + lr;
  const MlpWeights W = a.w;
  const int rows = a.t.rows;
  const BFrag<16> b0 = load_b<16>(W.pbF + mlp_w(0), w, ln);
  BFrag<256> b = load_b<256>(W.pbF + mlp_w(1), w, ln);
  if (tid < kMlpTile * kMlpInPad) {
    const int r = tid / kMlpInPad, f = tid % kMlpInPad, row = row0 + r;
    uint16_t v = 0;
    if (row < a.n && f < kMlpIn) {
      const int src = TRAIN && a.t.idx ? a.t.idx[row] : row;
      v = f2bf((a.x[(size_t)src * kMlpIn + f] - W.mean[f]) / W.scale[f]);
    }
    act[0][r][f] = v;
    if (TRAIN) a.t.h[0][part_at(rows, row, f)] = v;
  }
  __syncthreads();
  float gd[kMlpLayers - 1][4];  // GELU'(Z_l)
#pragma unroll
  for (int l = 0; l < kMlpLayers - 1; l++) {
    const f32x4 acc = l == 0 ? row_product<16>(&act[0][0][0], lr, lk, b0)
                             : row_product<256>(&act[l & 1][0][0], lr, lk, b);
    if (l >= 1 && l < kMlpLayers - 2) b = load_b<256>(W.pbF + mlp_w(l + 1), w, ln);
    if (l == kMlpLayers - 2 && w == 0) b = load_b<256>(W.pbF + mlp_w(l + 1), 0, ln);
    const float bias = W.p[mlp_b(l) + col];
    uint16_t h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float z = acc[j] + bias, e = gelu_erf(z);
      h[j] = f2bf(gelu(z, e));
      if (TRAIN) gd[l][j] = gelu_d(z, e);
      act[(l + 1) & 1][lk + j][col] = h[j];
    }
    if (TRAIN) store4(a.t.h[l + 1] + part_at(rows, row0 + lk, col), h);
    __syncthreads();
  }
  constexpr int last = kMlpLayers - 1;  // its input is act[last & 1]
  if (w == 0) {
    const f32x4 acc = row_product<256>(&act[last & 1][0][0], lr, lk, b);
    const float bias = W.p[mlp_b(last) + lr];
    for (int j = 0; j < 4; j++) outv[lk + j][lr] = acc[j] + bias;
  }
  if (!TRAIN) {
    __syncthreads();
    if (tid < kMlpTile * kMlpOut && row0 + tid / kMlpOut < a.n)
      a.out[(size_t)row0 * kMlpOut + tid] = outv[tid / kMlpOut][tid % kMlpOut];
    return;
  }
  const BFrag<16> d4 = load_b<16>(W.pbB + mlp_w(last), w, ln);
  b = load_b<256>(W.pbB + mlp_w(last - 1), w, ln);
  __syncthreads();
  // Gaussian NLL 0.5 ((y - mu) e^-s)^2 + s, mean over the batch's rows; s
  // clamped to [-12, 12] (its gradient is zero outside)
  if (w == 0) {
    float l = 0.0f;
    if (ln < kMlpTile) {
      const int row = row0 + ln;
      const float mu = outv[ln][0], s0 = outv[ln][1];
      const float s = fminf(12.0f, fmaxf(-12.0f, s0));
      const float r = a.t.y[a.t.idx ? a.t.idx[row] : row] - mu, e = expf(-2.0f * s);
      l = 0.5f * r * r * e + s;
      const float inv = 1.0f / (float)a.t.rows;
      const float dmu = -r * e * inv;
      const float ds = (s0 == s) ? (1.0f - r * r * e) * inv : 0.0f;
      for (int n = 0; n < kMlpOutPad; n++) {
        const uint16_t v = n == 0 ? f2bf(dmu) : (n == 1 ? f2bf(ds) : (uint16_t)0);
        act[(last + 1) & 1][ln][n] = v;
        a.t.dz[last][part_at(rows, row, n)] = v;
      }
    }
    for (int o = 8; o >= 1; o >>= 1) l += __shfl_xor(l, o, 64);
    if (ln == 0) atomicAdd(a.t.loss, l / (float)a.t.rows);
  }
  __syncthreads();
  // dZ_{l-1} = (dZ_l W_l^T) * GELU'(Z_{l-1})
#pragma unroll
  for (int l = last; l >= 1; l--) {
    const f32x4 acc = l == last ? row_product<16>(&act[(l + 1) & 1][0][0], lr, lk, d4)
                                : row_product<256>(&act[(l + 1) & 1][0][0], lr, lk, b);
    if (l < last && l > 1) b = load_b<256>(W.pbB + mlp_w(l - 1), w, ln);
    uint16_t d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      d[j] = f2bf(acc[j] * gd[l - 1][j]);
      act[l & 1][lk + j][col] = d[j];
    }
    store4(a.t.dz[l - 1] + part_at(rows, row0 + lk, col), d);
    __syncthreads();
  }
}

int launch_mlp_predict(const MlpWeights& w, const float* x, int n, float* out, hipStream_t s) {
  if (n <= 0) return 0;
  RowArgs a = {};
  a.w = w;
  a.x = x;
  a.n = n;
  a.out = out;
  hipLaunchKernelGGL(mlp_rows_kernel<false>, dim3((n + kMlpTile - 1) / kMlpTile),
                     dim3(64 * kRowWaves), 0, s, a);
  return (int)hipGetLastError();
}

int launch_mlp_train_rows(const MlpWeights& w, const MlpTrainRows& t, hipStream_t s) {
  if (t.rows <= 0 || t.rows % kMlpTile) return (int)hipErrorInvalidValue;
  RowArgs a = {};
  a.w = w;
  a.x = t.x;
  a.n = t.rows;
  a.t = t;
  hipLaunchKernelGGL(mlp_rows_kernel<true>, dim3(t.rows / kMlpTile), dim3(64 * kRowWaves), 0, s,
                     a);
  return (int)hipGetLastError();
}

// ---- weight gradients and Adam ----------------------------------------------
struct GradArgs {
  MlpTrainRows t;
  float* g;
  MlpAdam a;
};

// Parameter i's old values (none where the gradient is stored) and what its
// gradient does: it is stored, or Adam's step is taken with it; returns the
// updated weight.
struct Old {
  float p, m, v;
};
template <bool ADAM>
__device__ __forceinline__ Old old_at(const GradArgs& A, size_t i) {
  if (!ADAM) return Old{};
  return {A.a.p[i], A.a.m[i], A.a.v[i]};
}
template <bool ADAM>
__device__ __forceinline__ float use_grad(const GradArgs& A, size_t i, const Old& o, float gi) {
  if (!ADAM) {
    A.g[i] = gi;
    return 0.0f;
  }
  const MlpAdam& a = A.a;
  const float mi = a.b1 * o.m + (1.0f - a.b1) * gi;
  const float vi = a.b2 * o.v + (1.0f - a.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float w = o.p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  a.p[i] = w;
  return w;
}

// One wavefront's tile of dW_l: rows k0 .. k0 + 16 MT, columns n0 .. n0 + 16 NT,
// the sum over the batch's rows in order.  The next eight blocks of 16 rows
// are loaded while the current ones are multiplied.
constexpr int kGradAhead = 8;
template <int MT, int NT>
struct Blocks {
  bf16x4 a[kGradAhead][MT], b[kGradAhead][NT];
};

template <bool ADAM, int MT, int NT>
__device__ __forceinline__ void grad_tile(const GradArgs& A, int l, int k0, int n0) {
  const int ln = threadIdx.x & 63, lr = ln & 15, lk = (ln >> 4) * 4;
  const int rows = A.t.rows, nb = rows >> 4, K = mlp_K(l), N = mlp_N(l);
  const size_t off = mlp_w(l);
  const uint16_t* pa = A.t.h[l] + (size_t)(k0 >> 4) * nb * 256 + ln * 4;
  const uint16_t* pb = A.t.dz[l] + (size_t)(n0 >> 4) * nb * 256 + ln * 4;
  auto load = [&](Blocks<MT, NT>& f, int s0) {
#pragma unroll
    for (int u = 0; u < kGradAhead; u++)
      if (s0 + u < nb) {
#pragma unroll
        for (int t = 0; t < MT; t++)
          f.a[u][t] = *reinterpret_cast<const bf16x4*>(pa + ((size_t)t * nb + s0 + u) * 256);
#pragma unroll
        for (int t = 0; t < NT; t++)
          f.b[u][t] = *reinterpret_cast<const bf16x4*>(pb + ((size_t)t * nb + s0 + u) * 256);
      }
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Blocks<MT, NT>& f, int s0) {
#pragma unroll
    for (int u = 0; u < kGradAhead; u++)
      if (s0 + u < nb) {
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
          for (int b = 0; b < NT; b++)
            acc[a][b] =
                __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(f.a[u][a], f.b[u][b], acc[a][b], 0, 0, 0);
      }
  };
  Blocks<MT, NT> f0, f1;
  load(f0, 0);
  Old old[MT][NT][4];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        old[a][b][j] = old_at<ADAM>(A, off + (size_t)(k0 + 16 * a + lk + j) * N + n0 + 16 * b + lr);
  for (int s0 = 0; s0 < nb; s0 += 2 * kGradAhead) {
    load(f1, s0 + kGradAhead);
    multiply(f0, s0);
    load(f0, s0 + 2 * kGradAhead);
    multiply(f1, s0 + kGradAhead);
  }
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++) {
      const int n = n0 + 16 * b + lr, k = k0 + 16 * a + lk;
      uint16_t h[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        h[j] = f2bf(use_grad<ADAM>(A, off + (size_t)(k + j) * N + n, old[a][b][j], acc[a][b][j]));
        if (ADAM) A.a.pbB[off + frag_at(N, k + j, n)] = h[j];
      }
      if (ADAM) store4(A.a.pbF + off + frag_at(K, n, k), h);
    }
}

// 16 columns of db_l by one wavefront: 256 partial sums per column (of rows
// equal modulo 256) and a tree over them.
template <bool ADAM>
__device__ __forceinline__ void grad_bias(const GradArgs& A, int l, int n0) {
  const int ln = threadIdx.x & 63, nb = A.t.rows >> 4;
  const uint16_t* d = A.t.dz[l] + (size_t)(n0 >> 4) * nb * 256 + ln * 4;
  const size_t i = mlp_b(l) + n0 + (ln & 15);
  const Old old = old_at<ADAM>(A, i);
  float s[16][4];
#pragma unroll
  for (int u = 0; u < 16; u++)
#pragma unroll
    for (int j = 0; j < 4; j++) s[u][j] = 0.0f;
  for (int s0 = 0; s0 < nb; s0 += 16) {
#pragma unroll
    for (int u = 0; u < 16; u++)
      if (s0 + u < nb) {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(d + (size_t)(s0 + u) * 256);
#pragma unroll
        for (int j = 0; j < 4; j++) s[u][j] += bf2f((uint16_t)v[j]);
      }
  }
#pragma unroll
  for (int o = 8; o >= 1; o >>= 1)
#pragma unroll
    for (int u = 0; u < o; u++)
#pragma unroll
      for (int j = 0; j < 4; j++) s[u][j] += s[u + o][j];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    s[0][j] += __shfl_down(s[0][j], 32, 64);
    s[0][j] += __shfl_down(s[0][j], 16, 64);
  }
  const float g = (s[0][0] + s[0][2]) + (s[0][1] + s[0][3]);
  if (ln < 16) use_grad<ADAM>(A, i, old, g);
}

constexpr int kUnits0 = 8;                 // layer 0: 16 x 32 tiles
constexpr int kUnitsH = 64;                // layers 1-3: 32 x 32 tiles
constexpr int kUnits4 = 8;                 // layer 4: 32 x 16 tiles
constexpr int kTileUnits = kUnits0 + 3 * kUnitsH + kUnits4;
constexpr int kBiasUnits = 4 * (kMlpHidden / 16) + kMlpOutPad / 16;

// One wavefront per tile of a layer's weights or 16 columns of its bias, a
// workgroup each: 273 of them, one or two on every CU.
template <bool ADAM>
__global__ void __launch_bounds__(64) mlp_grad_kernel(GradArgs A) {
  int u = blockIdx.x;
  if (u < 3 * kUnitsH)
    return grad_tile<ADAM, 2, 2>(A, 1 + u / kUnitsH, 32 * (u % kUnitsH / 8), 32 * (u % 8));
  u -= 3 * kUnitsH;
  if (u < kUnits0) return grad_tile<ADAM, 1, 2>(A, 0, 0, 32 * u);
  u -= kUnits0;
  if (u < kUnits4) return grad_tile<ADAM, 2, 1>(A, 4, 32 * u, 0);
  u -= kUnits4;
  grad_bias<ADAM>(A, u / (kMlpHidden / 16), 16 * (u % (kMlpHidden / 16)));
}

int launch_mlp_grads(const MlpTrainRows& t, float* g, const MlpAdam& a, hipStream_t s) {
  if (t.rows <= 0 || t.rows % kMlpTile) return (int)hipErrorInvalidValue;
  GradArgs A = {t, g, a};
  const dim3 grid(kTileUnits + kBiasUnits);
  if (g)
    hipLaunchKernelGGL(mlp_grad_kernel<false>, grid, dim3(64), 0, s, A);
  else
    hipLaunchKernelGGL(mlp_grad_kernel<true>, grid, dim3(64), 0, s, A);
  return (int)hipGetLastError();
}

__global__ void mlp_copies_kernel(const float* p, uint16_t* pbF, uint16_t* pbB) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  for (int l = 0; l < kMlpLayers; l++) {
    const int K = mlp_K(l), N = mlp_N(l);
    const size_t off = mlp_w(l);
    if (i < off || i >= off + (size_t)K * N) continue;
    const int k = (int)((i - off) / N), n = (int)((i - off) % N);
    const uint16_t h = f2bf(p[i]);
    pbF[off + frag_at(K, n, k)] = h;
    pbB[off + frag_at(N, k, n)] = h;
  }
}

int launch_mlp_copies(const float* p, uint16_t* pbF, uint16_t* pbB, hipStream_t s) {
  hipLaunchKernelGGL(mlp_copies_kernel, dim3((unsigned)((kMlpTotal + 255) / 256)), dim3(256), 0, s,
                     p, pbF, pbB);
  return (int)hipGetLastError();
}

}  // namespace tl
