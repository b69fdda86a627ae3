// Surrogate network: a 14-256-256-256-256-2 MLP with GELU, BF16 weights and
// activations on the matrix cores, FP32 accumulation and FP32 master weights.
//
// Layer l computes Z_l = H_{l-1} W_l + b_l and H_l = GELU(Z_l) (the last layer
// is linear).  W_l is stored K x N row-major.  The input is padded from 14 to
// 16 features and the output from 2 to 16 columns; the padding stays zero.
// Outputs: mu = log(A_finite / A_point) and s = log(sigma).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tl {

constexpr int kMlpIn = 14;     // features
constexpr int kMlpInPad = 16;
constexpr int kMlpHidden = 256;
constexpr int kMlpOut = 2;
constexpr int kMlpOutPad = 16;
constexpr int kMlpLayers = 5;
constexpr int kMlpTile = 16;   // rows of a workgroup of the row kernel

constexpr int mlp_K(int l) { return l == 0 ? kMlpInPad : kMlpHidden; }
constexpr int mlp_N(int l) { return l == kMlpLayers - 1 ? kMlpOutPad : kMlpHidden; }

// Offsets of the layers' weights and biases in the flat (padded) parameter
// vector; dims of layer l: K_l x N_l.  The BF16 copies hold W_l at the same
// offset, in the orders of their products' fragments.
struct MlpLayout {
  int K[kMlpLayers], N[kMlpLayers];
  size_t w[kMlpLayers], b[kMlpLayers];
  size_t total;
};
MlpLayout mlp_layout();

// The BF16 weights as the row kernel reads them.
struct MlpWeights {
  const uint16_t* pbF;   // W_l for products over K_l (forward)
  const uint16_t* pbB;   // W_l for products over N_l (backward)
  const float* p;        // FP32 parameters (the biases)
  const float* mean;
  const float* scale;
};

// Inference of rows [0, n): x (n x 14), out (n x 2), device pointers.
int launch_mlp_predict(const MlpWeights& w, const float* x, int n, float* out, hipStream_t s);

// Forward and backward pass of `rows` rows (a multiple of 16): row r is row
// idx[r] of x and y (row r where idx is null).  Writes, for the weight
// gradients, the layers' inputs h[l] (rows x K_l) and pre-activation gradients
// dz[l] (rows x N_l), BF16 in the order of the gradients' fragments, and adds
// the mean loss to *loss.
struct MlpTrainRows {
  const float* x;
  const float* y;
  const int* idx;
  int rows;
  uint16_t* h[kMlpLayers];
  uint16_t* dz[kMlpLayers];
  float* loss;
};
int launch_mlp_train_rows(const MlpWeights& w, const MlpTrainRows& t, hipStream_t s);

// dW_l = H_{l-1}^T dZ_l and db_l (column sums of dZ_l) of every layer from
// h and dz; with g, stores them; else takes the Adam step with them: updates
// p, m, v and the BF16 copies.
struct MlpAdam {
  float *p, *m, *v;
  uint16_t *pbF, *pbB;
  float lr, b1, b2, eps, c1, c2;  // c1, c2: 1 - b1^t, 1 - b2^t
};
int launch_mlp_grads(const MlpTrainRows& t, float* g, const MlpAdam& a, hipStream_t s);

// BF16 copies (round to nearest even) of the padded parameters.
int launch_mlp_copies(const float* p, uint16_t* pbF, uint16_t* pbB, hipStream_t s);

// Rows of one tl_mlp_predict_noalloc call at most.
constexpr size_t kNoAllocRows = 4096;

}  // namespace tl
