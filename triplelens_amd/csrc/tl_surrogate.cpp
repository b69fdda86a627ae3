// Host side of the surrogate network (tl_mlp.h): parameters, training loop
// and inference on the GPU, behind the C ABI of include/tl_surrogate.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <mutex>
#include <numeric>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "tl_mlp.h"
#include "../../include/tl_surrogate.h"

using namespace tl;

namespace {

thread_local std::string g_mlp_err;

#define MCHK(x)                                                                    \
  do {                                                                             \
    hipError_t e_ = (hipError_t)(x);                                               \
    if (e_ != hipSuccess)                                                          \
      throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_));    \
  } while (0)

template <class F>
int mguard(F&& f) {
  g_mlp_err.clear();
  try {
    return f();
  } catch (const std::exception& e) {
    g_mlp_err = e.what();
    return -1;
  } catch (...) {
    g_mlp_err = "unknown error";
    return -1;
  }
}

template <class T>
struct Dev {
  T* p = nullptr;
  size_t n = 0;
  void ensure(size_t k) {
    if (k <= n) return;
    if (p) MCHK(hipFree(p));
    p = nullptr;
    n = 0;  // (should the allocation fail)
    MCHK(hipMalloc(&p, std::max<size_t>(k, 1) * sizeof(T)));
    n = k;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

// Rows whose device buffers a network keeps between calls: those of one piece
// of an inference, 4 MiB.
constexpr int kKeepRows = 1 << 16;

struct Mlp {
  std::mutex mu;
  hipStream_t stream = nullptr;
  MlpLayout L;
  Dev<float> p, g, m, v;   // FP32 master parameters, gradients, Adam moments
  Dev<uint16_t> pbF, pbB;   // BF16 copies, in the orders the products read
  Dev<float> mean, scale;  // feature standardisation
  int t = 0;               // Adam steps taken
  // workspaces: inference rows; a training set and one batch of it
  Dev<float> xin, out, y, loss, scratch;
  Dev<int> perm;
  Dev<uint16_t> h[kMlpLayers], dz[kMlpLayers];

  ~Mlp() {
    for (auto* d : {&p, &g, &m, &v, &mean, &scale, &out, &y, &xin, &loss, &scratch}) d->release();
    for (auto* d : {&pbF, &pbB}) d->release();
    for (auto& d : h) d.release();
    for (auto& d : dz) d.release();
    perm.release();
    if (stream) (void)hipStreamDestroy(stream);
  }

  // Gives back the rows of a training set beyond what an inference keeps.
  void drop_rows() {
    if (xin.n > (size_t)kKeepRows * kMlpIn) xin.release();
    if (y.n > (size_t)kKeepRows) y.release();
    if (perm.n > (size_t)kKeepRows) perm.release();
    if (loss.n > (size_t)kKeepRows) loss.release();
  }

  MlpWeights weights() const { return {pbF.p, pbB.p, p.p, mean.p, scale.p}; }

  // a training set of n rows on the GPU and the buffers of batches of it
  MlpTrainRows train_rows(int n, const float* x, const float* ys, int batch, int nLoss) {
    xin.ensure((size_t)n * kMlpIn);
    y.ensure(n);
    loss.ensure(nLoss);
    MCHK(hipMemcpyAsync(xin.p, x, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice,
                        stream));
    MCHK(hipMemcpyAsync(y.p, ys, (size_t)n * sizeof(float), hipMemcpyHostToDevice, stream));
    MCHK(hipMemsetAsync(loss.p, 0, nLoss * sizeof(float), stream));
    MlpTrainRows r;
    r.x = xin.p;
    r.y = y.p;
    r.idx = nullptr;
    r.rows = batch;
    r.loss = loss.p;
    for (int l = 0; l < kMlpLayers; l++) {
      h[l].ensure((size_t)batch * L.K[l]);
      dz[l].ensure((size_t)batch * L.N[l]);
      r.h[l] = h[l].p;
      r.dz[l] = dz[l].p;
    }
    return r;
  }
};

// logical parameter order: W1 (14 x 256), b1, W2, b2, W3, b3, W4, b4,
// W5 (256 x 2), b5 (2)
size_t logical_count() {
  return (size_t)kMlpIn * kMlpHidden + kMlpHidden +
         3 * ((size_t)kMlpHidden * kMlpHidden + kMlpHidden) + (size_t)kMlpHidden * kMlpOut + kMlpOut;
}

void to_logical(const MlpLayout& L, const std::vector<float>& pad, float* out) {
  size_t o = 0;
  for (int l = 0; l < kMlpLayers; l++) {
    const int Kr = l == 0 ? kMlpIn : L.K[l];
    const int Nr = l == kMlpLayers - 1 ? kMlpOut : L.N[l];
    for (int k = 0; k < Kr; k++)
      for (int n = 0; n < Nr; n++) out[o++] = pad[L.w[l] + (size_t)k * L.N[l] + n];
    for (int n = 0; n < Nr; n++) out[o++] = pad[L.b[l] + n];
  }
}

void from_logical(const MlpLayout& L, const float* in, std::vector<float>& pad) {
  pad.assign(L.total, 0.0f);
  size_t o = 0;
  for (int l = 0; l < kMlpLayers; l++) {
    const int Kr = l == 0 ? kMlpIn : L.K[l];
    const int Nr = l == kMlpLayers - 1 ? kMlpOut : L.N[l];
    for (int k = 0; k < Kr; k++)
      for (int n = 0; n < Nr; n++) pad[L.w[l] + (size_t)k * L.N[l] + n] = in[o++];
    for (int n = 0; n < Nr; n++) pad[L.b[l] + n] = in[o++];
  }
}

void upload_params(Mlp& M, const std::vector<float>& pad) {
  MCHK(hipMemcpy(M.p.p, pad.data(), pad.size() * sizeof(float), hipMemcpyHostToDevice));
  MCHK(launch_mlp_copies(M.p.p, M.pbF.p, M.pbB.p, M.stream));
  MCHK(hipStreamSynchronize(M.stream));
}

Mlp* checked(void* h) {
  if (!h) throw std::invalid_argument("null network");
  return static_cast<Mlp*>(h);
}

}  // namespace

extern "C" {

void* tl_mlp_new(unsigned long long seed) {
  Mlp* M = nullptr;
  mguard([&] {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
      throw std::runtime_error("no HIP device available: the surrogate needs a gfx950 GPU");
    M = new Mlp();
    MCHK(hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking));
    M->L = mlp_layout();
    const size_t n = M->L.total;
    M->p.ensure(n);
    M->g.ensure(n);
    M->m.ensure(n);
    M->v.ensure(n);
    M->pbF.ensure(n);
    M->pbB.ensure(n);
    M->scratch.ensure(kNoAllocRows * kMlpOut);
    M->mean.ensure(kMlpIn);
    M->scale.ensure(kMlpIn);
    MCHK(hipMemset(M->m.p, 0, n * sizeof(float)));
    MCHK(hipMemset(M->v.p, 0, n * sizeof(float)));
    MCHK(hipMemset(M->g.p, 0, n * sizeof(float)));
    std::vector<float> ones(kMlpIn, 1.0f), zeros(kMlpIn, 0.0f);
    MCHK(hipMemcpy(M->mean.p, zeros.data(), kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    MCHK(hipMemcpy(M->scale.p, ones.data(), kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    // He initialisation of the real weights; padding and biases zero
    std::mt19937_64 rng(seed ? seed : 1);
    std::vector<float> pad(n, 0.0f);
    for (int l = 0; l < kMlpLayers; l++) {
      const int Kr = l == 0 ? kMlpIn : M->L.K[l];
      const int Nr = l == kMlpLayers - 1 ? kMlpOut : M->L.N[l];
      const float sd = std::sqrt(2.0f / (float)Kr) * (l == kMlpLayers - 1 ? 0.1f : 1.0f);
      std::normal_distribution<float> nd(0.0f, sd);
      for (int k = 0; k < Kr; k++)
        for (int c = 0; c < Nr; c++) pad[M->L.w[l] + (size_t)k * M->L.N[l] + c] = nd(rng);
    }
    upload_params(*M, pad);
    return 0;
  });
  return M;
}

void tl_mlp_delete(void* h) { delete static_cast<Mlp*>(h); }

long tl_mlp_param_count(void) { return (long)logical_count(); }

int tl_mlp_set_scaling(void* h, const float* mean, const float* scale) {
  return mguard([&] {
    Mlp* M = checked(h);
    std::lock_guard<std::mutex> lock(M->mu);
    for (int f = 0; f < kMlpIn; f++)
      if (!(scale[f] > 0.0f) || !std::isfinite(mean[f])) throw std::invalid_argument("bad scaling");
    MCHK(hipMemcpy(M->mean.p, mean, kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    MCHK(hipMemcpy(M->scale.p, scale, kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    return 0;
  });
}

int tl_mlp_get_params(void* h, float* out) {
  return mguard([&] {
    Mlp* M = checked(h);
    std::lock_guard<std::mutex> lock(M->mu);
    std::vector<float> pad(M->L.total);
    MCHK(hipMemcpy(pad.data(), M->p.p, pad.size() * sizeof(float), hipMemcpyDeviceToHost));
    to_logical(M->L, pad, out);
    return 0;
  });
}

int tl_mlp_set_params(void* h, const float* in) {
  return mguard([&] {
    Mlp* M = checked(h);
    std::lock_guard<std::mutex> lock(M->mu);
    std::vector<float> pad;
    from_logical(M->L, in, pad);
    upload_params(*M, pad);
    return 0;
  });
}

int tl_mlp_predict(void* h, int n, const float* x, float* out) {
  return mguard([&] {
    Mlp* M = checked(h);
    if (n < 0 || (n > 0 && (!x || !out))) throw std::invalid_argument("bad arguments");
    std::lock_guard<std::mutex> lock(M->mu);
    const int chunk = kKeepRows;
    const size_t most = (size_t)std::min(n, chunk);
    M->xin.ensure(most * kMlpIn);
    M->out.ensure(most * kMlpOut);
    for (int r0 = 0; r0 < n; r0 += chunk) {
      const int rows = std::min(chunk, n - r0);
      MCHK(hipMemcpyAsync(M->xin.p, x + (size_t)r0 * kMlpIn, (size_t)rows * kMlpIn * sizeof(float),
                          hipMemcpyHostToDevice, M->stream));
      MCHK(launch_mlp_predict(M->weights(), M->xin.p, rows, M->out.p, M->stream));
      MCHK(hipMemcpyAsync(out + (size_t)r0 * kMlpOut, M->out.p,
                          (size_t)rows * kMlpOut * sizeof(float), hipMemcpyDeviceToHost,
                          M->stream));
      MCHK(hipStreamSynchronize(M->stream));
    }
    return 0;
  });
}

int tl_mlp_predict_noalloc(void* h, int n, const float* x, float* out) {
  return mguard([&] {
    Mlp* M = checked(h);
    if (n < 0 || (size_t)n > kNoAllocRows)
      throw std::invalid_argument("tl_mlp_predict_noalloc: n = " + std::to_string(n) +
                                  " rows; at most " + std::to_string(kNoAllocRows) +
                                  " fit its scratch array");
    if (n > 0 && (!x || !out)) throw std::invalid_argument("bad arguments");
    std::lock_guard<std::mutex> lock(M->mu);
    // rows are written while others are still read: a result that overlaps
    // the input goes through the scratch array
    const bool overlap = std::less<const float*>()(x, out + (size_t)n * kMlpOut) &&
                         std::less<const float*>()(out, x + (size_t)n * kMlpIn);
    float* o = overlap ? M->scratch.p : out;
    MCHK(launch_mlp_predict(M->weights(), x, n, o, M->stream));
    if (overlap)
      MCHK(hipMemcpyAsync(out, o, (size_t)n * kMlpOut * sizeof(float), hipMemcpyDeviceToDevice,
                          M->stream));
    MCHK(hipStreamSynchronize(M->stream));
    return 0;
  });
}

int tl_mlp_grads(void* h, int n, const float* x, const float* y, float* grads, float* loss) {
  return mguard([&] {
    Mlp* M = checked(h);
    if (n <= 0 || n % 64 || !x || !y) throw std::invalid_argument("n must be a positive multiple of 64");
    std::lock_guard<std::mutex> lock(M->mu);
    const MlpTrainRows r = M->train_rows(n, x, y, n, 1);
    MCHK(launch_mlp_train_rows(M->weights(), r, M->stream));
    MCHK(launch_mlp_grads(r, M->g.p, MlpAdam{}, M->stream));
    std::vector<float> pad(M->L.total);
    float l = 0.0f;
    MCHK(hipMemcpyAsync(pad.data(), M->g.p, pad.size() * sizeof(float), hipMemcpyDeviceToHost,
                        M->stream));
    MCHK(hipMemcpyAsync(&l, M->loss.p, sizeof(float), hipMemcpyDeviceToHost, M->stream));
    MCHK(hipStreamSynchronize(M->stream));
    if (grads) to_logical(M->L, pad, grads);
    if (loss) *loss = l;
    return 0;
  });
}

int tl_mlp_train(void* h, int n, const float* x, const float* y, int steps, int batch, float lr,
                 unsigned long long seed, float* losses) {
  return mguard([&] {
    Mlp* M = checked(h);
    if (n <= 0 || !x || !y || steps < 0 || batch <= 0 || batch % 64 || batch > n)
      throw std::invalid_argument("bad training arguments (batch: a multiple of 64, <= n)");
    std::lock_guard<std::mutex> lock(M->mu);
    std::mt19937_64 rng(seed ? seed : 1);
    std::vector<int> perm(n);
    std::iota(perm.begin(), perm.end(), 0);
    size_t pos = n;
    // Steps that see part of the training set only take their rows along, in
    // order; else the whole set goes to the GPU once and batches index it.
    const size_t used = (size_t)steps * batch;
    const bool part = used < (size_t)n;
    std::vector<float> px, py;
    if (part) {
      std::shuffle(perm.begin(), perm.end(), rng);
      px.resize(used * kMlpIn);
      py.resize(used);
      for (size_t i = 0; i < used; i++) {
        std::memcpy(&px[i * kMlpIn], x + (size_t)perm[i] * kMlpIn, kMlpIn * sizeof(float));
        py[i] = y[perm[i]];
      }
      x = px.data();
      y = py.data();
    } else {
      M->perm.ensure(n);
    }
    MlpTrainRows r = M->train_rows(part ? (int)used : n, x, y, batch, std::max(1, steps));
    for (int s = 0; s < steps; s++) {
      if (part) {
        r.x = M->xin.p + (size_t)s * batch * kMlpIn;
        r.y = M->y.p + (size_t)s * batch;
      } else {
        if (pos + batch > (size_t)n) {
          std::shuffle(perm.begin(), perm.end(), rng);
          MCHK(hipMemcpyAsync(M->perm.p, perm.data(), (size_t)n * sizeof(int),
                              hipMemcpyHostToDevice, M->stream));
          // the next shuffle may not touch perm before this copy has read it
          MCHK(hipStreamSynchronize(M->stream));
          pos = 0;
        }
        r.idx = M->perm.p + pos;
        pos += batch;
      }
      r.loss = M->loss.p + s;
      M->t++;
      MlpAdam a = {M->p.p, M->m.p, M->v.p, M->pbF.p, M->pbB.p, lr, 0.9f, 0.999f, 1e-8f,
                   1.0f - powf(0.9f, (float)M->t), 1.0f - powf(0.999f, (float)M->t)};
      MCHK(launch_mlp_train_rows(M->weights(), r, M->stream));
      MCHK(launch_mlp_grads(r, nullptr, a, M->stream));
    }
    if (losses && steps > 0)
      MCHK(hipMemcpyAsync(losses, M->loss.p, (size_t)steps * sizeof(float), hipMemcpyDeviceToHost,
                          M->stream));
    MCHK(hipStreamSynchronize(M->stream));
    M->drop_rows();
    return 0;
  });
}

const char* tl_mlp_last_error(void) { return g_mlp_err.c_str(); }

}  // extern "C"
