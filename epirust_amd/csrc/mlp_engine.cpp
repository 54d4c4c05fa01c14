// Host runtime of the surrogate MLP (C ABI in include/epirust_gpu.h): widths
// w0 -> w1 -> ... -> wL, GELU after every hidden layer, identity output, MSE loss, Adam.
// Parameters are fp32 masters with bf16 copies; activations are bf16; every product runs on
// bf16 MFMA with fp32 accumulation, and a step's launches follow one another on the handle's
// stream with one wait at its end.
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <string>
#include <vector>

#include "epirust_gpu.h"
#include "mlp.hpp"

using namespace epi;

namespace {

thread_local std::string g_mlp_error;

int mfail(int code, const std::string& m) {
  g_mlp_error = m;
  return code;
}

#define MHIP(expr)                                                                                          \
  do {                                                                                                      \
    hipError_t e_ = (expr);                                                                                 \
    if (e_ != hipSuccess) return mfail(EPI_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

struct Buf {
  std::vector<void*> owned;
  template <class T>
  hipError_t get(T** p, size_t n) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
    if (e == hipSuccess) {
      owned.push_back(q);
      (void)hipMemset(q, 0, std::max<size_t>(n, 1) * sizeof(T));
    }
    *p = static_cast<T*>(q);
    return e;
  }
  ~Buf() {
    for (void* p : owned) (void)hipFree(p);
  }
};

}  // namespace

// Host buffers the handle copies a batch through (pinned, so that the host copies one part
// while another is on the bus), and the parts they are copied in.
constexpr size_t kStagingBytes = 8u << 20, kPartBytes = 640u << 10;
constexpr size_t kParts = 4;

struct epi_mlp {
  std::vector<int> w;  // widths, L+1
  int L = 0, max_batch = 0, step = 0;
  hipStream_t stream = nullptr;
  Buf mem;
  std::vector<float*> W, b, gW, gb, mW, vW, mb, vb, Z, dZ32;
  // bf16 matrices by rows and transposed (mlp.hpp): weights K x N, activations and gradients
  // batch x N; act16[l] is the input of layer l.
  std::vector<uint16_t*> W16, W16T, act16, act16T, dZ16, dZ16T;
  float* X = nullptr;  // the input where it does not fit h_x
  float* T = nullptr;
  float* Y = nullptr;
  // pinned: input, targets or outputs (null where a batch would not fit), loss parts
  float *h_x = nullptr, *h_t = nullptr, *h_loss = nullptr;
  float *d_x = nullptr, *d_loss = nullptr;                  // h_x and h_loss as the device sees them
  hipEvent_t copied[kParts] = {};                           // a part of the outputs is in h_t
  ~epi_mlp() {
    for (float* p : {h_x, h_t, h_loss})
      if (p) (void)hipHostFree(p);
    for (hipEvent_t e : copied)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
  size_t param_count() const {
    size_t n = 0;
    for (int l = 0; l < L; ++l) n += static_cast<size_t>(w[l]) * w[l + 1] + w[l + 1];
    return n;
  }
};

namespace {

// Layer l of the forward pass; `training` keeps what the backward pass reads.
int forward_layer(epi_mlp* m, int l, int B, bool training) {
  const int K = m->w[l], N = m->w[l + 1];
  MlpStage st{};
  MlpJob& j = st.job[0];
  j.A = m->act16[l];
  j.lda = mlp_pitch(K);
  j.M = B;
  j.N = N;
  j.K = K;
  j.Bt = m->W16T[l];
  j.ldb = mlp_pitch(K);
  j.bias = m->b[l];
  if (l < m->L - 1) {
    j.kind = MLP_HIDDEN;
    j.c = training ? m->Z[l] : nullptr;
    j.row = m->act16[l + 1];
    j.ld_row = mlp_pitch(N);
    j.col = training ? m->act16T[l + 1] : nullptr;
    j.ld_col = mlp_pitch(m->max_batch);
  } else if (training) {
    j.kind = MLP_LOSS;
    j.t = m->T;
    j.c = m->dZ32[l];
    j.row = m->dZ16[l];
    j.ld_row = mlp_pitch(N);
    j.col = m->dZ16T[l];
    j.ld_col = mlp_pitch(m->max_batch);
    j.parts = m->d_loss;
    j.inv_count = 1.0f / static_cast<float>(static_cast<int64_t>(B) * N);
  } else {
    j.kind = MLP_OUTPUT;
    j.c = m->Y;
  }
  MHIP(mlp_stage(st, 1, m->stream));
  return EPI_OK;
}

// dZ_{l-1} = (dZ_l * W_l^T) * GELU'(Z_{l-1}), l >= 1
MlpJob input_grad(const epi_mlp* m, int l, int B) {
  const int K = m->w[l], N = m->w[l + 1];
  MlpJob j{};
  j.kind = MLP_INPUT_GRAD;
  j.M = B;
  j.N = K;
  j.K = N;
  j.A = m->dZ16[l];
  j.lda = mlp_pitch(N);
  j.Bt = m->W16[l];
  j.ldb = mlp_pitch(N);
  j.z = m->Z[l - 1];
  j.c = m->dZ32[l - 1];
  j.row = m->dZ16[l - 1];
  j.ld_row = mlp_pitch(K);
  j.col = m->dZ16T[l - 1];
  j.ld_col = mlp_pitch(m->max_batch);
  return j;
}

// gW_l = act_l^T * dZ_l (K x N) and gb_l, or the Adam step with them
int weight_jobs(const epi_mlp* m, int l, int B, bool adam, MlpJob* out) {
  const int K = m->w[l], N = m->w[l + 1];
  MlpJob g{}, h{};
  g.kind = MLP_WEIGHT_GRAD;
  g.A = m->act16T[l];
  g.lda = mlp_pitch(m->max_batch);
  g.M = K;
  g.N = N;
  g.K = B;
  g.Bt = m->dZ16T[l];
  g.ldb = mlp_pitch(m->max_batch);
  g.adam = h.adam = adam;
  if (adam) {
    g.w = m->W[l];
    g.m = m->mW[l];
    g.v = m->vW[l];
    g.row = m->W16[l];
    g.ld_row = mlp_pitch(N);
    g.col = m->W16T[l];
    g.ld_col = mlp_pitch(K);
    h.w = m->b[l];
    h.m = m->mb[l];
    h.v = m->vb[l];
  } else {
    g.c = m->gW[l];
    h.c = m->gb[l];
  }
  h.kind = MLP_BIAS_GRAD;
  h.N = N;
  h.K = B;
  h.z = m->dZ32[l];
  out[0] = g;
  out[1] = h;
  return 2;
}

// The backward pass, with an Adam step of every parameter when `adam` is set. The input
// gradient of layer l reads W_l before the next stage's Adam step changes it.
int backward(epi_mlp* m, int B, const AdamArgs* adam) {
  MlpStage st{};
  if (adam) st.adam = *adam;
  for (int l = m->L - 1; l >= 1; --l) {
    int n = 0;
    st.job[n++] = input_grad(m, l, B);
    if (l < m->L - 1) n += weight_jobs(m, l + 1, B, adam != nullptr, st.job + n);
    MHIP(mlp_stage(st, n, m->stream));
  }
  int n = 0;
  if (m->L > 1) n += weight_jobs(m, 1, B, adam != nullptr, st.job + n);
  n += weight_jobs(m, 0, B, adam != nullptr, st.job + n);
  MHIP(mlp_stage(st, n, m->stream));
  return EPI_OK;
}

hipError_t pack_weights(epi_mlp* m, int l) {
  const int K = m->w[l], N = m->w[l + 1];
  return mlp_pack(m->W[l], K, N, m->W16[l], mlp_pitch(N), m->W16T[l], mlp_pitch(K), m->stream);
}

// Loss parts of the largest batch or any smaller one: a wave takes four tiles only above a
// number of tiles, so a smaller batch may write more.
size_t most_loss_parts(int B, int N) { return static_cast<size_t>((B + 31) / 32) * ((N + 31) / 32); }

// Values of a part when n of them are copied in at most kParts parts.
size_t part_of(size_t n) { return std::max(kPartBytes / 4, (n + kParts - 1) / kParts); }

// n targets to the device through pinned memory, or by a plain copy where a batch does not
// fit it. (The loss stage reading the pinned memory itself took as long as the copy and its
// own time together.)
int load_targets(epi_mlp* m, const float* t, size_t n) {
  if (!m->h_t) {
    MHIP(hipMemcpyAsync(m->T, t, n * 4, hipMemcpyHostToDevice, m->stream));
    return EPI_OK;
  }
  for (size_t at = 0, part = part_of(n); at < n; at += part) {
    const size_t k = std::min(part, n - at);
    std::memcpy(m->h_t + at, t + at, k * 4);
    MHIP(hipMemcpyAsync(m->T + at, m->h_t + at, k * 4, hipMemcpyHostToDevice, m->stream));
  }
  return EPI_OK;
}

// n outputs to the caller the same way, once the stream has made them.
int store_outputs(epi_mlp* m, float* y, size_t n) {
  if (!m->h_t) {
    MHIP(hipMemcpyAsync(y, m->Y, n * 4, hipMemcpyDeviceToHost, m->stream));
    MHIP(hipStreamSynchronize(m->stream));
    return EPI_OK;
  }
  const size_t part = part_of(n);
  for (size_t at = 0, i = 0; at < n; at += part, ++i) {
    MHIP(hipMemcpyAsync(m->h_t + at, m->Y + at, std::min(part, n - at) * 4, hipMemcpyDeviceToHost, m->stream));
    MHIP(hipEventRecord(m->copied[i], m->stream));
  }
  for (size_t at = 0, i = 0; at < n; at += part, ++i) {
    MHIP(hipEventSynchronize(m->copied[i]));
    std::memcpy(y + at, m->h_t + at, std::min(part, n - at) * 4);
  }
  return EPI_OK;
}

// The batch's input to bf16. Where it fits the pinned buffer the kernel reads it there: a
// few values a sample, less than a copy's own cost.
int load_input(epi_mlp* m, const float* x, int B) {
  if (B <= 0 || B > m->max_batch) return mfail(EPI_ERR_ARG, "batch out of range");
  const size_t n = static_cast<size_t>(B) * m->w[0];
  const float* src = m->d_x;
  if (src) {
    std::memcpy(m->h_x, x, n * 4);
  } else {
    MHIP(hipMemcpyAsync(m->X, x, n * 4, hipMemcpyHostToDevice, m->stream));
    src = m->X;
  }
  MHIP(mlp_pack(src, B, m->w[0], m->act16[0], mlp_pitch(m->w[0]), m->act16T[0], mlp_pitch(m->max_batch), m->stream));
  return EPI_OK;
}

// Forward pass, loss and backward pass of a batch. The targets are staged while the hidden
// layers run.
int train_pass(epi_mlp* m, const float* x, const float* t, int B, const AdamArgs* adam, float* loss) {
  int rc = load_input(m, x, B);
  for (int l = 0; !rc && l < m->L - 1; ++l) rc = forward_layer(m, l, B, true);
  if (!rc) rc = load_targets(m, t, static_cast<size_t>(B) * m->w[m->L]);
  if (!rc) rc = forward_layer(m, m->L - 1, B, true);
  if (!rc) rc = backward(m, B, adam);
  if (rc) {
    (void)hipStreamSynchronize(m->stream);  // the copies may still read the caller's arrays
    return rc;
  }
  MHIP(hipStreamSynchronize(m->stream));
  if (loss) {
    double s = 0;
    for (uint32_t i = 0, n = mlp_loss_parts(B, m->w[m->L]); i < n; ++i) s += m->h_loss[i];
    *loss = static_cast<float>(s);
  }
  return EPI_OK;
}

}  // namespace

extern "C" {

const char* epi_mlp_last_error(void) { return g_mlp_error.c_str(); }

int epi_mlp_create(const uint32_t* widths, uint32_t n_widths, uint64_t seed, uint32_t max_batch, epi_mlp** out) {
  if (!widths || n_widths < 2 || !out || max_batch == 0) return mfail(EPI_ERR_ARG, "bad arguments");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return mfail(EPI_ERR_DEVICE, "no HIP device available");
  std::unique_ptr<epi_mlp> m(new epi_mlp());
  for (uint32_t i = 0; i < n_widths; ++i) {
    if (widths[i] == 0 || widths[i] > 65536) return mfail(EPI_ERR_ARG, "layer width out of range");
    m->w.push_back(static_cast<int>(widths[i]));
  }
  m->L = static_cast<int>(n_widths) - 1;
  m->max_batch = static_cast<int>(max_batch);
  MHIP(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
  const int L = m->L, B = m->max_batch;
  m->W.resize(L); m->b.resize(L); m->gW.resize(L); m->gb.resize(L); m->mW.resize(L); m->vW.resize(L);
  m->mb.resize(L); m->vb.resize(L); m->Z.resize(L); m->dZ32.resize(L); m->W16.resize(L); m->W16T.resize(L);
  m->dZ16.resize(L); m->dZ16T.resize(L); m->act16.resize(L); m->act16T.resize(L);
  const auto by_rows = [](size_t rows, size_t cols) {
    return static_cast<size_t>(mlp_rows(static_cast<int>(rows))) * mlp_pitch(static_cast<int>(cols));
  };
  std::mt19937_64 rng(seed);
  for (int l = 0; l < L; ++l) {
    const size_t K = m->w[l], N = m->w[l + 1];
    MHIP(m->mem.get(&m->W[l], K * N));
    MHIP(m->mem.get(&m->W16[l], by_rows(K, N)));
    MHIP(m->mem.get(&m->W16T[l], by_rows(N, K)));
    MHIP(m->mem.get(&m->b[l], N));
    MHIP(m->mem.get(&m->gW[l], K * N));
    MHIP(m->mem.get(&m->gb[l], N));
    MHIP(m->mem.get(&m->mW[l], K * N));
    MHIP(m->mem.get(&m->vW[l], K * N));
    MHIP(m->mem.get(&m->mb[l], N));
    MHIP(m->mem.get(&m->vb[l], N));
    MHIP(m->mem.get(&m->Z[l], static_cast<size_t>(B) * N));
    MHIP(m->mem.get(&m->dZ32[l], static_cast<size_t>(B) * N));
    MHIP(m->mem.get(&m->dZ16[l], by_rows(B, N)));
    MHIP(m->mem.get(&m->dZ16T[l], by_rows(N, B)));
    MHIP(m->mem.get(&m->act16[l], by_rows(B, K)));
    MHIP(m->mem.get(&m->act16T[l], by_rows(K, B)));
    // He-normal initialisation for GELU layers, biases zero
    std::normal_distribution<float> nd(0.0f, std::sqrt(2.0f / static_cast<float>(K)));
    std::vector<float> w(K * N);
    for (auto& v : w) v = nd(rng);
    MHIP(hipMemcpy(m->W[l], w.data(), w.size() * 4, hipMemcpyHostToDevice));
    MHIP(pack_weights(m.get(), l));
  }
  MHIP(m->mem.get(&m->Y, static_cast<size_t>(B) * m->w[L]));
  MHIP(m->mem.get(&m->T, static_cast<size_t>(B) * m->w[L]));
  const auto pinned = [](float** p, size_t bytes) {
    return hipHostMalloc(reinterpret_cast<void**>(p), std::max<size_t>(bytes, 4), hipHostMallocDefault);
  };
  const size_t x_bytes = static_cast<size_t>(B) * m->w[0] * 4, t_bytes = static_cast<size_t>(B) * m->w[L] * 4;
  if (x_bytes <= kStagingBytes) {
    MHIP(pinned(&m->h_x, x_bytes));
    MHIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&m->d_x), m->h_x, 0));
  } else {
    MHIP(m->mem.get(&m->X, static_cast<size_t>(B) * m->w[0]));
  }
  if (t_bytes <= kStagingBytes) MHIP(pinned(&m->h_t, t_bytes));
  for (hipEvent_t& e : m->copied) MHIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  MHIP(pinned(&m->h_loss, most_loss_parts(B, m->w[L]) * 4));
  MHIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&m->d_loss), m->h_loss, 0));
  MHIP(hipStreamSynchronize(nullptr));  // the clears ran there
  MHIP(hipStreamSynchronize(m->stream));
  *out = m.release();
  return EPI_OK;
}

void epi_mlp_destroy(epi_mlp* m) { delete m; }

uint64_t epi_mlp_param_count(epi_mlp* m) { return m ? m->param_count() : 0; }

int epi_mlp_get_params(epi_mlp* m, float* out, uint64_t n) {
  if (!m || !out || n != m->param_count()) return mfail(EPI_ERR_ARG, "parameter count mismatch");
  size_t o = 0;
  for (int l = 0; l < m->L; ++l) {
    const size_t kn = static_cast<size_t>(m->w[l]) * m->w[l + 1];
    MHIP(hipMemcpy(out + o, m->W[l], kn * 4, hipMemcpyDeviceToHost));
    o += kn;
    MHIP(hipMemcpy(out + o, m->b[l], m->w[l + 1] * 4, hipMemcpyDeviceToHost));
    o += m->w[l + 1];
  }
  return EPI_OK;
}

int epi_mlp_set_params(epi_mlp* m, const float* in, uint64_t n) {
  if (!m || !in || n != m->param_count()) return mfail(EPI_ERR_ARG, "parameter count mismatch");
  size_t o = 0;
  for (int l = 0; l < m->L; ++l) {
    const size_t kn = static_cast<size_t>(m->w[l]) * m->w[l + 1];
    MHIP(hipMemcpy(m->W[l], in + o, kn * 4, hipMemcpyHostToDevice));
    MHIP(pack_weights(m, l));
    o += kn;
    MHIP(hipMemcpy(m->b[l], in + o, m->w[l + 1] * 4, hipMemcpyHostToDevice));
    o += m->w[l + 1];
  }
  m->step = 0;
  for (int l = 0; l < m->L; ++l) {
    const size_t kn = static_cast<size_t>(m->w[l]) * m->w[l + 1];
    MHIP(hipMemsetAsync(m->mW[l], 0, kn * 4, m->stream));
    MHIP(hipMemsetAsync(m->vW[l], 0, kn * 4, m->stream));
    MHIP(hipMemsetAsync(m->mb[l], 0, m->w[l + 1] * 4, m->stream));
    MHIP(hipMemsetAsync(m->vb[l], 0, m->w[l + 1] * 4, m->stream));
  }
  MHIP(hipStreamSynchronize(m->stream));
  return EPI_OK;
}

int epi_mlp_forward(epi_mlp* m, const float* x, uint32_t batch, float* y) {
  if (!m || !x || !y) return mfail(EPI_ERR_ARG, "null argument");
  const int B = static_cast<int>(batch);
  int rc = load_input(m, x, B);
  for (int l = 0; !rc && l < m->L; ++l) rc = forward_layer(m, l, B, false);
  if (rc) {
    (void)hipStreamSynchronize(m->stream);
    return rc;
  }
  return store_outputs(m, y, static_cast<size_t>(batch) * m->w[m->L]);
}

int epi_mlp_gradients(epi_mlp* m, const float* x, const float* t, uint32_t batch, float* grads, float* loss) {
  if (!m || !x || !t || !grads) return mfail(EPI_ERR_ARG, "null argument");
  const int rc = train_pass(m, x, t, static_cast<int>(batch), nullptr, loss);
  if (rc) return rc;
  size_t o = 0;
  for (int l = 0; l < m->L; ++l) {
    const size_t kn = static_cast<size_t>(m->w[l]) * m->w[l + 1];
    MHIP(hipMemcpy(grads + o, m->gW[l], kn * 4, hipMemcpyDeviceToHost));
    o += kn;
    MHIP(hipMemcpy(grads + o, m->gb[l], m->w[l + 1] * 4, hipMemcpyDeviceToHost));
    o += m->w[l + 1];
  }
  return EPI_OK;
}

int epi_mlp_train_step(epi_mlp* m, const float* x, const float* t, uint32_t batch, float lr, float* loss) {
  if (!m || !x || !t) return mfail(EPI_ERR_ARG, "null argument");
  const float b1 = 0.9f, b2 = 0.999f, k = static_cast<float>(m->step + 1);
  const AdamArgs adam{lr, b1, b2, 1e-8f, 1.0f - std::pow(b1, k), 1.0f - std::pow(b2, k)};
  const int rc = train_pass(m, x, t, static_cast<int>(batch), &adam, loss);
  if (rc) return rc;
  ++m->step;
  return EPI_OK;
}

int epi_gemm_bf16(const uint16_t* A, const uint16_t* B, float* C, int M, int N, int K, int trans_a, int trans_b) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return mfail(EPI_ERR_ARG, "bad arguments");
  uint16_t *dA = nullptr, *dB = nullptr;
  float* dC = nullptr;
  Buf mem;
  MHIP(mem.get(&dA, static_cast<size_t>(M) * K));
  MHIP(mem.get(&dB, static_cast<size_t>(K) * N));
  MHIP(mem.get(&dC, static_cast<size_t>(M) * N));
  MHIP(hipMemcpy(dA, A, static_cast<size_t>(M) * K * 2, hipMemcpyHostToDevice));
  MHIP(hipMemcpy(dB, B, static_cast<size_t>(K) * N * 2, hipMemcpyHostToDevice));
  GemmArgs g{};
  g.A = dA;
  g.B = dB;
  // A is stored M x K row-major unless trans_a (then K x M); likewise B
  g.lda_m = trans_a ? 1 : K;
  g.lda_k = trans_a ? M : 1;
  g.ldb_k = trans_b ? 1 : N;
  g.ldb_n = trans_b ? K : 1;
  g.M = M;
  g.N = N;
  g.K = K;
  g.C = dC;
  MHIP(mlp_gemm(g, nullptr));
  MHIP(hipDeviceSynchronize());
  MHIP(hipMemcpy(C, dC, static_cast<size_t>(M) * N * 4, hipMemcpyDeviceToHost));
  return EPI_OK;
}

}  // extern "C"
