// Temperature surrogate: a 5-128-128-128-128-1 MLP with SiLU, BF16 operands on
// the gfx950 matrix cores (v_mfma_f32_32x32x16_bf16) and FP32 accumulation.
//
// Inference is one kernel, k_mlp_fused: the weights sit in LDS and a wave
// carries 64 rows through the whole network in registers.  A training step is
// two: k_train takes 64 rows per work-group through the forward and backward
// passes and leaves the work-group's share of the weight gradients, k_reduce
// adds the shares and applies Adam.  Both read the weights as bf16 images in
// the order the matrix instructions take them (NetImage), which whatever
// changes the parameters rewrites.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/amca3d.h"
#include "surrogate.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

namespace mlpk {

constexpr int kIn = 5, kHid = 128, kLayers = 5;
constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kPad = 8;  // bf16 elements of padding per LDS row
constexpr int kThreads = 256;

// parameter vector layout: W1[5][128] b1[128] W2[128][128] b2 W3 b3 W4 b4 W5[128][1] b5[1]
constexpr int kFanIn[kLayers] = {kIn, kHid, kHid, kHid, kHid};
constexpr int kFanOut[kLayers] = {kHid, kHid, kHid, kHid, 1};

struct Layout {
  int w[kLayers], b[kLayers];
  int total;
  __host__ __device__ Layout() {
    int o = 0;
    for (int l = 0; l < kLayers; l++) {
      w[l] = o;
      o += kFanIn[l] * kFanOut[l];
      b[l] = o;
      o += kFanOut[l];
    }
    total = o;
  }
};

// v_rcp_f32 (1 ulp) in place of the IEEE divide sequence: the result is
// rounded to bf16 or feeds an fp32 gradient, far coarser than the reciprocal.
__device__ __forceinline__ float sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}

// C = opA(A) * opB(B), operands rounded to BF16 when staged into LDS:
// amca_mlp_gemm_selftest, the lane layouts of the matrix instruction that the network's
// kernels use, against any operands (they do not run this kernel).  opA(A)[m][k] = TrA ? A[k*lda + m] :
// A[m*lda + k]; opB(B)[k][n] = TrB ? B[n*ldb + k] : B[k*ldb + n].  A work-group of
// 4 waves owns a 128 x 128 block of C (ldc = N), each wave 32 rows and four
// 32 x 32 MFMA tiles; elements outside the matrices stage as zero.
template <bool TrA, bool TrB>
__global__ void __launch_bounds__(kThreads)
k_gemm(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, int M, int N,
       int K, float* __restrict__ C) {
  __shared__ __bf16 As[kBM][kBK + kPad];
  __shared__ __bf16 Bs[kBN][kBK + kPad];  // n-major: Bs[n][k]
  const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  floatx16 acc[4];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[t][i] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += kBK) {
#pragma unroll
    for (int q = 0; q < (kBM * kBK) / kThreads; q++) {
      const int idx = threadIdx.x + q * kThreads;
      const int mm = TrA ? idx % kBM : idx / kBK, kk = TrA ? idx / kBM : idx % kBK;
      const int gm = m0 + mm, gk = k0 + kk;
      const bool in = gm < M && gk < K;
      const size_t o = in ? (TrA ? (size_t)gk * lda + gm : (size_t)gm * lda + gk) : 0;
      As[mm][kk] = (__bf16)(in ? A[o] : 0.0f);
    }
#pragma unroll
    for (int q = 0; q < (kBN * kBK) / kThreads; q++) {
      const int idx = threadIdx.x + q * kThreads;
      const int nn = TrB ? idx / kBK : idx % kBN, kk = TrB ? idx % kBK : idx / kBN;
      const int gn = n0 + nn, gk = k0 + kk;
      const bool in = gn < N && gk < K;
      const size_t o = in ? (TrB ? (size_t)gn * ldb + gk : (size_t)gk * ldb + gn) : 0;
      Bs[nn][kk] = (__bf16)(in ? B[o] : 0.0f);
    }
    __syncthreads();
    // two MFMA k-steps of 16: lane holds A[row = lane%32][k = (lane/32)*8 ..+8]
    // and B[k = (lane/32)*8 ..+8][col = lane%32]
#pragma unroll
    for (int ks = 0; ks < kBK; ks += 16) {
      const int kq = ks + (lane >> 5) * 8;
      bf16x8 a;
#pragma unroll
      for (int j = 0; j < 8; j++) a[j] = As[wave * 32 + (lane & 31)][kq + j];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        bf16x8 b;
#pragma unroll
        for (int j = 0; j < 8; j++) b[j] = Bs[t * 32 + (lane & 31)][kq + j];
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // D layout: element i of lane l is row (i/4)*8 + (l/32)*4 + i%4, column l%32
#pragma unroll
  for (int t = 0; t < 4; t++) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int m = m0 + wave * 32 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3);
      const int n = n0 + t * 32 + (lane & 31);
      if (m < M && n < N) C[(size_t)m * N + n] = acc[t][i];
    }
  }
}

}  // namespace mlpk

namespace mlpk {
// fused inference (defined with the sampler below)
enum FusedMode : int {
  kRowsScaled = 0,  // rows of X -> network output, activations rounded scaled by -log2(e)
  kLattice = 1,     // lattice points of (d, s, g) -> temperatures, the same rounding
  kRows = 2,        // rows of X -> network output, activations rounded as they are
};
struct NetImage;
size_t net_image_bytes();
hipError_t fused_setup();
hipError_t launch_pack(const float* p, NetImage* img, float* m, float* v, hipStream_t st);
// training (defined at the end of the kernels): one 64-row group per work-group
// and pass, at most one work-group per CU
constexpr int kTrainRows = 64;
constexpr int kPartStride = 50440;  // floats of one work-group's gradient share (16-byte rows)
struct Adam {
  float *m, *v;  // moments, or null: k_reduce leaves the gradients alone
  float lr, c1, c2;
};
hipError_t launch_train(const float* p, NetImage* img, int blocks, int n, const float* X,
                        const float* Y, float* part, float* part_loss, hipStream_t st);
hipError_t launch_reduce(int blocks, const float* part, const float* part_loss, float* p,
                         float* grads, float* loss, const Adam& adam, NetImage* img,
                         hipStream_t st);
hipError_t launch_fused(FusedMode mode, const NetImage* img, int cus, long long n, const float* X,
                        float* out, const amca_surrogate_desc& d, const amca_scan& s,
                        const SurLattice& g, hipStream_t st);
hipError_t launch_fused_timed(amca_mlp* h, FusedMode mode, long long n, const float* X, float* out,
                              const amca_surrogate_desc& d, const amca_scan& s,
                              const SurLattice& g);
}  // namespace mlpk

using namespace mlpk;

constexpr int kLossSteps = 4096;  // steps whose losses stay on the device between copies

struct amca_mlp {
  hipStream_t stream = nullptr;
  int device = -1;          // the device current at create
  int cus = 256;            // its compute units
  Layout lay;
  float* params = nullptr;  // FP32 master copy
  NetImage* image = nullptr;  // the same weights in the kernels' order (rewritten whenever
                              // the parameters change)
  float* grads = nullptr;
  float* adam_m = nullptr;
  float* adam_v = nullptr;
  long long adam_t = 0;
  // rows of host-pointer calls
  int rows_cap = 0;
  float* X = nullptr;            // [rows_cap][5]
  float* Y = nullptr;            // [rows_cap]
  float* T = nullptr;            // outputs [rows_cap]
  // training: the work-groups' gradient shares and losses, and a stretch of
  // per-step losses
  int part_cap = 0;              // work-groups
  float* part = nullptr;         // [part_cap][kPartStride]
  float* part_loss = nullptr;    // [part_cap]
  float* loss = nullptr;         // [kLossSteps]
  // device-resident training set (amca_surrogate_sample)
  float* setX = nullptr;
  float* setY = nullptr;
  long long set_n = 0;
  std::vector<void*> allocs;
  // HIP events around the fused kernel's launches (amca_mlp_enable_timing)
  bool timing = false;
  hipEvent_t ev[2] = {nullptr, nullptr};
  double fused_ms = 0.0;
  long long fused_launches = 0, fused_rows = 0;
  ~amca_mlp() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* p : allocs) (void)hipFree(p);
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

thread_local std::string g_mlp_error;

amca_status mlp_fail(amca_status s, const std::string& m) {
  g_mlp_error = m;
  return s;
}

#define MLP_HIP(expr)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return mlp_fail(AMCA_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
  } while (0)

#define MLP_TRY(expr)             \
  do {                            \
    amca_status s_ = (expr);      \
    if (s_ != AMCA_OK) return s_; \
  } while (0)

template <class T>
amca_status mlp_alloc(amca_mlp* h, T** p, size_t n) {
  void* q = nullptr;
  MLP_HIP(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
  h->allocs.push_back(q);
  *p = static_cast<T*>(q);
  return AMCA_OK;
}

void mlp_release(amca_mlp* h, void* p) {
  if (!p) return;
  for (auto& a : h->allocs)
    if (a == p) {
      (void)hipFree(a);
      a = nullptr;
    }
}

// input and output rows of the calls that take host pointers
amca_status ensure_rows(amca_mlp* h, int n) {
  if (n <= h->rows_cap) return AMCA_OK;
  MLP_HIP(hipStreamSynchronize(h->stream));
  h->rows_cap = 0;
  for (float** p : {&h->X, &h->Y, &h->T}) {
    mlp_release(h, *p);
    *p = nullptr;
  }
  MLP_TRY(mlp_alloc(h, &h->X, (size_t)n * kIn));
  MLP_TRY(mlp_alloc(h, &h->Y, (size_t)n));
  MLP_TRY(mlp_alloc(h, &h->T, (size_t)n));
  h->rows_cap = n;
  return AMCA_OK;
}

// work-groups of a training pass over n rows, their shares allocated
amca_status train_blocks(amca_mlp* h, int n, int* blocks) {
  *blocks = std::min((n + kTrainRows - 1) / kTrainRows, h->cus);
  if (*blocks <= h->part_cap) return AMCA_OK;
  MLP_HIP(hipStreamSynchronize(h->stream));
  h->part_cap = 0;
  for (float** p : {&h->part, &h->part_loss}) {
    mlp_release(h, *p);
    *p = nullptr;
  }
  MLP_TRY(mlp_alloc(h, &h->part, (size_t)*blocks * kPartStride));
  MLP_TRY(mlp_alloc(h, &h->part_loss, (size_t)*blocks));
  h->part_cap = *blocks;
  return AMCA_OK;
}

// the parameters from host memory, Adam's moments from zero, and the weight
// images, all on the network's stream and complete on return
amca_status load_params(amca_mlp* h, const float* p) {
  const size_t bytes = sizeof(float) * h->lay.total;
  MLP_HIP(hipMemcpyAsync(h->params, p, bytes, hipMemcpyHostToDevice, h->stream));
  h->adam_t = 0;
  MLP_HIP(launch_pack(h->params, h->image, h->adam_m, h->adam_v, h->stream));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

// network outputs of n device rows, enqueued on the network's stream
amca_status infer(amca_mlp* h, long long n, const float* X, float* T) {
  MLP_HIP(launch_fused(kRows, h->image, h->cus, n, X, T, amca_surrogate_desc{}, amca_scan{},
                       SurLattice{}, h->stream));
  return AMCA_OK;
}

}  // namespace

extern "C" {

const char* amca_mlp_last_error(void) { return g_mlp_error.c_str(); }

int32_t amca_mlp_param_count(void) { return Layout().total; }

amca_status amca_mlp_create(uint64_t seed, amca_mlp** out) {
  if (!out) return mlp_fail(AMCA_ERR_INVALID, "null argument");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return mlp_fail(AMCA_ERR_NO_DEVICE, "no HIP device visible");
  auto* h = new amca_mlp();
  amca_status st = AMCA_OK;
  do {
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "stream");
      break;
    }
    if (hipGetDevice(&h->device) != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "hipGetDevice");
      break;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, h->device) ==
            hipSuccess && cus > 0)
      h->cus = cus;
    if (fused_setup() != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "LDS size of the fused kernel");
      break;
    }
    unsigned char* img = nullptr;
    if ((st = mlp_alloc(h, &img, net_image_bytes())) != AMCA_OK) break;
    h->image = reinterpret_cast<NetImage*>(img);
    const int P = h->lay.total;
    if ((st = mlp_alloc(h, &h->params, P)) != AMCA_OK) break;
    if ((st = mlp_alloc(h, &h->grads, P)) != AMCA_OK) break;
    if ((st = mlp_alloc(h, &h->adam_m, P)) != AMCA_OK) break;
    if ((st = mlp_alloc(h, &h->adam_v, P)) != AMCA_OK) break;
    if ((st = mlp_alloc(h, &h->loss, kLossSteps)) != AMCA_OK) break;
    // He-uniform weights for SiLU layers, zero biases
    std::mt19937_64 rng(seed);
    std::vector<float> p(P, 0.0f);
    for (int l = 0; l < kLayers; l++) {
      const float a = std::sqrt(6.0f / (float)kFanIn[l]);
      std::uniform_real_distribution<float> U(-a, a);
      for (int i = 0; i < kFanIn[l] * kFanOut[l]; i++) p[h->lay.w[l] + i] = U(rng);
    }
    // on the network's stream, which does not wait for the null stream; the image's
    // padding stays zero
    if (hipMemsetAsync(h->image, 0, net_image_bytes(), h->stream) != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "upload");
      break;
    }
    st = load_params(h, p.data());
  } while (0);
  if (st != AMCA_OK) {
    delete h;
    return st;
  }
  *out = h;
  return AMCA_OK;
}

amca_status amca_mlp_destroy(amca_mlp* h) {
  delete h;
  return AMCA_OK;
}

amca_status amca_mlp_set_params(amca_mlp* h, const float* p) {
  if (!h || !p) return mlp_fail(AMCA_ERR_INVALID, "null argument");
  return load_params(h, p);
}

amca_status amca_mlp_get_params(amca_mlp* h, float* p) {
  if (!h || !p) return mlp_fail(AMCA_ERR_INVALID, "null argument");
  MLP_HIP(hipStreamSynchronize(h->stream));
  MLP_HIP(hipMemcpy(p, h->params, sizeof(float) * h->lay.total, hipMemcpyDeviceToHost));
  return AMCA_OK;
}

amca_status amca_mlp_forward(amca_mlp* h, int32_t n, const float* x5, float* t) {
  if (!h || n < 1 || !x5 || !t) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  MLP_TRY(ensure_rows(h, n));
  MLP_HIP(hipMemcpyAsync(h->X, x5, sizeof(float) * kIn * n, hipMemcpyHostToDevice, h->stream));
  MLP_TRY(infer(h, n, h->X, h->T));
  MLP_HIP(hipMemcpyAsync(t, h->T, sizeof(float) * n, hipMemcpyDeviceToHost, h->stream));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

amca_status amca_mlp_gradients(amca_mlp* h, int32_t n, const float* x5, const float* y,
                               float* grads, float* loss) {
  if (!h || n < 1 || !x5 || !y) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  MLP_TRY(ensure_rows(h, n));
  int blocks = 0;
  MLP_TRY(train_blocks(h, n, &blocks));
  MLP_HIP(hipMemcpyAsync(h->X, x5, sizeof(float) * kIn * n, hipMemcpyHostToDevice, h->stream));
  MLP_HIP(hipMemcpyAsync(h->Y, y, sizeof(float) * n, hipMemcpyHostToDevice, h->stream));
  MLP_HIP(launch_train(h->params, h->image, blocks, n, h->X, h->Y, h->part, h->part_loss,
                       h->stream));
  MLP_HIP(launch_reduce(blocks, h->part, h->part_loss, h->params, h->grads, h->loss, Adam{},
                        h->image, h->stream));
  if (grads)
    MLP_HIP(hipMemcpyAsync(grads, h->grads, sizeof(float) * h->lay.total, hipMemcpyDeviceToHost,
                           h->stream));
  float l = 0.0f;
  MLP_HIP(hipMemcpyAsync(&l, h->loss, sizeof(float), hipMemcpyDeviceToHost, h->stream));
  MLP_HIP(hipStreamSynchronize(h->stream));
  if (loss) *loss = l / (float)n;
  return AMCA_OK;
}

// One Adam step per batch over device-resident samples X[n][5], Y[n], read in
// place.  The losses stay on the device until kLossSteps of them are there or
// the last step is queued, so no step waits for the host.
amca_status amca_mlp_train_device(amca_mlp* h, int64_t n, const float* dX, const float* dY,
                                  int32_t batch, int32_t steps, float lr, uint64_t seed,
                                  float* loss_trace) {
  if (!h || n < batch || batch < 1 || steps < 0 || !dX || !dY)
    return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  int blocks = 0;
  MLP_TRY(train_blocks(h, batch, &blocks));
  std::mt19937_64 rng(seed);
  const long long nb = n / batch;
  for (int it = 0; it < steps; it++) {
    const long long b = (long long)(rng() % (unsigned long long)nb);
    MLP_HIP(launch_train(h->params, h->image, blocks, batch, dX + (size_t)b * batch * kIn,
                         dY + (size_t)b * batch, h->part, h->part_loss, h->stream));
    h->adam_t++;
    const float b1 = 0.9f, b2 = 0.999f;
    const Adam adam{h->adam_m, h->adam_v, lr, 1.0f - std::pow(b1, (float)h->adam_t),
                    1.0f - std::pow(b2, (float)h->adam_t)};
    const int slot = it % kLossSteps;
    MLP_HIP(launch_reduce(blocks, h->part, h->part_loss, h->params, h->grads, h->loss + slot, adam,
                          h->image, h->stream));
    if (loss_trace && (slot == kLossSteps - 1 || it == steps - 1)) {
      float* out = loss_trace + (it - slot);
      MLP_HIP(hipMemcpyAsync(out, h->loss, sizeof(float) * (slot + 1), hipMemcpyDeviceToHost,
                             h->stream));
      MLP_HIP(hipStreamSynchronize(h->stream));
      for (int q = 0; q <= slot; q++) out[q] /= (float)batch;
    }
  }
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

amca_status amca_mlp_forward_fused(amca_mlp* h, int32_t n, const float* x5, float* t) {
  if (!h || n < 1 || !x5 || !t) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  MLP_TRY(ensure_rows(h, n));
  MLP_HIP(hipMemcpyAsync(h->X, x5, sizeof(float) * kIn * n, hipMemcpyHostToDevice, h->stream));
  MLP_HIP(launch_fused_timed(h, kRowsScaled, n, h->X, h->T, amca_surrogate_desc{}, amca_scan{},
                             SurLattice{}));
  MLP_HIP(hipMemcpyAsync(t, h->T, sizeof(float) * n, hipMemcpyDeviceToHost, h->stream));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

amca_status amca_mlp_enable_timing(amca_mlp* h, int32_t on) {
  if (!h) return mlp_fail(AMCA_ERR_INVALID, "null handle");
  for (hipEvent_t& e : h->ev)
    if (!e) MLP_HIP(hipEventCreate(&e));
  h->timing = on != 0;
  h->fused_ms = 0.0;
  h->fused_launches = h->fused_rows = 0;
  return AMCA_OK;
}

amca_status amca_mlp_fused_times(amca_mlp* h, double* ms, int64_t* launches, int64_t* rows) {
  if (!h || !ms || !launches || !rows) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  *ms = h->fused_ms;
  *launches = h->fused_launches;
  *rows = h->fused_rows;
  return AMCA_OK;
}

// Device rows in place: one launch, no copies and no workspace.
amca_status amca_mlp_forward_device(amca_mlp* h, int64_t n, const float* dX, float* dT) {
  if (!h || n < 1 || !dX || !dT) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  MLP_TRY(infer(h, n, dX, dT));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

amca_status amca_mlp_forward_device_noalloc(amca_mlp* h, int64_t n, const float* dX, float* dT) {
  if (!h || n < 1 || !dX || !dT) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  if (n > AMCA_MLP_NOALLOC_MAX_ROWS)
    return mlp_fail(AMCA_ERR_INVALID, "n = " + std::to_string(n) +
                                          " rows exceeds the no-allocation maximum of " +
                                          std::to_string(AMCA_MLP_NOALLOC_MAX_ROWS) +
                                          " rows per call");
  int dev = -1;
  MLP_HIP(hipGetDevice(&dev));
  if (dev != h->device)
    return mlp_fail(AMCA_ERR_INVALID, "make the network's device (" + std::to_string(h->device) +
                                          ") current before the call");
  MLP_TRY(infer(h, n, dX, dT));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

}  // extern "C"

extern "C" amca_status amca_mlp_gemm_selftest(int32_t M, int32_t N, int32_t K, int32_t trans_a,
                                              int32_t trans_b, const float* A, const float* B,
                                              float* C) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  float *dA = nullptr, *dB = nullptr, *dC = nullptr;
  amca_status st = AMCA_OK;
  hipStream_t s = nullptr;
  do {
    if (hipMalloc(&dA, sizeof(float) * M * K) != hipSuccess ||
        hipMalloc(&dB, sizeof(float) * K * N) != hipSuccess ||
        hipMalloc(&dC, sizeof(float) * M * N) != hipSuccess || hipStreamCreate(&s) != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "alloc");
      break;
    }
    (void)hipMemcpy(dA, A, sizeof(float) * M * K, hipMemcpyHostToDevice);
    (void)hipMemcpy(dB, B, sizeof(float) * K * N, hipMemcpyHostToDevice);
    const int lda = trans_a ? M : K, ldb = trans_b ? K : N;
    const dim3 grid((N + kBN - 1) / kBN, (M + kBM - 1) / kBM), block(kThreads);
    if (!trans_a && !trans_b)
      hipLaunchKernelGGL((k_gemm<false, false>), grid, block, 0, s, dA, lda, dB, ldb, M, N, K, dC);
    else if (trans_a && !trans_b)
      hipLaunchKernelGGL((k_gemm<true, false>), grid, block, 0, s, dA, lda, dB, ldb, M, N, K, dC);
    else if (!trans_a && trans_b)
      hipLaunchKernelGGL((k_gemm<false, true>), grid, block, 0, s, dA, lda, dB, ldb, M, N, K, dC);
    else
      hipLaunchKernelGGL((k_gemm<true, true>), grid, block, 0, s, dA, lda, dB, ldb, M, N, K, dC);
    const hipError_t r = hipGetLastError();
    if (r != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
      st = mlp_fail(AMCA_ERR_HIP, "gemm");
      break;
    }
    (void)hipMemcpy(C, dC, sizeof(float) * M * N, hipMemcpyDeviceToHost);
  } while (0);
  if (dA) (void)hipFree(dA);
  if (dB) (void)hipFree(dB);
  if (dC) (void)hipFree(dC);
  if (s) (void)hipStreamDestroy(s);
  return st;
}

// ===========================================================================
// Training data and lattice evaluation of the temperature surrogate.


namespace mlpk {

struct Sampler {
  amca_surrogate_desc d;
  amca_scan s[16];
  int n_scans;
};

__device__ __forceinline__ unsigned long long splitmix(unsigned long long& st) {
  unsigned long long z = (st += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double unit(unsigned long long& st) {
  return (double)(splitmix(st) >> 11) * (1.0 / 9007199254740992.0);
}

__device__ __forceinline__ double rosenthal(const amca_surrogate_desc& d, const amca_scan& s,
                                            double x, double y, double z, double t) {
  const double xi = x - (s.x_start + s.v * t);
  const double dy = y - s.y_c, dz = z - d.z_top;
  double R = sqrt(xi * xi + dy * dy + dz * dz);
  if (R < d.r_min) R = d.r_min;
  return d.T0 + d.eta * s.P / (2.0 * 3.14159265358979323846 * d.k) / R *
                    exp(-s.v * (R + xi) / (2.0 * d.alpha));
}

// the coupled domain's FE path at (x, y, z, t): nodal frames of the source at
// t_f and t_f+1, linear in time (void rule), hex8 in space
__device__ double fe_temperature(const amca_surrogate_desc& d, const amca_scan& s, double x,
                                 double y, double z, double t) {
  int e[3];
  double p[3];
  const double o[3] = {d.fx0, d.fy0, d.fz0};
  const int n[3] = {d.fnx, d.fny, d.fnz};
  const double q[3] = {x, y, z};
  for (int a = 0; a < 3; a++) {
    int i = (int)floor((q[a] - o[a]) / d.fdx);
    i = i < 0 ? 0 : (i > n[a] - 2 ? n[a] - 2 : i);
    e[a] = i;
    p[a] = 2.0 * ((q[a] - (o[a] + i * d.fdx)) / d.fdx) - 1.0;
  }
  int f = (int)floor(t / d.frame_dt);
  f = f < 0 ? 0 : (f > d.n_frames - 2 ? d.n_frames - 2 : f);
  const double r = (t - f * d.frame_dt) / d.frame_dt;
  const double xi = p[0], eta = p[1], zeta = p[2];
  const double sf[8] = {
      0.125 * (1.0 - eta) * (1.0 - xi) * (1.0 - zeta), 0.125 * (1.0 - eta) * (1.0 + xi) * (1.0 - zeta),
      0.125 * (1.0 + eta) * (1.0 + xi) * (1.0 - zeta), 0.125 * (1.0 + eta) * (1.0 - xi) * (1.0 - zeta),
      0.125 * (1.0 - eta) * (1.0 - xi) * (1.0 + zeta), 0.125 * (1.0 - eta) * (1.0 + xi) * (1.0 + zeta),
      0.125 * (1.0 + eta) * (1.0 + xi) * (1.0 + zeta), 0.125 * (1.0 + eta) * (1.0 - xi) * (1.0 + zeta)};
  const int di[8] = {0, 1, 1, 0, 0, 1, 1, 0}, dj[8] = {0, 0, 1, 1, 0, 0, 1, 1},
            dk[8] = {0, 0, 0, 0, 1, 1, 1, 1};
  double T = 0.0;
  for (int m = 0; m < 8; m++) {
    const double nx = d.fx0 + (e[0] + di[m]) * d.fdx, ny = d.fy0 + (e[1] + dj[m]) * d.fdx,
                 nz = d.fz0 + (e[2] + dk[m]) * d.fdx;
    const double th1 = rosenthal(d, s, nx, ny, nz, f * d.frame_dt);
    const double th0 = rosenthal(d, s, nx, ny, nz, (f + 1) * d.frame_dt);
    const double v = d.void_temperature;
    const double th = (th0 <= v) ? v : ((th1 <= v) ? th0 : r * (th0 - th1) + th1);
    T += sf[m] * th;
  }
  return T;
}

__device__ __forceinline__ void inputs(const amca_surrogate_desc& d, const amca_scan& s, double x,
                                       double y, double z, double t, float* o) {
  o[0] = (float)((x - s.x_start - s.v * t) / d.xi_scale);
  o[1] = (float)((y - s.y_c) / d.y_scale);
  o[2] = (float)((z - d.z_top) / d.z_scale);
  o[3] = (float)(s.P / d.P_scale);
  o[4] = (float)(s.v / d.v_scale);
}

__device__ __host__ inline double to_target(const amca_surrogate_desc& d, double T) {
  const double u = (fmin(T, d.T_clip) - d.T_ref) / d.T_scale;
  return d.log_target ? log1p(fmax(u, 0.0)) : u;
}
__device__ __host__ inline double from_target(const amca_surrogate_desc& d, double y) {
  return d.T_ref + d.T_scale * (d.log_target ? expm1(y) : y);
}

__global__ void k_sample(Sampler S, long long n, double near_fraction, unsigned long long seed,
                         float* __restrict__ X, float* __restrict__ Y) {
  const amca_surrogate_desc& d = S.d;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    unsigned long long st = seed ^ ((unsigned long long)i * 0xd1b54a32d192ed03ull);
    const amca_scan& s = S.s[i % S.n_scans];
    const double t = unit(st) * (d.n_frames - 1) * d.frame_dt;
    const double lx = (d.fnx - 1) * d.fdx, ly = (d.fny - 1) * d.fdx, lz = (d.fnz - 1) * d.fdx;
    double x, y, z;
    if (unit(st) < near_fraction) {
      // close behind the source, where the field varies: 40 xi_scale behind,
      // 4 ahead, 8 y_scale across, 8 z_scale deep
      x = s.x_start + s.v * t + (unit(st) * 44.0 - 40.0) * d.xi_scale;
      y = s.y_c + (unit(st) * 2.0 - 1.0) * 8.0 * d.y_scale;
      z = d.z_top - unit(st) * 8.0 * d.z_scale;
    } else {
      x = d.fx0 + unit(st) * lx;
      y = d.fy0 + unit(st) * ly;
      z = d.fz0 + unit(st) * lz;
    }
    x = fmin(fmax(x, d.fx0), d.fx0 + lx);
    y = fmin(fmax(y, d.fy0), d.fy0 + ly);
    z = fmin(fmax(z, d.fz0), d.fz0 + lz);
    const double T = fe_temperature(d, s, x, y, z, t);
    inputs(d, s, x, y, z, t, X + 5 * i);
    Y[i] = (float)to_target(d, T);
  }
}

// ---------------------------------------------------------------------------
// Fused inference: the whole network per 64 rows in one wave (two halves of 32
// whose MFMAs and SiLU epilogues interleave), weights in LDS, activations in
// registers.  Layer l computes D'[out][row] = W_l^T act^T with
// v_mfma_f32_32x32x16_bf16 (A = weights, rows = output features; B =
// activations, columns = batch rows).  The accumulator of a 32 x 32 tile holds,
// in lane L and register i, output feature (i/4)*8 + (L/32)*4 + i%4 of batch
// row L%32: after bias, SiLU and BF16 rounding, registers 8s..8s+7 of tile t
// are exactly the B operand of the next layer's k-step 2t+s, provided that
// k-step's k order is the one those registers carry.  The weights are laid out
// in LDS in that order, so no activation moves between lanes.
//   k-step ks, lane group g (= L/32), element ii  <->  input feature
//   16*ks + 8*(ii/4) + 4*g + ii%4
// The hidden layers carry y = -log2(e) z instead of the pre-activation z, so
// that sigmoid(z) = 1 / (1 + 2^y) is one v_exp_f32 and one v_rcp_f32 with no
// scaling multiply: the stored activation is a' = y sigmoid(z) = -log2(e)
// silu(z), whose factor cancels against the -log2(e) the next layer's bias
// carries (y_next = W a' - log2(e) b = -log2(e) z_next).  Layer 1 scales its
// accumulator once (one FMA with the scaled bias); layer 5 is an MFMA with W5
// in every row of A and scales its output by -1/log2(e) before adding b5.  The
// biases of layers 2..4 are loaded into the accumulators before the first
// MFMA, so those layers add no bias either.
// Inputs and weights round to BF16; the activations round to BF16 as scaled
// values.  kRows keeps the unscaled form z sigmoid(z) instead (one multiply
// more per activation), which rounds the activations where training does.

constexpr int kFusedWaves = 8;
constexpr int kWtStride = kHid + 8;  // bf16 per LDS row (padding spreads the banks)

struct alignas(16) FusedLds {
  __bf16 wt[3][kHid][kWtStride];  // layers 2..4: wt[l][out][16*ks + 8*g + ii]
  __bf16 w1t[kHid][8];            // layer 1: W1[k][out] for k < 5, zero above
  float b[4][kHid];               // biases of layers 1..4, times -log2(e)
  __bf16 w5[8][2][8];             // W5 in BF16, as the A fragment of k-step ks, lane group g
  float b5;
};

// FusedLds as every work-group copies it into LDS, kept in device memory and
// rewritten when the parameters change, and the biases without the scaling for
// kRows.  Building it from the FP32 parameters in every work-group (a
// transposing gather of 50 K values, each rounded) cost more than a small call.
struct FusedImage {
  FusedLds lds;
  float raw_b[4][kHid];
};
static_assert(offsetof(FusedLds, b) % 16 == 0 && sizeof(FusedLds::b) % 16 == 0 &&
                  offsetof(FusedImage, raw_b) % 16 == 0,
              "the image is copied in 16-byte pieces");

// The hidden layers' weights as the B operands of k_train, 8 values per lane and
// k-step: wf for the forward pass (k = input, column = output feature), wb for
// the backward pass (k = output, column = input feature); w1f is layer 1, its k
// rows above the five inputs zero.
struct NetImage {
  FusedImage f;
  __bf16 wf[3][4][8][64][8];  // [layer][column tile][k-step][lane][k]
  __bf16 wb[3][4][8][64][8];
  __bf16 w1f[4][64][8];
};
static_assert(offsetof(NetImage, wf) % 16 == 0, "operands are read 16 bytes at a time");
size_t net_image_bytes() { return sizeof(NetImage); }

constexpr float kNegLog2e = -1.4426950408889634f;
constexpr float kNegLn2 = -0.6931471805599453f;  // -1/log2(e)

__device__ __forceinline__ int fused_feature(int ks, int g, int ii) {
  return 16 * ks + 8 * (ii >> 2) + 4 * g + (ii & 3);
}

// parameter offsets of the layered layout: W1 at 0, b1 at 640; layer l >= 2
// (0-based 1..3) at 768 + (l-1) * 16512, its bias 16384 further; W5, b5 last
__device__ __forceinline__ int fused_w(int l) { return l == 0 ? 0 : 768 + (l - 1) * 16512; }
__device__ __forceinline__ int fused_b(int l) { return l == 0 ? 640 : fused_w(l) + kHid * kHid; }

// parameter i into its places in the images
__device__ __forceinline__ void pack_param(NetImage& N, int i, float v) {
  FusedImage& I = N.f;
  FusedLds& L = I.lds;
  if (i < kIn * kHid) {
    const int in = i / kHid, out = i % kHid;
    L.w1t[out][in] = (__bf16)v;
    N.w1f[out >> 5][out & 31][in] = (__bf16)v;
    return;
  }
  const int w5 = fused_b(3) + kHid;
  if (i >= w5) {
    const int in = i - w5;
    if (in == kHid) {
      L.b5 = v;
    } else {
      const int r = in & 15;  // in = 16 ks + 8 (ii / 4) + 4 g + ii % 4
      L.w5[in >> 4][(r >> 2) & 1][4 * (r >> 3) + (r & 3)] = (__bf16)v;
    }
    return;
  }
  int l = 0, q = i - fused_b(0);
  if (q >= kHid) {
    l = 1 + (q - kHid) / (kHid * kHid + kHid);
    q = i - fused_w(l);
  } else {
    q += kHid * kHid;  // a bias of layer 1, in the place of the other layers' biases
  }
  if (q >= kHid * kHid) {
    I.raw_b[l][q - kHid * kHid] = v;
    L.b[l][q - kHid * kHid] = kNegLog2e * v;
    return;
  }
  const int in = q / kHid, out = q % kHid, r = in & 15;
  L.wt[l - 1][out][16 * (in >> 4) + 8 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3)] = (__bf16)v;
  N.wf[l - 1][out >> 5][in >> 4][((in >> 3) & 1) * 32 + (out & 31)][in & 7] = (__bf16)v;
  N.wb[l - 1][in >> 5][out >> 4][((out >> 3) & 1) * 32 + (in & 31)][out & 7] = (__bf16)v;
}

// The images of all parameters, and Adam's moments from zero.
__global__ void __launch_bounds__(kThreads) k_pack(const float* __restrict__ p,
                                                   NetImage* __restrict__ img,
                                                   float* __restrict__ m, float* __restrict__ v) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= fused_b(3) + 2 * kHid + 1) return;
  pack_param(*img, i, p[i]);
  m[i] = 0.0f;
  v[i] = 0.0f;
}

hipError_t launch_pack(const float* p, NetImage* img, float* m, float* v, hipStream_t st) {
  const int n = Layout().total;
  hipLaunchKernelGGL(k_pack, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, st, p, img, m,
                     v);
  return hipGetLastError();
}

template <bool kScaled>
__device__ __forceinline__ void fused_load(const FusedImage* __restrict__ img, FusedLds& L) {
  constexpr int kPieces = (int)((sizeof(FusedLds) + 15) / 16);
  constexpr int kPer = (kPieces + 64 * kFusedWaves - 1) / (64 * kFusedWaves);
  constexpr int kB0 = (int)(offsetof(FusedLds, b) / 16), kB1 = kB0 + (int)(sizeof(L.b) / 16);
  const uint4* src = reinterpret_cast<const uint4*>(img);
  const uint4* raw = reinterpret_cast<const uint4*>(&img->raw_b[0][0]) - kB0;
  uint4* dst = reinterpret_cast<uint4*>(&L);
  uint4 v[kPer];
#pragma unroll
  for (int x = 0; x < kPer; x++) {
    const int q = threadIdx.x + x * 64 * kFusedWaves;
    v[x] = make_uint4(0u, 0u, 0u, 0u);
    if (q < kPieces) v[x] = (!kScaled && q >= kB0 && q < kB1) ? raw[q] : src[q];
  }
#pragma unroll
  for (int x = 0; x < kPer; x++) {
    const int q = threadIdx.x + x * 64 * kFusedWaves;
    if (q < kPieces) dst[q] = v[x];
  }
  __syncthreads();
}

// Chunk ks of the epilogue: a' = y / (1 + 2^y) of the eight accumulator
// registers 8(ks%2).. of tile ks/2, rounded to BF16, into the next layer's B
// operand bop[ks]; kFirst: y = -log2(e) acc + bias (layer 1), else y = acc.
// Unscaled: a = z / (1 + 2^(-log2(e) z)), z = acc + bias (layer 1) or acc.
template <bool kFirst, bool kScaled>
__device__ __forceinline__ void fused_epi_chunk(const floatx16* acc, const float* bias, int g,
                                                int ks, bf16x8* bop) {
  const int t = ks >> 1, s = ks & 1;
#pragma unroll
  for (int ii = 0; ii < 8; ii++) {
    float y = acc[t][8 * s + ii];
    if (kFirst) {
      const float b = bias[fused_feature(ks, g, ii)];
      y = kScaled ? fmaf(y, kNegLog2e, b) : y + b;
    }
    const float e = __builtin_amdgcn_exp2f(kScaled ? y : kNegLog2e * y);
    bop[ks][ii] = (__bf16)(y * __builtin_amdgcn_rcpf(1.0f + e));
  }
}

// One phase of the two-half schedule: the 32 MFMAs of hidden layer l + 2
// (l = 0..2) for half P, interleaved with the epilogue of the previous layer
// of half Q, which needs no MFMA result of this phase.  The accumulators of P
// start at the layer's bias (register 4q+j of tile ot holds output feature
// 32 ot + 8 q + 4 g + j); the weight fragments of k-step ks+1 are read from
// LDS while those of k-step ks feed the MFMAs.
template <bool kFirstEpi, bool kScaled>
__device__ __forceinline__ void fused_phase(const FusedLds& L, int l, int r, int g,
                                            floatx16* accP, const bf16x8* bopP,
                                            const floatx16* accQ, bf16x8* bopQ) {
#pragma unroll
  for (int ot = 0; ot < 4; ot++) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float4 b = *reinterpret_cast<const float4*>(&L.b[l + 1][32 * ot + 8 * q + 4 * g]);
      accP[ot][4 * q] = b.x;
      accP[ot][4 * q + 1] = b.y;
      accP[ot][4 * q + 2] = b.z;
      accP[ot][4 * q + 3] = b.w;
    }
  }
  const __bf16* wl = &L.wt[l][r][8 * g];
  bf16x8 a[2][4];
#pragma unroll
  for (int ot = 0; ot < 4; ot++)
    a[0][ot] = *reinterpret_cast<const bf16x8*>(wl + 32 * ot * kWtStride);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = 0; ks < 8; ks++) {
    if (ks + 1 < 8) {
#pragma unroll
      for (int ot = 0; ot < 4; ot++)
        a[(ks + 1) & 1][ot] =
            *reinterpret_cast<const bf16x8*>(wl + 32 * ot * kWtStride + 16 * (ks + 1));
    }
#pragma unroll
    for (int ot = 0; ot < 4; ot++)
      accP[ot] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks & 1][ot], bopP[ks], accP[ot], 0, 0, 0);
    fused_epi_chunk<kFirstEpi, kScaled>(accQ, L.b[0], g, ks, bopQ);
    // LDS reads first, then each MFMA followed by a share of the epilogue
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
    for (int m = 0; m < 4; m++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Layer 5 of half P (8 MFMAs, A = W5 in every row, so every accumulator
// register of lane L holds the output of row L % 32), optionally interleaved
// with the last epilogue of half Q.
template <bool kEpi, bool kScaled>
__device__ __forceinline__ float fused_out(const FusedLds& L, int g, const bf16x8* bopP,
                                           const floatx16* accQ, bf16x8* bopQ) {
  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.0f;
#pragma unroll
  for (int ks = 0; ks < 8; ks++) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(&L.w5[ks][g][0]);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bopP[ks], acc, 0, 0, 0);
    if (kEpi) {
      fused_epi_chunk<false, kScaled>(accQ, nullptr, g, ks, bopQ);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 40, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  return kScaled ? fmaf(acc[0], kNegLn2, L.b5) : acc[0] + L.b5;
}

// Network output (the training target scale) of the 64 rows whose inputs the
// lanes hold in x[0..4] (lane L: row L of the group), returned in lane L.
// Half X is rows 0..31, half Y rows 32..63; each runs the whole network, and
// the MFMAs of one half overlap the SiLU epilogue of the other.
template <bool kScaled>
__device__ __forceinline__ float fused_rows(const FusedLds& L, const float* x) {
  const int lane = threadIdx.x & 63, g = lane >> 5, r = lane & 31;
  floatx16 accX[4], accY[4];
  bf16x8 bopX[8], bopY[8];
  // layer 1: K = 5, padded to one k-step of 16.  Half X takes k 0..7 (lane
  // group 0 holds its rows), half Y k 8..15 (lane group 1); the weight rows
  // repeat in both k halves and the other half's inputs are zero.
  bf16x8 bx, by;
#pragma unroll
  for (int ii = 0; ii < 8; ii++) {
    const __bf16 v = (__bf16)(ii < kIn ? x[ii] : 0.0f);
    bx[ii] = g == 0 ? v : (__bf16)0.0f;
    by[ii] = g == 1 ? v : (__bf16)0.0f;
  }
#pragma unroll
  for (int ot = 0; ot < 4; ot++) {
    const bf16x8 w = *reinterpret_cast<const bf16x8*>(&L.w1t[32 * ot + r][0]);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      accX[ot][i] = 0.0f;
      accY[ot][i] = 0.0f;
    }
    accX[ot] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, bx, accX[ot], 0, 0, 0);
    accY[ot] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, by, accY[ot], 0, 0, 0);
  }
#pragma unroll
  for (int ks = 0; ks < 8; ks++) fused_epi_chunk<true, kScaled>(accX, L.b[0], g, ks, bopX);
  // hidden layers 2..4
  fused_phase<true, kScaled>(L, 0, r, g, accX, bopX, accY, bopY);
  fused_phase<false, kScaled>(L, 0, r, g, accY, bopY, accX, bopX);
  fused_phase<false, kScaled>(L, 1, r, g, accX, bopX, accY, bopY);
  fused_phase<false, kScaled>(L, 1, r, g, accY, bopY, accX, bopX);
  fused_phase<false, kScaled>(L, 2, r, g, accX, bopX, accY, bopY);
  fused_phase<false, kScaled>(L, 2, r, g, accY, bopY, accX, bopX);
  const float tx = fused_out<true, kScaled>(L, g, bopX, accY, bopY);
  const float ty = fused_out<false, kScaled>(L, g, bopY, nullptr, nullptr);
  return g == 0 ? tx : ty;
}

// Bound by the SiLU epilogue's two transcendentals per activation (rows in and
// out are 24 bytes against 99 840 flop).  Every inference call runs here: rows
// that went through one tiled GEMM per layer, the activations through memory,
// took 1417 us for 1 000 003 rows and 95 us for 300 (five launches); in this
// kernel 154 us (646 TFLOP/s) and 23.5 us.
// 64-row groups over the work-groups: group gr goes to work-group gr % gridDim,
// so that a call of a few hundred rows spreads over as many CUs instead of
// filling one work-group's eight waves.
template <int kMode>
__global__ void __launch_bounds__(64 * kFusedWaves)
k_mlp_fused(const FusedImage* __restrict__ img, long long n, const float* __restrict__ X,
            float* __restrict__ out, amca_surrogate_desc d, amca_scan s, SurLattice g) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  FusedLds& L = *reinterpret_cast<FusedLds*>(lds_raw);
  fused_load<kMode != kRows>(img, L);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long groups = (n + 63) / 64;
  for (long long gr = blockIdx.x + (long long)wave * gridDim.x; gr < groups;
       gr += (long long)gridDim.x * kFusedWaves) {
    const long long row = gr * 64 + lane;
    float x[kIn] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (row < n) {
      if (kMode != kLattice) {
#pragma unroll
        for (int q = 0; q < kIn; q++) x[q] = X[row * kIn + q];
      } else {
        const int i = (int)(row % g.nxi);
        const int j = (int)((row / g.nxi) % g.ny);
        const int k = (int)(row / ((long long)g.nxi * g.ny));
        inputs(d, s, g.xi0 + i * g.dxi + s.x_start, g.y0 + j * g.dy, g.z0 + k * g.dz, 0.0, x);
      }
    }
    const float t = fused_rows<kMode != kRows>(L, x);
    if (row < n) out[row] = kMode != kLattice ? t : (float)from_target(d, (double)t);
  }
}

hipError_t train_setup();

hipError_t fused_setup() {
  for (const void* f : {(const void*)k_mlp_fused<kRowsScaled>, (const void*)k_mlp_fused<kLattice>,
                        (const void*)k_mlp_fused<kRows>}) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)sizeof(FusedLds));
    if (e != hipSuccess) return e;
  }
  return train_setup();
}

// One work-group per CU at most (its weights fill two thirds of the LDS, so
// more would only load them again when a CU comes free).
hipError_t launch_fused(FusedMode mode, const NetImage* img, int cus, long long n, const float* X,
                        float* out, const amca_surrogate_desc& d, const amca_scan& s,
                        const SurLattice& g, hipStream_t st) {
  const dim3 grid((unsigned)std::max(1LL, std::min((n + 63) / 64, (long long)cus)));
  const dim3 block(64 * kFusedWaves);
  const size_t lds = sizeof(FusedLds);
  const FusedImage* f = &img->f;
  if (mode == kRowsScaled)
    hipLaunchKernelGGL(k_mlp_fused<kRowsScaled>, grid, block, lds, st, f, n, X, out, d, s, g);
  else if (mode == kLattice)
    hipLaunchKernelGGL(k_mlp_fused<kLattice>, grid, block, lds, st, f, n, X, out, d, s, g);
  else
    hipLaunchKernelGGL(k_mlp_fused<kRows>, grid, block, lds, st, f, n, X, out, d, s, g);
  return hipGetLastError();
}

// launch_fused, bracketed by HIP events on the handle's stream when timing is
// on (the launch is waited for and its duration added to the totals)
hipError_t launch_fused_timed(amca_mlp* h, FusedMode mode, long long n, const float* X, float* out,
                              const amca_surrogate_desc& d, const amca_scan& s,
                              const SurLattice& g) {
  if (!h->timing) return launch_fused(mode, h->image, h->cus, n, X, out, d, s, g, h->stream);
  hipError_t e = hipEventRecord(h->ev[0], h->stream);
  if (e == hipSuccess) e = launch_fused(mode, h->image, h->cus, n, X, out, d, s, g, h->stream);
  if (e == hipSuccess) e = hipEventRecord(h->ev[1], h->stream);
  if (e == hipSuccess) e = hipEventSynchronize(h->ev[1]);
  float ms = 0.0f;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, h->ev[0], h->ev[1]);
  if (e == hipSuccess) {
    h->fused_ms += ms;
    h->fused_launches++;
    h->fused_rows += n;
  }
  return e;
}

// ---------------------------------------------------------------------------
// Training.  A work-group of four waves takes 64 rows through the network and
// back.  Wave w owns the 32 features f = 32 w + lane % 32 of every layer, for
// both 32-row tiles: with rows as M and features as N, its accumulators hold
// rows 32 rt + 8 (i / 4) + 4 (lane / 32) + i % 4 of feature f, and silu'(z) of
// every layer stays there (FP32) from the forward to the backward pass.
// Activations and dZ go through LDS in two layouts: [row][feature], the A
// operand of the next layer (or of dZ W^T), and [feature][row], the operands of
// the weight gradients A^T dZ, whose k is the row.  The work-group's gradients
// go to its own row of `part`; a work-group that takes more than one group of
// rows starts each weight-gradient tile from what it left there.  Weights come
// straight from L2 as matrix operands: every wave reads other tiles, so LDS
// would not save a byte.  Operands round to BF16 at the matrix instructions, dZ
// and the bias gradients are FP32 up to there, and the sums run in a fixed
// order, so the gradients are the same on every run.
//
// Bound by the latency of its chain of layers (one work-group per CU, 16
// barriers a group of rows).  One GEMM launch per layer and direction, with the
// activations, dZ and atomic gradient sums through memory, took 285 us per step
// of 8192 rows; k_train and k_reduce take 40 us.
struct TrainLds {
  __bf16 act[kTrainRows][kHid + 8];      // [row][feature]: activations, then dZ
  __bf16 at[4][kHid][kTrainRows + 8];    // [feature][row] of the four activations
  __bf16 xt[32][kTrainRows + 8];         // [input][row], rows above the five inputs zero
  __bf16 dzt[kHid][kTrainRows + 8];      // [feature][row] of dZ
  float w5[kHid];                        // W5, rounded to BF16
  float dT[kTrainRows];
  float sum[2][4];
};
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// 32 values of feature f (both row tiles) into the two LDS layouts
__device__ __forceinline__ void train_store(TrainLds& S, __bf16 (*t)[kTrainRows + 8], int f, int g,
                                            const floatx16* v) {
#pragma unroll
  for (int rt = 0; rt < 2; rt++) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int row = 32 * rt + 8 * q + 4 * g;
      bf16x4 x;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        x[j] = (__bf16)v[rt][4 * q + j];
        S.act[row + j][f] = x[j];
      }
      *reinterpret_cast<bf16x4*>(&t[f][row]) = x;
    }
  }
}

// acc[rt] += S.act rows of tile rt times the 128 x 32 operand tile b
__device__ __forceinline__ void train_mfma(const TrainLds& S, const bf16x8* __restrict__ b, int lane,
                                           floatx16* acc) {
  const int c = lane & 31, g = lane >> 5;
  bf16x8 w[8];
#pragma unroll
  for (int ks = 0; ks < 8; ks++) w[ks] = b[64 * ks + lane];
#pragma unroll
  for (int ks = 0; ks < 8; ks++) {
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&S.act[32 * rt + c][16 * ks + 8 * g]);
      acc[rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w[ks], acc[rt], 0, 0, 0);
    }
  }
}

// A phase boundary of k_train.  The scheduling barrier keeps the next phase's
// loads behind it: hoisted, the weights of every layer would sit in registers.
__device__ __forceinline__ void train_sync() {
  __syncthreads();
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ void __launch_bounds__(kThreads, 1)
k_train(const float* __restrict__ p, const NetImage* __restrict__ img, int n,
        const float* __restrict__ X, const float* __restrict__ Y, float* __restrict__ part,
        float* __restrict__ part_loss) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  TrainLds& S = *reinterpret_cast<TrainLds*>(lds_raw);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int c = lane & 31, g = lane >> 5, f = 32 * w + c;
  const int off_w5 = fused_b(3) + kHid;
  float* __restrict__ out = part + (size_t)blockIdx.x * kPartStride;
  if (t < kHid) S.w5[t] = (float)(__bf16)p[off_w5 + t];
  for (int q = t; q < 32 * (kTrainRows + 8); q += kThreads) (&S.xt[0][0])[q] = (__bf16)0.0f;
  const float b5 = p[off_w5 + kHid], inv_n = 2.0f / (float)n;
  const bf16x8 w1 = *reinterpret_cast<const bf16x8*>(&img->w1f[w][lane][0]);
  float bias[4], db[4];
#pragma unroll
  for (int l = 0; l < 4; l++) {
    bias[l] = p[fused_b(l) + f];
    db[l] = 0.0f;
  }
  float dw5 = 0.0f, db5 = 0.0f, loss = 0.0f;
  const int groups = (n + kTrainRows - 1) / kTrainRows;
  for (int gr = blockIdx.x; gr < groups; gr += gridDim.x) {
    const bool first = gr == (int)blockIdx.x;
    const int base = gr * kTrainRows;
    // opaque to the compiler, or it keeps every layer's weights and every
    // address of the loop in registers across the groups, and spills
    const NetImage* im = img;
    asm volatile("" : "+s"(im), "+v"(c), "+v"(g), "+v"(f));
    train_sync();  // xt cleared; the last group's reads done
    // layer 1: K = 5 in one k-step of 16
    bf16x8 xa[2];
    floatx16 z[4][2];
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
      const int r = base + 32 * rt + c;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float v = 0.0f;
        if (j < kIn && g == 0 && r < n) v = X[(size_t)r * kIn + j];
        xa[rt][j] = (__bf16)v;
      }
      if (w == 0 && g == 0)
#pragma unroll
        for (int j = 0; j < kIn; j++) S.xt[j][32 * rt + c] = xa[rt][j];
#pragma unroll
      for (int i = 0; i < 16; i++) z[0][rt][i] = bias[0];
      z[0][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[rt], w1, z[0][rt], 0, 0, 0);
    }
    floatx16 a[2];
#pragma unroll
    for (int l = 0; l < 4; l++) {
      if (l > 0) {
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
          for (int i = 0; i < 16; i++) z[l][rt][i] = bias[l];
        train_mfma(S, reinterpret_cast<const bf16x8*>(&im->wf[l - 1][w][0][0][0]), lane, z[l]);
        train_sync();  // the layer's input is read
      }
#pragma unroll
      for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const float v = z[l][rt][i], sg = sigmoid(v);
          a[rt][i] = v * sg;
          z[l][rt][i] = sg * (1.0f + v * (1.0f - sg));  // silu'(z), all the way back needs
        }
      train_store(S, S.at[l], f, g, a);
      train_sync();
    }
    // layer 5 and the loss: four threads per row, 32 features each
    {
      const int row = t >> 2, q = t & 3;
      float s = 0.0f;
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(&S.act[row][32 * q + 8 * x]);
#pragma unroll
        for (int j = 0; j < 8; j++) s = fmaf((float)v[j], S.w5[32 * q + 8 * x + j], s);
      }
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      float r = 0.0f;
      if (base + row < n) r = (s + b5) - Y[base + row];
      if (q == 0) {
        S.dT[row] = inv_n * r;  // the gradient of the mean squared error
        db5 += inv_n * r;
        loss += r * r;
      }
    }
    train_sync();
    // dW5 = A4^T dT: two threads per feature, 32 rows each
    {
      const int fe = t >> 1, h = t & 1;
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(&S.at[3][fe][32 * h + 8 * x]);
#pragma unroll
        for (int j = 0; j < 8; j++) dw5 = fmaf((float)v[j], S.dT[32 * h + 8 * x + j], dw5);
      }
    }
    // dZ4 = dT W5^T silu'(Z4)
    const float w5 = S.w5[f];
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 32 * rt + 8 * (i >> 2) + 4 * g + (i & 3);
        a[rt][i] = S.dT[row] * w5 * z[3][rt][i];
        db[3] += a[rt][i];
      }
    train_store(S, S.dzt, f, g, a);
    train_sync();
#pragma unroll
    for (int l = 3; l >= 0; l--) {
      // dW = A^T dZ: input tile w against the four output tiles (layer 1: the
      // inputs against output tile w)
      if (l > 0) {
        bf16x8 av[4];
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
          av[ks] = *reinterpret_cast<const bf16x8*>(&S.at[l - 1][f][16 * ks + 8 * g]);
#pragma unroll
        for (int ot = 0; ot < 4; ot++) {
          float* o = out + fused_w(l) + (32 * w + 4 * g) * kHid + 32 * ot + c;
          floatx16 acc;
#pragma unroll
          for (int i = 0; i < 16; i++)
            acc[i] = first ? 0.0f : o[(8 * (i >> 2) + (i & 3)) * kHid];
#pragma unroll
          for (int ks = 0; ks < 4; ks++) {
            const bf16x8 b =
                *reinterpret_cast<const bf16x8*>(&S.dzt[32 * ot + c][16 * ks + 8 * g]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[ks], b, acc, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 16; i++) o[(8 * (i >> 2) + (i & 3)) * kHid] = acc[i];
        }
        __builtin_amdgcn_sched_barrier(0);
        // dZ of the layer below
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
          for (int i = 0; i < 16; i++) a[rt][i] = 0.0f;
        train_mfma(S, reinterpret_cast<const bf16x8*>(&im->wb[l - 1][w][0][0][0]), lane, a);
        train_sync();  // dZ is read
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
          for (int i = 0; i < 16; i++) {
            a[rt][i] *= z[l - 1][rt][i];
            db[l - 1] += a[rt][i];
          }
        train_store(S, S.dzt, f, g, a);
        train_sync();
      } else {
        floatx16 acc;
        float* o = out + f;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
          const bf16x8 av = *reinterpret_cast<const bf16x8*>(&S.xt[c][16 * ks + 8 * g]);
          const bf16x8 b = *reinterpret_cast<const bf16x8*>(&S.dzt[f][16 * ks + 8 * g]);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, b, acc, 0, 0, 0);
        }
        // inputs 0..3 are elements 0..3 of lane group 0, input 4 element 0 of group 1
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (g == 0 || i == 0) {
            float* q = o + (4 * g + i) * kHid;
            *q = (first ? 0.0f : *q) + acc[i];
          }
      }
    }
  }
#pragma unroll
  for (int l = 0; l < 4; l++) {
    const float v = db[l] + __shfl_xor(db[l], 32, 64);
    if (g == 0) out[fused_b(l) + f] = v;
  }
  dw5 += __shfl_xor(dw5, 1, 64);
  if ((t & 1) == 0) out[off_w5 + (t >> 1)] = dw5;
  loss = wave_sum_f(loss);
  db5 = wave_sum_f(db5);
  if (lane == 0) {
    S.sum[0][w] = loss;
    S.sum[1][w] = db5;
  }
  __syncthreads();
  if (t == 0) {
    part_loss[blockIdx.x] = (S.sum[0][0] + S.sum[0][1]) + (S.sum[0][2] + S.sum[0][3]);
    out[off_w5 + kHid] = (S.sum[1][0] + S.sum[1][1]) + (S.sum[1][2] + S.sum[1][3]);
  }
}

hipError_t train_setup() {
  return hipFuncSetAttribute((const void*)k_train, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)sizeof(TrainLds));
}

// Gradient i = the sum of the work-groups' shares, each wave a quarter of them
// in order; with Adam's moments the parameter and its places in the images
// follow at once.  Bound by the read of the shares (26 MB for 8192 rows, mostly
// from L2 and the memory-side cache).
__global__ void __launch_bounds__(kThreads)
k_reduce(int blocks, const float* __restrict__ part, const float* __restrict__ part_loss,
         float* __restrict__ p, float* __restrict__ grads, float* __restrict__ loss, Adam adam,
         NetImage* __restrict__ img) {
  __shared__ float s_sum[kThreads / 64][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  const int total = fused_b(3) + 2 * kHid + 1;
  float s = 0.0f;
  if (i < total) {
    const float* q = part + i;
    int b = w;
    for (; b + 28 < blocks; b += 32) {
      float v[8];
#pragma unroll
      for (int x = 0; x < 8; x++) v[x] = q[(size_t)(b + 4 * x) * kPartStride];
#pragma unroll
      for (int x = 0; x < 8; x++) s += v[x];
    }
    for (; b < blocks; b += 4) s += q[(size_t)b * kPartStride];
  }
  s_sum[w][lane] = s;
  if (blockIdx.x == 0 && w == 1) {
    float l = 0.0f;
    for (int b = lane; b < blocks; b += 64) l += part_loss[b];
    l = wave_sum_f(l);
    if (lane == 0) *loss = l;
  }
  __syncthreads();
  if (w != 0 || i >= total) return;
  const float gi = (s_sum[0][lane] + s_sum[1][lane]) + (s_sum[2][lane] + s_sum[3][lane]);
  grads[i] = gi;
  if (!adam.m) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float mi = b1 * adam.m[i] + (1.0f - b1) * gi;
  const float vi = b2 * adam.v[i] + (1.0f - b2) * gi * gi;
  adam.m[i] = mi;
  adam.v[i] = vi;
  const float v = p[i] - adam.lr * (mi / adam.c1) / (sqrtf(vi / adam.c2) + eps);
  p[i] = v;
  pack_param(*img, i, v);
}

hipError_t launch_train(const float* p, NetImage* img, int blocks, int n, const float* X,
                        const float* Y, float* part, float* part_loss, hipStream_t st) {
  hipLaunchKernelGGL(k_train, dim3(blocks), dim3(kThreads), sizeof(TrainLds), st, p, img, n, X, Y,
                     part, part_loss);
  return hipGetLastError();
}

hipError_t launch_reduce(int blocks, const float* part, const float* part_loss, float* p,
                         float* grads, float* loss, const Adam& adam, NetImage* img,
                         hipStream_t st) {
  const int n = Layout().total;
  hipLaunchKernelGGL(k_reduce, dim3((n + 63) / 64), dim3(kThreads), 0, st, blocks, part, part_loss,
                     p, grads, loss, adam, img);
  return hipGetLastError();
}

__global__ void k_eval_points(amca_surrogate_desc d, amca_scan s, int n, const double* __restrict__ p,
                              float* __restrict__ X, double* __restrict__ Tfe) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const double x = p[4 * r], y = p[4 * r + 1], z = p[4 * r + 2], t = p[4 * r + 3];
  inputs(d, s, x, y, z, t, X + 5 * r);
  Tfe[r] = fe_temperature(d, s, x, y, z, t);
}

}  // namespace mlpk

const char* surrogate_error() { return g_mlp_error.c_str(); }

amca_status surrogate_eval_lattice(amca_mlp* h, const amca_surrogate_desc& d, const amca_scan& s,
                                   const SurLattice& g, float* out) {
  const long long total = (long long)g.nxi * g.ny * g.nz;
  MLP_HIP(launch_fused_timed(h, kLattice, total, nullptr, out, d, s, g));
  MLP_HIP(hipStreamSynchronize(h->stream));
  return AMCA_OK;
}

extern "C" {

amca_status amca_surrogate_sample(amca_mlp* h, const amca_surrogate_desc* d, const amca_scan* scans,
                                  int32_t n_scans, int64_t n, double near_fraction, uint64_t seed) {
  if (!h || !d || !scans || n_scans < 1 || n_scans > 16 || n < 1)
    return mlp_fail(AMCA_ERR_INVALID, "bad arguments (1..16 scans)");
  if (d->fnx < 2 || d->fny < 2 || d->fnz < 2 || d->n_frames < 2 || !(d->fdx > 0) ||
      !(d->frame_dt > 0) || !(d->xi_scale > 0) || !(d->T_scale > 0))
    return mlp_fail(AMCA_ERR_INVALID, "bad surrogate description");
  MLP_HIP(hipStreamSynchronize(h->stream));
  mlp_release(h, h->setX);
  mlp_release(h, h->setY);
  h->setX = h->setY = nullptr;
  h->set_n = 0;
  MLP_TRY(mlp_alloc(h, &h->setX, (size_t)n * kIn));
  MLP_TRY(mlp_alloc(h, &h->setY, (size_t)n));
  Sampler S;
  S.d = *d;
  S.n_scans = n_scans;
  for (int i = 0; i < n_scans; i++) S.s[i] = scans[i];
  const long long blocks = std::min<long long>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_sample, dim3((unsigned)blocks), dim3(256), 0, h->stream, S, (long long)n,
                     near_fraction, (unsigned long long)seed, h->setX, h->setY);
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipStreamSynchronize(h->stream));
  h->set_n = n;
  return AMCA_OK;
}

amca_status amca_surrogate_train(amca_mlp* h, int32_t batch, int32_t steps, float lr, uint64_t seed,
                                 float* loss_trace) {
  if (!h || !h->set_n) return mlp_fail(AMCA_ERR_INVALID, "no training set: call amca_surrogate_sample");
  return amca_mlp_train_device(h, h->set_n, h->setX, h->setY, batch, steps, lr, seed, loss_trace);
}

amca_status amca_surrogate_eval_lattice(amca_mlp* h, const amca_surrogate_desc* d,
                                        const amca_scan* s, int32_t nxi, double xi0, double dxi,
                                        int32_t ny, double y0, double dy, int32_t nz, double z0,
                                        double dz, float* out) {
  if (!h || !d || !s || !out || nxi < 1 || ny < 1 || nz < 1)
    return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  const long long n = (long long)nxi * ny * nz;
  float* dev = nullptr;
  MLP_HIP(hipMalloc(&dev, sizeof(float) * n));
  const SurLattice g{xi0, dxi, nxi, y0, dy, ny, z0, dz, nz};
  amca_status st = surrogate_eval_lattice(h, *d, *s, g, dev);
  if (st == AMCA_OK && hipMemcpy(out, dev, sizeof(float) * n, hipMemcpyDeviceToHost) != hipSuccess)
    st = mlp_fail(AMCA_ERR_HIP, "readback");
  (void)hipFree(dev);
  return st;
}

amca_status amca_surrogate_eval(amca_mlp* h, const amca_surrogate_desc* d, const amca_scan* s,
                                int32_t n, const double* xyzt, double* Ts, double* Tfe) {
  if (!h || !d || !s || n < 1 || !xyzt || !Ts || !Tfe) return mlp_fail(AMCA_ERR_INVALID, "bad arguments");
  MLP_TRY(ensure_rows(h, n));
  double *dp = nullptr, *dfe = nullptr;
  MLP_HIP(hipMalloc(&dp, sizeof(double) * 4 * n));
  MLP_HIP(hipMalloc(&dfe, sizeof(double) * n));
  amca_status st = AMCA_OK;
  std::vector<float> t(n);
  do {
    if (hipMemcpy(dp, xyzt, sizeof(double) * 4 * n, hipMemcpyHostToDevice) != hipSuccess) { st = mlp_fail(AMCA_ERR_HIP, "copy"); break; }
    hipLaunchKernelGGL(k_eval_points, dim3((n + 255) / 256), dim3(256), 0, h->stream, *d, *s, n, dp,
                       h->X, dfe);
    if ((st = infer(h, n, h->X, h->T)) != AMCA_OK) break;
    if (hipMemcpyAsync(t.data(), h->T, sizeof(float) * n, hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
        hipMemcpyAsync(Tfe, dfe, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
        hipStreamSynchronize(h->stream) != hipSuccess) { st = mlp_fail(AMCA_ERR_HIP, "readback"); break; }
    for (int i = 0; i < n; i++) Ts[i] = from_target(*d, (double)t[i]);
  } while (0);
  (void)hipFree(dp);
  (void)hipFree(dfe);
  return st;
}

}  // extern "C"
