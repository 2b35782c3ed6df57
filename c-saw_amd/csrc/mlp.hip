// Learned cost model: HIP forward, backward and SGD kernels for the
// 16 -> 64 -> 64 -> CSAW_NUM_VARIANTS MLP (BF16 weights, FP32 accumulate).
//
// The model is tiny, so the kernels are plain VALU code in FP32: forward and
// activation gradients run one wave per sample (lane j owns hidden unit j),
// the weight gradients one lane per parameter.  Every sum is a serial chain in
// a fixed order (inputs, hidden units, samples of the minibatch), so results
// are deterministic and do not depend on the launch shape.  SGD keeps an FP32
// master copy and re-rounds the BF16 working weights after each step.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "graph.hpp"
#include "mlp.hpp"
#include "plan.hpp"

namespace csaw {

constexpr int kMlpThreads = 256;

__device__ __forceinline__ float lane_f32(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// 64 consecutive bf16 weights (16-byte aligned) widened to FP32
template <int N>
__device__ __forceinline__ void load_row(const uint16_t* __restrict__ w, float* f) {
  const uint4* q = reinterpret_cast<const uint4*>(w);
#pragma unroll
  for (int k = 0; k < N / 8; ++k) {
    const uint4 t = q[k];
    const uint32_t u[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      f[8 * k + 2 * c] = __uint_as_float(u[c] << 16);
      f[8 * k + 2 * c + 1] = __uint_as_float(u[c] & 0xffff0000u);
    }
  }
}

// Forward pass of rows idx[0 .. n) (idx null: rows 0 .. n), one wave per row:
// lane j computes hidden unit j, the previous layer's values reach it by
// v_readlane in input order, so each sum is the same serial FMA chain one
// lane per sample would run.  The wave keeps its rows of the weights in
// registers.  BWD: also
//   dY = M (Y - T) / cnt; dH2 = (W3^T dY) * [H2 > 0]; dH1 = (W2^T dH2) * [H1 > 0]
// and the inputs, activations and gradients of the row for k_mlp_params.
// Null outputs are not written.
// Bound: latency of the chains (about 420 dependent FMAs a row).  One lane per
// row ran a 256-row minibatch in a single workgroup with its 64-value arrays in
// scratch: 94 us forward and 358 us backward; a wave per row spreads it over
// 256 workgroups and takes 5.2 us for both.
template <bool BWD>
__global__ __launch_bounds__(kWave) void k_mlp_rows(const uint16_t* __restrict__ w, const float* __restrict__ X,
                                                    const int32_t* __restrict__ idx, int64_t n,
                                                    const float* __restrict__ T, const float* __restrict__ M,
                                                    float inv_cnt, float* __restrict__ Y, float* __restrict__ Xb,
                                                    float* __restrict__ H1, float* __restrict__ H2,
                                                    float* __restrict__ dY, float* __restrict__ dH1,
                                                    float* __restrict__ dH2, float* __restrict__ loss_s) {
  const int j = lane_id();
  const int jo = j < kMlpOut ? j : 0;  // output unit of the lanes that have one
  float w1[kMlpIn], w2[kMlpHid], w3[kMlpHid], w2t[kMlpHid], w3t[kMlpOut];
  load_row<kMlpIn>(w + kMlpW1 + j * kMlpIn, w1);
  load_row<kMlpHid>(w + kMlpW2 + j * kMlpHid, w2);
  load_row<kMlpHid>(w + kMlpW3 + jo * kMlpHid, w3);
  const float b1 = bf16_to_f32(w[kMlpB1 + j]), b2 = bf16_to_f32(w[kMlpB2 + j]), b3 = bf16_to_f32(w[kMlpB3 + jo]);
  if (BWD) {
#pragma unroll
    for (int i = 0; i < kMlpHid; ++i) w2t[i] = bf16_to_f32(w[kMlpW2 + i * kMlpHid + j]);
#pragma unroll
    for (int i = 0; i < kMlpOut; ++i) w3t[i] = bf16_to_f32(w[kMlpW3 + i * kMlpHid + j]);
  }
  for (int64_t s = blockIdx.x; s < n; s += gridDim.x) {
    const int64_t r = idx ? idx[s] : s;
    const float x = X[r * kMlpIn + (j & (kMlpIn - 1))];
    float t = 0.f, m = 0.f;
    if (BWD) {
      t = T[r * kMlpOut + jo];
      m = M[r * kMlpOut + jo];
    }
    float a = b1;
#pragma unroll
    for (int i = 0; i < kMlpIn; ++i) a = fmaf(w1[i], lane_f32(x, i), a);
    const float h1 = a > 0.f ? a : 0.f;
    a = b2;
#pragma unroll
    for (int i = 0; i < kMlpHid; ++i) a = fmaf(w2[i], lane_f32(h1, i), a);
    const float h2 = a > 0.f ? a : 0.f;
    a = b3;
#pragma unroll
    for (int i = 0; i < kMlpHid; ++i) a = fmaf(w3[i], lane_f32(h2, i), a);
    if (Y && j < kMlpOut) Y[s * kMlpOut + j] = a;
    if (!BWD) continue;
    const float e = a - t;
    const float dy = m != 0.f ? e * inv_cnt : 0.f;
    const float le = m != 0.f ? 0.5f * e * e : 0.f;
    float l = 0.f;
#pragma unroll
    for (int k = 0; k < kMlpOut; ++k) l += lane_f32(le, k);
    if (j == 0) loss_s[s] = l * inv_cnt;
    if (!dH1) continue;
    float g = 0.f;
#pragma unroll
    for (int k = 0; k < kMlpOut; ++k) g = fmaf(w3t[k], lane_f32(dy, k), g);
    const float d2 = h2 > 0.f ? g : 0.f;
    g = 0.f;
#pragma unroll
    for (int k = 0; k < kMlpHid; ++k) g = fmaf(w2t[k], lane_f32(d2, k), g);
    const float d1 = h1 > 0.f ? g : 0.f;
    if (j < kMlpIn) Xb[s * kMlpIn + j] = x;
    if (j < kMlpOut) dY[s * kMlpOut + j] = dy;
    H1[s * kMlpHid + j] = h1;
    H2[s * kMlpHid + j] = h2;
    dH1[s * kMlpHid + j] = d1;
    dH2[s * kMlpHid + j] = d2;
  }
}

// Gradient of each parameter, one lane per parameter summing A[s] * B[s] over
// the rows in order, and with SGD its update in place of storing it.
// A workgroup owns the parameters that share a B tile (columns a0 .. a0 + NA of
// A against all WB columns of B; NA = 0: biases, the sums of B's columns) and
// stages kParamRows rows of it in LDS with wide coalesced loads, the next rows'
// loads in flight while the lanes run their chains from LDS.
// Bound: latency, of the first tile (the rows were written by other XCDs) and of
// each tile's round of store, barrier and sum; the 256 dependent FMAs of a chain
// are about 1 us of it.  For 256 rows: 88 us with a lane's pairs loaded from
// memory one by one, 26 us with 32 pairs loaded ahead, 15 us from LDS with the
// tile widths as run-time values, 12.3 us as constants, 10.9 us staged by sixteen
// waves (one wave a workgroup, four times the workgroups: 28 us).
constexpr int kParamRows = 128;
constexpr int kParamThreads = 1024;  // all stage, the first four waves sum
constexpr int kParamGrid = 25;
struct ParamOut {
  float *grad, *master;
  uint16_t* wb;
  float lr;
};

template <bool SGD, int WB, int NA, int SA>
__device__ __forceinline__ void param_tile(int64_t n, const float* __restrict__ B, const float* __restrict__ A, float* tb,
                                           float* ta, int ca, int cb, int p, const ParamOut& O) {
  const int tid = threadIdx.x;
  constexpr int kQuads = (kParamRows * WB / 4 + kParamThreads - 1) / kParamThreads;  // float4s of a B tile per thread
  constexpr int kSingles = (kParamRows * NA + kParamThreads - 1) / kParamThreads;
  float4 qb[kQuads];
  float qa[kSingles > 0 ? kSingles : 1];
  // quads past the last row end inside the array's padding (256 bytes)
  auto load = [&](int64_t s0) {
    const int rows = (int)(n - s0 < kParamRows ? n - s0 : kParamRows);
    const float4* src = reinterpret_cast<const float4*>(B + s0 * WB);
#pragma unroll
    for (int k = 0; k < kQuads; ++k)
      if (k * kParamThreads + tid < (rows * WB + 3) / 4) qb[k] = src[k * kParamThreads + tid];
    if constexpr (NA > 0) {
      const float* asrc = A + s0 * SA;
#pragma unroll
      for (int k = 0; k < kSingles; ++k) {
        const int i = k * kParamThreads + tid;
        if (i < rows * NA) qa[k] = asrc[(i / NA) * SA + i % NA];
      }
    }
  };
  float acc = 0.f;
  load(0);
  const float old = SGD && p >= 0 ? O.master[p] : 0.f;  // not after the chain
  for (int64_t s0 = 0; s0 < n; s0 += kParamRows) {
    const int rows = (int)(n - s0 < kParamRows ? n - s0 : kParamRows);
#pragma unroll
    for (int k = 0; k < kQuads; ++k)
      if (k * kParamThreads + tid < (rows * WB + 3) / 4) reinterpret_cast<float4*>(tb)[k * kParamThreads + tid] = qb[k];
#pragma unroll
    for (int k = 0; k < kSingles; ++k)
      if (k * kParamThreads + tid < rows * NA) ta[k * kParamThreads + tid] = qa[k];
    __syncthreads();
    if (s0 + kParamRows < n) load(s0 + kParamRows);
    if (p >= 0) {
      const float *pa = ta + ca, *pb = tb + cb;
      auto row = [&](int r) { acc = NA > 0 ? fmaf(pa[r * NA], pb[r * WB], acc) : acc + pb[r * WB]; };
      int r = 0;
      for (; r + 32 <= rows; r += 32) {
#pragma unroll
        for (int k = 0; k < 32; ++k) row(r + k);
      }
      for (; r < rows; ++r) row(r);
    }
    __syncthreads();
  }
  if (p < 0) return;
  if (SGD) {
    const float v = old - O.lr * acc;
    O.master[p] = v;
    O.wb[p] = f32_to_bf16(v);
  } else {
    O.grad[p] = acc;
  }
}

template <bool SGD>
__global__ __launch_bounds__(kParamThreads) void k_mlp_params(int64_t n, const float* __restrict__ Xb,
                                                            const float* __restrict__ H1, const float* __restrict__ H2,
                                                            const float* __restrict__ dY, const float* __restrict__ dH1,
                                                            const float* __restrict__ dH2, ParamOut O) {
  __shared__ __align__(16) float tb[kParamRows * kMlpHid];
  __shared__ __align__(16) float ta[kParamRows * kMlpIn];
  const int b = blockIdx.x, lane = lane_id(), wid = threadIdx.x / kWave;
  const int bias_p = wid == 0 ? lane : -1;
  if (b < 16) {  // W2, rows 4b .. 4b + 3
    param_tile<SGD, kMlpHid, 4, kMlpHid>(n, H1, dH2 + 4 * b, tb, ta, wid, lane,
                                         wid < 4 ? kMlpW2 + (4 * b + wid) * kMlpHid + lane : -1, O);
  } else if (b < 20) {  // W1, sixteen rows
    const int a0 = 16 * (b - 16), ca = 4 * wid + lane / kMlpIn, cb = lane % kMlpIn;
    param_tile<SGD, kMlpIn, 16, kMlpHid>(n, Xb, dH1 + a0, tb, ta, ca, cb,
                                         wid < 4 ? kMlpW1 + (a0 + ca) * kMlpIn + cb : -1, O);
  } else if (b == 20) {  // W3, rows 0 .. 3
    param_tile<SGD, kMlpHid, 4, kMlpOut>(n, H2, dY, tb, ta, wid, lane,
                                         wid < 4 ? kMlpW3 + wid * kMlpHid + lane : -1, O);
  } else if (b == 21) {  // W3, row 4
    param_tile<SGD, kMlpHid, 1, kMlpOut>(n, H2, dY + 4, tb, ta, 0, lane, wid == 0 ? kMlpW3 + 4 * kMlpHid + lane : -1, O);
  } else if (b < 24) {  // b1, b2
    param_tile<SGD, kMlpHid, 0, 0>(n, b == 22 ? dH1 : dH2, nullptr, tb, ta, 0, lane,
                                   bias_p >= 0 ? (b == 22 ? kMlpB1 : kMlpB2) + lane : -1, O);
  } else {  // b3
    param_tile<SGD, kMlpOut, 0, 0>(n, dY, nullptr, tb, ta, 0, lane, bias_p >= 0 && lane < kMlpOut ? kMlpB3 + lane : -1, O);
  }
}

__global__ void k_mlp_round(const float* __restrict__ master, uint16_t* __restrict__ wb) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < kMlpParams; p += gridDim.x * blockDim.x)
    wb[p] = f32_to_bf16(master[p]);
}

// single-workgroup ordered sum
__global__ __launch_bounds__(kMlpThreads) void k_sum(const float* __restrict__ x, int64_t n, float* __restrict__ out) {
  __shared__ float part[kMlpThreads];
  float a = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += kMlpThreads) a += x[i];
  part[threadIdx.x] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int i = 0; i < kMlpThreads; ++i) s += part[i];
    *out = s;
  }
}

}  // namespace csaw

using namespace csaw;

struct csaw_mlp {
  std::vector<float> master;  // host mirror of the FP32 master weights
  float* d_master = nullptr;
  uint16_t* d_w = nullptr;
  hipStream_t stream = nullptr;
  int num_cu = 0;
};

namespace csaw {
int mlp_upload_bf16(const csaw_mlp* m, uint16_t* dst) {
  CSAW_HIP(hipMemcpy(dst, m->d_w, sizeof(uint16_t) * kMlpParams, hipMemcpyDeviceToDevice));
  return CSAW_OK;
}
}  // namespace csaw

// Device work of one call, carved from one allocation: data rows X, T, M and
// their order, the per-row state of a minibatch, and the losses.
struct MlpWork {
  char* slab = nullptr;
  float *X = nullptr, *T = nullptr, *M = nullptr, *Xb = nullptr, *H1 = nullptr, *H2 = nullptr, *Y = nullptr;
  float *dY = nullptr, *dH1 = nullptr, *dH2 = nullptr, *grad = nullptr, *loss_s = nullptr, *loss = nullptr;
  int32_t* idx = nullptr;
  ~MlpWork() { (void)hipFree(slab); }
};

// n_data rows, n_batch of them with gradients at a time (0: forward only)
static int mlp_alloc_work(MlpWork& w, int64_t n_data, int64_t n_batch) {
  for (int pass = 0; pass < 2; ++pass) {
    int64_t at = 0;
    auto part = [&](auto** p, int64_t count) {
      if (w.slab) *p = reinterpret_cast<std::remove_reference_t<decltype(*p)>>(w.slab + at);
      at += (count * 4 + 255) & ~(int64_t)255;
    };
    part(&w.X, n_data * kMlpIn);
    if (n_batch > 0) {
      part(&w.T, n_data * kMlpOut);
      part(&w.M, n_data * kMlpOut);
      part(&w.idx, n_data);
      part(&w.Xb, n_batch * kMlpIn);
      part(&w.H1, n_batch * kMlpHid);
      part(&w.H2, n_batch * kMlpHid);
      part(&w.dY, n_batch * kMlpOut);
      part(&w.dH1, n_batch * kMlpHid);
      part(&w.dH2, n_batch * kMlpHid);
      part(&w.grad, kMlpParams);
      part(&w.loss_s, n_data);
      part(&w.loss, 1);
    } else {
      part(&w.Y, n_data * kMlpOut);
    }
    if (!w.slab) CSAW_HIP(device_malloc(&w.slab, at));
  }
  return CSAW_OK;
}

// one wave per row: every row its own workgroup up to 8 per CU
static int rows_grid(const csaw_mlp* m, int64_t n) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(n, (int64_t)m->num_cu * 8));
}

// losses (and with grads the per-row gradients) of rows idx[0 .. n)
static int mlp_rows_loss(csaw_mlp* m, MlpWork& w, const int32_t* idx, int64_t n, float inv_cnt, bool grads) {
  k_mlp_rows<true><<<rows_grid(m, n), kWave, 0, m->stream>>>(m->d_w, w.X, idx, n, w.T, w.M, inv_cnt, nullptr, w.Xb,
                                                             w.H1, w.H2, w.dY, grads ? w.dH1 : nullptr, w.dH2,
                                                             w.loss_s);
  CSAW_LAUNCH_CHECK();
  return CSAW_OK;
}

static int mlp_sum_loss(csaw_mlp* m, MlpWork& w, int64_t n) {
  k_sum<<<1, kMlpThreads, 0, m->stream>>>(w.loss_s, n, w.loss);
  CSAW_LAUNCH_CHECK();
  return CSAW_OK;
}

extern "C" int csaw_mlp_num_params(void) { return kMlpParams; }

extern "C" int csaw_mlp_create(uint64_t init_key, csaw_mlp** out) {
  if (!out) return CSAW_ERR_INVALID_ARG;
  *out = nullptr;
  csaw_mlp* m = new csaw_mlp();
  m->master.assign(kMlpParams, 0.f);
  // He-uniform initialisation from Philox (domain kDomExplore, word 2 = 1)
  auto fill = [&](int off, int rows, int cols) {
    const float lim = std::sqrt(6.0f / (float)cols);
    for (int i = 0; i < rows * cols; ++i) {
      const U4 o = philox4x32_10((uint32_t)(off + i), 0u, 1u, kDomExplore << 28, (uint32_t)init_key,
                                 (uint32_t)(init_key >> 32));
      const float u = (float)(o.x >> 8) * 5.9604644775390625e-08f;
      m->master[off + i] = (2.f * u - 1.f) * lim;
    }
  };
  fill(kMlpW1, kMlpHid, kMlpIn);
  fill(kMlpW2, kMlpHid, kMlpHid);
  fill(kMlpW3, kMlpOut, kMlpHid);
  auto body = [&]() -> int {
    CSAW_TRY(device_init(&m->num_cu));
    CSAW_HIP(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    CSAW_HIP(device_malloc(&m->d_master, sizeof(float) * kMlpParams));
    CSAW_HIP(device_malloc(&m->d_w, sizeof(uint16_t) * kMlpParams));
    return csaw_mlp_set_params(m, m->master.data());
  };
  int st = body();
  if (st != CSAW_OK) {
    csaw_mlp_destroy(m);
    return st;
  }
  *out = m;
  return CSAW_OK;
}

extern "C" int csaw_mlp_destroy(csaw_mlp* m) {
  if (!m) return CSAW_OK;
  (void)hipFree(m->d_master);
  (void)hipFree(m->d_w);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return CSAW_OK;
}

extern "C" int csaw_mlp_get_params(const csaw_mlp* m, float* params) {
  if (!m || !params) return CSAW_ERR_INVALID_ARG;
  CSAW_HIP(hipMemcpy(params, m->d_master, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
  return CSAW_OK;
}

extern "C" int csaw_mlp_set_params(csaw_mlp* m, const float* params) {
  if (!m || !params) return CSAW_ERR_INVALID_ARG;
  if (params != m->master.data()) m->master.assign(params, params + kMlpParams);
  CSAW_HIP(hipMemcpy(m->d_master, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
  k_mlp_round<<<(kMlpParams + 255) / 256, 256, 0, m->stream>>>(m->d_master, m->d_w);
  CSAW_LAUNCH_CHECK();
  CSAW_HIP(hipStreamSynchronize(m->stream));
  return CSAW_OK;
}

extern "C" int csaw_mlp_forward(csaw_mlp* m, const float* X, int64_t n, float* Y) {
  if (!m || n < 0 || (n > 0 && (!X || !Y))) return CSAW_ERR_INVALID_ARG;
  if (n == 0) return CSAW_OK;
  MlpWork w;
  CSAW_TRY(mlp_alloc_work(w, n, 0));
  CSAW_HIP(hipMemcpy(w.X, X, sizeof(float) * n * kMlpIn, hipMemcpyHostToDevice));
  k_mlp_rows<false><<<rows_grid(m, n), kWave, 0, m->stream>>>(m->d_w, w.X, nullptr, n, nullptr, nullptr, 0.f, w.Y,
                                                              nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                              nullptr);
  CSAW_LAUNCH_CHECK();
  CSAW_HIP(hipStreamSynchronize(m->stream));
  CSAW_HIP(hipMemcpy(Y, w.Y, sizeof(float) * n * kMlpOut, hipMemcpyDeviceToHost));
  return CSAW_OK;
}

static double mask_count(const float* M, int64_t n) {
  double c = 0;
  for (int64_t i = 0; i < n * kMlpOut; ++i) c += M[i] != 0.f ? 1.0 : 0.0;
  return c;
}

extern "C" int csaw_mlp_grad(csaw_mlp* m, const float* X, const float* T, const float* M, int64_t n, float* loss,
                             float* grad) {
  if (!m || n <= 0 || !X || !T || !M) return CSAW_ERR_INVALID_ARG;
  MlpWork w;
  CSAW_TRY(mlp_alloc_work(w, n, n));
  CSAW_HIP(hipMemcpy(w.X, X, sizeof(float) * n * kMlpIn, hipMemcpyHostToDevice));
  CSAW_HIP(hipMemcpy(w.T, T, sizeof(float) * n * kMlpOut, hipMemcpyHostToDevice));
  CSAW_HIP(hipMemcpy(w.M, M, sizeof(float) * n * kMlpOut, hipMemcpyHostToDevice));
  const double cnt = mask_count(M, n);
  CSAW_TRY(mlp_rows_loss(m, w, nullptr, n, cnt > 0 ? (float)(1.0 / cnt) : 0.f, true));
  k_mlp_params<false><<<kParamGrid, kParamThreads, 0, m->stream>>>(n, w.Xb, w.H1, w.H2, w.dY, w.dH1, w.dH2,
                                                                 ParamOut{w.grad, nullptr, nullptr, 0.f});
  CSAW_LAUNCH_CHECK();
  CSAW_TRY(mlp_sum_loss(m, w, n));
  CSAW_HIP(hipStreamSynchronize(m->stream));
  if (loss) CSAW_HIP(hipMemcpy(loss, w.loss, sizeof(float), hipMemcpyDeviceToHost));
  if (grad) CSAW_HIP(hipMemcpy(grad, w.grad, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
  return CSAW_OK;
}

extern "C" int csaw_mlp_train(csaw_mlp* m, const float* X, const float* T, const float* M, int64_t n, int32_t epochs,
                              int32_t batch, float lr, uint64_t shuffle_key, float* final_loss) {
  if (!m || n <= 0 || !X || !T || !M || epochs < 0 || batch <= 0) return CSAW_ERR_INVALID_ARG;
  MlpWork w;
  const int64_t nb = std::min<int64_t>(batch, n);
  CSAW_TRY(mlp_alloc_work(w, n, nb));
  CSAW_HIP(hipMemcpy(w.X, X, sizeof(float) * n * kMlpIn, hipMemcpyHostToDevice));
  CSAW_HIP(hipMemcpy(w.T, T, sizeof(float) * n * kMlpOut, hipMemcpyHostToDevice));
  CSAW_HIP(hipMemcpy(w.M, M, sizeof(float) * n * kMlpOut, hipMemcpyHostToDevice));
  std::vector<int32_t> perm(n);
  for (int64_t i = 0; i < n; ++i) perm[i] = (int32_t)i;
  float last = 0.f;
  for (int32_t ep = 0; ep < epochs; ++ep) {
    // Fisher-Yates with Philox draws
    for (int64_t i = n - 1; i > 0; --i) {
      const U4 o = philox4x32_10((uint32_t)i, (uint32_t)ep, 2u, kDomExplore << 28, (uint32_t)shuffle_key,
                                 (uint32_t)(shuffle_key >> 32));
      const int64_t j = (int64_t)mulhi64(philox_t64(o), (uint64_t)(i + 1));
      std::swap(perm[i], perm[j]);
    }
    CSAW_HIP(hipMemcpyAsync(w.idx, perm.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, m->stream));
    for (int64_t b = 0; b < n; b += nb) {
      const int64_t cnt_rows = std::min<int64_t>(nb, n - b);
      double cnt = 0;
      for (int64_t s = 0; s < cnt_rows; ++s)
        for (int j = 0; j < kMlpOut; ++j) cnt += M[(int64_t)perm[b + s] * kMlpOut + j] != 0.f ? 1.0 : 0.0;
      if (cnt == 0) continue;
      CSAW_TRY(mlp_rows_loss(m, w, w.idx + b, cnt_rows, (float)(1.0 / cnt), true));
      k_mlp_params<true><<<kParamGrid, kParamThreads, 0, m->stream>>>(cnt_rows, w.Xb, w.H1, w.H2, w.dY, w.dH1, w.dH2,
                                                                    ParamOut{nullptr, m->d_master, m->d_w, lr});
      CSAW_LAUNCH_CHECK();
    }
  }
  // full-data loss
  if (final_loss) {
    const double cnt = mask_count(M, n);
    CSAW_TRY(mlp_rows_loss(m, w, nullptr, n, cnt > 0 ? (float)(1.0 / cnt) : 0.f, false));
    CSAW_TRY(mlp_sum_loss(m, w, n));
    CSAW_HIP(hipStreamSynchronize(m->stream));
    CSAW_HIP(hipMemcpy(&last, w.loss, sizeof(float), hipMemcpyDeviceToHost));
    *final_loss = last;
  }
  CSAW_HIP(hipStreamSynchronize(m->stream));
  m->master.resize(kMlpParams);
  CSAW_HIP(hipMemcpy(m->master.data(), m->d_master, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
  return CSAW_OK;
}
