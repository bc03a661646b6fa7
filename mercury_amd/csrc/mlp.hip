// mlp.hip -- the surrogate network: fully connected layers with bf16
// weights (fp32 master copy for Adam) and fp32 activations, trained on the
// device by hand-written forward, backward and Adam kernels.  Every GEMM
// runs on the matrix cores with bf16 operands (activations and gradients
// rounded to nearest even as they enter it) and fp32 accumulation.
//
// Layer l: Z_l = A_{l-1} W_l^T + b_l, A_l = gelu(Z_l) on hidden layers,
// A_L = Z_L.  gelu(x) = 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3))).
// Loss = mean over the batch of 0.5 (A_L - target)^2.  Adam follows Kingma
// & Ba (2015), Algorithm 1 (bias-corrected moments).
//
// Networks of up to kDenseMaxLayers layers of at most kDenseMaxWidth units
// (the surrogate is 64-256-256-1) run as the fused kernels of mh_dense.h:
// one launch forward, two per training step.  Wider ones, and large batches of
// narrow ones on device buffers (forward_by_layers), run a launch per
// layer and direction: 64x64 output tiles, 256 threads (four waves of 2x2
// 16x16 MFMA blocks), K in steps of 32 staged through LDS as bf16.  Weight
// gradients reduce over the batch in row splits whose partials are summed in
// order; bias gradients (column sums of the fp32 gradients) likewise, so
// every reduction has a fixed order and training is deterministic, with the
// same bits on both paths.
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "mercury_hip.h"
#include "mh_internal.h"
#include "mh_dense.h"

// Scratch of mh_mlp_forward_noalloc: the hidden activations of one call, in
// two halves that alternate between layers.  Every device holds its own
// copy (MH_MLP_SCRATCH_FLOATS floats, 16 MiB) until the process ends.  In
// host code this name stands for a host-side shadow, not a device address:
// kernels take the address hipGetSymbolAddress gives on each device.
static __device__ __align__(256) float scratch[MH_MLP_SCRATCH_FLOATS];

struct mh_mlp {
  int device = 0;
  float* scratch = nullptr;   // device address of ::scratch on `device`
  std::vector<int> sizes;     // n_layers + 1
  std::vector<size_t> w_off;  // offset of W_l in the parameter vector; b_l follows W_l
  size_t n_params = 0;
  Dev<float> params, grads, m, v;
  bool fused = false;         // every layer fits the fused kernels
  DenseShape shape{};         // fused: the layers and where their packed weights lie
  Dev<uint16_t> pack;         // fused: bf16 weights in the kernels' operand order
  std::vector<Dev<uint16_t>> X16, D16;  // fused: weight-gradient operands of a batch
  std::vector<Dev<float>> delta;        // fused: gradients of every layer's output
  Dev<__hip_bfloat16> w16;    // bf16 copy of the parameter vector for the layer-by-layer kernels (weights used)
  std::vector<Dev<float>> Z, A, dA;  // per layer activations / gradients
  Dev<float> x, t, dY, terms, data_x, data_t;
  Dev<float> epoch_terms;     // loss terms of every batch of a training run's last epoch
  Dev<float> part;            // split-K partials of the weight and bias gradients
  Dev<int> idx;
  int batch_cap = 0;
  int adam_t = 0;
  hipStream_t stream = nullptr;
  ~mh_mlp() {
    if (stream) (void)hipStreamDestroy(stream);
  }
  int L() const { return static_cast<int>(sizes.size()) - 1; }
  size_t b_off(int l) const { return w_off[l] + static_cast<size_t>(sizes[l + 1]) * sizes[l]; }
};

namespace {

// weight and bias gradients reduce over the batch in up to this many row
// splits (at least 64 rows each), summed in order
constexpr int kMlpSplit = 8;

// Row splits of a batch of B for the weight and bias gradients.
int mlp_splits(int B) { return std::max(1, std::min(kMlpSplit, B / 64)); }

void ensure_batch(mh_mlp* net, int B) {
  if (B <= net->batch_cap) return;
  const int L = net->L();
  if (net->fused) {
    // operands are padded to whole slices of 32 rows per split: their size
    // is not monotonic in B, so a bound for every smaller batch is kept
    const size_t rows = static_cast<size_t>(B) + 32 * kMlpSplit;
    net->X16.resize(L);
    net->D16.resize(L);
    net->delta.resize(L);
    for (int l = 0; l < L; l++) {
      net->X16[l].ensure(rows * ((net->sizes[l] + 15) / 16 * 16));
      net->D16[l].ensure(rows * ((net->sizes[l + 1] + 15) / 16 * 16));
      net->delta[l].ensure(static_cast<size_t>(B) * net->sizes[l + 1]);
    }
    net->x.ensure(static_cast<size_t>(B) * net->sizes[0]);
    net->t.ensure(static_cast<size_t>(B) * net->sizes[L]);
    net->terms.ensure(static_cast<size_t>(B) * net->sizes[L]);
    net->batch_cap = B;
    return;
  }
  net->Z.resize(L);
  net->A.resize(L);
  net->dA.resize(L + 1);
  for (int l = 0; l < L; l++) {
    net->Z[l].ensure(static_cast<size_t>(B) * net->sizes[l + 1]);
    net->A[l].ensure(static_cast<size_t>(B) * net->sizes[l + 1]);
  }
  for (int l = 0; l <= L; l++) net->dA[l].ensure(static_cast<size_t>(B) * net->sizes[l]);
  net->x.ensure(static_cast<size_t>(B) * net->sizes[0]);
  net->t.ensure(static_cast<size_t>(B) * net->sizes[L]);
  net->dY.ensure(static_cast<size_t>(B) * net->sizes[L]);
  net->terms.ensure(static_cast<size_t>(B) * net->sizes[L]);
  net->batch_cap = B;
}

// Brings the device weights (packed, or the bf16 copy) up to date with the
// fp32 parameters.
void refresh_weights(mh_mlp* net) {
  if (net->fused) {
    PackList list{net->L(), {}};
    std::copy_n(net->shape.layer, net->L(), list.layer);
    launch_pack(list, net->params.p, net->pack.p, reinterpret_cast<uint16_t*>(net->w16.p), net->stream);
  } else {
    hipLaunchKernelGGL(to_bf16, dim3((net->n_params + 255) / 256), dim3(256), 0, net->stream, net->params.p,
                       net->w16.p, static_cast<int>(net->n_params));
  }
  hipcheck(hipGetLastError(), "weights");
}

// Whether a forward pass on device buffers that may not allocate takes the
// layer-by-layer kernels though the network is fused.
bool forward_by_layers(const mh_mlp* net, const float* x, int B, const float* y) {
  const int L = net->L(), in = net->sizes.front(), out = net->sizes.back();
  // y overlaps x: a fused workgroup would write rows that another still reads
  // (the layers' last kernel starts when all of x has been read)
  const size_t nx = static_cast<size_t>(B) * in * sizeof(float), ny = static_cast<size_t>(B) * out * sizeof(float);
  const uintptr_t ax = reinterpret_cast<uintptr_t>(x), ay = reinterpret_cast<uintptr_t>(y);
  if (L > 1 && ax < ay + ny && ay < ax + nx) return true;
  // Large batches of narrow networks: the fused kernel computes 256 units a
  // layer whatever the width (0.16 ns per row and layer once the chip is full),
  // the layers' kernels have one launch per layer (about 5 us) and then the
  // time of their own widths.  MI355X, us fused and by layers: 8-8-1 at 16384
  // rows 10.7 and 10.8, at 65536 37 and 12; 64-64-64-1 at 16384 15.7 and 18.6,
  // at 32768 29.5 and 21; 32-100-1 at 20480 20.0 and 18.3.  One layer: 64-1 at
  // 8192 rows 4.3 and 4.4, at 12288 5.7 and 4.4, at 65536 12.3 and 5.6; 64-256
  // at 16384 9.9 and 8.0, at 24576 12.5 and 12.8; 128-128 at 24576 9.6 and
  // 8.4, at 32768 10.5 and 11.1; 128-256 at 12288 9.0 and 8.5, at 16384 10.0
  // and 11.0; 256-1 at 65536 16.0 and 16.9.  (Networks of a hidden layer of 128
  // units or more stay under 16384 rows: the scratch array's limit.)
  if (L > 1) return B > 16384;
  // (one layer of 128 x 128 and more: fused from 4.1e8 products on)
  const size_t macs = static_cast<size_t>(in) * out;
  return B > 8192 && in < 256 && (macs < 128 * 128 || macs * B <= 410000000u);
}

// Fused forward of B rows on the device, x -> y.  A workgroup reads every
// packed weight from L2, so large batches take taller row tiles; small ones
// take 16 rows, as long as one workgroup per CU covers them.  64-256-256-1
// on MI355X, us with tiles of 16 / 32 / 64 rows: 4096 rows 7.7 / 10.9 / 18.6
// (the layer-by-layer kernels 13.9), 8192 rows 13.6 / 10.9 / 18.5, 16384
// rows 25.7 / 20.6 / 18.6, 65536 rows 98 / 78 / 70.
void fused_forward(mh_mlp* net, const float* x, int B, float* y, hipStream_t s) {
  if (B <= 4096) launch_dense_net<1, false>(net->shape, net->params.p, net->pack.p, x, B, y, DenseTrain{}, s);
  else if (B <= 8192) launch_dense_net<2, false>(net->shape, net->params.p, net->pack.p, x, B, y, DenseTrain{}, s);
  else launch_dense_net<4, false>(net->shape, net->params.p, net->pack.p, x, B, y, DenseTrain{}, s);
}

// Fused loss terms and gradients of a batch: batch row r is row x_idx[r] of
// x and t_idx[r] of target (null: r).  Gradients go to net->grads, or with
// `adam` straight into the parameters.
void fused_backward(mh_mlp* net, const float* x, const float* target, const int* idx, int B, float* terms,
                    const AdamArgs* adam) {
  DenseTrain tr{};
  tr.rs = row_splits(B, mlp_splits(B));
  tr.x_idx = idx;
  tr.t_idx = idx;
  tr.target = target;
  tr.inv_b = 1.0f / B;
  tr.terms = terms;
  for (int l = 0; l < net->L(); l++) {
    tr.X[l] = net->X16[l].p;
    tr.D[l] = net->D16[l].p;
    tr.delta[l] = net->delta[l].p;
  }
  launch_dense_net<1, true>(net->shape, net->params.p, net->pack.p, x, B, nullptr, tr, net->stream);
  if (adam) launch_dense_wgrad<4, 1, true>(net->shape, tr, *adam, nullptr, net->stream);
  else launch_dense_wgrad<4, 1, false>(net->shape, tr, AdamArgs{}, net->grads.p, net->stream);
}

// Forward of a batch already in net->x (or `in`): activations in A[l].
void forward(mh_mlp* net, const float* in, int B) {
  const int L = net->L();
  const float* prev = in;
  for (int l = 0; l < L; l++) {
    const int ni = net->sizes[l], no = net->sizes[l + 1];
    const __hip_bfloat16* W = net->w16.p + net->w_off[l];
    const float* b = net->params.p + net->b_off(l);
    if (l < L - 1)
      hipLaunchKernelGGL((gemm<float, __hip_bfloat16, false, true, 1>), grid_for(B, no), dim3(256), 0,
                         net->stream, prev, ni, W, ni, net->A[l].p, no, B, no, ni, b, net->Z[l].p,
                         static_cast<const float*>(nullptr));
    else
      hipLaunchKernelGGL((gemm<float, __hip_bfloat16, false, true, 2>), grid_for(B, no), dim3(256), 0,
                         net->stream, prev, ni, W, ni, net->A[l].p, no, B, no, ni, b,
                         static_cast<float*>(nullptr), static_cast<const float*>(nullptr));
    hipcheck(hipGetLastError(), "mlp forward");
    prev = net->A[l].p;
  }
}

// Backward from dY (already (Y - T)/B): gradients into net->grads, or with
// to_adam their split partials into net->part at the parameters' offsets,
// n_params apart, for adam_step_splits to sum.
void backward(mh_mlp* net, const float* in, int B, bool to_adam = false) {
  const int L = net->L();
  const float* delta = net->dY.p;  // dLoss/dZ_l for the current layer
  for (int l = L - 1; l >= 0; l--) {
    const int ni = net->sizes[l], no = net->sizes[l + 1];
    const float* a_prev = l == 0 ? in : net->A[l - 1].p;
    float* gW = net->grads.p + net->w_off[l];
    float* gb = net->grads.p + net->b_off(l);
    // gW[no x ni] = delta^T[no x B] a_prev[B x ni] and gb = column sums of
    // delta, each as S row-split partials summed in order
    const int S = mlp_splits(B);
    const int rows = (B + S - 1) / S;
    float* pW = to_adam ? net->part.p + net->w_off[l] : net->part.p;
    float* pb = to_adam ? net->part.p + net->b_off(l) : net->part.p;
    const size_t sW = to_adam ? net->n_params : static_cast<size_t>(no) * ni;
    const size_t sb = to_adam ? net->n_params : static_cast<size_t>(no);
    hipLaunchKernelGGL((wgrad_l<StridedB<float, false>>), dim3((ni + kTile - 1) / kTile, (no + kTile - 1) / kTile, S),
                       dim3(256), 0, net->stream, delta, no, StridedB<float, false>{a_prev, ni}, ni, B, rows, pW,
                       sW);
    if (!to_adam)
      hipLaunchKernelGGL(sum_splits, dim3((no * ni + 255) / 256), dim3(256), 0, net->stream, net->part.p, no * ni,
                         S, gW);
    hipLaunchKernelGGL(col_partial, dim3((no + kColTile - 1) / kColTile, S), dim3(kColThreads), 0, net->stream,
                       delta, B, no, rows, pb, sb);
    if (!to_adam)
      hipLaunchKernelGGL(sum_splits, dim3((no + 255) / 256), dim3(256), 0, net->stream, net->part.p, no, S, gb);
    if (l > 0) {
      // delta_prev[B x ni] = (delta[B x no] W[no x ni]) * gelu'(Z_{l-1})
      const __hip_bfloat16* W = net->w16.p + net->w_off[l];
      hipLaunchKernelGGL((gemm<float, __hip_bfloat16, false, false, 3>), grid_for(B, ni), dim3(256), 0,
                         net->stream, delta, no, W, ni, net->dA[l].p, ni, B, ni, no,
                         static_cast<const float*>(nullptr), static_cast<float*>(nullptr),
                         static_cast<const float*>(net->Z[l - 1].p));
      delta = net->dA[l].p;
    }
    hipcheck(hipGetLastError(), "mlp backward");
  }
}

float loss_and_grad(mh_mlp* net, const float* in, const float* target, int B) {
  const int L = net->L();
  const int n = B * net->sizes[L];
  if (net->fused) {
    fused_backward(net, in, target, nullptr, B, net->terms.p, nullptr);
  } else {
    forward(net, in, B);
    hipLaunchKernelGGL(loss_grad, dim3((n + 255) / 256), dim3(256), 0, net->stream, net->A[L - 1].p, target, n,
                       1.0f / B, net->dY.p, net->terms.p);
    backward(net, in, B);
  }
  std::vector<float> terms(n);
  hipcheck(hipMemcpyAsync(terms.data(), net->terms.p, n * sizeof(float), hipMemcpyDeviceToHost, net->stream),
           "D2H");
  hipcheck(hipStreamSynchronize(net->stream), "sync");
  double s = 0.0;
  for (float v : terms) s += v;
  return static_cast<float>(s / B);
}

int fail(const mh::Error& e) {
  mh::set_error(e.what());
  return e.code;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch[kMaxDevices] = {};

// Device address of `scratch` on `device` (current), resolved once per device.
float* scratch_address(int device) {
  if (device < 0 || device >= kMaxDevices) throw mh::Error(MH_ERR_ARG, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[device]) {
    void* p = nullptr;
    hipcheck(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    g_scratch[device] = static_cast<float*>(p);
  }
  return g_scratch[device];
}

}  // namespace

extern "C" {

int mh_mlp_create(int device, int n_layers, const int* sizes, uint64_t seed, mh_mlp** out) {
  try {
    if (!out || !sizes || n_layers < 1) throw mh::Error(MH_ERR_ARG, "invalid layer list");
    auto net = std::make_unique<mh_mlp>();
    net->device = device;
    hipcheck(hipSetDevice(device), "hipSetDevice");
    net->scratch = scratch_address(device);
    hipcheck(hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking), "stream");
    net->sizes.assign(sizes, sizes + n_layers + 1);
    for (int l = 0; l <= n_layers; l++)
      if (sizes[l] < 1) throw mh::Error(MH_ERR_ARG, "layer sizes must be >= 1");
    size_t off = 0;
    for (int l = 0; l < n_layers; l++) {
      net->w_off.push_back(off);
      off += static_cast<size_t>(sizes[l + 1]) * sizes[l] + sizes[l + 1];
    }
    net->n_params = off;
    net->fused = n_layers <= kDenseMaxLayers && *std::max_element(sizes, sizes + n_layers + 1) <= kDenseMaxWidth;
    if (net->fused) {
      int at = 0;
      net->shape.L = n_layers;
      for (int l = 0; l < n_layers; l++) {
        PackedLayer& p = net->shape.layer[l];
        p.out = sizes[l + 1];
        p.in = p.c = sizes[l];
        p.w_off = static_cast<int>(net->w_off[l]);
        p.b_off = static_cast<int>(net->b_off(l));
        at = pack_layout(p, at);
      }
      net->shape.zero = at;
      at += 8;
      net->pack.ensure(at);
      hipLaunchKernelGGL(fill_zero_u16, dim3((at + 255) / 256), dim3(256), 0, net->stream, net->pack.p, at);
    } else {
      size_t widest = 0;
      for (int l = 0; l < n_layers; l++) widest = std::max<size_t>(widest, static_cast<size_t>(sizes[l]) * sizes[l + 1]);
      // split partials of one tensor, or of every parameter for adam_step_splits
      net->part.ensure(static_cast<size_t>(kMlpSplit) * std::max(widest, net->n_params));
    }
    net->w16.ensure(off);
    // He-uniform weights (bound sqrt(6 / fan_in)), zero biases
    std::mt19937_64 rng(seed);
    std::vector<float> p(off, 0.f);
    for (int l = 0; l < n_layers; l++) {
      const float bound = std::sqrt(6.0f / sizes[l]);
      std::uniform_real_distribution<float> u(-bound, bound);
      const size_t nw = static_cast<size_t>(sizes[l + 1]) * sizes[l];
      for (size_t i = 0; i < nw; i++) p[net->w_off[l] + i] = u(rng);
    }
    net->params.ensure(off);
    net->grads.ensure(off);
    net->m.ensure(off);
    net->v.ensure(off);
    std::vector<float> zeros(off, 0.f);
    hipcheck(hipMemcpy(net->params.p, p.data(), off * sizeof(float), hipMemcpyHostToDevice), "H2D");
    hipcheck(hipMemcpy(net->m.p, zeros.data(), off * sizeof(float), hipMemcpyHostToDevice), "H2D");
    hipcheck(hipMemcpy(net->v.p, zeros.data(), off * sizeof(float), hipMemcpyHostToDevice), "H2D");
    refresh_weights(net.get());
    hipcheck(hipStreamSynchronize(net->stream), "init");
    *out = net.release();
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_destroy(mh_mlp* net) {
  delete net;
  return MH_OK;
}

int mh_mlp_param_count(const mh_mlp* net) { return net ? static_cast<int>(net->n_params) : MH_ERR_ARG; }

int mh_mlp_get_params(const mh_mlp* net, float* out) {
  try {
    if (!net || !out) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipMemcpy(out, net->params.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost), "D2H");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_set_params(mh_mlp* net, const float* in) {
  try {
    if (!net || !in) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    hipcheck(hipMemcpy(net->params.p, in, net->n_params * sizeof(float), hipMemcpyHostToDevice), "H2D");
    refresh_weights(net);
    hipcheck(hipStreamSynchronize(net->stream), "set params");
    net->adam_t = 0;
    std::vector<float> zeros(net->n_params, 0.f);
    hipcheck(hipMemcpy(net->m.p, zeros.data(), zeros.size() * sizeof(float), hipMemcpyHostToDevice), "H2D");
    hipcheck(hipMemcpy(net->v.p, zeros.data(), zeros.size() * sizeof(float), hipMemcpyHostToDevice), "H2D");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_forward(mh_mlp* net, const float* x, int batch, float* y) {
  try {
    if (!net || (batch > 0 && (!x || !y)) || batch < 0) throw mh::Error(MH_ERR_ARG, "null argument");
    if (batch == 0) return MH_OK;
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    const int L = net->L();
    const int chunk = 8192;
    if (net->fused) {
      // rows go up in pieces, each followed by its kernel, so all but the
      // last piece's kernel runs while the host stages the next; results
      // come back in one copy per round
      const int ni = net->sizes[0], no = net->sizes[L], round = 16 * chunk;
      net->x.ensure(static_cast<size_t>(std::min(batch, round)) * ni);
      net->dY.ensure(static_cast<size_t>(std::min(batch, round)) * no);
      for (int r0 = 0; r0 < batch; r0 += round) {
        const int rows = std::min(round, batch - r0);
        for (int b0 = 0; b0 < rows; b0 += chunk) {
          const int B = std::min(chunk, rows - b0);
          hipcheck(hipMemcpyAsync(net->x.p + static_cast<size_t>(b0) * ni, x + static_cast<size_t>(r0 + b0) * ni,
                                  static_cast<size_t>(B) * ni * sizeof(float), hipMemcpyHostToDevice, net->stream),
                   "H2D");
          fused_forward(net, net->x.p + static_cast<size_t>(b0) * ni, B, net->dY.p + static_cast<size_t>(b0) * no,
                        net->stream);
        }
        hipcheck(hipMemcpyAsync(y + static_cast<size_t>(r0) * no, net->dY.p, static_cast<size_t>(rows) * no * sizeof(float),
                                hipMemcpyDeviceToHost, net->stream), "D2H");
      }
      hipcheck(hipStreamSynchronize(net->stream), "sync");
      return MH_OK;
    }
    ensure_batch(net, std::min(batch, chunk));
    for (int b0 = 0; b0 < batch; b0 += chunk) {
      const int B = std::min(chunk, batch - b0);
      hipcheck(hipMemcpyAsync(net->x.p, x + static_cast<size_t>(b0) * net->sizes[0],
                              static_cast<size_t>(B) * net->sizes[0] * sizeof(float), hipMemcpyHostToDevice,
                              net->stream), "H2D");
      forward(net, net->x.p, B);
      hipcheck(hipMemcpyAsync(y + static_cast<size_t>(b0) * net->sizes[L], net->A[L - 1].p,
                              static_cast<size_t>(B) * net->sizes[L] * sizeof(float), hipMemcpyDeviceToHost,
                              net->stream), "D2H");
    }
    hipcheck(hipStreamSynchronize(net->stream), "sync");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_forward_noalloc(mh_mlp* net, const float* x, int batch, float* y, void* stream) {
  try {
    if (!net || batch < 0 || (batch > 0 && (!x || !y))) throw mh::Error(MH_ERR_ARG, "null argument");
    if (batch == 0) return MH_OK;
    const int L = net->L();
    size_t widest = 0;
    for (int l = 1; l < L; l++) widest = std::max<size_t>(widest, net->sizes[l]);
    const size_t half = MH_MLP_SCRATCH_FLOATS / 2;
    if (static_cast<size_t>(batch) * widest > half)
      throw mh::Error(MH_ERR_RANGE, "batch x widest hidden layer (" + std::to_string(batch) + " x " +
                                        std::to_string(widest) + ") over the scratch array's half (" +
                                        std::to_string(half) + " floats)");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    hipStream_t s = stream ? static_cast<hipStream_t>(stream) : net->stream;
    if (net->fused && !forward_by_layers(net, x, batch, y)) {
      fused_forward(net, x, batch, y, s);
      return MH_OK;
    }
    const float* prev = x;
    for (int l = 0; l < L; l++) {
      const int ni = net->sizes[l], no = net->sizes[l + 1];
      const __hip_bfloat16* W = net->w16.p + net->w_off[l];
      const float* b = net->params.p + net->b_off(l);
      float* out = l == L - 1 ? y : net->scratch + (l % 2) * half;
      if (l < L - 1)
        hipLaunchKernelGGL((gemm<float, __hip_bfloat16, false, true, 4>), grid_for(batch, no), dim3(256), 0, s,
                           prev, ni, W, ni, out, no, batch, no, ni, b, static_cast<float*>(nullptr),
                           static_cast<const float*>(nullptr));
      else
        hipLaunchKernelGGL((gemm<float, __hip_bfloat16, false, true, 2>), grid_for(batch, no), dim3(256), 0, s,
                           prev, ni, W, ni, out, no, batch, no, ni, b, static_cast<float*>(nullptr),
                           static_cast<const float*>(nullptr));
      hipcheck(hipGetLastError(), "mlp forward (no-alloc)");
      prev = out;
    }
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_loss_grad(mh_mlp* net, const float* x, const float* target, int batch, float* loss, float* grad) {
  try {
    if (!net || !x || !target || batch < 1) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    ensure_batch(net, batch);
    const int L = net->L();
    hipcheck(hipMemcpyAsync(net->x.p, x, static_cast<size_t>(batch) * net->sizes[0] * sizeof(float),
                            hipMemcpyHostToDevice, net->stream), "H2D");
    hipcheck(hipMemcpyAsync(net->t.p, target, static_cast<size_t>(batch) * net->sizes[L] * sizeof(float),
                            hipMemcpyHostToDevice, net->stream), "H2D");
    const float l = loss_and_grad(net, net->x.p, net->t.p, batch);
    if (loss) *loss = l;
    if (grad)
      hipcheck(hipMemcpy(grad, net->grads.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost), "D2H");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_mlp_train(mh_mlp* net, const float* x, const float* target, int n, int batch, int n_epochs, float lr,
                 uint64_t seed, float* final_loss) {
  try {
    if (!net || !x || !target || n < 1 || batch < 1 || n_epochs < 0) throw mh::Error(MH_ERR_ARG, "bad arguments");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    const int L = net->L();
    const int ni = net->sizes[0], no = net->sizes[L];
    batch = std::min(batch, n);
    ensure_batch(net, batch);
    net->data_x.ensure(static_cast<size_t>(n) * ni);
    net->data_t.ensure(static_cast<size_t>(n) * no);
    net->idx.ensure(n);
    hipcheck(hipMemcpyAsync(net->data_x.p, x, static_cast<size_t>(n) * ni * sizeof(float), hipMemcpyHostToDevice,
                            net->stream), "H2D");
    hipcheck(hipMemcpyAsync(net->data_t.p, target, static_cast<size_t>(n) * no * sizeof(float),
                            hipMemcpyHostToDevice, net->stream), "H2D");
    std::mt19937_64 rng(seed);
    std::vector<int> perm(n);
    // the last epoch keeps every batch's loss terms on the device, so no
    // batch waits for a copy to the host; they are summed after the loop
    const int n_batches = n / batch;
    const size_t nt = static_cast<size_t>(batch) * no;
    net->epoch_terms.ensure(static_cast<size_t>(n_batches) * nt);
    int batches = 0;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int ep = 0; ep < n_epochs; ep++) {
      for (int i = 0; i < n; i++) perm[i] = i;
      std::shuffle(perm.begin(), perm.end(), rng);
      hipcheck(hipMemcpyAsync(net->idx.p, perm.data(), n * sizeof(int), hipMemcpyHostToDevice, net->stream), "H2D");
      const bool last = ep == n_epochs - 1;
      for (int b0 = 0; b0 + batch <= n; b0 += batch) {
        float* terms = last ? net->epoch_terms.p + batches * nt : net->terms.p;
        net->adam_t++;
        const float bc1 = 1.f - std::pow(b1, static_cast<float>(net->adam_t));
        const float bc2 = 1.f - std::pow(b2, static_cast<float>(net->adam_t));
        if (last) batches++;
        if (net->fused) {
          const AdamArgs adam{net->params.p, net->m.p, net->v.p, net->pack.p, lr, b1, b2, eps, bc1, bc2};
          fused_backward(net, net->data_x.p, net->data_t.p, net->idx.p + b0, batch, terms, &adam);
          continue;
        }
        hipLaunchKernelGGL(gather_rows, dim3(batch), dim3(64), 0, net->stream, net->data_x.p, net->idx.p + b0,
                           batch, ni, net->x.p);
        hipLaunchKernelGGL(gather_rows, dim3(batch), dim3(64), 0, net->stream, net->data_t.p, net->idx.p + b0,
                           batch, no, net->t.p);
        forward(net, net->x.p, batch);
        hipLaunchKernelGGL(loss_grad, dim3((static_cast<int>(nt) + 255) / 256), dim3(256), 0, net->stream,
                           net->A[L - 1].p, net->t.p, static_cast<int>(nt), 1.0f / batch, net->dY.p, terms);
        backward(net, net->x.p, batch, true);
        hipLaunchKernelGGL(adam_step_splits, dim3((net->n_params + 255) / 256), dim3(256), 0, net->stream,
                           net->params.p, net->part.p, mlp_splits(batch), net->n_params, net->m.p, net->v.p,
                           net->w16.p, static_cast<int>(net->n_params), lr, b1, b2, eps, bc1, bc2);
        hipcheck(hipGetLastError(), "train step");
      }
    }
    // the fused update keeps the packed weights only
    if (net->fused && n_epochs > 0)
      hipLaunchKernelGGL(to_bf16, dim3((net->n_params + 255) / 256), dim3(256), 0, net->stream, net->params.p,
                         net->w16.p, static_cast<int>(net->n_params));
    // the last epoch's mean over batches of each batch's summed terms / batch
    std::vector<float> terms(static_cast<size_t>(batches) * nt);
    if (batches)
      hipcheck(hipMemcpyAsync(terms.data(), net->epoch_terms.p, terms.size() * sizeof(float),
                              hipMemcpyDeviceToHost, net->stream), "D2H");
    hipcheck(hipStreamSynchronize(net->stream), "sync");
    double epoch_loss = 0.0;
    for (int bi = 0; bi < batches; bi++) {
      double s = 0.0;
      for (size_t j = 0; j < nt; j++) s += terms[bi * nt + j];
      epoch_loss += s / batch;
    }
    if (batches) epoch_loss /= batches;
    if (final_loss) *final_loss = static_cast<float>(epoch_loss);
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

}  // extern "C"
