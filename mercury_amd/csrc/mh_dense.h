// mh_dense.h -- the surrogates' dense layers as two kernels: dense_net runs
// every layer of a row tile (forward, and in training the loss and the
// gradients of every layer's output) without leaving the workgroup, and
// dense_wgrad turns the operands it leaves into weight and bias gradients
// (or straight into Adam's update).  For networks of up to kDenseMaxLayers
// layers of at most kDenseMaxWidth units; wider ones, and large batches of
// narrow ones on device buffers, run layer by layer with the kernels of
// mh_nn_kernels.h.
//
// What bounds them: launches and latency, not arithmetic.  A step of the
// 64-256-256-1 network on 512 rows is 0.2 GFLOP; as 15 launches (a GEMM per
// layer and direction, column sums, batch assembly, loss, Adam) it took
// 82 us, each launch 3-11 us however little it did; as these two it takes
// 15 + 5.5 us and 2-3 us of gaps (an epoch of 30011 rows 5.05 -> 1.65 ms).
// Inside dense_net a full layer costs 3000 cycles of tanh (8 waves, 8 values
// a lane) and 2000 of reading 128 KB of weights through one CU's cache.
//
// Every product is v_mfma_f32_16x16x32_bf16 with k in ascending slices of
// 32, the operand positions and the order of every sum as in
// mh_nn_kernels.h, so both paths give the same bits.
#pragma once

#include "mh_nn_kernels.h"

namespace {

constexpr int kDenseMaxLayers = 4;
constexpr int kDenseMaxWidth = 256;
constexpr int kActPitch = kDenseMaxWidth + 8;  // bf16 per LDS row: an odd count of 16-byte units, so the
                                               // 16 rows of an operand read fall on different banks

// Packed weights: the bf16 weights in the order the matrix cores read them,
// one 1 KB block per (slice of 32 k, tile of 16 n), lane l's 8 values (n =
// l % 16, k = 8 (l / 16) ..) at 16 l.  A layer W [out x in], in = offsets x
// C (dense layers: one offset, C = in), has two packings: fwd with k = the
// input index and n = the output, and bwd with k = offset x out + output
// and n = the channel.  Blocks are padded with zeros.
struct PackedLayer {
  int out, in, c;      // c: channels per kernel offset (dense: in)
  int w_off, b_off;    // in the parameter vector
  int fwd, bwd;        // element offsets in the packed array
};

__host__ __device__ inline int packed_blocks(int k, int n) { return ((k + 31) / 32) * ((n + 15) / 16); }

// Lays out the packings of a layer from `at` and returns the end.
inline int pack_layout(PackedLayer& p, int at) {
  p.fwd = at;
  at += 512 * packed_blocks(p.in, p.out);
  p.bwd = at;
  at += 512 * packed_blocks(p.in / p.c * p.out, p.c);
  return at;
}

__device__ __forceinline__ int packed_index(int k, int n, int n_tiles) {
  return (((k >> 5) * n_tiles + (n >> 4)) * 64 + ((k & 31) >> 3) * 16 + (n & 15)) * 8 + (k & 7);
}

// A weight as bf16: round to nearest even, and NaN stays NaN (bf16_bits takes
// finite values only).
__device__ __forceinline__ uint16_t weight_bits(float w) {
  return w != w ? static_cast<uint16_t>(__float_as_uint(w) >> 16 | 0x40u) : bf16_bits(w);
}

// Stores weight (o, i) in both packings.
__device__ __forceinline__ void pack_store(const PackedLayer& p, uint16_t* pack, int o, int i, float w) {
  const uint16_t b = weight_bits(w);
  pack[p.fwd + packed_index(i, o, (p.out + 15) >> 4)] = b;
  const int k = i / p.c, c = i - k * p.c;
  pack[p.bwd + packed_index(k * p.out + o, c, (p.c + 15) >> 4)] = b;
}

// The packings of every layer of a network from its fp32 parameters.  plain
// (may be null): the bf16 weights as they lie in the parameter vector.
constexpr int kPackLayers = 6;
static_assert(kDenseMaxLayers <= kPackLayers, "a fused network packs in one launch");
struct PackList {
  int n;
  PackedLayer layer[kPackLayers];
};
__global__ void pack_layers(PackList list, const float* params, uint16_t* pack, uint16_t* plain) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
  for (int l = 0; l < kPackLayers; ++l) {
    if (l >= list.n) return;
    const PackedLayer& p = list.layer[l];
    if (e < p.out * p.in) {
      const float w = params[p.w_off + e];
      pack_store(p, pack, e / p.in, e % p.in, w);
      if (plain) plain[p.w_off + e] = weight_bits(w);
      return;
    }
    e -= p.out * p.in;
  }
}
inline void launch_pack(const PackList& list, const float* params, uint16_t* pack, uint16_t* plain, hipStream_t s) {
  int n = 0;
  for (int l = 0; l < list.n; l++) n += list.layer[l].out * list.layer[l].in;
  hipLaunchKernelGGL(pack_layers, dim3((n + 255) / 256), dim3(256), 0, s, list, params, pack, plain);
}

__global__ void fill_zero_u16(uint16_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

struct DenseShape {
  int L;
  int zero;  // element offset of 8 zeros in the packed array
  PackedLayer layer[kDenseMaxLayers];
};

// A batch of B rows reduces in `splits` runs of `rows` rows, each in slices
// of 32 rows counted from its start (`slices` per run).  Operands of the
// weight gradients are kept in the order their kernel reads them: element
// (row, n) of an [B x N] matrix at its slice's block (slice, n / 16), lane
// 16 (row in slice / 8) + n % 16, value row % 8.
struct RowSplits {
  int B, splits, rows, slices;
};
inline RowSplits row_splits(int B, int splits) {
  const int rows = (B + splits - 1) / splits;
  return RowSplits{B, splits, rows, (rows + 31) / 32};
}
// Where rows row .. row + 3 (row a multiple of 4) of such an operand lie:
// element (row + r, 16 t + c) at slice(r) * tiles * 512 + t * 512 + c * 8 +
// at(r).  Runs of a multiple of 4 rows keep the four in one 8-byte store.
struct OperandRows {
  bool whole;        // the four are consecutive values of one lane
  int n;             // rows inside the batch
  int slice[4], at[4];
};
__device__ __forceinline__ OperandRows operand_rows(const RowSplits& rs, int row) {
  OperandRows o;
  o.n = min(4, max(0, rs.B - row));
  o.whole = (rs.rows & 3) == 0 && o.n == 4;
  int s = row / rs.rows, local = row - s * rs.rows;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    o.slice[r] = s * rs.slices + (local >> 5);
    o.at[r] = ((local & 31) >> 3) * 128 + (local & 7);
    if (++local == rs.rows) {
      local = 0;
      ++s;
    }
  }
  return o;
}
__device__ __forceinline__ uint2 pack4(const uint16_t (&v)[4]) {
  return make_uint2(v[0] | static_cast<uint32_t>(v[1]) << 16, v[2] | static_cast<uint32_t>(v[3]) << 16);
}
__device__ __forceinline__ void operand_store4(const OperandRows& o, uint16_t* p, int t, int c, int tiles,
                                               uint2 v) {
  if (o.whole) {
    *reinterpret_cast<uint2*>(p + (static_cast<size_t>(o.slice[0]) * tiles + t) * 512 + o.at[0] + 8 * c) = v;
  } else {
    const uint32_t u[4] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16};
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < o.n)
        p[(static_cast<size_t>(o.slice[r]) * tiles + t) * 512 + o.at[r] + 8 * c] = static_cast<uint16_t>(u[r]);
  }
}

// Training buffers of dense_net and dense_wgrad.
struct DenseTrain {
  RowSplits rs;
  const int* x_idx;                    // batch row -> row of x (null: the same)
  const int* t_idx;                    // batch row -> row of target (null: the same)
  const float* target;
  float inv_b;
  float* terms;                        // 0.5 (y - t)^2 per output
  uint16_t* X[kDenseMaxLayers];        // input of layer l, as a weight-gradient operand
  uint16_t* D[kDenseMaxLayers];        // loss gradient of layer l's output, likewise
  float* delta[kDenseMaxLayers];       // and in fp32, [B x out], for the bias sums
  float* dx;                           // gradient of the input, [B x in]; null: not wanted (one layer: has to be)
};

// Every layer for 16 MT rows per workgroup (8 waves, output tiles w and w + 8
// of 16 units each): x [rows x in] -> y [B x out].  TRAIN: also the loss
// terms, the gradients of every layer's output (the last from y and the
// target) and the weight gradients' operands.  Activations alternate between
// two LDS buffers as bf16 (what the products round them to).  The slope of
// gelu shares its tanh and waits in LDS where the unit's gradient will
// stand: the backward products of layer l + 1 have the tiles of the forward
// products of layer l, so a lane reads what it wrote.
//
// The kernel is a chain of latencies, so the packed blocks of the layer
// after next are requested as soon as a layer's products have read theirs,
// by loads without conditions (a wave without a tile, or a slice past the
// layer's, reads one 16-byte word of zeros): behind a branch the compiler
// cannot count the loads in flight and waits for all of them.  For the same
// reason results are stored after the last layer (stores and loads share a
// counter), no register may spill (a reload waits for every load before
// it), and the layer count is a template parameter: the sizes are then
// kernel arguments read up front.
constexpr int kDenseThreads = 512;
template <int L, int MT, bool TRAIN>
__global__ __launch_bounds__(kDenseThreads) void dense_net(DenseShape sh, const float* __restrict__ params,
                                                           const uint16_t* __restrict__ pack,
                                                           const float* __restrict__ x, int B, float* __restrict__ y,
                                                           DenseTrain tr) {
  static_assert(!TRAIN || MT == 1, "training tiles are 16 rows");
  constexpr int kStages = TRAIN ? 2 * L : L;  // forward layers, then backward ones (the last only for dx)
  constexpr int kSlices = kDenseMaxWidth / 32;
  constexpr int T = kDenseMaxWidth / 16 / (kDenseThreads / 64);  // output tiles per wave
  __shared__ __align__(16) uint16_t act[2][16 * MT][kActPitch];
  __shared__ __align__(16) float grad[TRAIN ? L : 1][TRAIN ? 16 : 1][TRAIN ? kDenseMaxWidth : 1];
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * 16 * MT;
  int tile[T], n[T];  // this wave's tiles and this lane's units, in every layer
#pragma unroll
  for (int i = 0; i < T; ++i) {
    tile[i] = wave + kDenseThreads / 64 * i;
    n[i] = 16 * tile[i] + c16;
  }
  int in_[L], out_[L];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    in_[l] = sh.layer[l].in;
    out_[l] = sh.layer[l].out;
  }

  // target rows (indices first: what they feed is the longest chain of loads)
  int src[4] = {};
  if constexpr (TRAIN) {
#pragma unroll
    for (int r = 0; r < 4; ++r) src[r] = min(row0 + 4 * q + r, B - 1);
    if (tr.t_idx)
#pragma unroll
      for (int r = 0; r < 4; ++r) src[r] = tr.t_idx[src[r]];
  }
  bf16x8_t w[2][T][kSlices];
  auto fetch = [&](int st, int s0, int s1) {
    const bool fwd = st < L;
    const int l = fwd ? st : 2 * L - 1 - st;
    const int ks = ((fwd ? in_[l] : out_[l]) + 31) >> 5, nt = ((fwd ? out_[l] : in_[l]) + 15) >> 4;
    const int first = fwd ? sh.layer[l].fwd : sh.layer[l].bwd;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const uint32_t base = 2u * static_cast<uint32_t>(first + tile[i] * 512) + 16u * lane;
      const int mine = tile[i] < nt ? ks : 0;
#pragma unroll
      for (int s = s0; s < s1; ++s) {
        const uint32_t at = s < mine ? base + static_cast<uint32_t>(s * nt) * 1024u : 2u * sh.zero;
        w[st & 1][i][s] =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(reinterpret_cast<const char*>(pack) + at));
      }
    }
  };
  // the first layer's blocks travel while the row indices do
  fetch(0, 0, kSlices);
  float bias[L][T], target[T][4];
#pragma unroll
  for (int l = 0; l < L; ++l)
#pragma unroll
    for (int i = 0; i < T; ++i) bias[l][i] = params[sh.layer[l].b_off + min(n[i], out_[l] - 1)];
  if constexpr (TRAIN) {
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        target[i][r] = tr.target[static_cast<size_t>(src[r]) * out_[L - 1] + min(n[i], out_[L - 1] - 1)];
  }
  // input rows as bf16, zeros past the batch and past the width
  const int n_in = in_[0];
  const bool vec = n_in % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
  for (int e = tid; e < 16 * MT * 32; e += kDenseThreads) {
    const int r = e >> 5, k = 8 * (e & 31), row = row0 + r;
    u16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (row < B && k < n_in) {
      int from = row;
      if constexpr (TRAIN)
        if (tr.x_idx) from = tr.x_idx[row];
      const float* p = x + static_cast<size_t>(from) * n_in + k;
      if (vec) v = ld8_bf16_a16(p);
      else
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k + j < n_in) v[j] = bf16_bits(p[j]);
    }
    *reinterpret_cast<u16x8_t*>(&act[0][r][k]) = v;
  }
  if (L > 1) fetch(1, 0, kSlices);
  // operands for the stores at the end: every layer's input and output
  // gradient
  uint2 xo[TRAIN ? L : 1][T], go[TRAIN ? L : 1][T];
  lds_barrier();
  if constexpr (TRAIN) {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const uint16_t v[4] = {act[0][4 * q][n[i]], act[0][4 * q + 1][n[i]], act[0][4 * q + 2][n[i]],
                             act[0][4 * q + 3][n[i]]};
      xo[0][i] = pack4(v);
    }
  }

#pragma unroll
  for (int st = 0; st < kStages; ++st) {
    const bool fwd = st < L;
    const int l = fwd ? st : 2 * L - 1 - st;
    if (TRAIN && st == kStages - 1 && (L == 1 || !tr.dx)) break;
    const int no = fwd ? out_[l] : in_[l];
    const uint16_t (*a)[kActPitch] = act[st & 1];
    uint16_t (*b)[kActPitch] = act[1 - (st & 1)];
    f32x4_t acc[T][MT];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[i][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // every slice of 256 inputs, with zeros on both sides past the layer's
    // own: no branch between the LDS reads and the products
#pragma unroll
    for (int s = 0; s < kSlices; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const bf16x8_t av =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(&a[16 * m + c16][32 * s + 8 * q]));
#pragma unroll
        for (int i = 0; i < T; ++i)
          acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, w[st & 1][i][s], acc[i][m], 0, 0, 0);
      }
    // every wave writes its columns of the next layer's input: zeros past
    // the last unit
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const bool in = n[i] < no;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        // the requests go out between the tiles' arithmetic: a wave that
        // issues them in one run stalls until the cache has taken them
        constexpr int kRuns = T * MT;
        if (st + 2 < kStages) fetch(st + 2, (i * MT + m) * kSlices / kRuns, (i * MT + m + 1) * kSlices / kRuns);
        const int row = row0 + 16 * m + 4 * q;
        uint16_t o[4];
        if (fwd && l + 1 < L) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = acc[i][m][r] + bias[l][i], th = gelu_tanh(v);
            o[r] = in ? bf16_bits(gelu_f(v, th)) : uint16_t(0);
            if constexpr (TRAIN) grad[TRAIN ? l : 0][4 * q + r][n[i]] = gelu_grad(v, th);
          }
          if constexpr (TRAIN) xo[l + 1 < L ? l + 1 : 0][i] = pack4(o);
        } else if (!TRAIN) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (in && row + r < B) y[static_cast<size_t>(row + r) * no + n[i]] = acc[i][m][r] + bias[l][i];
        } else if (fwd) {
          // dY = (y - t) / B; the target's registers keep the error for the
          // loss terms
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float e = (acc[i][m][r] + bias[l][i]) - target[i][r];
            const float d = in && row + r < B ? e * tr.inv_b : 0.f;
            target[i][r] = e;
            grad[TRAIN ? l : 0][4 * q + r][n[i]] = d;
            o[r] = bf16_bits(d);
          }
          go[TRAIN ? l : 0][i] = pack4(o);
        } else if (l > 0) {
          // dLoss/dZ_{l-1} = (dLoss/dZ_l W_l) gelu'(Z_{l-1})
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float& g = grad[TRAIN && l > 0 ? l - 1 : 0][4 * q + r][n[i]];  // the slope until now
            const float d = in ? acc[i][m][r] * g : 0.f;
            g = d;
            o[r] = bf16_bits(d);
          }
          go[TRAIN && l > 0 ? l - 1 : 0][i] = pack4(o);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (in && row + r < B) tr.dx[static_cast<size_t>(row + r) * no + n[i]] = acc[i][m][r];
        }
        if (st + 1 < kStages)
#pragma unroll
          for (int r = 0; r < 4; ++r) b[16 * m + 4 * q + r][n[i]] = o[r];
      }
    }
    if (st + 1 < kStages) lds_barrier();
  }

  if constexpr (TRAIN) {
    const int row = row0 + 4 * q;
    const OperandRows rows = operand_rows(tr.rs, row);
#pragma unroll
    for (int l = 0; l < L; ++l) {
      const int ti = (in_[l] + 15) >> 4, to = (out_[l] + 15) >> 4;
#pragma unroll
      for (int i = 0; i < T; ++i) {
        if (tile[i] < ti) operand_store4(rows, tr.X[l], tile[i], c16, ti, xo[l][i]);
        if (tile[i] < to) operand_store4(rows, tr.D[l], tile[i], c16, to, go[l][i]);
        if (l == L - 1 && n[i] < out_[l])
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (row + r < B) tr.terms[static_cast<size_t>(row + r) * out_[l] + n[i]] = 0.5f * target[i][r] * target[i][r];
      }
    }
    lds_barrier();
    const int rows_here = min(16, B - row0);
#pragma unroll
    for (int l = 0; l < L; ++l) {
      float* out = tr.delta[l] + static_cast<size_t>(row0) * out_[l];
      if (out_[l] == kDenseMaxWidth) {
#pragma unroll
        for (int e = 0; e < 16 * kDenseMaxWidth / 4 / kDenseThreads; ++e) {
          const int at = 4 * (tid + e * kDenseThreads);
          if (at < rows_here * kDenseMaxWidth)
            *reinterpret_cast<float4*>(out + at) = *reinterpret_cast<const float4*>(&grad[l][0][0] + at);
        }
      } else {
        for (int e = tid; e < rows_here * out_[l]; e += kDenseThreads) out[e] = grad[l][e / out_[l]][e % out_[l]];
      }
    }
  }
}

struct AdamArgs {
  float *p, *m, *v;
  uint16_t* pack;
  float lr, b1, b2, eps, bc1, bc2;
};

// Weight and bias gradients of every layer from dense_net's operands.  A
// weight workgroup (8 waves) takes 16 outputs x 16 JT inputs: wave w
// computes the partial products of splits w, w + 8, .. (SR of them), and
// the partials are added through LDS in ascending split order, the order of
// sum_splits and adam_step_splits.  A bias workgroup sums 16 columns of
// delta, the row groups of every split in parallel, then added in
// col_partial's order.  ADAM: the parameters are updated in place (with
// their packings), so no gradient or partial reaches memory; otherwise
// gradients go to `grads`.  The parameters and moments are requested before
// the products: the kernel is a few memory latencies long.
constexpr int kWgThreads = 512;
inline int dense_wgrad_blocks(const DenseShape& sh, int jt) {
  int n = 0;
  for (int l = 0; l < sh.L; ++l)
    n += ((sh.layer[l].out + 15) / 16) * ((sh.layer[l].in + 16 * jt - 1) / (16 * jt) + 1);
  return n;
}
template <int L, int JT, int SR, bool ADAM>
__global__ __launch_bounds__(kWgThreads) void dense_wgrad(DenseShape sh, DenseTrain tr, AdamArgs ad,
                                                          float* __restrict__ grads) {
  constexpr int kCols = 16 * JT, kSplits = 8 * SR, kPer = (16 * kCols + kWgThreads - 1) / kWgThreads;
  __shared__ float part[kSplits][16][kCols + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const RowSplits& rs = tr.rs;
  // the layer, and the tile or bias run, of this workgroup
  int b = blockIdx.x, it = 0, jg = 0;
  bool bias = false, found = false;
  PackedLayer p{};
  const uint16_t *D = nullptr, *X = nullptr;
  const float* delta = nullptr;
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const PackedLayer& pl = sh.layer[l];
    const int jn = (pl.in + kCols - 1) / kCols, on = (pl.out + 15) / 16;
    if (!found && b < on * (jn + 1)) {
      found = true;
      it = b / (jn + 1);
      jg = b - it * (jn + 1);
      bias = jg == jn;
      p = pl;
      D = tr.D[l];
      X = tr.X[l];
      delta = tr.delta[l];
    }
    b -= on * (jn + 1);
  }
  auto load = [&](int index, float (&pmv)[3]) {
    if constexpr (ADAM) {
      pmv[0] = ad.p[index];
      pmv[1] = ad.m[index];
      pmv[2] = ad.v[index];
    }
  };
  // returns the new parameter
  auto finish = [&](int index, float g, const float (&pmv)[3]) {
    if constexpr (ADAM) {
      float m = pmv[1], v = pmv[2], w = pmv[0];
      adam_update(g, w, m, v, ad.lr, ad.b1, ad.b2, ad.eps, ad.bc1, ad.bc2);
      ad.p[index] = w;
      ad.m[index] = m;
      ad.v[index] = v;
      return w;
    } else {
      grads[index] = g;
      return g;
    }
  };
  if (bias) {
    // (split, row group) sums of 16 columns, [splits * 16][16]
    float (*acc)[16] = reinterpret_cast<float (*)[16]>(&part[0][0][0]);
    static_assert(sizeof(part) >= kSplits * 16 * 16 * sizeof(float), "bias sums fit the partials' buffer");
    const int c = tid & 15, n = 16 * it + c;
    float pmv[3] = {};
    if (tid < 16 && n < p.out) load(p.b_off + n, pmv);
    // U (split, group) sums at a time, their loads in flight together (no
    // conditions: a row outside its split is read elsewhere and adds +0)
    constexpr int U = 8;
    for (int u0 = tid >> 4; u0 < rs.splits * 16; u0 += U * (kWgThreads / 16)) {
      float sum[U] = {};
      for (int i = 0; i < rs.rows; i += 16) {
        float v[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int u = u0 + k * (kWgThreads / 16), r = (u >> 4) * rs.rows + (u & 15) + i;
          v[k] = delta[static_cast<size_t>(min(r, rs.B - 1)) * p.out + min(n, p.out - 1)];
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int u = u0 + k * (kWgThreads / 16), in_split = (u & 15) + i;
          sum[k] += in_split < rs.rows && (u >> 4) * rs.rows + in_split < rs.B ? v[k] : 0.f;
        }
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int u = u0 + k * (kWgThreads / 16);
        if (u < rs.splits * 16) acc[u][c] = sum[k];
      }
    }
    lds_barrier();
    for (int u = tid; u < rs.splits * 16; u += kWgThreads) {
      const int s = u >> 4, cc = u & 15;
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) t += acc[16 * s + k][cc];
      acc[16 * s][cc] = t;
    }
    lds_barrier();
    if (tid < 16 && n < p.out) {
      float g = 0.f;
#pragma unroll 8
      for (int s = 0; s < rs.splits; ++s) g += acc[16 * s][c];
      finish(p.b_off + n, g, pmv);
    }
    return;
  }
  float pmv[kPer][3] = {};
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int e = tid + k * kWgThreads, o = 16 * it + e / kCols, i = kCols * jg + e % kCols;
    if (e < 16 * kCols && o < p.out && i < p.in) load(p.w_off + o * p.in + i, pmv[k]);
  }
  const int nti = (p.out + 15) >> 4, ntj = (p.in + 15) >> 4;
  // The operands of SR splits (one slice each), or of SR slices of one split
  // at a time, are requested together, without conditions: rows outside the
  // split were never written, and count as zeros.
  f32x4_t acc[SR][JT];
#pragma unroll
  for (int k = 0; k < SR; ++k)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[k][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  struct Operands {
    u16x8_t d, x[JT];
  };
  auto request = [&](int s, int sl) {
    const size_t slice = static_cast<size_t>(min(s, rs.splits - 1)) * rs.slices + min(sl, rs.slices - 1);
    Operands o;
    o.d = *reinterpret_cast<const u16x8_t*>(D + (slice * nti + it) * 512 + 8 * lane);
#pragma unroll
    for (int j = 0; j < JT; ++j)
      o.x[j] = *reinterpret_cast<const u16x8_t*>(X + (slice * ntj + min(jg * JT + j, ntj - 1)) * 512 + 8 * lane);
    return o;
  };
  auto products = [&](int s, int sl, Operands& o, f32x4_t (&c)[JT]) {
    const int nr = s < rs.splits ? min(rs.B - s * rs.rows, rs.rows) - 32 * sl : 0;  // rows of the slice
    if (nr <= 0) return;
    if (nr < 32) {
      const int valid = nr - 8 * (lane >> 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o.d[e] = e < valid ? o.d[e] : uint16_t(0);
#pragma unroll
        for (int j = 0; j < JT; ++j) o.x[j][e] = e < valid ? o.x[j][e] : uint16_t(0);
      }
    }
#pragma unroll
    for (int j = 0; j < JT; ++j)
      c[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, o.d),
                                                     __builtin_bit_cast(bf16x8_t, o.x[j]), c[j], 0, 0, 0);
  };
  constexpr int kRound = SR > 2 ? SR : 2;
  Operands o[kRound];
  if (rs.slices == 1 && SR > 1) {
#pragma unroll
    for (int k = 0; k < SR; ++k) o[k] = request(wave + 8 * k, 0);
#pragma unroll
    for (int k = 0; k < SR; ++k) products(wave + 8 * k, 0, o[k], acc[k]);
  } else {
#pragma unroll
    for (int k = 0; k < SR; ++k)
      for (int sl = 0; sl < rs.slices; sl += kRound) {
#pragma unroll
        for (int u = 0; u < kRound; ++u) o[u] = request(wave + 8 * k, sl + u);
#pragma unroll
        for (int u = 0; u < kRound; ++u)
          if (sl + u < rs.slices) products(wave + 8 * k, sl + u, o[u], acc[k]);
      }
  }
#pragma unroll
  for (int k = 0; k < SR; ++k)
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave + 8 * k][4 * (lane >> 4) + r][16 * j + (lane & 15)] = acc[k][j][r];
  lds_barrier();
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int e = tid + k * kWgThreads, r = e / kCols, c = e % kCols, o = 16 * it + r, i = kCols * jg + c;
    if (e >= 16 * kCols || o >= p.out || i >= p.in) continue;
    float g = 0.f;
#pragma unroll 8
    for (int s = 0; s < kSplits; ++s)
      if (s < rs.splits) g += part[s][r][c];
    const float w = finish(p.w_off + o * p.in + i, g, pmv[k]);
    if constexpr (ADAM) pack_store(p, ad.pack, o, i, w);
  }
}

// dense_net and dense_wgrad of a network of L layers, and for any layer count.
template <int L, int MT, bool TRAIN>
void launch_dense_net_of(const DenseShape& sh, const float* params, const uint16_t* pack, const float* x, int B,
                         float* y, const DenseTrain& tr, hipStream_t s) {
  // a network of one layer has no stage before the input gradient in which
  // its weights could be requested
  if (L == 1 && tr.dx) throw mh::Error(MH_ERR_INTERNAL, "input gradient of a one-layer network");
  hipLaunchKernelGGL((dense_net<L, MT, TRAIN>), dim3((B + 16 * MT - 1) / (16 * MT)), dim3(kDenseThreads), 0, s, sh,
                     params, pack, x, B, y, tr);
  hipcheck(hipGetLastError(), "dense layers");
}
template <int L, int JT, int SR, bool ADAM>
void launch_dense_wgrad_of(const DenseShape& sh, const DenseTrain& tr, const AdamArgs& ad, float* grads,
                           hipStream_t s) {
  hipLaunchKernelGGL((dense_wgrad<L, JT, SR, ADAM>), dim3(dense_wgrad_blocks(sh, JT)), dim3(kWgThreads), 0, s, sh, tr,
                     ad, grads);
  hipcheck(hipGetLastError(), "dense weight gradients");
}
template <int MT, bool TRAIN>
void launch_dense_net(const DenseShape& sh, const float* params, const uint16_t* pack, const float* x, int B, float* y,
                      const DenseTrain& tr, hipStream_t s) {
  switch (sh.L) {
    case 1: return launch_dense_net_of<1, MT, TRAIN>(sh, params, pack, x, B, y, tr, s);
    case 2: return launch_dense_net_of<2, MT, TRAIN>(sh, params, pack, x, B, y, tr, s);
    case 3: return launch_dense_net_of<3, MT, TRAIN>(sh, params, pack, x, B, y, tr, s);
    default: launch_dense_net_of<4, MT, TRAIN>(sh, params, pack, x, B, y, tr, s);
  }
}
template <int JT, int SR, bool ADAM>
void launch_dense_wgrad(const DenseShape& sh, const DenseTrain& tr, const AdamArgs& ad, float* grads, hipStream_t s) {
  switch (sh.L) {
    case 1: return launch_dense_wgrad_of<1, JT, SR, ADAM>(sh, tr, ad, grads, s);
    case 2: return launch_dense_wgrad_of<2, JT, SR, ADAM>(sh, tr, ad, grads, s);
    case 3: return launch_dense_wgrad_of<3, JT, SR, ADAM>(sh, tr, ad, grads, s);
    default: launch_dense_wgrad_of<4, JT, SR, ADAM>(sh, tr, ad, grads, s);
  }
}

}  // namespace
