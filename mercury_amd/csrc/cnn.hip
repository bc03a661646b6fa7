// cnn.hip -- convolutional surrogate for voxel genomes: a learned 64-d
// feature extractor in front of the surrogate MLP (64 -> 256 -> 256 -> 1).
//
// Input: a genome, one material index (0 = empty, 1..4) per voxel of an 8^3
// grid, voxel (x, y, z) at x + 8 (y + 8 z).  Network:
//   conv1  3x3x3, 5 (one-hot materials) -> 32, zero padding, GELU
//   conv2  3x3x3, 32 -> 32, GELU
//   pool   2x2x2 average, 8^3 -> 4^3
//   conv3  3x3x3, 32 -> 64, GELU
//   mean over the 4^3 positions -> 64 features
//   dense  64 -> 256 GELU -> 256 GELU -> 1
// Three kernels carry the convolutions, every product on the matrix cores
// (v_mfma_f32_16x16x32_bf16: bf16 operands, fp32 accumulate):
//   conv_features  one genome per workgroup, conv1 to the 64 features, its
//                  activations in LDS from layer to layer;
//   conv_backward  one genome per workgroup, from the features' gradient to
//                  dLoss/dZ of conv3, conv2 and conv1;
//   conv_wgrad     weight and bias gradients, reduced over the batch in
//                  kSplit row splits per layer;
// and the dense head runs in the kernels of mh_dense.h.  Products are
// im2col GEMMs whose operands are read from zero-padded LDS grids, k in
// ascending slices of 32 (column k*C + c for kernel offset
// k = (dz+1)*9 + (dy+1)*3 + (dx+1)), and every reduction has a fixed order,
// so training is deterministic.  Weights are bf16 with an fp32 master copy
// for Adam; activations and gradients enter every product rounded to bf16,
// with fp32 accumulation.  Loss = mean 0.5 (y - target)^2.
//
// What the layer-by-layer form cost (a GEMM or column sum per launch, fp32
// activations through memory, 64-wide tiles half empty at 32 channels): 35
// launches and 812 us per training step of 256 genomes, 0.67 us per scored
// genome.  As these kernels, on MI355X: 129 us of kernels per step
// (conv_features 35, conv_wgrad 35, conv_backward 26, the head's two 15 and
// 11, conv_update 6), 0.064 us per scored genome.  conv_features is bound by
// the 36 900 tanh of a genome (VALU issue: 0.85 wave64 instructions per
// CU-cycle, where plain FP32 chains reach 0.88-0.92; the matrix cores are busy
// 27 % of the time), the training kernels, one genome per CU at this batch, by
// the latency of their chains.
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "mercury_hip.h"
#include "mh_internal.h"
#include "mh_dense.h"

namespace {

constexpr int kG = 8, kP1 = kG * kG * kG;        // genome grid and positions
constexpr int kG2 = kG / 2, kP2 = kG2 * kG2 * kG2;
constexpr int kC0 = 5, kC1 = 32, kC2 = 32, kC3 = 64, kH = 256;
constexpr int kK1 = 27 * kC0, kK2 = 27 * kC1, kK3 = 27 * kC2;
constexpr int kSplit = 64;                        // split-K partials for weight gradients

// Offsets of a padded grid of side S for kernel offset k.
template <int S>
__host__ __device__ constexpr int offset3(int k) { return (k / 9 - 1) * S * S + ((k / 3) % 3 - 1) * S + (k % 3 - 1); }

// 8^3 activations of 32 channels in LDS: bf16, a border of zeros, 64 bytes
// per position whose four 16-byte octets are permuted by the position (by
// bit 2 of x and bit 0 of y), so that the 16 positions an operand read
// covers (two rows of x) fall on different banks.  A kernel offset changes
// a lane's permutation only through x and the parity of y: six base
// addresses serve all 27 offsets and 4 row tiles as immediate offsets.
constexpr int kP = 10, kVol = kP * kP * kP;      // padded side and positions
constexpr int kRowB = 64 * kP, kPlaneB = 64 * kP * kP;
__device__ __forceinline__ int swz8(int yp, int xp) { return ((xp >> 2) & 1) | ((yp & 1) << 1); }
// 4^3 grids likewise: side 6; 32 channels permuted by y, 64 channels by x
// and y.
constexpr int kQ = 6, kVolQ = kQ * kQ * kQ;
__device__ __forceinline__ int swz4(int yp) { return yp & 3; }
__device__ __forceinline__ int swz4w(int yp, int xp) { return ((xp >> 1) & 1) | ((yp & 3) << 1); }

// The grids' operand bases of a wave's plane z = wave: row r16 of a 16-row
// tile is y = 2 t + r16 / 8, x = r16 % 8; base[dx + 1][dy & 1].
struct GridBase {
  int at[3][2];
  __device__ GridBase(int wave, int lane) {
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int xp = (r & 7) + dx, yp = (r >> 3) + 1 + p;  // parity of y + 1 + dy
        at[dx][p] = wave * kPlaneB + (r >> 3) * kRowB + xp * 64 + ((q ^ swz8(yp, xp)) << 4);
      }
  }
};

// acc[t][j] += sum over the 27 offsets of grid rows (shifted by +offset, or
// -offset with REV) times the packed blocks [27][2]: 64 positions x 32
// outputs per wave.  Blocks are requested three offsets ahead.
template <bool REV>
__device__ __forceinline__ void conv_products(const unsigned char* grid, const GridBase& base,
                                              const uint16_t* __restrict__ w, int lane, f32x4_t (&acc)[4][2]) {
  constexpr int kAhead = 3;
  bf16x8_t b[kAhead][2];
  auto load = [&](int k) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      b[k % kAhead][j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + (2 * k + j) * 512 + 8 * lane));
  };
#pragma unroll
  for (int k = 0; k < kAhead; ++k) load(k);
#pragma unroll
  for (int k = 0; k < 27; ++k) {
    const int o = REV ? 26 - k : k, dz = o / 9, dy = (o / 3) % 3, dx = o % 3;
    bf16x8_t a[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      a[t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(
                                              grid + base.at[dx][(dy + 1) & 1] + dz * kPlaneB + (dy + 2 * t) * kRowB));
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[k % kAhead][j], acc[t][j], 0, 0, 0);
    if (k + kAhead < 27) load(k + kAhead);
  }
}

// Writes this lane's four values (x = 4 (q & 1) .. + 3 of row y = 2 t + q / 2,
// channel 16 j + c16) of plane `wave` into an 8^3 grid.
struct GridStore {
  int at[2][2];  // [r == 3][j]
  __device__ GridStore(int wave, int lane) {
    const int q = lane >> 4, c = lane & 15, yp = (q >> 1) + 1;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int xp = 4 * (q & 1) + 1 + 3 * e;
        at[e][j] = (wave + 1) * kPlaneB + yp * kRowB + (4 * (q & 1) + 1) * 64 +
                   (((2 * j + (c >> 3)) ^ swz8(yp, xp)) << 4) + 2 * (c & 7);
      }
  }
  __device__ void put(unsigned char* grid, int t, int j, const uint16_t (&v)[4]) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<uint16_t*>(grid + at[r == 3][j] + 2 * t * kRowB + 64 * r) = v[r];
  }
};

__device__ __forceinline__ void zero_lds(void* p, int bytes, int threads) {
  uint4* q = reinterpret_cast<uint4*>(p);
  for (int i = threadIdx.x; i < bytes / 16; i += threads) q[i] = make_uint4(0u, 0u, 0u, 0u);
}

// A genome's voxels: values above 4 hold no channel, like the border.
constexpr int kNoMaterial = 16;
__device__ __forceinline__ uint32_t clean_voxel(uint32_t v) { return v > 4u ? kNoMaterial : v; }

struct ConvNet {
  PackedLayer l1, l2, l3;
  const float* params;
  const uint16_t* pack;
  const uint8_t* genomes;
  const int* idx;  // batch row -> genome (null: the same)
};
// Per genome: slopes of gelu in the accumulators' order (float4 per lane),
// overwritten in place by the layer's gradient, which has the same order;
// operands of the weight gradients in bf16, the form every reader takes.
struct ConvTrain {
  float4 *s1, *s2;       // [genome][wave 8][t 4][j 2][lane 64]: dLoss/dZ after conv_backward
  float4* s3;            // [genome][tile 16][lane 64]
  uint16_t* a1;          // [genome][channel 32][position 512]: conv1 output
  uint16_t* p2;          // [genome][position 64][channel 32]: pooled conv2 output
  uint16_t *d1, *d2;     // as a1: dLoss/dZ of conv1, conv2
  float* d3;             // [genome][position 64][channel 64]
  const float* dfeat;    // [genome][64]
};

// One genome per workgroup (8 waves, wave w the plane z = w): conv1, conv2,
// pooling, conv3 and the mean over positions -> feat [B][64].  78 KB of LDS,
// so two workgroups share a CU.  TRAIN: also the slopes of gelu and the
// weight gradients' operands.
template <bool TRAIN>
__global__ __launch_bounds__(512, 4) void conv_features(ConvNet net, float* __restrict__ feat, ConvTrain tr) {
  __shared__ __align__(16) unsigned char grid[64 * kVol];   // conv1 output; later pooling sums and conv3 output
  __shared__ __align__(16) unsigned char gridq[64 * kVolQ]; // pooled conv2 output
  __shared__ __align__(16) uint8_t vox[kVol + 8];           // materials with a border
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x;
  const uint8_t* g = net.genomes + static_cast<size_t>(net.idx ? net.idx[n] : n) * kP1;
  const uint32_t voxel = clean_voxel(g[tid]);
  f32x4_t acc[4][2];
  float bias1[2], bias2[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    bias1[j] = net.params[net.l1.b_off + 16 * j + c16];
    bias2[j] = net.params[net.l2.b_off + 16 * j + c16];
  }
  zero_lds(grid, 64 * kVol, 512);
  zero_lds(gridq, 64 * kVolQ, 512);
  for (int i = tid; i < (kVol + 8) / 4; i += 512) reinterpret_cast<uint32_t*>(vox)[i] = 0x01010101u * kNoMaterial;
  lds_barrier();
  vox[((tid >> 6) + 1) * 100 + (((tid >> 3) & 7) + 1) * 10 + (tid & 7) + 1] = static_cast<uint8_t>(voxel);
  lds_barrier();

  // conv1: the one-hot columns 8 k' .. 8 k' + 7 of a row span at most three
  // kernel offsets (5 channels each); each voxel sets one bit of the eight,
  // and the bits become bf16 ones.  The border's value sets bits outside.
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[t][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  {
    const int p0 = (wave + 1) * 100 + ((c16 >> 3) + 1) * 10 + (c16 & 7) + 1;
    const uint16_t* w = net.pack + net.l1.fwd;
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      bf16x8_t b[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + (2 * s + j) * 512 + 8 * lane));
      const int kk = 32 * s + 8 * q, k0 = kk / kC0, c0 = kk - k0 * kC0;
      const uint8_t* v[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int k = k0 + i;
        // past the last offset the weights are zeros: any voxel will do
        v[i] = vox + p0 + (k < 27 ? offset3<kP>(k) : 0);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t m = 1u << ((v[0][20 * t] - c0) & 31) | 1u << ((v[1][20 * t] + kC0 - c0) & 31) |
                           1u << ((v[2][20 * t] + 2 * kC0 - c0) & 31);
        uint4 a;
        uint32_t* aw = &a.x;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          aw[i] = (static_cast<uint32_t>(static_cast<int32_t>(m << (31 - 2 * i)) >> 31) & 0x3f80u) |
                  (static_cast<uint32_t>(static_cast<int32_t>(m << (30 - 2 * i)) >> 31) & 0x3f800000u);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), b[j], acc[t][j], 0, 0, 0);
      }
    }
  }
  const GridStore store(wave, lane);
  const size_t frag = (static_cast<size_t>(n) * 8 + wave) * 8;  // [t][j] blocks of 64 lanes
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      uint16_t o[4];
      float sl[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = acc[t][j][r] + bias1[j], th = gelu_tanh(z);
        o[r] = bf16_bits(gelu_f(z, th));
        sl[r] = TRAIN ? gelu_grad(z, th) : 0.f;
      }
      store.put(grid, t, j, o);
      if constexpr (TRAIN) {
        tr.s1[(frag + 2 * t + j) * 64 + lane] = make_float4(sl[0], sl[1], sl[2], sl[3]);
        *reinterpret_cast<uint2*>(tr.a1 + (static_cast<size_t>(n) * kC1 + 16 * j + c16) * kP1 + 64 * wave + 16 * t + 4 * q) =
            pack4(o);
      }
      acc[t][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  lds_barrier();

  conv_products<false>(grid, GridBase(wave, lane), net.pack + net.l2.fwd, lane, acc);
  lds_barrier();  // the grid is free

  // gelu, then the 2x2x2 means, each summed z, y, x ascending from +0: an
  // even plane's lanes add their row's pair and the next row's (in lane +
  // 32), the odd plane above goes on from their sum
  float* sums = reinterpret_cast<float*>(grid);  // [Z 4][Y 4][X 4][32]
  float row2[4][2][4];                           // odd planes: this row's 4 values, then the next row's, per (t, j)
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float a[4], sl[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = acc[t][j][r] + bias2[j], th = gelu_tanh(z);
        a[r] = gelu_f(z, th);
        sl[r] = TRAIN ? gelu_grad(z, th) : 0.f;
      }
      if constexpr (TRAIN) tr.s2[(frag + 2 * t + j) * 64 + lane] = make_float4(sl[0], sl[1], sl[2], sl[3]);
#pragma unroll
      for (int r = 0; r < 4; ++r) row2[t][j][r] = a[r];
    }
  const int sum_at = ((wave >> 1) * 16 + 2 * (q & 1)) * 32 + c16;  // + (4 t + h) * 32 + 16 j
  auto pooled = [&](int t, int j, int h, float from) {
    const float a0 = row2[t][j][2 * h], a1 = row2[t][j][2 * h + 1];
    const float b0 = __shfl_xor(a0, 32), b1 = __shfl_xor(a1, 32);
    return (((from + a0) + a1) + b0) + b1;
  };
  if ((wave & 1) == 0)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float s = pooled(t, j, h, 0.f);
          if (q < 2) sums[sum_at + (4 * t + h) * 32 + 16 * j] = s;
        }
  lds_barrier();
  if ((wave & 1) == 1)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float s = pooled(t, j, h, sums[sum_at + (4 * t + h) * 32 + 16 * j]);
          const int zp = (wave >> 1) + 1, yp = t + 1, xp = 2 * (q & 1) + h + 1;
          if (q < 2)
            *reinterpret_cast<uint16_t*>(gridq + ((zp * kQ + yp) * kQ + xp) * 64 +
                                         (((2 * j + (c16 >> 3)) ^ swz4(yp)) << 4) + 2 * (c16 & 7)) = bf16_bits(0.125f * s);
        }
  lds_barrier();
  if (TRAIN && tid < 256) {
    const int p = tid >> 2, o = tid & 3, yp = ((p >> 2) & 3) + 1;
    const int at = (((p >> 4) + 1) * kQ + yp) * kQ + (p & 3) + 1;
    *reinterpret_cast<uint4*>(tr.p2 + (static_cast<size_t>(n) * kP2 + p) * kC2 + 8 * o) =
        *reinterpret_cast<const uint4*>(gridq + at * 64 + ((o ^ swz4(yp)) << 4));
  }

  // conv3: wave -> output tile w % 4, planes 2 (w / 4) and the next
  {
    const int nt = wave & 3, m0 = 2 * (wave >> 2);
    const uint16_t* w = net.pack + net.l3.fwd + nt * 512 + 8 * lane;
    const float bias = net.params[net.l3.b_off + 16 * nt + c16];
    int base[3];
#pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
      const int yp = (c16 >> 2) + dy;
      base[dy] = ((m0 * kQ + yp) * kQ + (c16 & 3)) * 64 + ((q ^ swz4(yp)) << 4);
    }
    f32x4_t c[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int kAhead = 6;
    bf16x8_t b[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) b[k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + 2048 * k));
#pragma unroll
    for (int k = 0; k < 27; ++k) {
      const int dz = k / 9, dy = (k / 3) % 3, dx = k % 3;
#pragma unroll
      for (int m = 0; m < 2; ++m)
        c[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(gridq + base[dy] + ((dz + m) * kQ * kQ + dx) * 64)),
            b[k % kAhead], c[m], 0, 0, 0);
      if (k + kAhead < 27)
        b[k % kAhead] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + 2048 * (k + kAhead)));
    }
    float* out = reinterpret_cast<float*>(grid) + 4096;  // [position 64][64], past the pooling sums
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      float sl[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = c[m][r] + bias, th = gelu_tanh(z);
        out[(16 * (m0 + m) + 4 * q + r) * kC3 + 16 * nt + c16] = gelu_f(z, th);
        sl[r] = TRAIN ? gelu_grad(z, th) : 0.f;
      }
      if constexpr (TRAIN)
        tr.s3[(static_cast<size_t>(n) * 16 + 4 * (m0 + m) + nt) * 64 + lane] = make_float4(sl[0], sl[1], sl[2], sl[3]);
    }
  }
  lds_barrier();
  if (tid < kC3) {  // positions in ascending order
    const float* in = reinterpret_cast<const float*>(grid) + 4096;
    float s = 0.f;
#pragma unroll 16
    for (int p = 0; p < kP2; ++p) s += in[p * kC3 + tid];
    feat[static_cast<size_t>(n) * kC3 + tid] = s * (1.0f / kP2);
  }
}

// One genome per workgroup: dLoss/dZ of conv3 (from the features' gradient),
// conv2 and conv1, each the gradient of the layer's output times the slope
// of gelu.  Input gradients are products over (kernel offset, output
// channel) of the shifted gradients, read from padded grids as in
// conv_features.  The 64-channel grid of conv3's gradient and the grid of
// conv2's share their LDS.
__global__ __launch_bounds__(512, 2) void conv_backward(ConvNet net, ConvTrain tr) {
  __shared__ __align__(16) unsigned char grid[64 * kVol];  // conv3's gradient (128 B per position), then conv2's
  __shared__ float dpool[kP2][kC2];
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x;
  const size_t frag = (static_cast<size_t>(n) * 8 + wave) * 8;
  {
    const int nt = wave & 3, m0 = 2 * (wave >> 2), o = 16 * nt + c16;
    const float df = tr.dfeat[static_cast<size_t>(n) * kC3 + o] * (1.0f / kP2);
    float4 sl[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) sl[m] = tr.s3[(static_cast<size_t>(n) * 16 + 4 * (m0 + m) + nt) * 64 + lane];
    zero_lds(grid, 128 * kVolQ, 512);
    lds_barrier();
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const float s[4] = {sl[m].x, sl[m].y, sl[m].z, sl[m].w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d = df * s[r];
        const int zp = m0 + m + 1, yp = q + 1, xp = r + 1;
        *reinterpret_cast<uint16_t*>(grid + ((zp * kQ + yp) * kQ + xp) * 128 + (((o >> 3) ^ swz4w(yp, xp)) << 4) +
                                     2 * (o & 7)) = bf16_bits(d);
        tr.d3[(static_cast<size_t>(n) * kP2 + 16 * (m0 + m) + 4 * q + r) * kC3 + o] = d;
      }
    }
  }
  lds_barrier();
  {  // wave -> plane w / 2, channels 16 (w % 2) ..; 54 slices: offset, half of the outputs
    const int mt = wave >> 1, nt = wave & 1;
    const uint16_t* w = net.pack + net.l3.bwd + nt * 512 + 8 * lane;
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
    constexpr int kAhead = 8;
    bf16x8_t b[kAhead];
#pragma unroll
    for (int s = 0; s < kAhead; ++s) b[s] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + 1024 * s));
#pragma unroll
    for (int s = 0; s < 54; ++s) {
      const int o = 26 - s / 2, dz = o / 9, dy = (o / 3) % 3, dx = o % 3;
      const int yp = (c16 >> 2) + dy, xp = (c16 & 3) + dx;
      const int at = (((mt + dz) * kQ + yp) * kQ + xp) * 128 + (((4 * (s & 1) + q) ^ swz4w(yp, xp)) << 4);
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(grid + at)), b[s % kAhead], c, 0, 0, 0);
      if (s + kAhead < 54)
        b[s % kAhead] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(w + 1024 * (s + kAhead)));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) dpool[16 * mt + 4 * q + r][16 * nt + c16] = c[r];
  }
  lds_barrier();
  zero_lds(grid, 64 * kVol, 512);
  lds_barrier();
  const GridStore store(wave, lane);
  auto leave = [&](int t, int j, const float (&d)[4], float4* s, uint16_t* dT, uint16_t (&o)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = bf16_bits(d[r]);
    s[(frag + 2 * t + j) * 64 + lane] = make_float4(d[0], d[1], d[2], d[3]);
    *reinterpret_cast<uint2*>(dT + (static_cast<size_t>(n) * 32 + 16 * j + c16) * kP1 + 64 * wave + 16 * t + 4 * q) = pack4(o);
  };
  float4 sl[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) sl[t][j] = tr.s2[(frag + 2 * t + j) * 64 + lane];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float s[4] = {sl[t][j].x, sl[t][j].y, sl[t][j].z, sl[t][j].w};
      float d[4];
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        d[r] = 0.125f * dpool[((wave >> 1) * 4 + t) * 4 + 2 * (q & 1) + (r >> 1)][16 * j + c16] * s[r];
      leave(t, j, d, tr.s2, tr.d2, o);
      store.put(grid, t, j, o);
    }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) sl[t][j] = tr.s1[(frag + 2 * t + j) * 64 + lane];
  lds_barrier();
  f32x4_t acc[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[t][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  conv_products<true>(grid, GridBase(wave, lane), net.pack + net.l2.bwd, lane, acc);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float s[4] = {sl[t][j].x, sl[t][j].y, sl[t][j].z, sl[t][j].w};
      float d[4];
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) d[r] = acc[t][j][r] * s[r];
      leave(t, j, d, tr.s1, tr.d1, o);
    }
}

// Weight and bias gradients of the convolutions: blockIdx.y = role, x =
// split.  A layer's rows (genome, position) reduce in kSplit runs of M /
// kSplit rows, each in ascending slices of 32; partials go to part[split]
// at the parameters' offsets, `stride` apart.  Runs of the 8^3 layers are
// whole rows of x (8 positions, an octet: the 8 k values of a lane), so
// operands are octets of the transposed gradients and activations in LDS; a
// lane's three x offsets are its octet shifted by one value in registers.
enum { kRoleConv2 = 0, kRoleConv3 = 3, kRoleConv1 = 6, kRoleBias2 = 7, kRoleBias1 = 8, kRoles = 9 };
constexpr int kOctPitch = 65 * 16;  // bytes per channel of 64 octets: an odd count of 16-byte units

// Bias gradient of an 8^3 layer from its fp32 gradient in accumulator order:
// the split's rows in 16 groups (row mod 16 from its start), each summed in
// ascending order, then the groups.
__device__ __forceinline__ void conv_bias(const float4* d, int B, int split, float* part, unsigned char* lds) {
  float (*acc)[32] = reinterpret_cast<float (*)[32]>(lds);
  const int tid = threadIdx.x, r0 = 8 * B * split, r1 = r0 + 8 * B;
  if (tid < 128) {
    const int j = tid >> 6, lane = tid & 63, q = lane >> 4;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    // 16-row tiles; a run starts and ends at a multiple of 8 rows, so a
    // lane's four rows are in it or not together
    const int t0 = r0 >> 4, t1 = (r1 + 15) >> 4;
    // the loads carry no condition, so 16 of them are in flight together;
    // adding +0 for a row outside leaves a sum that started at +0 unchanged
    for (int t = t0; t < t1; t += 16) {
      float4 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = d[(static_cast<size_t>(min(t + u, t1 - 1)) * 2 + j) * 64 + lane];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int row = 16 * (t + u) + 4 * q;
        const bool in = row >= r0 && row < r1;
        s[0] += in ? v[u].x : 0.f;
        s[1] += in ? v[u].y : 0.f;
        s[2] += in ? v[u].z : 0.f;
        s[3] += in ? v[u].w : 0.f;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[(4 * q + r - r0) & 15][16 * j + (lane & 15)] = s[r];
  }
  lds_barrier();
  if (tid < 32) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += acc[k][tid];
    part[tid] = t;
  }
}

// Stages octets [c0, c0 + count) of a transposed gradient [genome][32][64
// octets] into LDS [32][kOctPitch], zeros past count.
struct OctetStage {
  uint4 v[4];
  __device__ void load(const uint16_t* d, int c0, int count) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = threadIdx.x + 512 * i, o = u >> 6, e = u & 63, id = c0 + min(e, count - 1);
      v[i] = *reinterpret_cast<const uint4*>(d + ((static_cast<size_t>(id >> 6) * 32 + o) * 64 + (id & 63)) * 8);
    }
  }
  __device__ void put(unsigned char* lds, int count) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = threadIdx.x + 512 * i, o = u >> 6, e = u & 63;
      *reinterpret_cast<uint4*>(lds + o * kOctPitch + e * 16) = e < count ? v[i] : make_uint4(0u, 0u, 0u, 0u);
    }
  }
};

__device__ __forceinline__ void wgrad_conv2(const ConvTrain& tr, int B, int split, int dz, float* part,
                                            unsigned char* lds) {
  unsigned char* sd = lds;                       // gradient octets
  unsigned char* sx = lds + 32 * kOctPitch;      // conv1 outputs of two genomes, by parity
  unsigned char* zero = sx + 64 * kOctPitch;     // 16 bytes of zeros
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dy = (wave >> 1) - 1, ct = wave & 1;  // waves 0 .. 5
  const int begin = B * split, end = begin + B;   // octets
  if (tid == 0) *reinterpret_cast<uint4*>(zero) = make_uint4(0u, 0u, 0u, 0u);
  f32x4_t acc[3][2];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[i][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  OctetStage d, x;
  auto genome = [&](int g) { x.load(tr.a1 + static_cast<size_t>(g) * 32 * kP1, 0, 64); };
  auto put_genome = [&](int g) { x.put(sx + (g & 1) * 32 * kOctPitch, 64); };
  // the first chunk's genomes, at most two
  int loaded = begin >> 6;
  genome(loaded);
  d.load(tr.d2, begin, min(64, end - begin));
  put_genome(loaded);
  if (((min(begin + 64, end) - 1) >> 6) > loaded) {
    genome(++loaded);
    put_genome(loaded);
  }
  bool fresh = false;  // x holds the next chunk's new genome
  for (int c0 = begin; c0 < end; c0 += 64) {
    const int count = min(64, end - c0);
    d.put(sd, count);
    if (fresh) put_genome(loaded);
    lds_barrier();
    fresh = false;
    if (c0 + 64 < end) {
      const int next = min(64, end - c0 - 64);
      d.load(tr.d2, c0 + 64, next);
      if (((c0 + 64 + next - 1) >> 6) > loaded) {  // at most one genome further
        genome(++loaded);
        fresh = true;
      }
    }
    if (wave < 6)
#pragma unroll 4
      for (int e0 = 0; e0 < count; e0 += 4) {
        const int e = e0 + q, id = c0 + e, zz = ((id >> 3) & 7) + dz, yy = (id & 7) + dy;
        const bool in = e < count && zz >= 0 && zz < 8 && yy >= 0 && yy < 8;
        const unsigned char* xp =
            in ? sx + ((id >> 6) & 1) * 32 * kOctPitch + (16 * ct + c16) * kOctPitch + (8 * zz + yy) * 16 : zero;
        const uint4 v = *reinterpret_cast<const uint4*>(xp);
        bf16x8_t a[2];
#pragma unroll
        for (int m = 0; m < 2; ++m)
          a[m] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(sd + (16 * m + c16) * kOctPitch + e * 16));
        const uint32_t s01 = __builtin_amdgcn_alignbit(v.y, v.x, 16), s12 = __builtin_amdgcn_alignbit(v.z, v.y, 16),
                       s23 = __builtin_amdgcn_alignbit(v.w, v.z, 16);
        const uint4 b[3] = {make_uint4(v.x << 16, s01, s12, s23), v, make_uint4(s01, s12, s23, v.w >> 16)};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int m = 0; m < 2; ++m)
            acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], __builtin_bit_cast(bf16x8_t, b[i]), acc[i][m], 0, 0, 0);
      }
    lds_barrier();
  }
  if (wave < 6)
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(16 * m + 4 * q + r) * kK2 + ((dz + 1) * 9 + (dy + 1) * 3 + i) * kC1 + 16 * ct + c16] = acc[i][m][r];
}

// The one-hot genome's columns: column 16 nt + c16 is material c at kernel
// offset k; its octet is 8 voxels of a padded row compared with c, byte by
// byte (a byte of 0x80 - (voxel ^ c) keeps its top bit only where equal),
// spread to bf16 ones (0x3f80).
__device__ __forceinline__ void wgrad_conv1(const ConvNet& net, const ConvTrain& tr, int B, int split, float* part,
                                            unsigned char* lds) {
  unsigned char* sd = lds;
  unsigned char* sg = lds + 32 * kOctPitch;  // two genomes by parity: 10 x 10 rows of 16 bytes, x at byte 1 + x
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int begin = B * split, end = begin + B;
  constexpr int kSlot = kP * kP * 16;
  for (int i = tid; i < 2 * kSlot / 4; i += 512) reinterpret_cast<uint32_t*>(sg)[i] = 0x01010101u * kNoMaterial;
  // wave w: column tile w, both halves of the outputs; tile 8's halves on
  // waves 0 and 1
  constexpr int kT = 2;
  int row_off[kT], shift[kT];
  uint32_t want[kT];
#pragma unroll
  for (int i = 0; i < kT; ++i) {
    const int col = min(16 * (i == 0 ? wave : 8) + c16, kK1 - 1), k = col / kC0, c = col - k * kC0;
    row_off[i] = ((k / 9) * kP + (k / 3) % 3) * 16;
    shift[i] = k % 3;
    want[i] = 0x01010101u * c;
  }
  f32x4_t acc[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  OctetStage d;
  lds_barrier();
  auto get_genome = [&](int g) {
    return net.genomes[static_cast<size_t>(net.idx ? net.idx[g] : g) * kP1 + tid];
  };
  auto put_genome = [&](int g, uint32_t v) {
    sg[(g & 1) * kSlot + ((((tid >> 6) + 1) * kP + ((tid >> 3) & 7) + 1) * 16) + 1 + (tid & 7)] =
        static_cast<uint8_t>(clean_voxel(v));
  };
  // a chunk of 64 octets reaches at most one genome past those in LDS: the
  // next one is on its way while a chunk is worked on
  int loaded = begin >> 6;
  const int last = (end - 1) >> 6;
  d.load(tr.d1, begin, min(64, end - begin));
  put_genome(loaded, get_genome(loaded));
  uint32_t next = get_genome(min(loaded + 1, last));
  for (int c0 = begin; c0 < end; c0 += 64) {
    const int count = min(64, end - c0);
    d.put(sd, count);
    if (((c0 + count - 1) >> 6) > loaded) {
      ++loaded;
      put_genome(loaded, next);
      next = get_genome(min(loaded + 1, last));
    }
    lds_barrier();
    if (c0 + 64 < end) d.load(tr.d1, c0 + 64, min(64, end - c0 - 64));
#pragma unroll 4
    for (int e0 = 0; e0 < count; e0 += 4) {
      const int e = e0 + q, id = c0 + min(e, count - 1);
      const unsigned char* rows = sg + ((id >> 6) & 1) * kSlot + (((id >> 3) & 7) * kP + (id & 7)) * 16;
      bf16x8_t a[2];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        a[m] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(sd + (16 * m + c16) * kOctPitch + e * 16));
      auto column = [&](int i) {
        const uint4 v = *reinterpret_cast<const uint4*>(rows + row_off[i]);
        uint4 o;
        uint32_t* ow = &o.x;
        const uint32_t w[2] = {__builtin_amdgcn_alignbyte(v.y, v.x, shift[i]), __builtin_amdgcn_alignbyte(v.z, v.y, shift[i])};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t m = (0x80808080u - (w[h] ^ want[i])) & 0x80808080u, hi = (m >> 1) - (m >> 7);
          ow[2 * h] = __builtin_amdgcn_perm(hi, m, 0x05010400u);
          ow[2 * h + 1] = __builtin_amdgcn_perm(hi, m, 0x07030602u);
        }
        return __builtin_bit_cast(bf16x8_t, o);
      };
      const bf16x8_t b = column(0);
#pragma unroll
      for (int m = 0; m < 2; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b, acc[m], 0, 0, 0);
      if (wave < 2) acc[2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wave ? a[1] : a[0], column(1), acc[2], 0, 0, 0);
    }
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int m = i < 2 ? i : wave, col = 16 * (i < 2 ? wave : 8) + c16;
    if ((i < 2 || wave < 2) && col < kK1)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(16 * m + 4 * q + r) * kK1 + col] = acc[i][r];
  }
}

// conv3: runs of B rows start anywhere, so the gradient is transposed into
// LDS from the run's start (64 rows at a time) and the pooled activations
// (two genomes by parity, channel-major with a border) are gathered value by
// value.  The group dz = -1 also sums the bias from the fp32 values as it
// stages them.
__device__ __forceinline__ void wgrad_conv3(const ConvTrain& tr, int B, int split, int dz, float* part, float* part_b,
                                            unsigned char* lds) {
  constexpr int kPitchD = 144, kPitchX = 2 * kVolQ, kSlot = 32 * kPitchX;
  unsigned char* sd = lds;                                                    // [64 outputs][72 rows]
  unsigned char* sx = lds + 64 * kPitchD;                                     // [2][32 channels][216]
  float (*sb)[64] = reinterpret_cast<float (*)[64]>(sx + 2 * kSlot);          // bias sums [16][64]
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dy = (wave >> 1) - 1, ct = wave & 1;  // waves 0 .. 5
  const int begin = B * split, end = begin + B;
  const int c = tid & 63, g0 = tid >> 6;
  f32x4_t acc[3][4];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[i][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float bias[2] = {0.f, 0.f};
  zero_lds(sx, 2 * kSlot, 512);
  lds_barrier();
  const int last = (end - 1) >> 6;
  auto get_genome = [&](int g) {  // threads 0 .. 255: 8 channels of a position
    return *reinterpret_cast<const uint4*>(tr.p2 + (static_cast<size_t>(g) * kP2 + ((tid >> 2) & 63)) * kC2 + 8 * (tid & 3));
  };
  auto put_genome = [&](int g, uint4 w) {
    if (tid >= 256) return;
    const int p = tid >> 2, o = tid & 3;
    const int at = (((p >> 4) + 1) * kQ + ((p >> 2) & 3) + 1) * kQ + (p & 3) + 1;
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 8; ++i)
      *reinterpret_cast<uint16_t*>(sx + (g & 1) * kSlot + (8 * o + i) * kPitchX + 2 * at) =
          static_cast<uint16_t>(i & 1 ? u[i >> 1] >> 16 : u[i >> 1]);
  };
  float v[8];
  auto get_rows = [&](int c0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = tr.d3[static_cast<size_t>(min(c0 + g0 + 8 * i, end - 1)) * kC3 + c];
  };
  // as in wgrad_conv1: the next rows and genome travel while a chunk is
  // worked on
  int loaded = begin >> 6;
  get_rows(begin);
  put_genome(loaded, get_genome(loaded));
  uint4 next = get_genome(min(loaded + 1, last));
  for (int c0 = begin; c0 < end; c0 += 64) {
    const int count = min(64, end - c0);
    if (((c0 + count - 1) >> 6) > loaded) {
      ++loaded;
      put_genome(loaded, next);
      next = get_genome(min(loaded + 1, last));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = g0 + 8 * i;
      const bool in = row < count;
      if (in) bias[i & 1] += v[i];
      *reinterpret_cast<uint16_t*>(sd + c * kPitchD + 2 * row) = in ? bf16_bits(v[i]) : uint16_t(0);
    }
    get_rows(min(c0 + 64, end - 1));
    lds_barrier();
    if (wave < 6)
      for (int e0 = 0; 8 * e0 < count; e0 += 4) {
        bf16x8_t a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
          a[m] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u16x8_t*>(sd + (16 * m + c16) * kPitchD + (e0 + q) * 16));
        const unsigned char* at[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int row = c0 + min(8 * (e0 + q) + i, count - 1);
          at[i] = sx + ((row >> 6) & 1) * kSlot + (16 * ct + c16) * kPitchX +
                  2 * (((((row >> 4) & 3) + 1 + dz) * kQ + ((row >> 2) & 3) + 1 + dy) * kQ + (row & 3));
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          u16x8_t b;
#pragma unroll
          for (int k = 0; k < 8; ++k) b[k] = *reinterpret_cast<const uint16_t*>(at[k] + 2 * i);
#pragma unroll
          for (int m = 0; m < 4; ++m)
            acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], __builtin_bit_cast(bf16x8_t, b), acc[i][m], 0, 0, 0);
        }
      }
    lds_barrier();
  }
  if (wave < 6)
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(16 * m + 4 * q + r) * kK3 + ((dz + 1) * 9 + (dy + 1) * 3 + i) * kC2 + 16 * ct + c16] = acc[i][m][r];
  if (dz == -1) {
    sb[g0][c] = bias[0];
    sb[g0 + 8][c] = bias[1];
    lds_barrier();
    if (tid < 64) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) t += sb[k][tid];
      part_b[tid] = t;
    }
  }
}

__global__ __launch_bounds__(512) void conv_wgrad(ConvNet net, ConvTrain tr, int B, float* __restrict__ part,
                                                  size_t stride) {
  __shared__ __align__(16) unsigned char lds[96 * kOctPitch + 16];
  const int split = blockIdx.x, role = blockIdx.y;
  float* out = part + split * stride;
  if (role < kRoleConv3) wgrad_conv2(tr, B, split, role - kRoleConv2 - 1, out + net.l2.w_off, lds);
  else if (role < kRoleConv1)
    wgrad_conv3(tr, B, split, role - kRoleConv3 - 1, out + net.l3.w_off, out + net.l3.b_off, lds);
  else if (role == kRoleConv1) wgrad_conv1(net, tr, B, split, out + net.l1.w_off, lds);
  else if (role == kRoleBias2) conv_bias(tr.s2, B, split, out + net.l2.b_off, lds);
  else conv_bias(tr.s1, B, split, out + net.l1.b_off, lds);
}

// The convolutions' parameters: each gradient summed from its partials in
// ascending split order, then Adam's update and the packed weights (ADAM),
// or the gradient itself.
template <bool ADAM>
__global__ __launch_bounds__(256) void conv_update(ConvNet net, const float* __restrict__ part, int n, AdamArgs ad,
                                                   float* __restrict__ grads) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float p = 0.f, m = 0.f, v = 0.f;
  if constexpr (ADAM) {
    p = ad.p[i];
    m = ad.m[i];
    v = ad.v[i];
  }
  float g = 0.f;
#pragma unroll 32
  for (int k = 0; k < kSplit; ++k) g += part[static_cast<size_t>(k) * n + i];
  if constexpr (!ADAM) {
    grads[i] = g;
    return;
  }
  adam_update(g, p, m, v, ad.lr, ad.b1, ad.b2, ad.eps, ad.bc1, ad.bc2);
  ad.p[i] = p;
  ad.m[i] = m;
  ad.v[i] = v;
  const PackedLayer& l = i < net.l2.w_off ? net.l1 : i < net.l3.w_off ? net.l2 : net.l3;
  const int e = i - l.w_off;
  if (e < l.out * l.in) pack_store(l, ad.pack, e / l.in, e % l.in, p);
}

unsigned blocks_for(size_t n) { return static_cast<unsigned>((n + 255) / 256); }

struct LayerShape {
  int out, in;  // weight [out x in], bias [out]
};
constexpr LayerShape kLayers[] = {{kC1, kK1}, {kC2, kK2}, {kC3, kK3}, {kH, kC3}, {kH, kH}, {1, kH}};
constexpr int kNL = 6, kHeadL = 3;

}  // namespace

struct mh_cnn {
  int device = 0;
  hipStream_t stream = nullptr;
  size_t w_off[kNL] = {}, b_off[kNL] = {};
  size_t n_params = 0;
  size_t n_conv = 0;          // parameters of the convolutions (they come first)
  PackedLayer conv[3];
  DenseShape head{};
  Dev<float> params, grads, m, v, part;
  Dev<uint16_t> pack;         // bf16 weights in the kernels' operand order
  int cap = 0;
  Dev<uint8_t> g;
  Dev<float> feat, y, t;
  // training, per genome of a batch
  Dev<float4> s1, s2, s3;
  Dev<uint16_t> a1, p2, d1, d2;
  Dev<float> d3, dfeat, terms;
  Dev<uint16_t> hx[3], hd[3];  // the head's weight-gradient operands
  Dev<float> hdelta[3];
  Dev<float> epoch_terms;  // loss terms of every batch of a training run's last epoch
  Dev<uint8_t> data_g;
  Dev<float> data_t;
  Dev<int> idx;
  int adam_t = 0;
  ~mh_cnn() {
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

void ensure(mh_cnn* net, int B) {
  if (B <= net->cap) return;
  const size_t n = B, R1 = n * kP1, R2 = n * kP2;
  net->g.ensure(R1);
  net->t.ensure(n);
  net->feat.ensure(n * kC3);
  net->s1.ensure(R1 * kC1 / 4);
  net->s2.ensure(R1 * kC2 / 4);
  net->s3.ensure(R2 * kC3 / 4);
  net->a1.ensure(R1 * kC1);
  net->p2.ensure(R2 * kC2);
  net->d1.ensure(R1 * kC1);
  net->d2.ensure(R1 * kC2);
  net->d3.ensure(R2 * kC3);
  net->dfeat.ensure(n * kC3);
  net->terms.ensure(n);
  // the head's operands hold whole slices of 32 rows per split
  const size_t rows = n + 32 * kSplit;
  for (int l = 0; l < 3; l++) {
    net->hx[l].ensure(rows * net->head.layer[l].in);
    net->hd[l].ensure(rows * ((net->head.layer[l].out + 15) / 16 * 16));
    net->hdelta[l].ensure(n * net->head.layer[l].out);
  }
  net->cap = B;
}

ConvNet conv_net(const mh_cnn* net, const uint8_t* genomes, const int* idx) {
  return ConvNet{net->conv[0], net->conv[1], net->conv[2], net->params.p, net->pack.p, genomes, idx};
}

// y [B] of the genomes on the device (chunks of up to 4096: 16-row tiles in
// the head, as mh_mlp_forward's)
void forward(mh_cnn* net, const uint8_t* genomes, int B, float* feat, float* y) {
  hipLaunchKernelGGL((conv_features<false>), dim3(B), dim3(512), 0, net->stream, conv_net(net, genomes, nullptr), feat,
                     ConvTrain{});
  launch_dense_net_of<kHeadL, 1, false>(net->head, net->params.p, net->pack.p, feat, B, y, DenseTrain{}, net->stream);
  hipcheck(hipGetLastError(), "cnn forward");
}

// Loss terms (into `terms`, B floats on the device) and gradients of a batch
// whose row r is genome idx[r] and target idx[r] (null: r): into net->grads,
// or with `adam` straight into the parameters.
void loss_backward_to(mh_cnn* net, const uint8_t* genomes, const float* target, const int* idx, int B, float* terms,
                      const AdamArgs* adam) {
  hipStream_t s = net->stream;
  const ConvNet cn = conv_net(net, genomes, idx);
  ConvTrain ct{net->s1.p, net->s2.p, net->s3.p, net->a1.p, net->p2.p, net->d1.p, net->d2.p, net->d3.p, net->dfeat.p};
  hipLaunchKernelGGL((conv_features<true>), dim3(B), dim3(512), 0, s, cn, net->feat.p, ct);
  DenseTrain tr{};
  tr.rs = row_splits(B, kSplit);
  tr.t_idx = idx;
  tr.target = target;
  tr.inv_b = 1.0f / B;
  tr.terms = terms;
  tr.dx = net->dfeat.p;
  for (int l = 0; l < 3; l++) {
    tr.X[l] = net->hx[l].p;
    tr.D[l] = net->hd[l].p;
    tr.delta[l] = net->hdelta[l].p;
  }
  launch_dense_net_of<kHeadL, 1, true>(net->head, net->params.p, net->pack.p, net->feat.p, B, nullptr, tr, s);
  hipLaunchKernelGGL(conv_backward, dim3(B), dim3(512), 0, s, cn, ct);
  const AdamArgs ad = adam ? *adam : AdamArgs{};
  if (adam) launch_dense_wgrad_of<kHeadL, 1, 8, true>(net->head, tr, ad, nullptr, s);
  else launch_dense_wgrad_of<kHeadL, 1, 8, false>(net->head, tr, ad, net->grads.p, s);
  hipLaunchKernelGGL(conv_wgrad, dim3(kSplit, kRoles), dim3(512), 0, s, cn, ct, B, net->part.p, net->n_conv);
  const int n = static_cast<int>(net->n_conv);
  if (adam)
    hipLaunchKernelGGL((conv_update<true>), dim3(blocks_for(n)), dim3(256), 0, s, cn, net->part.p, n, ad,
                       static_cast<float*>(nullptr));
  else
    hipLaunchKernelGGL((conv_update<false>), dim3(blocks_for(n)), dim3(256), 0, s, cn, net->part.p, n, ad, net->grads.p);
  hipcheck(hipGetLastError(), "cnn training step");
}

// The packed weights of every layer from the fp32 parameters.
void refresh_weights(mh_cnn* net) {
  PackList list{kNL, {}};
  static_assert(kNL <= kPackLayers, "every layer in one launch");
  for (int l = 0; l < kNL; l++) list.layer[l] = l < 3 ? net->conv[l] : net->head.layer[l - 3];
  launch_pack(list, net->params.p, net->pack.p, nullptr, net->stream);
  hipcheck(hipGetLastError(), "weights");
}

// A batch's loss from its B terms on the host: their sum in order / B.
float batch_loss(const float* terms, int B) {
  double sum = 0.0;
  for (int i = 0; i < B; i++) sum += terms[i];
  return static_cast<float>(sum / B);
}

int fail(const mh::Error& e) {
  mh::set_error(e.what());
  return e.code;
}

}  // namespace

extern "C" {

int mh_cnn_create(int device, uint64_t seed, mh_cnn** out) {
  try {
    if (!out) throw mh::Error(MH_ERR_ARG, "null argument");
    auto net = std::make_unique<mh_cnn>();
    net->device = device;
    hipcheck(hipSetDevice(device), "hipSetDevice");
    hipcheck(hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking), "stream");
    size_t off = 0;
    int at = 0;
    for (int l = 0; l < kNL; l++) {
      net->w_off[l] = off;
      off += static_cast<size_t>(kLayers[l].out) * kLayers[l].in;
      net->b_off[l] = off;
      off += kLayers[l].out;
      PackedLayer& p = l < 3 ? net->conv[l] : net->head.layer[l - 3];
      p.out = kLayers[l].out;
      p.in = kLayers[l].in;
      p.c = l < 3 ? kLayers[l].in / 27 : kLayers[l].in;
      p.w_off = static_cast<int>(net->w_off[l]);
      p.b_off = static_cast<int>(net->b_off[l]);
      at = pack_layout(p, at);
    }
    net->n_params = off;
    net->n_conv = net->w_off[3];
    net->head.L = kHeadL;
    net->head.zero = at;
    at += 8;
    // He-uniform weights (bound sqrt(6 / fan_in)), zero biases
    std::mt19937_64 rng(seed);
    std::vector<float> p(off, 0.f);
    for (int l = 0; l < kNL; l++) {
      std::uniform_real_distribution<float> u(-std::sqrt(6.0f / kLayers[l].in), std::sqrt(6.0f / kLayers[l].in));
      for (size_t i = 0; i < static_cast<size_t>(kLayers[l].out) * kLayers[l].in; i++) p[net->w_off[l] + i] = u(rng);
    }
    net->params.ensure(off);
    net->grads.ensure(off);
    net->m.ensure(off);
    net->v.ensure(off);
    net->pack.ensure(at);
    net->part.ensure(static_cast<size_t>(kSplit) * net->n_conv);
    hipLaunchKernelGGL(fill_zero_u16, dim3(blocks_for(at)), dim3(256), 0, net->stream, net->pack.p, at);
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

int mh_cnn_destroy(mh_cnn* net) {
  delete net;
  return MH_OK;
}

int mh_cnn_param_count(const mh_cnn* net) { return net ? static_cast<int>(net->n_params) : MH_ERR_ARG; }

int mh_cnn_get_params(const mh_cnn* net, float* out) {
  try {
    if (!net || !out) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    hipcheck(hipMemcpy(out, net->params.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost), "D2H");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_cnn_set_params(mh_cnn* net, const float* in) {
  try {
    if (!net || !in) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    hipcheck(hipMemcpy(net->params.p, in, net->n_params * sizeof(float), hipMemcpyHostToDevice), "H2D");
    std::vector<float> zeros(net->n_params, 0.f);
    hipcheck(hipMemcpy(net->m.p, zeros.data(), net->n_params * sizeof(float), hipMemcpyHostToDevice), "H2D");
    hipcheck(hipMemcpy(net->v.p, zeros.data(), net->n_params * sizeof(float), hipMemcpyHostToDevice), "H2D");
    net->adam_t = 0;
    refresh_weights(net);
    hipcheck(hipStreamSynchronize(net->stream), "set params");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_cnn_forward(mh_cnn* net, const uint8_t* genomes, int n, float* y) {
  try {
    if (!net || n < 0 || (n > 0 && (!genomes || !y))) throw mh::Error(MH_ERR_ARG, "null argument");
    if (n == 0) return MH_OK;
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    // genomes go up in pieces, each followed by its kernels, so the host
    // stages a piece while the previous one is scored; results come back in
    // one copy per round
    const int chunk = 4096, round = 16 * chunk;
    net->data_g.ensure(static_cast<size_t>(std::min(n, round)) * kP1);
    net->feat.ensure(static_cast<size_t>(std::min(n, chunk)) * kC3);
    net->y.ensure(std::min(n, round));
    for (int r0 = 0; r0 < n; r0 += round) {
      const int rows = std::min(round, n - r0);
      for (int b0 = 0; b0 < rows; b0 += chunk) {
        const int B = std::min(chunk, rows - b0);
        uint8_t* g = net->data_g.p + static_cast<size_t>(b0) * kP1;
        hipcheck(hipMemcpyAsync(g, genomes + static_cast<size_t>(r0 + b0) * kP1, static_cast<size_t>(B) * kP1,
                                hipMemcpyHostToDevice, net->stream), "H2D");
        forward(net, g, B, net->feat.p, net->y.p + b0);
      }
      hipcheck(hipMemcpyAsync(y + r0, net->y.p, rows * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
    }
    hipcheck(hipStreamSynchronize(net->stream), "sync");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_cnn_loss_grad(mh_cnn* net, const uint8_t* genomes, const float* target, int n, float* loss, float* grad) {
  try {
    if (!net || !genomes || !target || n < 1) throw mh::Error(MH_ERR_ARG, "null argument");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    ensure(net, n);
    hipcheck(hipMemcpyAsync(net->g.p, genomes, static_cast<size_t>(n) * kP1, hipMemcpyHostToDevice, net->stream),
             "H2D");
    hipcheck(hipMemcpyAsync(net->t.p, target, n * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
    loss_backward_to(net, net->g.p, net->t.p, nullptr, n, net->terms.p, nullptr);
    std::vector<float> terms(n);
    hipcheck(hipMemcpyAsync(terms.data(), net->terms.p, n * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
    hipcheck(hipStreamSynchronize(net->stream), "sync");
    if (loss) *loss = batch_loss(terms.data(), n);
    if (grad) hipcheck(hipMemcpy(grad, net->grads.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost), "D2H");
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

int mh_cnn_train(mh_cnn* net, const uint8_t* genomes, const float* target, int n, int batch, int n_epochs, float lr,
                 uint64_t seed, float* final_loss) {
  try {
    if (!net || !genomes || !target || n < 1 || batch < 1 || n_epochs < 0) throw mh::Error(MH_ERR_ARG, "bad arguments");
    hipcheck(hipSetDevice(net->device), "hipSetDevice");
    batch = std::min(batch, n);
    ensure(net, batch);
    net->data_g.ensure(static_cast<size_t>(n) * kP1);
    net->data_t.ensure(n);
    net->idx.ensure(n);
    hipcheck(hipMemcpyAsync(net->data_g.p, genomes, static_cast<size_t>(n) * kP1, hipMemcpyHostToDevice,
                            net->stream), "H2D");
    hipcheck(hipMemcpyAsync(net->data_t.p, target, n * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
    std::mt19937_64 rng(seed);
    std::vector<int> perm(n);
    // the last epoch keeps every batch's loss terms on the device, so no
    // batch waits for a copy to the host; they are summed after the loop
    const int n_batches = n / batch;
    net->epoch_terms.ensure(static_cast<size_t>(n_batches) * batch);
    int batches = 0;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int ep = 0; ep < n_epochs; ep++) {
      for (int i = 0; i < n; i++) perm[i] = i;
      std::shuffle(perm.begin(), perm.end(), rng);
      hipcheck(hipMemcpyAsync(net->idx.p, perm.data(), n * sizeof(int), hipMemcpyHostToDevice, net->stream), "H2D");
      const bool last = ep == n_epochs - 1;
      for (int b0 = 0; b0 + batch <= n; b0 += batch) {
        net->adam_t++;
        const float bc1 = 1.f - std::pow(b1, static_cast<float>(net->adam_t));
        const float bc2 = 1.f - std::pow(b2, static_cast<float>(net->adam_t));
        const AdamArgs adam{net->params.p, net->m.p, net->v.p, net->pack.p, lr, b1, b2, eps, bc1, bc2};
        loss_backward_to(net, net->data_g.p, net->data_t.p, net->idx.p + b0, batch,
                         last ? net->epoch_terms.p + static_cast<size_t>(batches) * batch : net->terms.p, &adam);
        if (last) batches++;
      }
    }
    // the last epoch's mean of the batch losses
    std::vector<float> terms(static_cast<size_t>(batches) * batch);
    if (batches)
      hipcheck(hipMemcpyAsync(terms.data(), net->epoch_terms.p, terms.size() * sizeof(float),
                              hipMemcpyDeviceToHost, net->stream), "D2H");
    hipcheck(hipStreamSynchronize(net->stream), "sync");
    double epoch_loss = 0.0;
    for (int bi = 0; bi < batches; bi++) epoch_loss += batch_loss(terms.data() + static_cast<size_t>(bi) * batch, batch);
    if (batches) epoch_loss /= batches;
    if (final_loss) *final_loss = static_cast<float>(epoch_loss);
    return MH_OK;
  } catch (const mh::Error& e) {
    return fail(e);
  }
}

}  // extern "C"
