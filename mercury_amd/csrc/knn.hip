// knn.hip -- K nearest neighbours of every mass of every robot, on the GPU.
//
// Replaces Triangulation::KNN (common/evolvables/knn.cu:62-144: dense M x M
// distance matrix + segmented radix sort per row).  Robots of up to 2048
// masses, from 6 neighbours on (16 under 64 masses): one wave per query, the
// robot's positions in the wave's registers; otherwise one lane per query, a
// scan over LDS tiles.  Distances are sqrtf(dx*dx + (dy*dy + dz*dz)) (Eigen's
// Vector3f::norm order, as KNN_CPU computes them, knn.cu:147-158); a zero
// distance -- the mass itself or a coincident mass -- counts as +inf
// (knn.cu:166-167); equal distances keep the lower index first, the order
// the reference's stable radix sort of index-ordered rows produces.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "mercury_hip.h"
#include "mh_internal.h"

namespace {

constexpr int kQueryBlock = 256;
constexpr int kTile = 1024;
constexpr int kMaxK = 32;

struct KnnTile {
  uint32_t mass_begin;  // robot's first mass (global)
  uint32_t n_mass;      // robot's mass count
  uint32_t query0;      // first query mass of this workgroup (robot-local)
  uint32_t out_begin;   // first output row (global mass index)
};

__global__ __launch_bounds__(kQueryBlock) void knn_tiles(const float* __restrict__ pos,
                                                         const KnnTile* __restrict__ tiles,
                                                         int K, uint16_t* __restrict__ nbr,
                                                         float* __restrict__ dist) {
  __shared__ float sx[kTile], sy[kTile], sz[kTile];
  const KnnTile t = tiles[blockIdx.x];
  const int q = static_cast<int>(t.query0) + static_cast<int>(threadIdx.x);
  const bool active = q < static_cast<int>(t.n_mass);
  float qx = 0.f, qy = 0.f, qz = 0.f;
  if (active) {
    const size_t g = 3u * (static_cast<size_t>(t.mass_begin) + q);
    qx = pos[g];
    qy = pos[g + 1];
    qz = pos[g + 2];
  }
  float bd[kMaxK];
  int bi[kMaxK];
#pragma unroll
  for (int k = 0; k < kMaxK; ++k) {
    bd[k] = INFINITY;
    bi[k] = 0x7fffffff;
  }
  float worst = INFINITY;  // bd[K - 1], kept in its own register
  for (int base = 0; base < static_cast<int>(t.n_mass); base += kTile) {
    const int n = min(kTile, static_cast<int>(t.n_mass) - base);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kQueryBlock) {
      const size_t g = 3u * (static_cast<size_t>(t.mass_begin) + base + i);
      sx[i] = pos[g];
      sy[i] = pos[g + 1];
      sz[i] = pos[g + 2];
    }
    __syncthreads();
    for (int c = 0; c < n; ++c) {
      const float dx = qx - sx[c], dy = qy - sy[c], dz = qz - sz[c];
      const float yz = dy * dy + dz * dz;
      float d = sqrtf(dx * dx + yz);
      if (d == 0.0f) d = INFINITY;
      // rows are ranked by (distance, index) and candidates arrive in index
      // order, so a candidate enters only if strictly closer than the K-th
      if (active && d < worst) {
        float cd = d;
        int ci = base + c;
        bool moving = false;
#pragma unroll
        for (int k = 0; k < kMaxK; ++k) {
          if (k < K) {
            const bool take = moving || cd < bd[k];
            const float td = bd[k];
            const int ti = bi[k];
            bd[k] = take ? cd : td;
            bi[k] = take ? ci : ti;
            cd = take ? td : cd;
            ci = take ? ti : ci;
            moving = take;
            if (k == K - 1) worst = bd[k];
          }
        }
      }
    }
  }
  if (active) {
    const size_t o = (static_cast<size_t>(t.out_begin) + q) * K;
#pragma unroll
    for (int k = 0; k < kMaxK; ++k)
      if (k < K) {
        nbr[o + k] = static_cast<uint16_t>(bi[k] == 0x7fffffff ? 0xffff : bi[k]);
        dist[o + k] = bd[k];
      }
  }
}

// One wave per query mass: lane l holds the candidates l, l + 64, .. (NC of
// them) in registers for all of its queries.  Squared distances are compared
// with a threshold T until it admits between K and 64 candidates (the last
// query's T, adjusted, is usually right at once: neighbours lie alike); those
// are compacted through LDS to one per lane, ranked by (distance, index) by
// counting, and the first K written.  The square root is taken of the
// admitted ones only: it is monotonic, and a candidate over T can share the
// K-th distance only if that distance is sqrtf(T) itself.  In that case, and
// where the search ends between two adjacent floats because more than 64
// candidates lie at one distance, the distances below that one D and the
// lowest indices at it are taken.
//
// What bounds it: VALU issue (per query 10 instructions for each 64 squared
// distances and 2 per try of T, then the ranking).  The scan spends its time
// on insertions: nearly every candidate enters the list of some lane of the
// wave, and an entry moves K pairs.  MI355X, K = 25, 384 robots of 200 to
// 2000 masses: the kernels 5.53 -> 0.99 ms, the call 11.6 -> 7.1 (the rest is
// allocations and copies of the results).  One robot of 2000 masses 3.3 ->
// 0.15 ms.  Clouds of few distinct points have few insertions, which the scan
// is fast at, and no threshold admits 64 of them; nearest_levels serves them
// (kernel, us, scan / this one, K = 6: 128 robots of 1100 masses at two points
// 185 / 151, 200 of 300 60 / 30; without it 437 and 62).  Still slower than
// the scan: robots of about 100 masses or fewer at few points (100 robots of
// 64 masses at two points, K = 6, 17 / 34), and some clouds of many scales (128
// of 1100 masses over 12 decades, K = 6, 523 / 572).
//   kWaveQueries: 64 queries per wave left small robots on too few waves
//     (the robots of at most 512 masses 219 us, at 16 per wave 55).
//   kWaveMinK: a short list is cheap to insert into: 128 robots of 1100
//     masses on a lattice, K = 6 1078 us by the scan and 973 by this kernel,
//     12 1743 and 1361.  Under kWaveSmall masses the wave is not full: calls
//     of 300 robots of 40 masses, K = 8, 119 and 123 us uniform, 98 and 109 all
//     at one point, K = 12 139 and 137, 111 and 123, K = 16 159 and 152.
//   kWaveMaxMasses: 32 candidates a lane take 221 VGPRs, two waves per SIMD.
constexpr int kWaveQueries = 16;  // per wave
constexpr int kWaveMaxMasses = 2048;
constexpr int kWaveMinK = 6;
constexpr uint32_t kWaveSmall = 64;
constexpr int kWaveMinKSmall = 16;
static_assert(kMaxK < 64, "admitted candidates fit a wave");

// orders a wave's own LDS accesses
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// the lanes below this one in m
__device__ __forceinline__ int lanes_below(uint64_t m) {
  return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                    __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
}

// Ranks the c <= 64 entries {distance, index} of kept by (distance, index);
// lane l returns the rank of entry l.  Fills the entries c .. 63.
__device__ __forceinline__ int wave_rank(float2* kept, int lane, int c, float d, int idx) {
  const uint64_t key = static_cast<uint64_t>(__float_as_uint(d)) << 32 | static_cast<uint32_t>(idx);
  kept[lane] = make_float2(d, __int_as_float(idx));
  wave_sync();
  int rank = 0;
  for (int j = 0; j < c; j += 4) {  // entries c .. 63 are past every key
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float2 e = kept[j + u];
      rank += (static_cast<uint64_t>(__float_as_uint(e.x)) << 32 | __float_as_uint(e.y)) < key;
    }
  }
  wave_sync();
  return rank;
}

// Clouds of few distinct points: the K nearest of the candidates s (squared
// distances, NaN: none) by one level of distance after the other, each in
// index order, into kept -- in rank order, nothing is left to sort.  False
// where three levels hold fewer than K (kept is then undefined).
template <int NC>
__device__ __forceinline__ bool nearest_levels(const float (&s)[NC], float2* kept, int lane, int K) {
  int base = 0;
  float after = 0.0f;  // squared distances up to here are in kept
  for (int level = 0; level < 3; ++level) {
    float m = INFINITY;
#pragma unroll
    for (int i = 0; i < NC; ++i) m = s[i] > after ? fminf(m, s[i]) : m;
    for (int off = 32; off > 0; off >>= 1) m = fminf(m, __shfl_xor(m, off));
    m = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m)));
    if (m == INFINITY) break;
    // the floats from m up with its root, one a lane
    const uint64_t roots = __builtin_amdgcn_ballot_w64(sqrtf(__uint_as_float(__float_as_uint(m) + lane)) == sqrtf(m));
    after = __uint_as_float(__float_as_uint(m) + 63 - __builtin_clzll(roots));
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      if (base >= K) break;
      const bool in = s[i] >= m && s[i] <= after;
      const uint64_t lanes = __builtin_amdgcn_ballot_w64(in);
      const int at = base + lanes_below(lanes);
      if (in && at < K) kept[at] = make_float2(s[i], __int_as_float(lane + 64 * i));
      base += __popcll(lanes);
    }
    if (base >= K) {
      wave_sync();
      return true;
    }
  }
  return false;
}

template <int NC>
__global__ __launch_bounds__(256, 2) void knn_waves(const float* __restrict__ pos, const KnnTile* __restrict__ tiles,
                                                    int K, uint16_t* __restrict__ nbr, float* __restrict__ dist) {
  __shared__ float2 kept_all[4][64];
  const KnnTile t = tiles[blockIdx.x];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float2* const kept = kept_all[wave];
  const int n = static_cast<int>(t.n_mass);
  const float* p = pos + 3u * static_cast<size_t>(t.mass_begin);
  float x[NC], y[NC], z[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = min(lane + 64 * i, n - 1);
    const bool in = lane + 64 * i < n;
    x[i] = in ? p[3 * c] : __builtin_nanf("");
    y[i] = p[3 * c + 1];
    z[i] = p[3 * c + 2];
  }
  const int q0 = static_cast<int>(t.query0) + wave * kWaveQueries;
  const int q_end = min(n, q0 + kWaveQueries);
  constexpr float kMax = 3.402823466e+38f;
  float T = 1.0f;  // threshold on the squared distance, 0 < T <= kMax
  bool tied = false;  // the last query had more than 64 candidates at one distance
  for (int q = q0; q < q_end; ++q) {
    const float qx = p[3 * q], qy = p[3 * q + 1], qz = p[3 * q + 2];
    // squared distances; NaN, which passes no comparison, for what is no
    // candidate: a zero distance, a lane past the robot's masses
    float s[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const float dx = qx - x[i], dy = qy - y[i], dz = qz - z[i];
      const float v = dx * dx + (dy * dy + dz * dz);
      s[i] = v > 0.0f ? v : __builtin_nanf("");
    }
    const size_t o = (static_cast<size_t>(t.out_begin) + q) * K;
    if (tied && nearest_levels<NC>(s, kept, lane, K)) {
      if (lane < K) {
        const float2 e = kept[lane];
        nbr[o + lane] = static_cast<uint16_t>(__float_as_int(e.y));
        dist[o + lane] = sqrtf(e.x);
      }
      wave_sync();
      continue;
    }
    tied = false;
    // lo admits too few, hi too many (bit patterns of positive floats order
    // as they do).  Every try lies strictly between and becomes one of them,
    // so the search ends.
    uint32_t lo = 0u, hi = __float_as_uint(kMax) + 1u;
    float D = 0.0f, grow = 2.0f, shrink = 0.25f;
    bool done = false, first = true;
    while (true) {
      int c = 0;
#pragma unroll
      for (int i = 0; i < NC; ++i) c += __popcll(__builtin_amdgcn_ballot_w64(s[i] <= T));
      const bool few = c < K && T < kMax;
      if (!few && c <= 64) {
        int base = 0;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
          const uint64_t m = __builtin_amdgcn_ballot_w64(s[i] <= T);
          if (s[i] <= T) kept[base + lanes_below(m)] = make_float2(s[i], __int_as_float(lane + 64 * i));
          base += __popcll(m);
        }
        wave_sync();
        float d = INFINITY;
        int idx = 0x7fffffff;
        if (lane < c) {
          const float2 e = kept[lane];
          d = sqrtf(e.x);
          idx = __float_as_int(e.y);
        }
        wave_sync();
        const int rank = wave_rank(kept, lane, c, d, idx);
        D = sqrtf(T);
        // the K-th distance must lie below every candidate left out
        if (T < kMax && __builtin_amdgcn_ballot_w64(lane < c && rank == K - 1 && !(d < D)) != 0ull) break;
        if (lane < c && rank < K) {
          nbr[o + rank] = static_cast<uint16_t>(idx);
          dist[o + rank] = d;
        }
        if (lane >= c && lane < K) {  // fewer than K candidates
          nbr[o + lane] = 0xffff;
          dist[o + lane] = INFINITY;
        }
        done = true;
        // the next query's guess: aim at the middle of the admitted range
        if (c < (K + 64) / 2 - 8) T = fminf(T * 1.12f, kMax);
        else if (c > (K + 64) / 2 + 8) T *= 0.92f;
        if (!(T > 0.0f)) T = 1.0f;
        break;
      }
      const uint32_t b = __float_as_uint(T);
      const bool top = !few && first;
      if (few) {
        lo = b;
      } else if (top) {
        // too many for the first time: down to the farthest one admitted
        first = false;
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < NC; ++i) m = s[i] <= T ? fmaxf(m, s[i]) : m;
        for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
        hi = __builtin_amdgcn_readfirstlane(__float_as_uint(m));
      } else {
        hi = b;
      }
      if (hi - lo <= 1u) {  // all between lo and hi lie at sqrtf(hi)
        T = __uint_as_float(hi);
        D = sqrtf(T);
        tied = true;
        break;
      }
      if (top) {  // and one float below it: many candidates may lie there
        T = __uint_as_float(hi - 1u);
      } else if (lo == 0u) {
        T *= shrink;
        shrink *= shrink;
        if (!(T > 0.0f)) T = __uint_as_float(1u);
      } else if (hi > __float_as_uint(kMax)) {
        T = fminf(T * grow, kMax);
        grow *= grow;
      } else {
        T = __uint_as_float(lo + (hi - lo) / 2u);
      }
    }
    if (done) continue;
    // fewer than K candidates below D, K or more up to it
    int below = 0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      s[i] = sqrtf(s[i]);
      const uint64_t m = __builtin_amdgcn_ballot_w64(s[i] < D);
      if (s[i] < D) kept[below + lanes_below(m)] = make_float2(s[i], __int_as_float(lane + 64 * i));
      below += __popcll(m);
    }
    int base = below;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(s[i] == D);
      const int at = base + lanes_below(m);
      if (s[i] == D && at < K) kept[at] = make_float2(D, __int_as_float(lane + 64 * i));
      base += __popcll(m);
    }
    wave_sync();
    float d = INFINITY;
    int idx = 0x7fffffff;
    if (lane < K) {
      const float2 e = kept[lane];
      d = e.x;
      idx = __float_as_int(e.y);
    }
    wave_sync();
    const int rank = wave_rank(kept, lane, K, d, idx);
    if (lane < K) {
      nbr[o + rank] = static_cast<uint16_t>(idx);
      dist[o + rank] = d;
    }
    T = fminf(T * 1.0001f, kMax);  // past this distance, which the next query may share
  }
}

int fail(int code, const std::string& m) {
  mh::set_error(m);
  return code;
}

}  // namespace

extern "C" {

int mh_knn_batch(int device, int n_robots, const uint32_t* mass_offset, const float* pos, int K,
                 uint16_t* nbr, float* dist) {
  if (n_robots < 0 || (n_robots > 0 && (!mass_offset || !pos || !nbr || !dist)))
    return fail(MH_ERR_ARG, "null argument");
  if (K < 1 || K > kMaxK) return fail(MH_ERR_RANGE, "K must be 1..32");
  if (n_robots == 0) return MH_OK;
  // tiles by kernel: knn_waves with 8, 16, 24 or 32 candidates a lane, then
  // the scan (larger robots, few neighbours)
  std::vector<KnnTile> kinds[5];
  for (int r = 0; r < n_robots; r++) {
    const uint32_t m = mass_offset[r + 1] - mass_offset[r];
    if (mass_offset[r + 1] < mass_offset[r]) return fail(MH_ERR_ARG, "offsets must be non-decreasing");
    if (m > 65535) return fail(MH_ERR_RANGE, "robot has more than 65535 masses");
    if (m > 0 && static_cast<int>(m) <= K) return fail(MH_ERR_RANGE, "robot has no more than K masses");
    const bool scan = m > kWaveMaxMasses || K < (m < kWaveSmall ? kWaveMinKSmall : kWaveMinK);
    std::vector<KnnTile>& kind = kinds[scan ? 4 : m <= 512 ? 0 : (m - 1) / 512];
    const uint32_t block = scan ? kQueryBlock : 4 * kWaveQueries;
    for (uint32_t q = 0; q < m; q += block) kind.push_back({mass_offset[r], m, q, mass_offset[r]});
  }
  std::vector<KnnTile> tiles;
  for (const auto& k : kinds) tiles.insert(tiles.end(), k.begin(), k.end());
  const size_t M = mass_offset[n_robots];
  if (tiles.empty()) return MH_OK;
  hipError_t e = hipSetDevice(device);
  if (e != hipSuccess) return fail(MH_ERR_HIP, std::string("hipSetDevice: ") + hipGetErrorString(e));
  float* d_pos = nullptr;
  float* d_dist = nullptr;
  uint16_t* d_nbr = nullptr;
  KnnTile* d_tiles = nullptr;
  auto cleanup = [&]() {
    hipFree(d_pos);
    hipFree(d_dist);
    hipFree(d_nbr);
    hipFree(d_tiles);
  };
  if ((e = hipMalloc(&d_pos, 3 * M * sizeof(float))) != hipSuccess ||
      (e = hipMalloc(&d_dist, M * K * sizeof(float))) != hipSuccess ||
      (e = hipMalloc(&d_nbr, M * K * sizeof(uint16_t))) != hipSuccess ||
      (e = hipMalloc(&d_tiles, tiles.size() * sizeof(KnnTile))) != hipSuccess) {
    cleanup();
    return fail(MH_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  }
  e = hipMemcpy(d_pos, pos, 3 * M * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(d_tiles, tiles.data(), tiles.size() * sizeof(KnnTile), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    using Kernel = void (*)(const float*, const KnnTile*, int, uint16_t*, float*);
    const Kernel kernels[5] = {knn_waves<8>, knn_waves<16>, knn_waves<24>, knn_waves<32>, knn_tiles};
    size_t at = 0;
    for (int k = 0; k < 5; k++) {
      if (!kinds[k].empty())
        hipLaunchKernelGGL(kernels[k], dim3(static_cast<unsigned>(kinds[k].size())), dim3(kQueryBlock), 0, nullptr,
                           d_pos, d_tiles + at, K, d_nbr, d_dist);
      at += kinds[k].size();
    }
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(nbr, d_nbr, M * K * sizeof(uint16_t), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(dist, d_dist, M * K * sizeof(float), hipMemcpyDeviceToHost);
  cleanup();
  if (e != hipSuccess) return fail(MH_ERR_HIP, std::string("knn: ") + hipGetErrorString(e));
  return MH_OK;
}

}  // extern "C"
