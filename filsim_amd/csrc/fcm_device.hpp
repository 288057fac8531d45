// fcm_device.hpp -- device pieces the FCM kernels share: Gaussian constants,
// segment records and tile lists, matrix-core steps.
#pragma once

#include "common.hpp"
#include "fcm_impl.hpp"

namespace fs {

constexpr double kPi = 3.14159265358979323846264338327950288;
constexpr int kCoef = 8;  // spread coefficients per segment (6 used)
constexpr int kMaxBinsPerTile = 64;

struct GaussConst {
  double dx, anorm, anorm2, anormdip, anormdip2, sigmadipsq;
  int ngd, ngdh, nx, ny, nz;
  int fine;  // FP32 tile weights: FP64, rounded
  // base-2 weights: g = anorm 2^(-xx^2 e2), gD = anormdip 2^(-xx^2 ed2),
  // e2 = log2(e) / anorm2, ed2 = log2(e) / anormdip2
  double e2, ed2;
  double nrsd;  // -1 / sigmadipsq
};

// What a tile needs of one segment: per axis the FP64 offset xx0 = (grid
// coordinate of stencil point 0) * dx - y (point i lies at xx0 + i dx), its
// id, stencil origin (10 bits per axis, x lowest) and spread coefficients
// (force, half torque: GA_setup).
template <typename T>
struct alignas(16) SegRec {
  double xx0[3];
  int id, org;
  T cf[6];
};
constexpr int kTileCap = 32;  // records in a tile's slab; the rest: pool
constexpr int kListBins = 128;  // bins a tile's list is gathered from
constexpr int kDirectMax = 4096;  // segments of tile lists without bins (LDS)
// steps of 1,024 segments over all rows of tiles, where the line to them lies
constexpr long kDirectRowSteps = 1024;
inline size_t rec_bytes(int tsz) {
  return tsz == 8 ? sizeof(SegRec<double>) : sizeof(SegRec<float>);
}

// Whether a stencil of ngd points starting at o overlaps the te points
// starting at p0 on a periodic axis of n points (o, p0 in [0, n)).
__device__ __forceinline__ bool stencil_meets(int o, int p0, int te, int ngd,
                                             int n) {
  int d = o - p0;
  if (d < 0) d += n;
  return d < te || d > n - ngd;
}

// Stages records [r0, r0 + n) of tile `tile` into s_rec: r0 = 0 copies the
// whole slab (issued before the count is known; entries past the count are
// never used), r0 >= kTileCap the tile's pool block. 256 threads.
template <typename T>
__device__ __forceinline__ void stage_tile_records(
    const SegRec<T> *__restrict__ slab, const SegRec<T> *__restrict__ pool,
    int tile, int ovf, int r0, int n, SegRec<T> *s_rec) {
  constexpr int W = sizeof(SegRec<T>) / 16;
  static_assert(kTileCap * W <= 256, "one 16-byte word per thread");
  const int4 *src =
      r0 == 0 ? reinterpret_cast<const int4 *>(slab + (size_t)tile * kTileCap)
              : reinterpret_cast<const int4 *>(pool + ovf + r0 - kTileCap);
  const int nw = (r0 == 0 ? kTileCap : n) * W;
  if ((int)threadIdx.x < nw)
    reinterpret_cast<int4 *>(s_rec)[threadIdx.x] = src[threadIdx.x];
}

// A tile's record count and this thread's 16-byte word of its slab, loaded
// ahead of use: the persistent tile kernels fetch the next tile's while
// they work on the current one.
template <typename T>
struct TilePrefetch {
  static constexpr int W = sizeof(SegRec<T>) / 16;
  int4 w;
  int cnt;
  __device__ __forceinline__ void load(const SegRec<T> *__restrict__ slab,
                                       const int *__restrict__ tcnt, int tile) {
    if ((int)threadIdx.x < kTileCap * W)
      w = reinterpret_cast<const int4 *>(slab + (size_t)tile * kTileCap)[threadIdx.x];
    cnt = tcnt[tile];
  }
  __device__ __forceinline__ void store(SegRec<T> *s_rec) const {
    if ((int)threadIdx.x < kTileCap * W)
      reinterpret_cast<int4 *>(s_rec)[threadIdx.x] = w;
  }
};

// One 16x16x4 matrix-core step D += A B in the real type, and the row of
// D held in accumulator element r of lane l (column l % 16): 4 (l / 16) + r
// for FP32, 4 r + l / 16 for FP64 (the instructions' output layouts).
template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 step(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) {
    return 4 * (lane >> 4) + r;
  }
};
template <>
struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 step(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) {
    return 4 * r + (lane >> 4);
  }
};

// Sums over the four 16-lane groups of four values at once: lane group q gets
// the total of v_q, (0 + 2) + (1 + 3). v_permlane32_swap exchanges the upper
// half of one register with the lower half of another, v_permlane16_swap the
// odd with the even rows of 16: five exchanges less than four butterflies,
// and none through LDS.
template <typename T>
__device__ __forceinline__ T lane_reduce4(T v0, T v1, T v2, T v3) {
  constexpr int W = sizeof(T) / 4;
  const auto swap = [](T &a, T &b, auto exchange) {
    unsigned ua[W], ub[W];
    __builtin_memcpy(ua, &a, sizeof(T));
    __builtin_memcpy(ub, &b, sizeof(T));
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const auto r = exchange(ua[w], ub[w]);
      ua[w] = r[0];
      ub[w] = r[1];
    }
    __builtin_memcpy(&a, ua, sizeof(T));
    __builtin_memcpy(&b, ub, sizeof(T));
  };
  const auto s32 = [](unsigned a, unsigned b) {
    return __builtin_amdgcn_permlane32_swap(a, b, false, false);
  };
  const auto s16 = [](unsigned a, unsigned b) {
    return __builtin_amdgcn_permlane16_swap(a, b, false, false);
  };
  swap(v0, v2, s32);
  swap(v1, v3, s32);
  T s = v0 + v2, t = v1 + v3;  // rows (v0, v0, v2, v2) and (v1, v1, v3, v3)
  swap(s, t, s16);
  return s + t;
}

// 2^t for t <= 0 in FP64: 2^(t - n) by its Taylor series on [-1/2, 1/2]
// (degree 13: remainder 4e-18) scaled by 2^n. What underflows is 0, NaN stays
// NaN. Half the instructions of exp(), whose range checks the weights do not
// need.
__device__ __forceinline__ double exp2_neg(double t) {
  t = t < -1100.0 ? -1100.0 : t;
  const double n = rint(t), f = (t - n) * 0.69314718055994530941723212145818;
  double p = 1.0 / 6227020800.0;
  p = fma(p, f, 1.0 / 479001600.0);
  p = fma(p, f, 1.0 / 39916800.0);
  p = fma(p, f, 1.0 / 3628800.0);
  p = fma(p, f, 1.0 / 362880.0);
  p = fma(p, f, 1.0 / 40320.0);
  p = fma(p, f, 1.0 / 5040.0);
  p = fma(p, f, 1.0 / 720.0);
  p = fma(p, f, 1.0 / 120.0);
  p = fma(p, f, 1.0 / 24.0);
  p = fma(p, f, 1.0 / 6.0);
  p = fma(p, f, 0.5);
  p = fma(p, f, 1.0);
  p = fma(p, f, 1.0);
  return ldexp(p, (int)n);
}

// Orders a wavefront's own LDS writes before its reads of them.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Tiles of te points that a stencil of ngd points can meet along an axis.
__host__ __device__ constexpr int stencil_tiles(int ngd, int te) {
  return (ngd + te - 2) / te + 1;
}
}  // namespace fs
