// fcm_run.hpp -- kernels and launch sequence of the FCM mobility solve, one
// translation unit per precision (fcm_f32.hip, fcm_f64.hip); the pipeline is
// described in fcm.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "fcm_device.hpp"
#include "fcm_impl.hpp"
#include "fft.hpp"
#include "scan.hpp"

namespace fs {

constexpr int kMaxNgd = 24;     // largest Gaussian support handled
constexpr int kCandChunk = 16;  // segments staged in LDS per spread chunk

// ---------------------------------------------------------------------
// prepare: tables [seg][9][ngd] (ga x,y,z | gd x,y,z | gr x,y,z), stencil
// origin (wrapped index of support point 0), bin, spread coefficients.
// ---------------------------------------------------------------------
// Grid cell holding coordinate y: truncation of y/dx, as
// FCMfunctions.cpp:565-567. A coordinate that is not finite or lies more
// than 2^30 cells out (a diverged iterate) gets cell s instead: no
// saturating conversion or signed overflow downstream, and such segments
// spread over many bins rather than piling into one (the order in a bin is
// quadratic in the bin's population). Its tables are then 0 or NaN.
__device__ __forceinline__ int stencil_cell(double y, double dx, int s) {
  const double cy = y / dx;
  return fabs(cy) < 1073741824.0 ? (int)cy : s;
}

// Wrapped index of support point 0 of the stencil around coordinate y.
__device__ __forceinline__ int stencil_origin(double y, double dx, int s,
                                              int ngdh, int n) {
  const int w = (stencil_cell(y, dx, s) - ngdh + 1) % n;
  return w < 0 ? w + n : w;
}

// Bin of tile (bx, by, bz): z fastest, so the bin-sorted segment list runs
// along the grid's contiguous axis and segments next to each other in it
// share cache lines of the real grids (interpolation reads them in list
// order). The spread enumerates its candidate bins by tile offset, so its
// summation order does not depend on this numbering.
__device__ __forceinline__ int spread_bin(int bx, int by, int bz, int nbx,
                                          int nby, int nbz) {
  return bz + nbz * (by + nby * bx);
}

template <typename T>
__global__ void k_prepare_tab(const int *__restrict__ act, int np, const double *__restrict__ Y,
                              GaussConst g, T *__restrict__ tab) {
  if (act && !*act) return;  // batched sweep: suspension converged
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)np * 3 * g.ngd) return;
  const int i = (int)(t % g.ngd), d = (int)((t / g.ngd) % 3),
            s = (int)(t / (3 * g.ngd));
  const double y = Y[3 * s + d];
  const int c = stencil_cell(y, g.dx, s);
  const int xg = c - g.ngdh + 1 + i;
  const double xx = ((double)xg) * g.dx - y;
  T *ts = tab + (size_t)s * 9 * g.ngd;
  ts[(0 + d) * g.ngd + i] = (T)(g.anorm * exp(-xx * xx / g.anorm2));
  ts[(3 + d) * g.ngd + i] = (T)(g.anormdip * exp(-xx * xx / g.anormdip2));
  ts[(6 + d) * g.ngd + i] = (T)(-xx / g.sigmadipsq);
}

template <typename T, typename GC = GaussConst>
__device__ __forceinline__ void d_prepare(const int *__restrict__ act, int np, const double *__restrict__ Y,
                          const double *__restrict__ F,
                          const double *__restrict__ Tq, GC g,
                          int tx, int ty, int tz, int nbx, int nby, int nbz,
                          int *__restrict__ origin, T *__restrict__ coef,
                          int *__restrict__ bin, int *__restrict__ bin_count,
                          int *__restrict__ slot) {
  if (act && !*act) return;  // batched sweep: suspension converged
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= np) return;
  const int nn[3] = {g.nx, g.ny, g.nz};
  int o[3];
  for (int d = 0; d < 3; ++d) {
    o[d] = stencil_origin(Y[3 * s + d], g.dx, s, g.ngdh, nn[d]);
    origin[3 * s + d] = o[d];
  }
  // spread coefficients of the vector path (the matrix-core path keeps them in
  // its records): F and half torque (GA_setup: GA = T/2 pattern), kCoef per
  // segment so a record is whole 16-byte words
  if (coef) {
    for (int d = 0; d < 3; ++d) {
      coef[kCoef * s + d] = (T)F[3 * s + d];
      coef[kCoef * s + 3 + d] = (T)(0.5 * Tq[3 * s + d]);
    }
    coef[kCoef * s + 6] = (T)0;
    coef[kCoef * s + 7] = (T)0;
  }
  int b = spread_bin(o[0] / tx, o[1] / ty, o[2] / tz, nbx, nby, nbz);
  bin[s] = b;
  slot[s] = atomicAdd(&bin_count[b], 1);
}
template <typename T>
__global__ void k_prepare(const int *__restrict__ act, int np, const double *__restrict__ Y,
                          const double *__restrict__ F,
                          const double *__restrict__ Tq, GaussConst g,
                          int tx, int ty, int tz, int nbx, int nby, int nbz,
                          int *__restrict__ origin, T *__restrict__ coef,
                          int *__restrict__ bin, int *__restrict__ bin_count,
                          int *__restrict__ slot) {
  d_prepare<T>(act, np, Y, F, Tq, g, tx, ty, tz, nbx, nby, nbz, origin, coef, bin, bin_count, slot);
}
// arguments of one suspension for k_prepare_multi
template <typename T>
struct A_prepare {
  const int *act;
  int np;
  const double *Y;
  const double *F;
  const double *Tq;
  GaussConst g;
  int tx;
  int ty;
  int tz;
  int nbx;
  int nby;
  int nbz;
  int *origin;
  T *coef;
  int *bin;
  int *bin_count;
  int *slot;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void k_prepare_multi(const A_prepare<T> *__restrict__ a) {
  const A_prepare<T> &A = a[blockIdx.z];
  d_prepare<T, const GaussConst &>(A.act, A.np, A.Y, A.F, A.Tq, A.g, A.tx, A.ty, A.tz, A.nbx, A.nby, A.nbz, A.origin, A.coef, A.bin, A.bin_count, A.slot);
}

__device__ __forceinline__ void d_scatter(int np, const int *__restrict__ bin,
                          const int *__restrict__ slot,
                          const int *__restrict__ start, int *__restrict__ ids) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= np) return;
  ids[start[bin[s]] + slot[s]] = s;
}
static __global__ void k_scatter(int np, const int *__restrict__ bin,
                          const int *__restrict__ slot,
                          const int *__restrict__ start, int *__restrict__ ids) {
  d_scatter(np, bin, slot, start, ids);
}
// arguments of one suspension for k_scatter_multi
struct A_scatter {
  int np;
  const int *bin;
  const int *slot;
  const int *start;
  int *ids;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
static __global__ void k_scatter_multi(const A_scatter *__restrict__ a) {
  const A_scatter &A = a[blockIdx.z];
  d_scatter(A.np, A.bin, A.slot, A.start, A.ids);
}

// Record of segment s, whose stencil origin is (o0, o1, o2).
template <typename T>
__device__ __forceinline__ SegRec<T> segment_record(
    int s, int o0, int o1, int o2, const double *__restrict__ Y,
    const double *__restrict__ F, const double *__restrict__ Tq, double dx,
    int ngdh) {
  SegRec<T> r;
  for (int d = 0; d < 3; ++d) {
    const double y = Y[3 * s + d];
    r.xx0[d] = ((double)(stencil_cell(y, dx, s) - ngdh + 1)) * dx - y;
    r.cf[d] = (T)F[3 * s + d];
    r.cf[3 + d] = (T)(0.5 * Tq[3 * s + d]);
  }
  r.id = s;
  r.org = o0 | (o1 << 10) | (o2 << 20);
  return r;
}

// Ascending segment order inside each bin (atomic slots are unordered): a
// thread per segment counts the smaller ids in its bin (ids, unordered) and
// writes its id to that place of sids, or (the matrix-core path) its record
// and packed stencil origin to that place of srec and sorg. A thread per bin
// sorting it by insertion is a chain of dependent loads and stores: all launches
// up to here 36 -> 22 us at 30k segments on 256^3, 63 -> 50 us at 240k on 512^3.
template <typename T>
__device__ __forceinline__ void d_bin_order(const int *__restrict__ act, int np,
                            const int *__restrict__ bin,
                            const int *__restrict__ start,
                            const int *__restrict__ ids,
                            const int *__restrict__ origin,
                            const double *__restrict__ Y,
                            const double *__restrict__ F,
                            const double *__restrict__ Tq, double dx,
                            int ngdh, SegRec<T> *__restrict__ srec,
                            int *__restrict__ sorg, int *__restrict__ sids) {
  if (act && !*act) return;  // batched sweep: suspension converged
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= np) return;
  const int b = bin[s];
  const int lo = start[b], hi = start[b + 1];
  int pos = lo;
  for (int i = lo; i < hi; ++i) pos += ids[i] < s;
  if (srec) {
    const SegRec<T> r = segment_record<T>(s, origin[3 * s], origin[3 * s + 1],
                                          origin[3 * s + 2], Y, F, Tq, dx, ngdh);
    srec[pos] = r;
    sorg[pos] = r.org;
  } else {
    sids[pos] = s;
  }
}
template <typename T>
__global__ void k_bin_order(const int *__restrict__ act, int np,
                            const int *__restrict__ bin,
                            const int *__restrict__ start,
                            const int *__restrict__ ids,
                            const int *__restrict__ origin,
                            const double *__restrict__ Y,
                            const double *__restrict__ F,
                            const double *__restrict__ Tq, double dx,
                            int ngdh, SegRec<T> *__restrict__ srec,
                            int *__restrict__ sorg, int *__restrict__ sids) {
  d_bin_order<T>(act, np, bin, start, ids, origin, Y, F, Tq, dx, ngdh, srec, sorg, sids);
}
// arguments of one suspension for k_bin_order_multi
template <typename T>
struct A_bin_order {
  const int *act;
  int np;
  const int *bin;
  const int *start;
  const int *ids;
  const int *origin;
  const double *Y;
  const double *F;
  const double *Tq;
  double dx;
  int ngdh;
  SegRec<T> *srec;
  int *sorg;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void k_bin_order_multi(const A_bin_order<T> *__restrict__ a) {
  const A_bin_order<T> &A = a[blockIdx.z];
  d_bin_order<T>(A.act, A.np, A.bin, A.start, A.ids, A.origin, A.Y, A.F, A.Tq, A.dx, A.ngdh, A.srec, A.sorg, nullptr);
}

// ---------------------------------------------------------------------
// spread (gather): one workgroup per grid tile of tx * ty * TZ points, one
// thread per (x, y) column owning TZ consecutive z points. Candidates (the
// segments whose stencil origin lies in the bins that can reach the tile)
// are staged in LDS in a fixed order (bins, then ascending segment id) with
// their z overlap precomputed; each thread tests x and y once per
// candidate and accumulates the z run in registers. Every grid point is
// written once: no atomics, no zeroing pass, deterministic.
// ---------------------------------------------------------------------
template <typename T, int TZ>
__global__ void __launch_bounds__(256)
    k_spread(const int *__restrict__ act, SpreadGeom G, const T *__restrict__ tab,
             const int *__restrict__ origin, const T *__restrict__ coef,
             const int *__restrict__ start, const int *__restrict__ ids,
             T *__restrict__ R) {
  if (act && !*act) return;  // batched sweep: suspension converged
  __shared__ int s_bstart[kMaxBinsPerTile + 1];
  __shared__ int s_bfirst[kMaxBinsPerTile];
  __shared__ int s_ntot;
  // candidate tables during the sum, the output tile during the store
  constexpr int kTabSz = kCandChunk * 9 * kMaxNgd;
  constexpr int kBufSz = kTabSz > 256 * TZ ? kTabSz : 256 * TZ;
  __shared__ T s_buf[kBufSz];
  __shared__ int s_org[kCandChunk][2];
  __shared__ int s_z[kCandChunk][3];  // zlo, zhi, stencil z index of z0
  __shared__ T s_coef[kCandChunk][6];
  __shared__ int s_cid[kCandChunk];

  const int ntiles = G.nbx * G.nby * G.nbz;
  // XCD-aware order: consecutive tiles land on the same XCD's L2.
  int bid = blockIdx.x;
  if ((ntiles & 7) == 0) bid = (bid & 7) * (ntiles >> 3) + (bid >> 3);
  const int bx = bid % G.nbx;
  const int by = (bid / G.nbx) % G.nby;
  const int bz = bid / (G.nbx * G.nby);
  const int ngd = G.ngd;

  const int cx = min(G.hx + 1, G.nbx), cy = min(G.hy + 1, G.nby),
            cz = min(G.hz + 1, G.nbz);
  const int nbins = cx * cy * cz;
  // the workgroup may have fewer threads (tx*ty) than bins: stride
  for (int t = threadIdx.x; t < nbins; t += blockDim.x) {
    int dz = t / (cx * cy), dy = (t / cx) % cy, dx = t % cx;
    int ix = ((bx - G.hx + dx) % G.nbx + G.nbx) % G.nbx;
    int iy = ((by - G.hy + dy) % G.nby + G.nby) % G.nby;
    int iz = ((bz - G.hz + dz) % G.nbz + G.nbz) % G.nbz;
    int b = spread_bin(ix, iy, iz, G.nbx, G.nby, G.nbz);
    s_bfirst[t] = start[b];
    s_bstart[t + 1] = start[b + 1] - start[b];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s_bstart[0] = 0;
    for (int t = 0; t < nbins; ++t) s_bstart[t + 1] += s_bstart[t];
    s_ntot = s_bstart[nbins];
  }
  __syncthreads();
  const int ntot = s_ntot;
  const int lx = threadIdx.x / G.ty, ly = threadIdx.x % G.ty;
  const bool active = lx < G.tx;
  const int px = bx * G.tx + lx, py = by * G.ty + ly, pz0 = bz * TZ;
  T acc[TZ][3];
#pragma unroll
  for (int k = 0; k < TZ; ++k) acc[k][0] = acc[k][1] = acc[k][2] = (T)0;

  for (int c0 = 0; c0 < ntot; c0 += kCandChunk) {
    const int nc = min(kCandChunk, ntot - c0);
    // candidate ids, origins, z overlap and coefficients: one thread each
    for (int c = threadIdx.x; c < nc; c += blockDim.x) {
      const int gc = c0 + c;
      int t = 0;
      while (gc >= s_bstart[t + 1]) ++t;
      const int s = ids[s_bfirst[t] + gc - s_bstart[t]];
      s_cid[c] = s;
      s_org[c][0] = origin[3 * s + 0];
      s_org[c][1] = origin[3 * s + 1];
      for (int r = 0; r < 6; ++r) s_coef[c][r] = coef[kCoef * s + r];
      // z overlap of the stencil [oz, oz+ngd) with [pz0, pz0+TZ) (mod nz;
      // nz >= TZ + ngd so at most one interval)
      const int oz = origin[3 * s + 2];
      int o = pz0 - oz;
      if (o < 0) o += G.nz;
      int zlo = 0, zhi = 0, izb = 0;
      if (o < ngd) {
        zhi = min(TZ, ngd - o);
        izb = o;
      } else if (o + TZ > G.nz) {
        zlo = G.nz - o;
        zhi = min(TZ, G.nz - o + ngd);
        izb = o - G.nz;
      }
      s_z[c][0] = zlo;
      s_z[c][1] = zhi;
      s_z[c][2] = izb;
    }
    __syncthreads();
    // tables: flat copy with independent loads in flight. e / tl via a
    // float reciprocal is exact here: (e + 0.5) / tl stays >= 0.5 / tl from
    // an integer and e < 2^13.
    {
      const int tl = 9 * ngd, ne = nc * tl;
      const float inv_tl = 1.0f / (float)tl;
#pragma unroll 4
      for (int e = threadIdx.x; e < ne; e += blockDim.x) {
        const int c = (int)(((float)e + 0.5f) * inv_tl);
        const int r = e - c * tl;
        s_buf[c * (9 * kMaxNgd) + r] = tab[(size_t)s_cid[c] * tl + r];
      }
    }
    __syncthreads();
    if (active) {
      for (int c = 0; c < nc; ++c) {
        int ix = px - s_org[c][0];
        if (ix < 0) ix += G.nx;
        int iy = py - s_org[c][1];
        if (iy < 0) iy += G.ny;
        if (ix >= ngd || iy >= ngd) continue;
        const int zlo = s_z[c][0], zhi = s_z[c][1], izb = s_z[c][2];
        const T *tb = s_buf + c * (9 * kMaxNgd);
        const T gxy = tb[0 * ngd + ix] * tb[1 * ngd + iy];
        const T dxy = tb[3 * ngd + ix] * tb[4 * ngd + iy];
        const T xx = tb[6 * ngd + ix], yy = tb[7 * ngd + iy];
        const T *cf = s_coef[c];
        // constant parts of the dipole terms (g = T/2 pattern, GA_setup)
        const T ax = cf[5] * yy, ay = -cf[5] * xx, az = cf[4] * xx - cf[3] * yy;
#pragma unroll
        for (int k = 0; k < TZ; ++k) {
          if (k >= zlo && k < zhi) {
            const int iz = izb + k;
            const T temp = gxy * tb[2 * ngd + iz];
            const T temp2 = dxy * tb[5 * ngd + iz];
            const T zz = tb[8 * ngd + iz];
            acc[k][0] += cf[0] * temp + (ax - cf[4] * zz) * temp2;
            acc[k][1] += cf[1] * temp + (cf[3] * zz + ay) * temp2;
            acc[k][2] += cf[2] * temp + az * temp2;
          }
        }
      }
    }
    __syncthreads();
  }
  // stage each component's tile in LDS (the table buffer is free now) and
  // write it with consecutive threads on consecutive z: runs of TZ values
  // instead of one address per lane per store
  const size_t N = (size_t)G.nx * G.ny * G.nz;
  T *stage = s_buf;
  const int nrow = G.tx * G.ty;
  for (int c = 0; c < 3; ++c) {
    if (active) {
#pragma unroll
      for (int k = 0; k < TZ; ++k) stage[threadIdx.x * TZ + k] = acc[k][c];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nrow * TZ; e += blockDim.x) {
      const int row = e / TZ, k = e - row * TZ;
      const int rx = bx * G.tx + row / G.ty, ry = by * G.ty + row % G.ty;
      R[(size_t)c * N + ((size_t)rx * G.ny + ry) * G.nz + pz0 + k] = stage[e];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------
// Matrix-core spread and interpolation work on 8 x 8 x 16 grid tiles.
// Per solve, k_tile_lists gives every tile the records of the segments
// whose stencil meets it; both kernels then load a tile's records in one
// round trip and form the Gaussian weights of those segments at the tile's
// own 8 + 8 + 16 axis points in LDS (no per-segment tables).
// ---------------------------------------------------------------------

// Block id -> tile (bx, by, bz): consecutive block ids on one XCD (blocks
// are dealt to the 8 XCDs round-robin) take a contiguous run of tiles, and
// z-neighbouring tiles, which share 128-byte lines of the grid, are next to
// each other in it when nbz is even.
__device__ __forceinline__ void tile_of_block(const SpreadGeom &G, int bid,
                                              int *bx, int *by, int *bz) {
  const int ntiles = G.nbx * G.nby * G.nbz;
  if ((ntiles & 7) == 0) bid = (bid & 7) * (ntiles >> 3) + (bid >> 3);
  if ((G.nbz & 1) == 0) {
    const int zl = bid & 1, r = bid >> 1;
    *bx = r % G.nbx;
    *by = (r / G.nbx) % G.nby;
    *bz = 2 * (r / (G.nbx * G.nby)) + zl;
  } else {
    *bx = bid % G.nbx;
    *by = (bid / G.nbx) % G.nby;
    *bz = bid / (G.nbx * G.nby);
  }
}

// One wavefront per tile (tile = 4 * block id + wave, x fastest): the
// segments of the bins that can reach the tile whose stencil meets it, in
// (neighbouring bin, position in bin) order; the test reads the packed
// origins (sorg), only kept segments' records are copied. The first
// kTileCap records go to the tile's slab, the rest to a block of the pool
// reserved with one atomic per tile (where the block lies varies between
// runs, the order inside it does not); tcnt = how many, tovf = the pool
// block. The pool holds np times the tiles one stencil can meet, a bound on
// the records of all tiles.
template <typename T, typename SG = SpreadGeom>
__device__ __forceinline__ void d_tile_lists(const int *__restrict__ act, SG G,
                 const int *__restrict__ start, const int *__restrict__ sorg,
                 const SegRec<T> *__restrict__ srec, SegRec<T> *__restrict__ slab,
                 int *__restrict__ tcnt, int *__restrict__ tovf,
                 SegRec<T> *__restrict__ pool, int *__restrict__ pool_top) {
  if (act && !*act) return;  // batched sweep: suspension converged
  __shared__ int s_pre[4][kListBins], s_first[4][kListBins];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ntiles = G.nbx * G.nby * G.nbz;
  const int tile = blockIdx.x * 4 + wave;
  if (tile >= ntiles) return;  // whole wave; no workgroup barrier below
  int *pre = s_pre[wave], *first = s_first[wave];
  const int bx = tile % G.nbx, by = (tile / G.nbx) % G.nby,
            bz = tile / (G.nbx * G.nby);
  const int cx = min(G.hx + 1, G.nbx), cy = min(G.hy + 1, G.nby),
            cz = min(G.hz + 1, G.nbz);
  const int nbins = cx * cy * cz;  // <= kListBins
  int total = 0;
  for (int k0 = 0; k0 < nbins; k0 += 64) {
    const int k = k0 + lane;
    int n = 0, f = 0;
    if (k < nbins) {
      const int dz = k / (cx * cy), dy = (k / cx) % cy, dx = k % cx;
      const int ix = ((bx - G.hx + dx) % G.nbx + G.nbx) % G.nbx;
      const int iy = ((by - G.hy + dy) % G.nby + G.nby) % G.nby;
      const int iz = ((bz - G.hz + dz) % G.nbz + G.nbz) % G.nbz;
      const int b = spread_bin(ix, iy, iz, G.nbx, G.nby, G.nbz);
      f = start[b];
      n = start[b + 1] - f;
    }
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off, 64);
      if (lane >= off) incl += t;
    }
    pre[k] = total + incl - n;
    first[k] = f;
    total += __shfl(incl, 63, 64);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int px0 = bx * G.tx, py0 = by * G.ty, pz0 = bz * G.tz;
  int kept = 0, base = 0;
  // pass 0 counts and fills the slab; pass 1 (a tile with more than
  // kTileCap records) fills its pool block
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1) {
      if (kept <= kTileCap) break;
      int b0 = 0;
      if (lane == 0) b0 = atomicAdd(pool_top, kept - kTileCap);
      base = __shfl(b0, 0, 64);
      kept = 0;
    }
    for (int j0 = 0; j0 < total; j0 += 64) {
      const int j = j0 + lane;
      bool keep = false;
      int pos = 0;
      if (j < total) {
        // the last bin whose first list position is <= j holds entry j
        int lo = 0, hi = nbins - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (pre[mid] <= j)
            lo = mid;
          else
            hi = mid - 1;
        }
        pos = first[lo] + j - pre[lo];
        const int org = sorg[pos];
        keep = stencil_meets(org & 1023, px0, min(G.tx, G.nx - px0), G.ngd, G.nx) &&
               stencil_meets((org >> 10) & 1023, py0, min(G.ty, G.ny - py0), G.ngd,
                             G.ny) &&
               stencil_meets(org >> 20, pz0, min(G.tz, G.nz - pz0), G.ngd, G.nz);
      }
      const unsigned long long kb = __ballot(keep);
      const int k = kept + __popcll(kb & ((1ull << lane) - 1ull));
      if (keep) {
        if (pass == 0 && k < kTileCap)
          slab[(size_t)tile * kTileCap + k] = srec[pos];
        else if (pass == 1 && k >= kTileCap)
          pool[base + k - kTileCap] = srec[pos];
      }
      kept += __popcll(kb);
    }
  }
  if (lane == 0) {
    tcnt[tile] = kept;
    tovf[tile] = base;
  }
}
template <typename T>
__global__ void __launch_bounds__(256)
    k_tile_lists(const int *__restrict__ act, SpreadGeom G,
                 const int *__restrict__ start, const int *__restrict__ sorg,
                 const SegRec<T> *__restrict__ srec, SegRec<T> *__restrict__ slab,
                 int *__restrict__ tcnt, int *__restrict__ tovf,
                 SegRec<T> *__restrict__ pool, int *__restrict__ pool_top) {
  d_tile_lists<T>(act, G, start, sorg, srec, slab, tcnt, tovf, pool, pool_top);
}
// arguments of one suspension for k_tile_lists_multi
template <typename T>
struct A_tile_lists {
  const int *act;
  SpreadGeom G;
  const int *start;
  const int *sorg;
  const SegRec<T> *srec;
  SegRec<T> *slab;
  int *tcnt;
  int *tovf;
  SegRec<T> *pool;
  int *pool_top;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void __launch_bounds__(256)
    k_tile_lists_multi(const A_tile_lists<T> *__restrict__ a) {
  const A_tile_lists<T> &A = a[blockIdx.z];
  d_tile_lists<T, const SpreadGeom &>(A.act, A.G, A.start, A.sorg, A.srec, A.slab, A.tcnt, A.tovf, A.pool, A.pool_top);
}

// The tile lists of few segments without bins: one workgroup per row of tiles
// along x (where the rows are few, several, each with a part of the tiles). Its
// threads form every segment's origin and keep, in ascending order, those whose
// stencil meets the row in y and z; then each wavefront fills the lists of tiles
// of the row (order, slab, pool and counts as above, except that a tile's
// segments are in ascending order over all bins). It
// replaces prepare, scan, scatter, order and list launches, whose time is
// latency at these sizes: 240 segments on 64^3 31 -> 16 us, 1,350 on 96^3 39 ->
// 20 us, 2,400 on 192^3 37 -> 28 us. The pool's counter is zeroed by
// k_interp_sum, which runs after the last use of the pool.
template <typename T, typename SG = SpreadGeom>
__device__ __forceinline__ void d_tile_lists_direct(
    const int *__restrict__ act, int np, SG G, double dx,
    const double *__restrict__ Y, const double *__restrict__ F,
    const double *__restrict__ Tq, int *__restrict__ origin,
    SegRec<T> *__restrict__ slab, int *__restrict__ tcnt,
    int *__restrict__ tovf, SegRec<T> *__restrict__ pool,
    int *__restrict__ pool_top) {
  if (act && !*act) return;  // batched sweep: suspension converged
  __shared__ int s_id[kDirectMax], s_org[kDirectMax];
  __shared__ int s_cnt[2][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int by = blockIdx.x % G.nby, bz = blockIdx.x / G.nby;
  const int ngdh = G.ngd / 2;
  int nrow = 0;  // segments that meet the row
  for (int s0 = 0, it = 0; s0 < np; s0 += 1024, ++it) {
    const int s = s0 + threadIdx.x;
    // one workgroup a round also stores the origins
    const bool own = it % (int)gridDim.x == (int)blockIdx.x && blockIdx.y == 0;
    bool keep = false;
    int org = 0;
    if (s < np) {
      const int oy = stencil_origin(Y[3 * s + 1], dx, s, ngdh, G.ny);
      const int oz = stencil_origin(Y[3 * s + 2], dx, s, ngdh, G.nz);
      keep = stencil_meets(oy, by * G.ty, min(G.ty, G.ny - by * G.ty), G.ngd, G.ny) &&
             stencil_meets(oz, bz * G.tz, min(G.tz, G.nz - bz * G.tz), G.ngd, G.nz);
      if (keep || own) {
        const int ox = stencil_origin(Y[3 * s], dx, s, ngdh, G.nx);
        org = ox | (oy << 10) | (oz << 20);
        if (own) {
          origin[3 * s] = ox;
          origin[3 * s + 1] = oy;
          origin[3 * s + 2] = oz;
        }
      }
    }
    const unsigned long long kb = __ballot(keep);
    if (lane == 0) s_cnt[it & 1][wave] = __popcll(kb);
    __syncthreads();
    int at = nrow;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int n = s_cnt[it & 1][w];
      if (w < wave) at += n;
      nrow += n;
    }
    if (keep) {
      at += __popcll(kb & below);
      s_id[at] = s;
      s_org[at] = org;
    }
  }
  __syncthreads();
  for (int bx = wave + 16 * blockIdx.y; bx < G.nbx; bx += 16 * gridDim.y) {
    const int tile = bx + G.nbx * blockIdx.x;
    int kept = 0, base = 0;
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1) {
        if (kept <= kTileCap) break;
        int b0 = 0;
        if (lane == 0) b0 = atomicAdd(pool_top, kept - kTileCap);
        base = __shfl(b0, 0, 64);
        kept = 0;
      }
      for (int j0 = 0; j0 < nrow; j0 += 64) {
        const int j = j0 + lane;
        const int org = j < nrow ? s_org[j] : 0;
        const bool keep =
            j < nrow && stencil_meets(org & 1023, bx * G.tx,
                                      min(G.tx, G.nx - bx * G.tx), G.ngd, G.nx);
        const unsigned long long kb = __ballot(keep);
        const int k = kept + __popcll(kb & below);
        if (keep && (pass == 0) == (k < kTileCap)) {
          const SegRec<T> r =
              segment_record<T>(s_id[j], org & 1023, (org >> 10) & 1023,
                                org >> 20, Y, F, Tq, dx, ngdh);
          if (pass == 0)
            slab[(size_t)tile * kTileCap + k] = r;
          else
            pool[base + k - kTileCap] = r;
        }
        kept += __popcll(kb);
      }
    }
    if (lane == 0) {
      tcnt[tile] = kept;
      tovf[tile] = base;
    }
  }
}
template <typename T>
__global__ void __launch_bounds__(1024)
    k_tile_lists_direct(const int *__restrict__ act, int np, SpreadGeom G,
                        double dx, const double *__restrict__ Y,
                        const double *__restrict__ F,
                        const double *__restrict__ Tq, int *__restrict__ origin,
                        SegRec<T> *__restrict__ slab, int *__restrict__ tcnt,
                        int *__restrict__ tovf, SegRec<T> *__restrict__ pool,
                        int *__restrict__ pool_top) {
  d_tile_lists_direct<T>(act, np, G, dx, Y, F, Tq, origin, slab, tcnt, tovf, pool, pool_top);
}
// arguments of one suspension for k_tile_lists_direct_multi
template <typename T>
struct A_tile_lists_direct {
  const int *act;
  int np;
  SpreadGeom G;
  double dx;
  const double *Y;
  const double *F;
  const double *Tq;
  int *origin;
  SegRec<T> *slab;
  int *tcnt;
  int *tovf;
  SegRec<T> *pool;
  int *pool_top;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void __launch_bounds__(1024)
    k_tile_lists_direct_multi(const A_tile_lists_direct<T> *__restrict__ a) {
  const A_tile_lists_direct<T> &A = a[blockIdx.z];
  d_tile_lists_direct<T, const SpreadGeom &>(A.act, A.np, A.G, A.dx, A.Y, A.F, A.Tq, A.origin, A.slab, A.tcnt, A.tovf, A.pool, A.pool_top);
}

// Gaussian weights of one segment at a tile's axis points. Point a: x
// (a < 8), y (8 <= a < 16), z (16 <= a < 32) of the tile starting at
// (px0, py0, pz0). w[a] = g (monopole), w[32 + a] = gD (dipole), w[64 + a]
// = its derivative h = gD (-xx / sigma_dip^2), zero off the stencil and past
// the axis' end (a cut tile); xx is formed in FP64, and so is the exponent (base
// 2). FP32 rounds it before the hardware exp2, or (fine) rounds the FP64 weight,
// as the vector path does.
// weights (96) + coefficients (6) per record; odd, so that 16 rows read at one
// point fall on different banks
constexpr int kTileW = 105;
template <typename T>
__device__ __forceinline__ void tile_weights(const GaussConst &g,
                                             const SegRec<T> &r, int a, int px0,
                                             int py0, int pz0, T *w) {
  const int d = a < 8 ? 0 : (a < 16 ? 1 : 2);
  const int p = d == 0 ? px0 + a : (d == 1 ? py0 + a - 8 : pz0 + a - 16);
  const int n = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
  int i = p - ((r.org >> (10 * d)) & 1023);
  if (i < 0) i += n;
  T ga = 0, gd = 0, h = 0;
  if (i < g.ngd && p < n) {
    const double x0 = d == 0 ? r.xx0[0] : (d == 1 ? r.xx0[1] : r.xx0[2]);
    const double xx = x0 + (double)i * g.dx;
    const double x2 = xx * xx;
    if constexpr (sizeof(T) == 8) {
      ga = g.anorm * exp2_neg(-x2 * g.e2);
      gd = g.anormdip * exp2_neg(-x2 * g.ed2);
    } else {
      if (g.fine) {
        ga = (float)(g.anorm * exp2_neg(-x2 * g.e2));
        gd = (float)(g.anormdip * exp2_neg(-x2 * g.ed2));
      } else {
        ga = (float)g.anorm * __builtin_amdgcn_exp2f((float)(-x2 * g.e2));
        gd = (float)g.anormdip * __builtin_amdgcn_exp2f((float)(-x2 * g.ed2));
      }
    }
    h = gd * (T)(xx * g.nrsd);
  }
  w[a] = ga;
  w[32 + a] = gd;
  w[64 + a] = h;
}

// Weights (and, with CF, coefficients) of records s_rec[c0 .. c0 + nc) into
// s_w[0 .. nc). 256 threads.
template <typename T, bool CF>
__device__ __forceinline__ void tile_chunk_weights(const GaussConst &g,
                                                   const SegRec<T> *s_rec,
                                                   int c0, int nc, int px0,
                                                   int py0, int pz0,
                                                   T (*s_w)[kTileW]) {
  for (int e = threadIdx.x; e < nc * 32; e += 256) {
    const int c = e >> 5, a = e & 31;
    tile_weights<T>(g, s_rec[c0 + c], a, px0, py0, pz0, s_w[c]);
  }
  if constexpr (CF) {
    for (int e = threadIdx.x; e < nc * 6; e += 256) {
      const int c = e / 6, k = e - 6 * c;
      s_w[c][96 + k] = s_rec[c0 + c].cf[k];
    }
  }
}

// A wavefront's candidates among rows s_w[0 .. nc): those with a stencil
// point in x columns 2 wave and 2 wave + 1 of the tile (non-zero monopole or
// dipole weight; the others add exact zeros there). Their rows go to wl[0 ..
// count), then pad entries of the zero row KC.
template <typename T, int KC>
__device__ __forceinline__ int wave_candidates(const T (*s_w)[kTileW], int nc,
                                               int wave, int lane, int pad,
                                               int *wl) {
  const T *w = s_w[lane < nc ? lane : KC];
  const bool mine =
      lane < nc && (w[2 * wave] != (T)0 || w[2 * wave + 1] != (T)0 ||
                    w[32 + 2 * wave] != (T)0 || w[33 + 2 * wave] != (T)0);
  const unsigned long long mm = __ballot(mine);
  const int n = __popcll(mm);
  if (mine) wl[__popcll(mm & ((1ull << lane) - 1ull))] = lane;
  if (lane < pad) wl[n + lane] = KC;
  wave_lds_fence();
  return n;
}

// ---------------------------------------------------------------------
// spread on the matrix cores: one workgroup per 8 x 8 x 16 tile,
// four wavefronts of 16 (x, y) points each. Per component the tile is
//   R[xy][z] = sum over candidates c and terms t of A_t[xy][c] * B_t[c][z]
// with the force term   A_0 = F * gx gy,                      B_0 = gz,
// and the torque terms  A_1 = (G_z gDx hy, -G_z hx gDy,
//                              G_y hx gDy - G_x gDx hy),       B_1 = gDz,
//                       A_2 = (-G_y, G_x, 0) gDx gDy,          B_2 = hz
// (h the derivative of the dipole Gaussian gD, G the half torque: the same
// sum as k_spread). Each MFMA 16x16x4 step takes four
// candidates of one term; lane l supplies A[xy = l % 16][c = l / 16] and
// B[c = l / 16][z = l % 16] and holds R[xy = Mfma<T>::row(l, r)][z = l % 16].
// Weights are zero off a candidate's stencil, and the entries that fill a
// wave's last step are the zero row. Candidates are summed in tile-list
// order: no atomics, no zeroing pass, every grid point written once.
// Bound by the matrix instructions and the latency of LDS reads and barriers
// (a tile's grid values are 25 to 50 KB a workgroup, written once): the
// matrix and vector units of a SIMD do not work at the same time here (12
// MFMA 162 ns, 64 FMA 68 ns, both 239 ns), so instructions count, wherever
// they run. 30k segments on 256^3 83 us FP32 / 151 us FP64 (with exp() for
// the FP64 weights and the candidates walked in a bit mask 83 / 156), 128^3
// FP64 39 -> 36 us. One wavefront to a tile, without barriers: 118 / 193 us.
// ---------------------------------------------------------------------
// Candidates per round (FP32 32, FP64 16: the same 13 KB of weights).
template <typename T>
constexpr int kMfmaChunk = sizeof(T) == 8 ? 16 : 32;

template <typename T, typename SG = SpreadGeom, typename GC = GaussConst>
__device__ __forceinline__ void d_spread_mfma(const int *__restrict__ act, SG G, GC g,
                  const SegRec<T> *__restrict__ slab,
                  const SegRec<T> *__restrict__ pool,
                  const int *__restrict__ tcnt, const int *__restrict__ tovf,
                  T *__restrict__ R) {
  typedef typename Mfma<T>::v4 v4;
  constexpr int KC = kMfmaChunk<T>;
  if (act && !*act) return;  // batched sweep: suspension converged
  __shared__ SegRec<T> s_rec[kTileCap];
  __shared__ T s_w[KC + 1][kTileW];  // row KC stays zero
  __shared__ int s_wl[4][KC + 4];    // each wave's candidate list

  int bx, by, bz;
  tile_of_block(G, blockIdx.x, &bx, &by, &bz);
  const int tile = bx + G.nbx * (by + G.nby * bz);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int q = lane >> 4, i16 = lane & 15;
  const int xy = wave * 16 + i16;  // this lane's A row
  const int lx = xy >> 3, ly = xy & 7, lz = i16;
  const int px0 = bx * 8, py0 = by * 8, pz0 = bz * 16;
  // the slab is copied while the count is still on its way
  stage_tile_records<T>(slab, pool, tile, 0, 0, 0, s_rec);
  for (int e = threadIdx.x; e < kTileW; e += 256) s_w[KC][e] = 0;
  const int cnt = tcnt[tile];
  const int ovf = cnt > kTileCap ? tovf[tile] : 0;
  v4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};

  for (int r0 = 0; r0 < cnt; r0 += kTileCap) {
    const int nb = min(kTileCap, cnt - r0);
    if (r0 > 0) {
      __syncthreads();  // the last round still reads s_rec
      stage_tile_records<T>(slab, pool, tile, ovf, r0, nb, s_rec);
    }
    __syncthreads();
    for (int c0 = 0; c0 < nb; c0 += KC) {
      const int nc = min(KC, nb - c0);
      tile_chunk_weights<T, true>(g, s_rec, c0, nc, px0, py0, pz0, s_w);
      __syncthreads();
      const int nw = wave_candidates<T, KC>(s_w, nc, wave, lane, 4, s_wl[wave]);
      for (int c4 = 0; c4 < nw; c4 += 4) {
        // lane group q takes the (c4 + q)-th candidate of the wave's list
        // (the zero row past its end)
        const T *w = s_w[s_wl[wave][c4 + q]];
        const T *cf = w + 96;
        const T gx = w[lx], dx = w[32 + lx], hx = w[64 + lx];
        const T gy = w[8 + ly], dy = w[40 + ly], hy = w[72 + ly];
        const T gz = w[16 + lz], dz = w[48 + lz], hz = w[80 + lz];
        const T gxy = gx * gy, dxy = dx * dy, dhy = dx * hy, hdy = hx * dy;
        acc0 = Mfma<T>::step(cf[0] * gxy, gz, acc0);
        acc1 = Mfma<T>::step(cf[1] * gxy, gz, acc1);
        acc2 = Mfma<T>::step(cf[2] * gxy, gz, acc2);
        acc0 = Mfma<T>::step(cf[5] * dhy, dz, acc0);
        acc1 = Mfma<T>::step(-cf[5] * hdy, dz, acc1);
        acc2 = Mfma<T>::step(cf[4] * hdy - cf[3] * dhy, dz, acc2);
        acc0 = Mfma<T>::step(-cf[4] * dxy, hz, acc0);
        acc1 = Mfma<T>::step(cf[3] * dxy, hz, acc1);
      }
      __syncthreads();  // the next round overwrites the weights
    }
  }
  // lane holds R[xy = wave*16 + Mfma<T>::row(lane, r)][z = i16]: 16 lanes
  // write 16 consecutive z of one (x, y) column
  const size_t N = (size_t)G.nx * G.ny * G.nz;
  const bool whole = px0 + 8 <= G.nx && py0 + 8 <= G.ny && pz0 + 16 <= G.nz;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int oxy = wave * 16 + Mfma<T>::row(lane, r);
    if (!whole && (px0 + (oxy >> 3) >= G.nx || py0 + (oxy & 7) >= G.ny ||
                   pz0 + i16 >= G.nz))
      continue;
    const size_t o = ((size_t)(px0 + (oxy >> 3)) * G.ny + py0 + (oxy & 7)) *
                         G.nz + pz0 + i16;
    R[o] = acc0[r];
    R[N + o] = acc1[r];
    R[2 * N + o] = acc2[r];
  }
}
template <typename T>
__global__ void __launch_bounds__(256)
    k_spread_mfma(const int *__restrict__ act, SpreadGeom G, GaussConst g,
                  const SegRec<T> *__restrict__ slab,
                  const SegRec<T> *__restrict__ pool,
                  const int *__restrict__ tcnt, const int *__restrict__ tovf,
                  T *__restrict__ R) {
  d_spread_mfma<T>(act, G, g, slab, pool, tcnt, tovf, R);
}
// arguments of one suspension for k_spread_mfma_multi
template <typename T>
struct A_spread_mfma {
  const int *act;
  SpreadGeom G;
  GaussConst g;
  const SegRec<T> *slab;
  const SegRec<T> *pool;
  const int *tcnt;
  const int *tovf;
  T *R;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void __launch_bounds__(256)
    k_spread_mfma_multi(const A_spread_mfma<T> *__restrict__ a) {
  const A_spread_mfma<T> &A = a[blockIdx.z];
  d_spread_mfma<T, const SpreadGeom &, const GaussConst &>(A.act, A.G, A.g, A.slab, A.pool, A.tcnt, A.tovf, A.R);
}
// ---------------------------------------------------------------------
// FFT passes. Half spectrum layout C[c][kz][y][x] (x fastest): the z pass
// writes it transposed so the x pass reads contiguous lines and the y pass
// reads runs of consecutive x.
// ---------------------------------------------------------------------

// Kernels of the FFT passes are instantiated on LOGN: n = 2^LOGN known at
// compile time (LOGN > 0) or taken from the plan (LOGN = 0).
template <typename T, int LOGN>
constexpr int kFftMaxThreads = LOGN > 0 ? 1024 : kGenMaxThreads<T>;
template <int LOGN>
__device__ __forceinline__ int fft_len(const FftPlan &pl) {
  if constexpr (LOGN > 0)
    return 1 << LOGN;
  else
    return pl.n;
}
template <int LOGN>
__device__ __forceinline__ int div_len(int e, const FftPlan &pl) {  // e / n
  if constexpr (LOGN > 0)
    return e >> LOGN;
  else
    return pl.dn.q(e);
}

// 16-byte global accesses of reals (float4 / double2); p must be 16-byte
// aligned.
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  using type = float4;
  static constexpr int n = 4, logn = 2;
};
template <>
struct Vec16<double> {
  using type = double2;
  static constexpr int n = 2, logn = 1;
};
template <typename T>
__device__ __forceinline__ void ld16(const T *p, T *out) {
  using V = typename Vec16<T>::type;
  const V v = *reinterpret_cast<const V *>(p);
  __builtin_memcpy(out, &v, 16);
}
// Non-temporal 16-byte load, for data read once that the solve does not
// read again before overwriting it (the z passes' inputs): the hint keeps it
// from displacing the grid the next pass reads from the Infinity Cache
// (measured at 256^3 FP32: spread, z passes and forward y pass 0.039 ms
// faster per solve; the interpolation, which shares 128-byte lines between
// neighbouring tiles through L2, loads normally).
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ void ld16_nt(const T *p, T *out) {
  const i32x4 v = __builtin_nontemporal_load(reinterpret_cast<const i32x4 *>(p));
  __builtin_memcpy(out, &v, 16);
}
template <typename T>
__device__ __forceinline__ T ld_nt(const T *p) {
  return __builtin_nontemporal_load(p);
}
template <typename T>
__device__ __forceinline__ void st16(T *p, const T *in) {
  using V = typename Vec16<T>::type;
  V v;
  __builtin_memcpy(&v, in, 16);
  *reinterpret_cast<V *>(p) = v;
}

// z forward: XB = 2P consecutive x rows at one y, as P complex sequences
// (row 2p in the real part, row 2p+1 in the imaginary part).
template <typename T, int LOGN, typename PL = FftPlan>
__device__ __forceinline__ void d_fft_z_r2c(const int *__restrict__ act, const T *__restrict__ R, cx<T> *__restrict__ C, PL pl,
                const cx<T> *__restrict__ twg, int nx, int ny, int P,
                FastDiv dXB, FastDiv dP) {
  if (act && !*act) return;  // batched sweep: suspension converged
  extern __shared__ unsigned char smem_raw[];
  const int n = fft_len<LOGN>(pl), nh = n / 2 + 1, XB = 2 * P;
  cx<T> *tw = reinterpret_cast<cx<T> *>(smem_raw);
  cx<T> *a = tw + n;
  const int comp = blockIdx.y;
  const int nxb = nx / XB;
  const int x0 = (blockIdx.x % nxb) * XB, y = blockIdx.x / nxb;
  const int pn = fft_padded_len(n);
  const T *Rc = R + (size_t)comp * nx * ny * n;
  cx<T> *Cc = C + (size_t)comp * nh * ny * nx;
  for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twg[i];
  const T half = (T)0.5;
  // the first stage reads both rows of a sequence straight from the grid;
  // the last one leaves the line in LDS for the split
  const T *row = Rc + ((size_t)x0 * ny + y) * n;
  const size_t rs = (size_t)ny * n;
  const LdsIO<T, true> io{a, 1, pn};
  __syncthreads();
  lds_fft<T, true, false, LOGN>(
      io, pl, P, tw,
      [&](int z, int p) {
        const T *r0 = row + 2 * p * rs + z;
        return cx<T>{ld_nt(r0), ld_nt(r0 + rs)};
      },
      io);
  __syncthreads();
  if constexpr (LOGN > 0) {
    // both rows of a sequence from the same two spectrum values, stored
    // as one 16-byte pair (FP32) or two (FP64) of consecutive x
    for (int e = threadIdx.x; e < nh * P; e += blockDim.x) {
      const int kz = dP.q(e), p = e - kz * P;
      const cx<T> z = a[p * pn + fft_pad(kz)];
      const cx<T> w = a[p * pn + fft_pad((n - kz) & (n - 1))];
      const T o[4] = {half * (z.x + w.x), half * (z.y - w.y),
                      half * (z.y + w.y), half * (w.x - z.x)};
      T *dst = reinterpret_cast<T *>(Cc + ((size_t)kz * ny + y) * nx + x0 + 2 * p);
      st16(dst, o);
      if constexpr (Vec16<T>::n == 2) st16(dst + 2, o + 2);
    }
  } else {
    for (int e = threadIdx.x; e < nh * XB; e += blockDim.x) {
      int kz = dXB.q(e), i = e - kz * XB;
      int p = i >> 1;
      cx<T> z = a[p * pn + fft_pad(kz)];
      cx<T> w = a[p * pn + fft_pad(kz == 0 ? 0 : n - kz)];
      cx<T> o = (i & 1) ? cx<T>{half * (z.y + w.y), half * (w.x - z.x)}
                        : cx<T>{half * (z.x + w.x), half * (z.y - w.y)};
      Cc[((size_t)kz * ny + y) * nx + x0 + i] = o;
    }
  }
}
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_z_r2c(const int *__restrict__ act, const T *__restrict__ R, cx<T> *__restrict__ C, FftPlan pl,
                const cx<T> *__restrict__ twg, int nx, int ny, int P,
                FastDiv dXB, FastDiv dP) {
  d_fft_z_r2c<T, LOGN>(act, R, C, pl, twg, nx, ny, P, dXB, dP);
}
// arguments of one suspension for k_fft_z_r2c_multi
template <typename T, int LOGN>
struct A_fft_z_r2c {
  const int *act;
  const T *R;
  cx<T> *C;
  FftPlan pl;
  const cx<T> *twg;
  int nx;
  int ny;
  int P;
  FastDiv dXB;
  FastDiv dP;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_z_r2c_multi(const A_fft_z_r2c<T, LOGN> *__restrict__ a) {
  const A_fft_z_r2c<T, LOGN> &A = a[blockIdx.z];
  d_fft_z_r2c<T, LOGN, const FftPlan &>(A.act, A.R, A.C, A.pl, A.twg, A.nx, A.ny, A.P, A.dXB, A.dP);
}

// z inverse: the mirror of k_fft_z_r2c.
template <typename T, int LOGN, typename PL = FftPlan>
__device__ __forceinline__ void d_fft_z_c2r(const int *__restrict__ act, const cx<T> *__restrict__ C, T *__restrict__ R, PL pl,
                const cx<T> *__restrict__ twg, int nx, int ny, int P,
                FastDiv dP) {
  if (act && !*act) return;  // batched sweep: suspension converged
  extern __shared__ unsigned char smem_raw[];
  const int n = fft_len<LOGN>(pl), nh = n / 2 + 1, XB = 2 * P;
  cx<T> *tw = reinterpret_cast<cx<T> *>(smem_raw);
  cx<T> *a = tw + n;
  const int comp = blockIdx.y;
  const int nxb = nx / XB;
  const int x0 = (blockIdx.x % nxb) * XB, y = blockIdx.x / nxb;
  const int pn = fft_padded_len(n);
  T *Rc = R + (size_t)comp * nx * ny * n;
  const cx<T> *Cc = C + (size_t)comp * nh * ny * nx;
  for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twg[i];
  for (int e = threadIdx.x; e < nh * P; e += blockDim.x) {
    int k = dP.q(e), p = e - k * P;
    const cx<T> *src = Cc + ((size_t)k * ny + y) * nx + x0 + 2 * p;
    cx<T> A, B;
    if constexpr (LOGN > 0) {  // x0 + 2p even: the pair is 16-byte aligned
      T u[4];
      ld16_nt(reinterpret_cast<const T *>(src), u);
      if constexpr (Vec16<T>::n == 2) ld16_nt(reinterpret_cast<const T *>(src) + 2, u + 2);
      A = {u[0], u[1]};
      B = {u[2], u[3]};
    } else {
      A = src[0];
      B = src[1];
    }
    if (k == 0 || 2 * k == n) {  // DC / Nyquist of a real line are real
      A.y = 0;
      B.y = 0;
    }
    a[p * pn + fft_pad(k)] = {A.x - B.y, A.y + B.x};
    if (k > 0 && 2 * k < n) a[p * pn + fft_pad(n - k)] = {A.x + B.y, B.x - A.y};
  }
  __syncthreads();
  // the last stage writes both rows of a sequence straight to the grid
  T *row = Rc + ((size_t)x0 * ny + y) * n;
  const size_t rs = (size_t)ny * n;
  const LdsIO<T, true> io{a, 1, pn};
  lds_fft<T, true, true, LOGN>(io, pl, P, tw, io,
                                  [&](int z, int p, cx<T> v) {
                                    T *r0 = row + 2 * p * rs + z;
                                    r0[0] = v.x;
                                    r0[rs] = v.y;
                                  });
}
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_z_c2r(const int *__restrict__ act, const cx<T> *__restrict__ C, T *__restrict__ R, FftPlan pl,
                const cx<T> *__restrict__ twg, int nx, int ny, int P,
                FastDiv dP) {
  d_fft_z_c2r<T, LOGN>(act, C, R, pl, twg, nx, ny, P, dP);
}
// arguments of one suspension for k_fft_z_c2r_multi
template <typename T, int LOGN>
struct A_fft_z_c2r {
  const int *act;
  const cx<T> *C;
  T *R;
  FftPlan pl;
  const cx<T> *twg;
  int nx;
  int ny;
  int P;
  FastDiv dP;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_z_c2r_multi(const A_fft_z_c2r<T, LOGN> *__restrict__ a) {
  const A_fft_z_c2r<T, LOGN> &A = a[blockIdx.z];
  d_fft_z_c2r<T, LOGN, const FftPlan &>(A.act, A.C, A.R, A.pl, A.twg, A.nx, A.ny, A.P, A.dP);
}

// y pass: one workgroup per (comp, kz, run of B consecutive x).
template <typename T, int LOGN, typename PL = FftPlan>
__device__ __forceinline__ void d_fft_y(const int *__restrict__ act, cx<T> *__restrict__ C, PL pl, const cx<T> *__restrict__ twg,
            int nx, int nh, int B, int inverse, FastDiv dB) {
  if (act && !*act) return;  // batched sweep: suspension converged
  extern __shared__ unsigned char smem_raw[];
  const int n = fft_len<LOGN>(pl);  // ny
  cx<T> *tw = reinterpret_cast<cx<T> *>(smem_raw);
  cx<T> *a = tw + n;
  const int nxb = nx / B;
  const int x0 = (blockIdx.x % nxb) * B, kz = blockIdx.x / nxb;
  const int comp = blockIdx.y;
  cx<T> *base = C + ((size_t)comp * nh + kz) * n * nx + x0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twg[i];
  // the first stage reads the columns straight from the spectrum, the last
  // one writes them back: LDS only between stages
  const LdsIO<T, false> io{a, B, 1};
  const auto ld = [&](int m, int col) { return base[(size_t)m * nx + col]; };
  const auto st = [&](int m, int col, cx<T> v) { base[(size_t)m * nx + col] = v; };
  __syncthreads();
  if (inverse)
    lds_fft<T, false, true, LOGN>(io, pl, B, tw, ld, st, dB);
  else
    lds_fft<T, false, false, LOGN>(io, pl, B, tw, ld, st, dB);
}
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_y(const int *__restrict__ act, cx<T> *__restrict__ C, FftPlan pl, const cx<T> *__restrict__ twg,
            int nx, int nh, int B, int inverse, FastDiv dB) {
  d_fft_y<T, LOGN>(act, C, pl, twg, nx, nh, B, inverse, dB);
}
// arguments of one suspension for k_fft_y_multi
template <typename T, int LOGN>
struct A_fft_y {
  const int *act;
  cx<T> *C;
  FftPlan pl;
  const cx<T> *twg;
  int nx;
  int nh;
  int B;
  int inverse;
  FastDiv dB;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T, int LOGN>
__global__ void __launch_bounds__((kFftMaxThreads<T, LOGN>))
    k_fft_y_multi(const A_fft_y<T, LOGN> *__restrict__ a) {
  const A_fft_y<T, LOGN> &A = a[blockIdx.z];
  d_fft_y<T, LOGN, const FftPlan &>(A.act, A.C, A.pl, A.twg, A.nx, A.nh, A.B, A.inverse, A.dB);
}

struct ProjConst {
  int nx, ny, nz, nh;
  double kfx, kfy, kfz;  // 2 pi / L per axis
  double scale;          // 1 / (N mu)
};

// Compile-time plans hold three lines' values a thread.
template <typename T, int LOGN>
constexpr int kXMaxThreads = LOGN > 0 ? 256 : kGenMaxThreads<T>;

// flow_solve (FCMfunctions.cpp:648-736) at wavenumber (x, y, kz): f[0..3) ->
// the velocity's.
template <typename T, typename PC>
__device__ __forceinline__ void project(const PC &pc, int x, int y, int kz,
                                        cx<T> &f1, cx<T> &f2, cx<T> &f3) {
  const T q1 = (T)(((x <= pc.nx / 2) ? x : x - pc.nx) * pc.kfx);
  const T q2 = (T)(((y <= pc.ny / 2) ? y : y - pc.ny) * pc.kfy);
  const T q3 = (T)(kz * pc.kfz);
  const T sc = (T)pc.scale;
  const T qq = q2 * q2 + q1 * q1 + (T)1e-18;
  const T norm = (T)1 / (qq + q3 * q3);
  cx<T> u1, u2, u3;
  T kf = (q1 * f1.x + q2 * f2.x + q3 * f3.x) * norm;
  u1.x = norm * (f1.x - q1 * kf) * sc;
  u2.x = norm * (f2.x - q2 * kf) * sc;
  u3.x = norm * (f3.x - q3 * kf) * sc;
  kf = (q1 * f1.y + q2 * f2.y + q3 * f3.y) * norm;
  u1.y = norm * (f1.y - q1 * kf) * sc;
  u2.y = norm * (f2.y - q2 * kf) * sc;
  u3.y = norm * (f3.y - q3 * kf) * sc;
  if (x == 0 && y == 0 && kz == 0) u1 = u2 = u3 = cx<T>{0, 0};
  f1 = u1;
  f2 = u2;
  f3 = u3;
}

// One stage of a compile-time plan on a thread's registers: radix 2^LR, span
// 2^LS of n = 2^LOGN; butterfly m of thread t is t + m * blockDim.x, lines
// contiguous in LDS.
template <typename T, int LOGN, int LR, int LS>
struct RegStage {
  static constexpr int R = 1 << LR, NB = kP2E / R, LNB = LOGN - LR, nb = 1 << LNB,
                       ns = 1 << LS, PN = fft_padded_len(1 << LOGN);
  static __device__ __forceinline__ int line(int m) {
    return (threadIdx.x + m * blockDim.x) >> LNB;
  }
  static __device__ __forceinline__ int j(int m) {
    return (threadIdx.x + m * blockDim.x) & (nb - 1);
  }
  static __device__ __forceinline__ int out(int m) {  // element of output 0
    return ((j(m) >> LS) << (LS + LR)) + (j(m) & (ns - 1));
  }
  static __device__ __forceinline__ void put(cx<T> *buf, const cx<T> *v) {
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      cx<T> *dst = buf + line(m) * PN;
      const int d = out(m);
#pragma unroll
      for (int r = 0; r < R; ++r)
        dst[ns % kFftPadGroup == 0 ? fft_pad(d) + fft_pad(r * ns)
                                   : fft_pad(d + r * ns)] = v[m * R + r];
    }
  }
  static __device__ __forceinline__ void get(const cx<T> *buf, cx<T> *v) {
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const cx<T> *src = buf + line(m) * PN;
      const int jj = j(m);
#pragma unroll
      for (int r = 0; r < R; ++r)
        v[m * R + r] = src[nb % kFftPadGroup == 0 ? fft_pad(jj) + fft_pad(r * nb)
                                                  : fft_pad(jj + r * nb)];
    }
  }
  template <bool INV>
  static __device__ __forceinline__ void butterflies(const cx<T> *tw, cx<T> *v) {
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      if constexpr (LS > 0) {
        const int k = j(m) & (ns - 1);
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = tw[(r * k) << (LOGN - LS - LR)];
          if constexpr (INV) w.y = -w.y;
          v[m * R + r] = cmul(v[m * R + r], w);
        }
      }
      dftR<T, R>(&v[m * R], INV);
    }
  }
};
// The stage that starts at span 2^LS, in the plan's order (FWD) or in the
// reversed one: log2 of its radix.
template <int LOGN>
constexpr int p2_log_radix(int ls, bool fwd) {
  int at = 0;
  int lr[16] = {}, n = 0;
  while (at < LOGN) {
    const int rem = LOGN - at;
    lr[n] = rem >= 3 ? 3 : rem >= 2 ? 2 : 1;
    at += lr[n++];
  }
  at = 0;
  for (int s = 0; s < n; ++s) {
    const int l = lr[fwd ? s : n - 1 - s];
    if (at == ls) return l;
    at += l;
  }
  return 0;
}
// Stages from span 2^LS on of three components' lines; the values come in the
// registers of the stage before it (or of this one for LS = 0).
template <typename T, int LOGN, bool INV, int LS>
__device__ __forceinline__ void x_stages(cx<T> *buf, const cx<T> *tw,
                                         cx<T> (*v)[kP2E]) {
  if constexpr (LS < LOGN) {
    constexpr int LR = p2_log_radix<LOGN>(LS, !INV);
    using S = RegStage<T, LOGN, LR, LS>;
#pragma unroll
    for (int c = 0; c < 3; ++c) S::template butterflies<INV>(tw, v[c]);
    if constexpr (LS + LR < LOGN) {
      using N = RegStage<T, LOGN, p2_log_radix<LOGN>(LS + LR, !INV), LS + LR>;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        __syncthreads();
        S::put(buf, v[c]);
        __syncthreads();
        N::get(buf, v[c]);
      }
      x_stages<T, LOGN, INV, LS + LR>(buf, tw, v);
    }
  }
}

// x pass + Stokes projection + inverse x pass: one workgroup per (kz, Q
// consecutive y). The first stage reads the lines straight from the spectrum
// and the last one writes them back. Compile-time plans keep the three
// components of a line in one thread's registers and pass them through one
// component's LDS buffer in turn (a wavefront needs 11 KB in FP32); the last
// forward stage, the projection and the first inverse stage work on registers
// (the inverse takes the radices in reverse, so its first stage starts from
// the elements the last forward one ends with). 256^3: FP32 95 -> 76 us, FP64
// 225 -> 145 us; 512^3 FP32 1,111 -> 697 us. The run-time plans' radices would
// need up to 200 registers for that (192^3: 73 -> 128 us): there the three
// components stay in LDS.
template <typename T, int LOGN, typename PL = FftPlan, typename PC = ProjConst>
__device__ __forceinline__ void d_fft_x_project(const int *__restrict__ act, cx<T> *__restrict__ C, PL pl,
                    const cx<T> *__restrict__ twg, PC pc, int Q,
                    FastDiv dQ) {
  if (act && !*act) return;  // batched sweep: suspension converged
  extern __shared__ unsigned char smem_raw[];
  const int n = fft_len<LOGN>(pl);  // nx
  const int nh = pc.nh;
  cx<T> *tw = reinterpret_cast<cx<T> *>(smem_raw);
  cx<T> *a = tw + n;
  const int nyb = pc.ny / Q;
  const int y0 = (blockIdx.x % nyb) * Q, kz = blockIdx.x / nyb;
  const size_t comp_stride = (size_t)nh * pc.ny * n;
  cx<T> *base = C + ((size_t)kz * pc.ny + y0) * n;
  for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twg[i];
  if constexpr (LOGN > 0) {
    using F = RegStage<T, LOGN, p2_log_radix<LOGN>(0, true), 0>;
    constexpr int LL = p2_log_radix<LOGN>(0, false);  // the last stage's
    using L = RegStage<T, LOGN, LL, LOGN - LL>;
    using O = RegStage<T, LOGN, p2_log_radix<LOGN>(0, true),
                       LOGN - p2_log_radix<LOGN>(0, true)>;
    cx<T> v[3][kP2E];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int m = 0; m < F::NB; ++m) {
        const cx<T> *src = base + c * comp_stride + F::line(m) * n + F::j(m);
#pragma unroll
        for (int r = 0; r < F::R; ++r) v[c][m * F::R + r] = src[r * F::nb];
      }
    x_stages<T, LOGN, false, 0>(a, tw, v);
#pragma unroll
    for (int m = 0; m < L::NB; ++m)
#pragma unroll
      for (int r = 0; r < L::R; ++r)
        project<T>(pc, L::j(m) + r * L::nb, y0 + L::line(m), kz,
                   v[0][m * L::R + r], v[1][m * L::R + r], v[2][m * L::R + r]);
    x_stages<T, LOGN, true, 0>(a, tw, v);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int m = 0; m < O::NB; ++m) {
        cx<T> *dst = base + c * comp_stride + O::line(m) * n + O::out(m);
#pragma unroll
        for (int r = 0; r < O::R; ++r) dst[r * O::ns] = v[c][m * O::R + r];
      }
  } else {
    const LdsIO<T, true> io{a, 1, fft_padded_len(n)};
    const auto at = [&](int x, int sq) -> cx<T> & {
      const int c = dQ.q(sq);
      return base[c * comp_stride + (size_t)(sq - c * Q) * n + x];
    };
    const auto ld = [&](int x, int sq) { return at(x, sq); };
    const auto st = [&](int x, int sq, cx<T> v) { at(x, sq) = v; };
    __syncthreads();
    lds_fft_plan<T, true, false>(io, pl, 3 * Q, tw, FastDiv{0, 0}, ld, io);
    __syncthreads();
    for (int e = threadIdx.x; e < Q * n; e += blockDim.x) {
      const int ql = div_len<LOGN>(e, pl), x = e - ql * n;
      cx<T> f[3] = {io(x, ql), io(x, Q + ql), io(x, 2 * Q + ql)};
      project<T>(pc, x, y0 + ql, kz, f[0], f[1], f[2]);
#pragma unroll
      for (int c = 0; c < 3; ++c) io(x, c * Q + ql, f[c]);
    }
    __syncthreads();
    lds_fft_plan<T, true, true>(io, pl, 3 * Q, tw, FastDiv{0, 0}, io, st);
  }
}
template <typename T, int LOGN>
__global__ void __launch_bounds__((kXMaxThreads<T, LOGN>))
    k_fft_x_project(const int *__restrict__ act, cx<T> *__restrict__ C, FftPlan pl,
                    const cx<T> *__restrict__ twg, ProjConst pc, int Q,
                    FastDiv dQ) {
  d_fft_x_project<T, LOGN>(act, C, pl, twg, pc, Q, dQ);
}
// arguments of one suspension for k_fft_x_project_multi
template <typename T, int LOGN>
struct A_fft_x_project {
  const int *act;
  cx<T> *C;
  FftPlan pl;
  const cx<T> *twg;
  ProjConst pc;
  int Q;
  FastDiv dQ;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T, int LOGN>
__global__ void __launch_bounds__((kXMaxThreads<T, LOGN>))
    k_fft_x_project_multi(const A_fft_x_project<T, LOGN> *__restrict__ a) {
  const A_fft_x_project<T, LOGN> &A = a[blockIdx.z];
  d_fft_x_project<T, LOGN, const FftPlan &, const ProjConst &>(A.act, A.C, A.pl, A.twg, A.pc, A.Q, A.dQ);
}

// ---------------------------------------------------------------------
// interpolation: one 64-lane wavefront per segment (segments in bin order
// so neighbours share L2 lines); each lane owns one z of the stencil and a
// share of its (x, y) columns, then the wavefront reduces.
// ---------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename T, int NGD>
__global__ void __launch_bounds__(256)
    k_interp(const int *__restrict__ act, int np, SpreadGeom G, double dx3, const T *__restrict__ tab,
             const int *__restrict__ origin, const int *__restrict__ ids,
             const T *__restrict__ R, double *__restrict__ V,
             double *__restrict__ W) {
  if (act && !*act) return;  // batched sweep: suspension converged
  constexpr int NC = NGD * NGD;          // (x, y) columns of a stencil
  constexpr int NP = NC * NGD;           // stencil points
  constexpr int PER = (NP + 63) / 64;    // points per lane
  __shared__ T s_gxy[4][NC], s_dxy[4][NC];
  __shared__ T s_z[4][3 * NGD];          // g_z, gD_z, grad_z
  __shared__ T s_xx[4][NGD], s_yy[4][NGD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // XCD-aware order: the 8 XCDs take contiguous runs of the bin-sorted
  // segment list, so neighbouring stencils share an L2
  const int nblk = (np + 3) / 4;
  const int q8 = (nblk + 7) / 8;
  const int b = (blockIdx.x & 7) * q8 + (blockIdx.x >> 3);
  const int w = b * 4 + wave;
  const bool valid = (b < nblk) && (w < np);
  const int s = valid ? ids[w] : 0;
  const T *ts = tab + (size_t)s * 9 * NGD;
  if (valid) {
    for (int c = lane; c < NC; c += 64) {
      int i = c / NGD, j = c - (c / NGD) * NGD;
      s_gxy[wave][c] = ts[0 * NGD + i] * ts[1 * NGD + j];
      s_dxy[wave][c] = ts[3 * NGD + i] * ts[4 * NGD + j];
    }
    for (int k = lane; k < NGD; k += 64) {
      s_z[wave][k] = ts[2 * NGD + k];
      s_z[wave][NGD + k] = ts[5 * NGD + k];
      s_z[wave][2 * NGD + k] = ts[8 * NGD + k];
      s_xx[wave][k] = ts[6 * NGD + k];
      s_yy[wave][k] = ts[7 * NGD + k];
    }
  }
  const int ox = valid ? origin[3 * s] : 0, oy = valid ? origin[3 * s + 1] : 0,
            oz = valid ? origin[3 * s + 2] : 0;
  __syncthreads();
  const size_t N = (size_t)G.nx * G.ny * G.nz;
  // NGD lanes per (x, y) column, KL columns per pass: lane (cl, k) keeps one
  // z (its weights and wrapped z are constants) and walks the columns
  // cl, cl + KL, ...; consecutive lanes still read consecutive z. The
  // stencil sums factor per lane into 9 running sums scaled by the lane's
  // z weights at the end:
  //   V   = g_z   sum gx gy u
  //   W_x = gd_z (sum d y u_z - z sum d u_y), d = gdx gdy, x, y, z the
  //   W_y = gd_z (z sum d u_x - sum d x u_z)   dipole gradient factors
  //   W_z = gd_z (sum d x u_y - sum d y u_x)
  constexpr int KL = 64 / NGD;
  constexpr int NPASS = (NC + KL - 1) / KL;
  constexpr int KLI = KL / NGD, KLJ = KL % NGD;
  constexpr int CH = 6;  // passes whose loads are in flight together
  const int cl = lane / NGD, kz = lane - cl * NGD;
  const bool on = valid && cl < KL;
  int zw = oz + (on ? kz : 0);
  if (zw >= G.nz) zw -= G.nz;
  const T gz = on ? s_z[wave][kz] : (T)0, gdz = on ? s_z[wave][NGD + kz] : (T)0,
          zk = on ? s_z[wave][2 * NGD + kz] : (T)0;
  int ci = cl / NGD, cj = cl % NGD;  // the next pass's column (i, j)
  T sg0 = 0, sg1 = 0, sg2 = 0, sd0 = 0, sd1 = 0;
  T sx1 = 0, sx2 = 0, sy0 = 0, sy2 = 0;
  for (int t0 = 0; t0 < NPASS; t0 += CH) {
    T ux[CH], uy[CH], uz[CH];
    int ic[CH], jc[CH];
    bool okc[CH];
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const bool ok = on && t0 + t < NPASS && ci < NGD;
      int ii = ox + (ok ? ci : 0);
      if (ii >= G.nx) ii -= G.nx;
      int jj = oy + (ok ? cj : 0);
      if (jj >= G.ny) jj -= G.ny;
      const size_t o = ((size_t)ii * G.ny + jj) * G.nz + zw;
      ux[t] = ok ? R[o] : (T)0;
      uy[t] = ok ? R[N + o] : (T)0;
      uz[t] = ok ? R[2 * N + o] : (T)0;
      ic[t] = ok ? ci : 0;
      jc[t] = ok ? cj : 0;
      okc[t] = ok;
      ci += KLI;
      cj += KLJ;
      if (cj >= NGD) {
        cj -= NGD;
        ++ci;
      }
    }
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const int c = ic[t] * NGD + jc[t];
      const T gxy = okc[t] ? s_gxy[wave][c] : (T)0;
      const T dxy = okc[t] ? s_dxy[wave][c] : (T)0;
      const T tx = dxy * s_xx[wave][ic[t]], ty = dxy * s_yy[wave][jc[t]];
      sg0 += gxy * ux[t];
      sg1 += gxy * uy[t];
      sg2 += gxy * uz[t];
      sd0 += dxy * ux[t];
      sd1 += dxy * uy[t];
      sx1 += tx * uy[t];
      sx2 += tx * uz[t];
      sy0 += ty * ux[t];
      sy2 += ty * uz[t];
    }
  }
  T v0 = gz * sg0, v1 = gz * sg1, v2 = gz * sg2;
  T w0 = gdz * (sy2 - zk * sd1);
  T w1 = gdz * (zk * sd0 - sx2);
  T w2 = gdz * (sx1 - sy0);
  v0 = wave_sum(v0);
  v1 = wave_sum(v1);
  v2 = wave_sum(v2);
  w0 = wave_sum(w0);
  w1 = wave_sum(w1);
  w2 = wave_sum(w2);
  if (valid && lane == 0) {
    V[3 * s + 0] = dx3 * (double)v0;
    V[3 * s + 1] = dx3 * (double)v1;
    V[3 * s + 2] = dx3 * (double)v2;
    W[3 * s + 0] = -0.5 * dx3 * (double)w0;
    W[3 * s + 1] = -0.5 * dx3 * (double)w1;
    W[3 * s + 2] = -0.5 * dx3 * (double)w2;
  }
}

// ---------------------------------------------------------------------
// interpolation on the matrix cores: the transpose of k_spread_mfma. One
// workgroup per 8 x 8 x 16 tile reads the tile's three velocity grids once
// (each lane four consecutive z of one (x, y) column per component) and,
// for the segments of its tile list (up to 32 per round; each wave takes
// those with a stencil point in its rows, 16 per group), contracts them
// with each segment's weights:
//   P_m[xy][c] = sum_z u_d[xy][z] b_m,c[z]   (per wave 16 xy rows x 16
//   segments, v_mfma 16x16x4 over z; 8 products m: u_0..2 with g_z,
//   u_0..2 with gD_z, u_0..1 with the derivative h_z)
// then weights each (x, y) row with the segment's x and y factors, sums
// the lane's rows, the four lane groups and the four waves in a fixed
// order, and stores the tile's 6 partial sums per segment in
// part[segment][component][slot] (slot = the tile's offset from the
// segment's origin tile). k_interp_sum adds a segment's slots in slot
// order: no atomics, results independent of scheduling.
// Latency bound: of the FP64 270 us at 30k segments on 256^3 that the form with
// four wavefronts a SIMD took, the products were 90, the weights' reads from
// LDS 100, making the weights 50 and the grid's loads 50, one after another. So
// three accumulators at a time, which leaves registers for wavefronts: FP32
// four a SIMD (125 -> 117 us; five the same, six spill: 170 us), FP64 three
// (297 -> 224 us, two the same, four spill: 269 us; 128^3 55 -> 43 us). One
// wavefront to a tile 257 / 140 us, and slower on small grids; weights read 16
// bytes at a time 313 / 125 us (spills).
// ---------------------------------------------------------------------
// Wavefronts a SIMD that the interpolation's registers leave room for.
template <typename T>
constexpr int kInterpWaves = sizeof(T) == 8 ? 3 : 4;

template <int NGD>
constexpr int kInterpSlots = stencil_tiles(NGD, 8) * stencil_tiles(NGD, 8) *
                             stencil_tiles(NGD, 16);

// Four consecutive reals at p (16-byte aligned).
template <typename T>
__device__ __forceinline__ void ld4(const T *p, T *out) {
  ld16(p, out);
  if constexpr (sizeof(T) == 8) ld16(p + 2, out + 2);
}

template <typename T, typename SG = SpreadGeom, typename GC = GaussConst>
__device__ __forceinline__ void d_interp_mfma(const int *__restrict__ act, SG G, GC g,
                  const SegRec<T> *__restrict__ slab,
                  const SegRec<T> *__restrict__ pool,
                  const int *__restrict__ tcnt, const int *__restrict__ tovf,
                  const T *__restrict__ R, T *__restrict__ part) {
  typedef typename Mfma<T>::v4 v4;
  constexpr int KC = kTileCap;  // candidates per round
  const int nslot = G.sx * G.sy * G.sz;
  if (act && !*act) return;  // batched sweep: suspension converged
  __shared__ SegRec<T> s_rec[kTileCap];
  __shared__ T s_w[KC + 1][kTileW];  // row KC stays zero
  __shared__ T s_red[4][KC][8];  // 6 sums; two more keep the stores uniform
  __shared__ int s_wl[4][KC + 16];  // each wave's candidate list

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int q = lane >> 4, i16 = lane & 15;
  const int ntiles = G.nbx * G.nby * G.nbz;
  const size_t N = (size_t)G.nx * G.ny * G.nz;
  for (int e = threadIdx.x; e < kTileW; e += 256) s_w[KC][e] = 0;
  // persistent: block b takes tiles b, b + gridDim.x, ... (gridDim.x <=
  // ntiles, a multiple of 8 so each block's tiles stay on its XCD's run)
  int v = blockIdx.x;
  TilePrefetch<T> pf;
  {
    int bx, by, bz;
    tile_of_block(G, v, &bx, &by, &bz);
    pf.load(slab, tcnt, bx + G.nbx * (by + G.nby * bz));
  }
  for (; v < ntiles; v += gridDim.x) {
    int bx, by, bz;
    tile_of_block(G, v, &bx, &by, &bz);
    const int tile = bx + G.nbx * (by + G.nby * bz);
    const int px0 = bx * 8, py0 = by * 8, pz0 = bz * 16;
    // A operands: u_d[xy = wave*16 + i16][z = pz0 + 4q + k] for K step k
    // (lane group q supplies z 4q .. 4q + 3); in flight during the weights
    T u[3][4];
    {
      const int xy = wave * 16 + i16;
      const size_t o = ((size_t)(px0 + (xy >> 3)) * G.ny + py0 + (xy & 7)) * G.nz +
                       pz0 + 4 * q;
      if (px0 + 8 <= G.nx && py0 + 8 <= G.ny && pz0 + 16 <= G.nz &&
          (sizeof(T) == 8 || (G.nz & 3) == 0)) {
        ld4(R + o, u[0]);
        ld4(R + N + o, u[1]);
        ld4(R + 2 * N + o, u[2]);
      } else {  // a cut tile, or lines that are not 16-byte aligned
        const bool in = px0 + (xy >> 3) < G.nx && py0 + (xy & 7) < G.ny;
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            u[d][k] = in && pz0 + 4 * q + k < G.nz ? R[d * N + o + k] : (T)0;
      }
    }
    const int cnt = pf.cnt;
    __syncthreads();  // the last tile is done with s_rec, s_w and s_red
    pf.store(s_rec);
    if (v + (int)gridDim.x < ntiles) {
      int nx_, ny_, nz_;
      tile_of_block(G, v + gridDim.x, &nx_, &ny_, &nz_);
      pf.load(slab, tcnt, nx_ + G.nbx * (ny_ + G.nby * nz_));
    }
    const int ovf = cnt > kTileCap ? tovf[tile] : 0;

    for (int r0 = 0; r0 < cnt; r0 += kTileCap) {
      const int nc = min(kTileCap, cnt - r0);
      if (r0 > 0) {
        __syncthreads();  // the last round still reads s_rec
        stage_tile_records<T>(slab, pool, tile, ovf, r0, nc, s_rec);
      }
      __syncthreads();
      tile_chunk_weights<T, false>(g, s_rec, 0, nc, px0, py0, pz0, s_w);
      __syncthreads();
      // the wave handles its own candidates, 16 per group, and leaves zeros
      // for the others
      {
        for (int e = lane; e < KC * 8; e += 64) (&s_red[wave][0][0])[e] = 0;
        const int nw = wave_candidates<T, KC>(s_w, nc, wave, lane, 16, s_wl[wave]);
        for (int g0 = 0; g0 < nw; g0 += 16) {
          // B operands: this lane's column is the wave's candidate g0 + i16
          const int c = s_wl[wave][g0 + i16];
          const T *w = s_w[c];
          // the monopole, dipole and derivative products one after another:
          // three accumulators live at a time leave room for twice the
          // wavefronts. Lane holds P[xy = wave*16 + row(lane, r)][candidate
          // c] and weights each row with the candidate's x/y factors.
          const v4 z4 = {0, 0, 0, 0};
          T v0 = 0, v1 = 0, v2 = 0, w0 = 0, w1 = 0, w2 = 0;
          {
            v4 p0 = z4, p1 = z4, p2 = z4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const T gz = w[16 + 4 * q + k];
              p0 = Mfma<T>::step(u[0][k], gz, p0);
              p1 = Mfma<T>::step(u[1][k], gz, p1);
              p2 = Mfma<T>::step(u[2][k], gz, p2);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int rxy = wave * 16 + Mfma<T>::row(lane, r);
              const T gxy = w[rxy >> 3] * w[8 + (rxy & 7)];
              v0 += gxy * p0[r];
              v1 += gxy * p1[r];
              v2 += gxy * p2[r];
            }
          }
          {
            v4 p0 = z4, p1 = z4, p2 = z4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const T dz = w[48 + 4 * q + k];
              p0 = Mfma<T>::step(u[0][k], dz, p0);
              p1 = Mfma<T>::step(u[1][k], dz, p1);
              p2 = Mfma<T>::step(u[2][k], dz, p2);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int rxy = wave * 16 + Mfma<T>::row(lane, r);
              const int x = rxy >> 3, y = rxy & 7;
              const T dhy = w[32 + x] * w[72 + y], hdy = w[64 + x] * w[40 + y];
              w0 += dhy * p2[r];
              w1 -= hdy * p2[r];
              w2 += hdy * p1[r] - dhy * p0[r];
            }
          }
          {
            v4 p0 = z4, p1 = z4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const T hz = w[80 + 4 * q + k];
              p0 = Mfma<T>::step(u[0][k], hz, p0);
              p1 = Mfma<T>::step(u[1][k], hz, p1);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int rxy = wave * 16 + Mfma<T>::row(lane, r);
              const T dxy = w[32 + (rxy >> 3)] * w[40 + (rxy & 7)];
              w0 -= dxy * p1[r];
              w1 += dxy * p0[r];
            }
          }
          // the four lane groups (rows) of the wave: group q gets sums q and
          // 4 + q
          const T a = lane_reduce4<T>(v0, v1, v2, w0);
          const T b = lane_reduce4<T>(w1, w2, (T)0, (T)0);
          if (c < KC) {
            s_red[wave][c][q] = a;
            s_red[wave][c][4 + q] = b;
          }
        }
      }
      __syncthreads();
      // the four waves in a fixed order
      if (threadIdx.x < KC * 6) {
        const int c = threadIdx.x / 6, m = threadIdx.x - 6 * c;
        if (c < nc) {
          const T sum = ((s_red[0][c][m] + s_red[1][c][m]) + s_red[2][c][m]) +
                        s_red[3][c][m];
          const SegRec<T> &rc = s_rec[c];
          int sx = bx - (rc.org & 1023) / 8, sy = by - ((rc.org >> 10) & 1023) / 8,
              sz = bz - (rc.org >> 20) / 16;
          if (sx < 0) sx += G.nbx;
          if (sy < 0) sy += G.nby;
          if (sz < 0) sz += G.nbz;
          part[((size_t)rc.id * 6 + m) * nslot + (sx * G.sy + sy) * G.sz + sz] = sum;
        }
      }
    }
  }
}
template <typename T>
__global__ void __launch_bounds__(256, kInterpWaves<T>)
    k_interp_mfma(const int *__restrict__ act, SpreadGeom G, GaussConst g,
                  const SegRec<T> *__restrict__ slab,
                  const SegRec<T> *__restrict__ pool,
                  const int *__restrict__ tcnt, const int *__restrict__ tovf,
                  const T *__restrict__ R, T *__restrict__ part) {
  d_interp_mfma<T>(act, G, g, slab, pool, tcnt, tovf, R, part);
}
// arguments of one suspension for k_interp_mfma_multi
template <typename T>
struct A_interp_mfma {
  const int *act;
  SpreadGeom G;
  GaussConst g;
  const SegRec<T> *slab;
  const SegRec<T> *pool;
  const int *tcnt;
  const int *tovf;
  const T *R;
  T *part;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T>
__global__ void __launch_bounds__(256, kInterpWaves<T>)
    k_interp_mfma_multi(const A_interp_mfma<T> *__restrict__ a) {
  const A_interp_mfma<T> &A = a[blockIdx.z];
  d_interp_mfma<T, const SpreadGeom &, const GaussConst &>(A.act, A.G, A.g, A.slab, A.pool, A.tcnt, A.tovf, A.R, A.part);
}

// One thread per (segment, component): adds the segment's tile partials in
// slot order (only the tiles its stencil meets, the ones k_interp_mfma
// wrote) and scales them: V = dx^3 sum, Omega = -dx^3 / 2 sum
// (particle_velocities / particle_rotations, FCMfunctions.cpp:740-808).
template <typename T, int NGD, typename SG = SpreadGeom>
__device__ __forceinline__ void d_interp_sum(const int *__restrict__ act, int np, SG G,
                             double dx3, const int *__restrict__ origin,
                             const T *__restrict__ part,
                             double *__restrict__ V, double *__restrict__ W,
                             int *__restrict__ pool_top) {
  constexpr int SX = stencil_tiles(NGD, 8), SZ = stencil_tiles(NGD, 16);
  constexpr int NSLOT = kInterpSlots<NGD>;
  if (act && !*act) return;  // batched sweep: suspension converged
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  // the pool's counter for the next solve
  if (e == 0) *pool_top = 0;
  const int s = e / 6, m = e - 6 * s;
  if (s >= np) return;
  const int ox = origin[3 * s], oy = origin[3 * s + 1], oz = origin[3 * s + 2];
  double acc = 0;
  if (G.sx == SX && G.sy == SX && G.sz == SZ) {
    // every slot is read (in range); the ones no tile wrote are not added
    T v[NSLOT];
    const T *pp = part + ((size_t)s * 6 + m) * NSLOT;
#pragma unroll
    for (int k = 0; k < NSLOT; ++k) v[k] = pp[k];
#pragma unroll
    for (int sx = 0; sx < SX; ++sx) {
      int tx = ox / 8 + sx;
      if (tx >= G.nbx) tx -= G.nbx;
      const bool mx = sx < G.nbx && stencil_meets(ox, tx * 8, 8, NGD, G.nx);
#pragma unroll
      for (int sy = 0; sy < SX; ++sy) {
        int ty = oy / 8 + sy;
        if (ty >= G.nby) ty -= G.nby;
        const bool my = sy < G.nby && stencil_meets(oy, ty * 8, 8, NGD, G.ny);
#pragma unroll
        for (int sz = 0; sz < SZ; ++sz) {
          int tz = oz / 16 + sz;
          if (tz >= G.nbz) tz -= G.nbz;
          const bool mz = sz < G.nbz && stencil_meets(oz, tz * 16, 16, NGD, G.nz);
          if (mx && my && mz) acc += (double)v[(sx * SX + sy) * SZ + sz];
        }
      }
    }
  } else {  // cut tiles, one slot more on their axes
    const T *pp = part + ((size_t)s * 6 + m) * (G.sx * G.sy * G.sz);
    for (int sx = 0; sx < min(G.sx, G.nbx); ++sx) {
      int tx = ox / 8 + sx;
      if (tx >= G.nbx) tx -= G.nbx;
      if (!stencil_meets(ox, tx * 8, min(8, G.nx - tx * 8), NGD, G.nx)) continue;
      for (int sy = 0; sy < min(G.sy, G.nby); ++sy) {
        int ty = oy / 8 + sy;
        if (ty >= G.nby) ty -= G.nby;
        if (!stencil_meets(oy, ty * 8, min(8, G.ny - ty * 8), NGD, G.ny)) continue;
        for (int sz = 0; sz < min(G.sz, G.nbz); ++sz) {
          int tz = oz / 16 + sz;
          if (tz >= G.nbz) tz -= G.nbz;
          if (stencil_meets(oz, tz * 16, min(16, G.nz - tz * 16), NGD, G.nz))
            acc += (double)pp[(sx * G.sy + sy) * G.sz + sz];
        }
      }
    }
  }
  if (m < 3)
    V[3 * s + m] = dx3 * acc;
  else
    W[3 * s + m - 3] = -0.5 * dx3 * acc;
}
template <typename T, int NGD>
__global__ void k_interp_sum(const int *__restrict__ act, int np, SpreadGeom G,
                             double dx3, const int *__restrict__ origin,
                             const T *__restrict__ part,
                             double *__restrict__ V, double *__restrict__ W,
                             int *__restrict__ pool_top) {
  d_interp_sum<T, NGD>(act, np, G, dx3, origin, part, V, W, pool_top);
}
// arguments of one suspension for k_interp_sum_multi
template <typename T, int NGD>
struct A_interp_sum {
  const int *act;
  int np;
  SpreadGeom G;
  double dx3;
  const int *origin;
  const T *part;
  double *V;
  double *W;
  int *pool_top;
};
// one launch for a group of suspensions with equal launch shapes:
// blockIdx.z selects the suspension
template <typename T, int NGD>
__global__ void k_interp_sum_multi(const A_interp_sum<T, NGD> *__restrict__ a) {
  const A_interp_sum<T, NGD> &A = a[blockIdx.z];
  d_interp_sum<T, NGD, const SpreadGeom &>(A.act, A.np, A.G, A.dx3, A.origin, A.part, A.V, A.W, A.pool_top);
}

// ---------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------
// Compile-time length of an FFT plan's kernels: n = 2^LOGN for the compile-time
// plans, LOGN = 0 for the run-time plan.
template <typename F>
static bool with_LOGN(const FftPlan &pl, F f) {
  if (pl.E == 0) {
    f(std::integral_constant<int, 0>{});
    return true;
  }
  switch (p2_log(pl.n)) {
    case 6: f(std::integral_constant<int, 6>{}); return true;
    case 7: f(std::integral_constant<int, 7>{}); return true;
    case 8: f(std::integral_constant<int, 8>{}); return true;
    case 9: f(std::integral_constant<int, 9>{}); return true;
  }
  return false;
}

template <typename F>
static bool with_TZ(int tz, F f) {
  switch (tz) {
    case 4: f(std::integral_constant<int, 4>{}); return true;
    case 5: f(std::integral_constant<int, 5>{}); return true;
    case 6: f(std::integral_constant<int, 6>{}); return true;
    case 8: f(std::integral_constant<int, 8>{}); return true;
    case 10: f(std::integral_constant<int, 10>{}); return true;
    case 12: f(std::integral_constant<int, 12>{}); return true;
    case 16: f(std::integral_constant<int, 16>{}); return true;
  }
  return false;
}

template <typename F>
static bool with_NGD(int ngd, F f) {
  switch (ngd) {
    case 6: f(std::integral_constant<int, 6>{}); return true;
    case 8: f(std::integral_constant<int, 8>{}); return true;
    case 10: f(std::integral_constant<int, 10>{}); return true;
    case 12: f(std::integral_constant<int, 12>{}); return true;
    case 16: f(std::integral_constant<int, 16>{}); return true;
    case 20: f(std::integral_constant<int, 20>{}); return true;
    case 24: f(std::integral_constant<int, 24>{}); return true;
  }
  return false;
}

template <typename T>
int set_fft_lds_attr(const FftPlan &plx, const FftPlan &ply,
                     const FftPlan &plz) {
  const int lds_max = 160 * 1024;
  bool ok = true;
  ok &= with_LOGN(plz, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    (void)hipFuncSetAttribute((const void *)k_fft_z_r2c<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    (void)hipFuncSetAttribute((const void *)k_fft_z_c2r<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    (void)hipFuncSetAttribute((const void *)k_fft_z_r2c_multi<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    (void)hipFuncSetAttribute((const void *)k_fft_z_c2r_multi<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
  });
  ok &= with_LOGN(ply, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    (void)hipFuncSetAttribute((const void *)k_fft_y<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    (void)hipFuncSetAttribute((const void *)k_fft_y_multi<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
  });
  ok &= with_LOGN(plx, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    (void)hipFuncSetAttribute((const void *)k_fft_x_project<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    (void)hipFuncSetAttribute((const void *)k_fft_x_project_multi<T, LL>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
  });
  FS_CHECK(ok, FS_ERR_ARG, "no FFT register tile for these sizes");
  return FS_OK;
}

// Blocks of a persistent tile kernel (256 threads): as many as are resident
// on the device at once, a multiple of 8, at most one per tile.
template <typename K>
static int persistent_blocks(K kernel, int ntiles) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
          hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 256, 0) !=
          hipSuccess ||
      per < 1 || cus < 1)
    return ntiles;
  long b = (long)cus * per;
  b = std::max(8L, b - b % 8);
  return (int)std::min<long>(b, ntiles);
}

// Resident blocks of the persistent interpolation.
template <typename T>
int interp_blocks(const FcmImpl &f) {
  return persistent_blocks(k_interp_mfma<T>, f.nbins);
}

// Workgroups per row of tiles of the lists without bins: up to 16 tiles (one a
// wavefront) each, where that fills the chip.
static int direct_parts(const SpreadGeom &g) {
  return std::max(1, std::min(ceil_div(g.nbx, 16), 256 / (g.nby * g.nbz)));
}

// Gaussian constants of the spread, tables and interpolation.
static GaussConst gauss_const(const FcmImpl &f, int np) {
  const fs_fcm_params &p = f.p;
  GaussConst g;
  g.fine = f.fine_weights(np);
  g.dx = p.dx;
  double sigmadipsq = p.sigma_dip * p.sigma_dip;
  g.sigmadipsq = sigmadipsq;
  g.anormdip = 1.0 / std::sqrt(2.0 * kPi * sigmadipsq);
  g.anormdip2 = 2.0 * sigmadipsq;
  double sigmasq = p.sigma * p.sigma;
  g.anorm = 1.0 / std::sqrt(2.0 * kPi * sigmasq);
  g.anorm2 = 2.0 * sigmasq;
  g.ngd = p.ngd;
  g.ngdh = p.ngd / 2;
  g.e2 = 1.4426950408889634074 / g.anorm2;
  g.ed2 = 1.4426950408889634074 / g.anormdip2;
  g.nrsd = -1.0 / sigmadipsq;
  g.nx = p.nx;
  g.ny = p.ny;
  g.nz = p.nz;
  return g;
}

// Constants of the Stokes projection (flow_solve).
static ProjConst proj_const(const fs_fcm_params &p) {
  ProjConst pc;
  pc.nx = p.nx;
  pc.ny = p.ny;
  pc.nz = p.nz;
  pc.nh = p.nz / 2 + 1;
  pc.kfx = 2.0 * kPi / (p.nx * p.dx);
  pc.kfy = 2.0 * kPi / (p.ny * p.dx);
  pc.kfz = 2.0 * kPi / (p.nz * p.dx);
  pc.scale = 1.0 / ((double)p.nx * p.ny * p.nz * p.mu);
  return pc;
}

template <typename T>
int FcmImpl::run(int np, const double *Y, const double *F, const double *Tq,
                 double *V, double *W, hipStream_t st) {
  const GaussConst g = gauss_const(*this, np);

  hipEvent_t *pset = nullptr;  // this solve's profiling events
  if (prof) {
    while (prof_ev.size() < prof_used + 7) {
      hipEvent_t e = nullptr;
      FS_HIP(hipEventCreate(&e));
      prof_ev.push_back(e);
    }
    pset = prof_ev.data() + prof_used;
    prof_used += 7;
  }
  auto mark = [&](int i) {
    if (timing) (void)hipEventRecord(ev[i], st);
    if (pset) (void)hipEventRecord(pset[i], st);
  };
  // kernel boundaries (timing only); a boundary not recorded in this solve
  // marks a kernel the path does not have
  for (int i = 0; i < 11; ++i) kev_used[i] = false;
  auto kmark = [&](int i) {
    if (timing) {
      (void)hipEventRecord(kev[i], st);
      kev_used[i] = true;
    }
  };
  mark(0);
  kmark(0);
  const int ntiles = nbins;
  if (lists_direct(np)) {
    kmark(1);
    hipLaunchKernelGGL(k_tile_lists_direct<T>,
                       dim3(geom.nby * geom.nbz, direct_parts(geom)), dim3(1024), 0, st, act, np, geom, p.dx, Y, F, Tq,
                       origin.as<int>(), tslab.as<SegRec<T>>(), tcnt.as<int>(),
                       tovf.as<int>(), tpool.as<SegRec<T>>(),
                       bin_count.as<int>() + nbins);
  } else {
    // bin counting sort. The scan also zeroes the counts (and the pool counter
    // after them) for the next solve: they start zeroed (set_geometry) and
    // every solve leaves them so, so no fill pass is needed.
    if (!mfma_spread)  // the matrix-core kernels form their weights per tile
      hipLaunchKernelGGL(k_prepare_tab<T>, dim3(ceil_div((long)np * 3 * p.ngd, 256)),
                         dim3(256), 0, st, act, np, Y, g, tab.as<T>());
    hipLaunchKernelGGL(k_prepare<T>, dim3(ceil_div(np, 64)), dim3(64), 0, st, act, np,
                       Y, F, Tq, g, geom.tx, geom.ty, geom.tz, geom.nbx, geom.nby,
                       geom.nbz, origin.as<int>(),
                       mfma_spread ? (T *)nullptr : coef.as<T>(), bin.as<int>(),
                       bin_count.as<int>(), slot.as<int>());
    if (nbins <= kScanOneMax)
      FS_TRY(device_scan_one(act, bin_count.as<int>(), nbins, bin_start.as<int>(), 1, st));
    else
      FS_TRY(device_scan(bin_count.as<int>(), nbins, bin_start.as<int>(),
                         scan_tmp.as<int>(), 1, st));
    hipLaunchKernelGGL(k_scatter, dim3(ceil_div(np, 256)), dim3(256), 0, st, np,
                       bin.as<int>(), slot.as<int>(), bin_start.as<int>(),
                       ids.as<int>());
    hipLaunchKernelGGL(k_bin_order<T>, dim3(ceil_div(np, 64)), dim3(64), 0, st,
                       act, np, bin.as<int>(), bin_start.as<int>(), ids.as<int>(),
                       origin.as<int>(), Y, F, Tq, p.dx, p.ngd / 2,
                       mfma_spread ? srec.as<SegRec<T>>() : (SegRec<T> *)nullptr,
                       sorg.as<int>(), sids.as<int>());
    kmark(1);
    if (mfma_spread)
      hipLaunchKernelGGL(k_tile_lists<T>, dim3(ceil_div(ntiles, 4)), dim3(256), 0, st,
                         act, geom, bin_start.as<int>(), (const int *)sorg.as<int>(),
                         srec.as<SegRec<T>>(),
                         tslab.as<SegRec<T>>(), tcnt.as<int>(), tovf.as<int>(),
                         tpool.as<SegRec<T>>(), bin_count.as<int>() + nbins);
  }
  mark(1);
  if (mfma_spread) kmark(2);
  bool okz = true;
  if (mfma_spread)
    hipLaunchKernelGGL(k_spread_mfma<T>, dim3(ntiles), dim3(256), 0, st, act, geom,
                       g, tslab.as<SegRec<T>>(), tpool.as<SegRec<T>>(),
                       tcnt.as<int>(), tovf.as<int>(), R.as<T>());
  if (!mfma_spread)
    okz = with_TZ(geom.tz, [&](auto z) {
      constexpr int TZ = decltype(z)::value;
      hipLaunchKernelGGL((k_spread<T, TZ>), dim3(ntiles), dim3(geom.tx * geom.ty),
                         0, st, act, geom, tab.as<T>(), origin.as<int>(), coef.as<T>(),
                         bin_start.as<int>(), sids.as<int>(), R.as<T>());
    });
  FS_CHECK(okz, FS_ERR_ARG, "spread dispatch failed");
  FS_LAUNCHED();
  mark(2);
  kmark(3);
  const int nh = p.nz / 2 + 1;
  const size_t csz = sizeof(cx<T>);
  bool ok = with_LOGN(plz, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    hipLaunchKernelGGL((k_fft_z_r2c<T, LL>), dim3(p.ny * (p.nx / (2 * zP)), 3),
                       dim3(fft_threads(plz, zP)),
                       csz * (p.nz + (size_t)zP * fft_padded_len(p.nz)), st, act,
                       R.as<T>(), C.as<cx<T>>(), plz, twz.as<cx<T>>(), p.nx,
                       p.ny, zP, make_div(2 * zP), make_div(zP));
  });
  kmark(4);
  ok &= with_LOGN(ply, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    hipLaunchKernelGGL((k_fft_y<T, LL>), dim3(nh * (p.nx / yB), 3),
                       dim3(fft_threads(ply, yB)), csz * (p.ny + (size_t)yB * fft_rowpad_len(p.ny)), st, act,
                       C.as<cx<T>>(), ply, twy.as<cx<T>>(), p.nx, nh, yB, 0,
                       make_div(yB));
  });
  FS_CHECK(ok, FS_ERR_ARG, "FFT dispatch failed");
  FS_LAUNCHED();
  mark(3);
  kmark(5);
  const ProjConst pc = proj_const(p);
  ok = with_LOGN(plx, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    hipLaunchKernelGGL((k_fft_x_project<T, LL>), dim3(nh * (p.ny / xQ)),
                       dim3(x_threads(plx, xQ)),
                       csz * x_lds_values(plx, xQ), st, act,
                       C.as<cx<T>>(),
                       plx, twx.as<cx<T>>(), pc, xQ, make_div(xQ));
  });
  FS_CHECK(ok, FS_ERR_ARG, "FFT dispatch failed");
  FS_LAUNCHED();
  mark(4);
  kmark(6);
  ok = with_LOGN(ply, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    hipLaunchKernelGGL((k_fft_y<T, LL>), dim3(nh * (p.nx / yB), 3),
                       dim3(fft_threads(ply, yB)), csz * (p.ny + (size_t)yB * fft_rowpad_len(p.ny)), st, act,
                       C.as<cx<T>>(), ply, twy.as<cx<T>>(), p.nx, nh, yB, 1,
                       make_div(yB));
  });
  kmark(7);
  ok &= with_LOGN(plz, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    hipLaunchKernelGGL((k_fft_z_c2r<T, LL>), dim3(p.ny * (p.nx / (2 * zP)), 3),
                       dim3(fft_threads(plz, zP)),
                       csz * (p.nz + (size_t)zP * fft_padded_len(p.nz)), st, act,
                       C.as<cx<T>>(), R.as<T>(), plz, twz.as<cx<T>>(), p.nx,
                       p.ny, zP, make_div(zP));
  });
  FS_CHECK(ok, FS_ERR_ARG, "FFT dispatch failed");
  FS_LAUNCHED();
  mark(5);
  kmark(8);
  double dx3 = p.dx * p.dx * p.dx;
  bool okn = with_NGD(p.ngd, [&](auto ng) {
    constexpr int NG = decltype(ng)::value;
    if (mfma_spread) {
      hipLaunchKernelGGL(k_interp_mfma<T>, dim3(grid_interp), dim3(256), 0,
                         st, act, geom, g, tslab.as<SegRec<T>>(),
                         tpool.as<SegRec<T>>(), tcnt.as<int>(), tovf.as<int>(),
                         R.as<T>(), ipart.as<T>());
      kmark(9);
      hipLaunchKernelGGL((k_interp_sum<T, NG>), dim3(ceil_div(6L * np, 256)),
                         dim3(256), 0, st, act, np, geom, dx3,
                         origin.as<int>(), ipart.as<T>(), V, W,
                         bin_count.as<int>() + nbins);
    } else {
      hipLaunchKernelGGL((k_interp<T, NG>),
                         dim3(8 * ceil_div(ceil_div(np, 4), 8)), dim3(256), 0,
                         st, act, np, geom, dx3, tab.as<T>(), origin.as<int>(),
                         sids.as<int>(), R.as<T>(), V, W);
    }
  });
  FS_CHECK(okn, FS_ERR_ARG, "interp dispatch failed");
  FS_LAUNCHED();
  mark(6);
  kmark(10);
  return FS_OK;
}

// ---------------------------------------------------------------------
// Batched sweep: the mobility solves of a group of suspensions with one
// launch per FCM stage. Members have equal launch shapes (same precision,
// grid, Gaussian support and tile/FFT shapes), so every stage's grid is the
// same for each member and blockIdx.z selects the member; the kernels are
// the single-solve kernels' bodies (the k_*_multi wrappers), so each
// member's results are bit-identical to its own solve. Segment counts may
// differ: segment-indexed stages launch for the largest and return past a
// member's own count. The argument tables are built once for fixed
// Y/F/T/V/W and loop-control pointers.
// ---------------------------------------------------------------------
struct A_scan_small {
  const int *act;
  int *cnt;
  int n;
  int *start;
};
// start[0..n] = exclusive scan of cnt[0..n) with one workgroup per member,
// which leaves cnt[0..n] zeroed as the single-solve path does: up to
// kScanOneMax bins the single-solve scan, else 1024-element chunks with a
// running carry
static __global__ void __launch_bounds__(1024)
    k_scan_small_multi(const A_scan_small *__restrict__ a) {
  const A_scan_small &A = a[blockIdx.z];
  if (A.n <= kScanOneMax) {
    d_scan_one(A.act, A.cnt, A.n, A.start, 1);
    return;
  }
  if (A.act && !*A.act) return;  // batched sweep: suspension converged
  __shared__ int s[1024];
  const int t = threadIdx.x;
  int carry = 0;
  for (int base = 0; base < A.n; base += 1024) {
    const int i = base + t;
    s[t] = (i < A.n) ? A.cnt[i] : 0;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      int v = (t >= off) ? s[t - off] : 0;
      __syncthreads();
      s[t] += v;
      __syncthreads();
    }
    if (i < A.n) {
      A.start[i] = carry + ((t == 0) ? 0 : s[t - 1]);
      A.cnt[i] = 0;
    }
    carry += s[1023];
    __syncthreads();  // s is rewritten by the next chunk
  }
  if (t == 0) {
    A.start[A.n] = carry;
    A.cnt[A.n] = 0;
  }
}

// One pass over the stages: with `host` set, appends each stage's argument
// table (256-byte aligned) and records its offset; otherwise launches each
// stage with its table in G.tab.
template <typename T>
int group_stages(FcmGroup &G, std::vector<char> *host, hipStream_t st) {
  const int S = (int)G.m.size();
  const FcmImpl &f0 = *G.m[0].fcm;
  const fs_fcm_params &p = f0.p;
  int npmax = 0;
  for (auto &m : G.m) npmax = std::max(npmax, m.np);
  const int nbins = f0.nbins, ntiles = f0.nbins, nh = p.nz / 2 + 1;
  const size_t csz = sizeof(cx<T>);
  size_t k = 0;  // stage index
  // table of stage k: build it (host) or return its device address
  auto table = [&](auto make) -> const void * {
    using A = decltype(make(G.m[0]));
    if (host) {
      size_t at = (host->size() + 255) & ~(size_t)255;
      host->resize(at + sizeof(A) * S);
      for (int i = 0; i < S; ++i) {
        A v = make(G.m[i]);
        std::memcpy(host->data() + at + sizeof(A) * i, &v, sizeof(A));
      }
      G.off.push_back(at);
      ++k;
      return nullptr;
    }
    return static_cast<const char *>(G.tab.p) + G.off[k++];
  };
  const GaussConst g = gauss_const(f0, G.m[0].np);
  const ProjConst pc = proj_const(p);
  const double dx3 = p.dx * p.dx * p.dx;
  if (f0.lists_direct(G.m[0].np)) {
    auto t = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_tile_lists_direct<T>{
          m.act, m.np, f.geom, p.dx, m.Y, m.F, m.T, f.origin.as<int>(),
          f.tslab.as<SegRec<T>>(), f.tcnt.as<int>(), f.tovf.as<int>(),
          f.tpool.as<SegRec<T>>(), f.bin_count.as<int>() + nbins};
    });
    if (!host)
      hipLaunchKernelGGL(k_tile_lists_direct_multi<T>,
                         dim3(f0.geom.nby * f0.geom.nbz, direct_parts(f0.geom), S),
                         dim3(1024), 0, st,
                         (const A_tile_lists_direct<T> *)t);
  } else {
    {
      auto t = table([&](const FcmGroupMember &m) {
        const FcmImpl &f = *m.fcm;
        return A_prepare<T>{m.act, m.np, m.Y, m.F, m.T, g, f.geom.tx, f.geom.ty,
                            f.geom.tz, f.geom.nbx, f.geom.nby, f.geom.nbz,
                            f.origin.as<int>(), nullptr, f.bin.as<int>(),
                            f.bin_count.as<int>(), f.slot.as<int>()};
      });
      if (!host)
        hipLaunchKernelGGL(k_prepare_multi<T>, dim3(ceil_div(npmax, 64), 1, S),
                           dim3(64), 0, st, (const A_prepare<T> *)t);
    }
    {
      auto t = table([&](const FcmGroupMember &m) {
        return A_scan_small{m.act, m.fcm->bin_count.as<int>(), nbins,
                            m.fcm->bin_start.as<int>()};
      });
      if (!host)
        hipLaunchKernelGGL(k_scan_small_multi, dim3(1, 1, S), dim3(1024), 0, st,
                           (const A_scan_small *)t);
    }
    {
      auto t = table([&](const FcmGroupMember &m) {
        const FcmImpl &f = *m.fcm;
        return A_scatter{m.np, f.bin.as<int>(), f.slot.as<int>(),
                         f.bin_start.as<int>(), f.ids.as<int>()};
      });
      if (!host)
        hipLaunchKernelGGL(k_scatter_multi, dim3(ceil_div(npmax, 256), 1, S),
                           dim3(256), 0, st, (const A_scatter *)t);
    }
    {
      auto t = table([&](const FcmGroupMember &m) {
        const FcmImpl &f = *m.fcm;
        return A_bin_order<T>{m.act, m.np, f.bin.as<int>(), f.bin_start.as<int>(),
                              f.ids.as<int>(), f.origin.as<int>(), m.Y, m.F, m.T,
                              p.dx, p.ngd / 2, f.srec.as<SegRec<T>>(),
                              f.sorg.as<int>()};
      });
      if (!host)
        hipLaunchKernelGGL(k_bin_order_multi<T>, dim3(ceil_div(npmax, 64), 1, S),
                           dim3(64), 0, st, (const A_bin_order<T> *)t);
      auto t2 = table([&](const FcmGroupMember &m) {
        const FcmImpl &f = *m.fcm;
        return A_tile_lists<T>{m.act, f.geom, f.bin_start.as<int>(), f.sorg.as<int>(),
                               f.srec.as<SegRec<T>>(), f.tslab.as<SegRec<T>>(),
                               f.tcnt.as<int>(), f.tovf.as<int>(),
                               f.tpool.as<SegRec<T>>(), f.bin_count.as<int>() + nbins};
      });
      if (!host)
        hipLaunchKernelGGL(k_tile_lists_multi<T>, dim3(ceil_div(ntiles, 4), 1, S),
                           dim3(256), 0, st, (const A_tile_lists<T> *)t2);
    }
  }
  {
    auto t = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_spread_mfma<T>{m.act, f.geom, g, f.tslab.as<SegRec<T>>(),
                              f.tpool.as<SegRec<T>>(), f.tcnt.as<int>(),
                              f.tovf.as<int>(), f.R.as<T>()};
    });
    if (!host)
      hipLaunchKernelGGL(k_spread_mfma_multi<T>, dim3(ntiles, 1, S), dim3(256), 0,
                         st, (const A_spread_mfma<T> *)t);
  }
  bool ok = with_LOGN(f0.plz, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    auto t = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_fft_z_r2c<T, LL>{m.act, f.R.as<T>(), f.C.as<cx<T>>(), f.plz,
                                    f.twz.as<cx<T>>(), p.nx, p.ny, f.zP,
                                    make_div(2 * f.zP), make_div(f.zP)};
    });
    if (!host)
      hipLaunchKernelGGL((k_fft_z_r2c_multi<T, LL>),
                         dim3(p.ny * (p.nx / (2 * f0.zP)), 3, S),
                         dim3(fft_threads(f0.plz, f0.zP)),
                         csz * (p.nz + (size_t)f0.zP * fft_padded_len(p.nz)), st,
                         (const A_fft_z_r2c<T, LL> *)t);
  });
  for (int inv = 0; inv < 2 && ok; ++inv) {
    ok &= with_LOGN(f0.ply, [&](auto l) {
      constexpr int LL = decltype(l)::value;
      auto t = table([&](const FcmGroupMember &m) {
        const FcmImpl &f = *m.fcm;
        return A_fft_y<T, LL>{m.act, f.C.as<cx<T>>(), f.ply, f.twy.as<cx<T>>(),
                                  p.nx, nh, f.yB, inv, make_div(f.yB)};
      });
      if (!host)
        hipLaunchKernelGGL((k_fft_y_multi<T, LL>),
                           dim3(nh * (p.nx / f0.yB), 3, S), dim3(fft_threads(f0.ply, f0.yB)),
                           csz * (p.ny + (size_t)f0.yB * fft_rowpad_len(p.ny)), st,
                           (const A_fft_y<T, LL> *)t);
    });
    if (inv == 0)
      ok &= with_LOGN(f0.plx, [&](auto l) {
        constexpr int LL = decltype(l)::value;
        auto t = table([&](const FcmGroupMember &m) {
          const FcmImpl &f = *m.fcm;
          return A_fft_x_project<T, LL>{m.act, f.C.as<cx<T>>(), f.plx,
                                            f.twx.as<cx<T>>(), pc, f.xQ,
                                            make_div(f.xQ)};
        });
        if (!host)
          hipLaunchKernelGGL((k_fft_x_project_multi<T, LL>),
                             dim3(nh * (p.ny / f0.xQ), 1, S),
                             dim3(x_threads(f0.plx, f0.xQ)),
                             csz * x_lds_values(f0.plx, f0.xQ),
                             st, (const A_fft_x_project<T, LL> *)t);
      });
  }
  ok &= with_LOGN(f0.plz, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    auto t = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_fft_z_c2r<T, LL>{m.act, f.C.as<cx<T>>(), f.R.as<T>(), f.plz,
                                    f.twz.as<cx<T>>(), p.nx, p.ny, f.zP,
                                    make_div(f.zP)};
    });
    if (!host)
      hipLaunchKernelGGL((k_fft_z_c2r_multi<T, LL>),
                         dim3(p.ny * (p.nx / (2 * f0.zP)), 3, S),
                         dim3(fft_threads(f0.plz, f0.zP)),
                         csz * (p.nz + (size_t)f0.zP * fft_padded_len(p.nz)), st,
                         (const A_fft_z_c2r<T, LL> *)t);
  });
  ok &= with_NGD(p.ngd, [&](auto ng) {
    constexpr int NG = decltype(ng)::value;
    auto t = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_interp_mfma<T>{m.act, f.geom, g, f.tslab.as<SegRec<T>>(),
                              f.tpool.as<SegRec<T>>(), f.tcnt.as<int>(),
                              f.tovf.as<int>(), f.R.as<T>(), f.ipart.as<T>()};
    });
    if (!host)
      hipLaunchKernelGGL(k_interp_mfma_multi<T>, dim3(f0.grid_interp, 1, S),
                         dim3(256), 0, st, (const A_interp_mfma<T> *)t);
    auto t2 = table([&](const FcmGroupMember &m) {
      const FcmImpl &f = *m.fcm;
      return A_interp_sum<T, NG>{m.act, m.np, f.geom, dx3, f.origin.as<int>(),
                                 f.ipart.as<T>(), m.V, m.W,
                                 f.bin_count.as<int>() + nbins};
    });
    if (!host)
      hipLaunchKernelGGL((k_interp_sum_multi<T, NG>),
                         dim3(ceil_div(6L * npmax, 256), 1, S), dim3(256), 0, st,
                         (const A_interp_sum<T, NG> *)t2);
  });
  FS_CHECK(ok, FS_ERR_ARG, "group FCM dispatch failed");
  if (!host) FS_LAUNCHED();
  return FS_OK;
}

}  // namespace fs
