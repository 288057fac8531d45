// scan.hpp -- device-wide exclusive scan of int counts (counting sorts of
// the spread bins and the barrier cells): block sums, then block-local scans
// with the block offsets; arrays of up to 16Ki counts in one workgroup instead.
#pragma once

#include "common.hpp"

namespace fs {

constexpr int kScanBlock = 1024;
constexpr int kScanMaxBlocks = 65536;  // up to 64Mi elements

namespace {  // each including translation unit gets its own kernels

// Four consecutive counts of a block (thread t of 256: lo + 4 t), zero past n.
__device__ __forceinline__ int4 scan_load(const int *__restrict__ cnt, int i,
                                          int n) {
  if (i + 4 <= n) return *reinterpret_cast<const int4 *>(cnt + i);
  return int4{i < n ? cnt[i] : 0, i + 1 < n ? cnt[i + 1] : 0,
              i + 2 < n ? cnt[i + 2] : 0, 0};
}

// Sum of v over 256 threads, on all of them.
__device__ __forceinline__ int scan_block_total(int v, int *wsum) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
  __syncthreads();
  return (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

__global__ void __launch_bounds__(256)
    k_scan_blocksum(const int *__restrict__ cnt, int n, int *__restrict__ bsum) {
  __shared__ int wsum[4];
  const int4 c = scan_load(cnt, blockIdx.x * kScanBlock + 4 * threadIdx.x, n);
  const int s = scan_block_total(c.x + c.y + c.z + c.w, wsum);
  if (threadIdx.x == 0) bsum[blockIdx.x] = s;
}

// Exclusive scan in place of nb block sums, 1024 at a time with a running
// carry; bsum[nb] = total.
__global__ void __launch_bounds__(1024) k_scan_top(int *__restrict__ bsum, int nb) {
  __shared__ int s[1024];
  const int t = threadIdx.x;
  int carry = 0;
  for (int base = 0; base < nb; base += 1024) {
    const int i = base + t;
    s[t] = (i < nb) ? bsum[i] : 0;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      int v = (t >= off) ? s[t - off] : 0;
      __syncthreads();
      s[t] += v;
      __syncthreads();
    }
    if (i < nb) bsum[i] = carry + ((t == 0) ? 0 : s[t - 1]);
    carry += s[1023];
    __syncthreads();  // s is rewritten by the next chunk
  }
  if (t == 0) bsum[nb] = carry;
}

// start of a block's 1,024 counts. bsum: the block sums, which the block adds
// up to its own (exclusive == 0), or their exclusive scan. clear != 0 zeroes
// the counts and the extra counter cnt[n] after they are read.
__global__ void __launch_bounds__(256)
    k_scan_apply(int *__restrict__ cnt, int n, const int *__restrict__ bsum,
                 int exclusive, int *__restrict__ start, int clear) {
  __shared__ int wsum[4], wpre[4];
  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int i = b * kScanBlock + 4 * t;
  const int4 c = scan_load(cnt, i, n);
  int base;
  if (exclusive) {
    base = bsum[b];
  } else {
    int v = 0;
    for (int k = t; k < b; k += 256) v += bsum[k];
    base = scan_block_total(v, wsum);
  }
  const int own = c.x + c.y + c.z + c.w;
  int x = own;  // inclusive prefix over the wavefront
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wpre[w] = x;
  __syncthreads();
  for (int k = 0; k < w; ++k) base += wpre[k];
  base += x - own;
  const int4 r = {base, base + c.x, base + c.x + c.y, base + c.x + c.y + c.z};
  if (i + 4 <= n) {
    *reinterpret_cast<int4 *>(start + i) = r;
    if (clear) *reinterpret_cast<int4 *>(cnt + i) = int4{0, 0, 0, 0};
  } else {
    const int v[4] = {r.x, r.y, r.z, r.w};
    for (int k = 0; k < 4; ++k)
      if (i + k < n) {
        start[i + k] = v[k];
        if (clear) cnt[i + k] = 0;
      }
  }
  if (b == (int)gridDim.x - 1 && t == 255) {
    start[n] = base + own;
    if (clear) cnt[n] = 0;
  }
}

// One-workgroup exclusive scan for short count arrays (n <= kScanOneMax):
// thread t holds the run [16 t, 16 t + 16) in registers (four 16-byte loads
// issued together), the 1024 run sums are scanned by wavefront prefix sums
// and one more over the 16 wavefront totals, then each thread writes its
// run's starts. With clear != 0 the counts cnt[0..n] (including the extra
// counter cnt[n]) are zeroed after they are read, so the next counting pass
// needs no fill kernel. act: loop-control flag (nullptr: always run; 0: the
// launch returns at once). cnt and start: 16-byte aligned.
constexpr int kScanOneMax = 16 * 1024;
__device__ __forceinline__ void d_scan_one(const int *__restrict__ act,
                                           int *__restrict__ cnt, int n,
                                           int *__restrict__ start, int clear) {
  if (act && !*act) return;
  __shared__ int wsum[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int lo = 16 * t;
  const bool full = lo + 16 <= n;
  int v[16];
  if (full) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 c = reinterpret_cast<const int4 *>(cnt + lo)[q];
      v[4 * q] = c.x;
      v[4 * q + 1] = c.y;
      v[4 * q + 2] = c.z;
      v[4 * q + 3] = c.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = lo + j < n ? cnt[lo + j] : 0;
  }
  int s = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) s += v[j];
  int x = s;  // inclusive prefix over the wavefront's runs
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  if (w == 0) {
    int u = lane < 16 ? wsum[lane] : 0;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      const int y = __shfl_up(u, off, 64);
      if (lane >= off) u += y;
    }
    if (lane < 16) wsum[lane] = u;
  }
  __syncthreads();
  int base = (w ? wsum[w - 1] : 0) + x - s;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int c = v[j];
    v[j] = base;
    base += c;
  }
  if (full) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      reinterpret_cast<int4 *>(start + lo)[q] =
          int4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      if (clear) reinterpret_cast<int4 *>(cnt + lo)[q] = int4{0, 0, 0, 0};
    }
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (lo + j < n) {
        start[lo + j] = v[j];
        if (clear) cnt[lo + j] = 0;
      }
  }
  if (t == 1023) start[n] = wsum[15];
  if (clear && t == 0) cnt[n] = 0;
}
__global__ void __launch_bounds__(1024)
    k_scan_one(const int *__restrict__ act, int *__restrict__ cnt, int n,
               int *__restrict__ start, int clear) {
  d_scan_one(act, cnt, n, start, clear);
}

}  // namespace

// start[0..n] = exclusive scan of cnt[0..n) in one workgroup (n <=
// kScanOneMax); clear != 0 also zeroes cnt[0..n].
inline int device_scan_one(const int *act, int *cnt, int n, int *start,
                           int clear, hipStream_t st) {
  FS_CHECK(n >= 1 && n <= kScanOneMax, FS_ERR_ARG,
           "one-workgroup scan of %d elements", n);
  hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(1024), 0, st, act, cnt, n, start,
                     clear);
  return FS_OK;
}

// start[0..n] = exclusive scan of cnt[0..n); scratch: >= n/1024 + 2 ints;
// clear != 0 also zeroes cnt[0..n]. Up to 4Mi counts a block adds the sums
// before its own itself (at most 16 loads a thread); above, a launch scans them
// first, which would take 6 us of latency for any number of sums. cnt and
// start: 16-byte aligned.
inline int device_scan(int *cnt, int n, int *start, int *scratch, int clear,
                       hipStream_t st) {
  const int nb = (n + kScanBlock - 1) / kScanBlock;
  FS_CHECK(nb >= 1 && nb <= kScanMaxBlocks, FS_ERR_ARG,
           "scan of %d elements too large", n);
  const int exclusive = nb > 4096;
  hipLaunchKernelGGL(k_scan_blocksum, dim3(nb), dim3(256), 0, st, cnt, n,
                     scratch);
  if (exclusive)
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, st, scratch, nb);
  hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(256), 0, st, cnt, n, scratch,
                     exclusive, start, clear);
  return FS_OK;
}

}  // namespace fs
