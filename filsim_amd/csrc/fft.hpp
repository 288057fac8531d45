// fft.hpp -- mixed-radix Stockham FFT exchanged through LDS.
//
// Replaces FFTW 2.1.5 rfftwnd (FCMfunctions.cpp:16-19, 360-406). A workgroup
// transforms `ncols` sequences of length n held in LDS; element (m, col) lives
// at buf[m*sm + col*sc]. A stage of radix R has n/R butterflies per
// sequence: butterfly j reads inputs j + r*n/R, twiddles them by
// W_{ns R}^{r (j mod ns)} and writes outputs (j/ns)*ns*R + (j mod ns) + r*ns
// (decimation in time, autosorting: the result is in natural order).
// Stages run in place: every thread holds its butterflies' values in
// registers across the barrier that separates the reads from the writes, so
// one LDS buffer holds the data. Transforms are unnormalised; sign -1
// forward, +1 inverse.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace fs {

constexpr int kMaxStages = 12;

// Division by a launch constant d without the integer divide sequence:
// q = (t * m) >> 32 with m = floor(2^32 / d) + 1 is exact for t < 2^16 and
// 1 <= d <= 2^16 (the error t * (m - 2^32/d) / 2^32 < 2^-16 <= 1/d never
// crosses an integer); every FFT index here is below 2^16.
struct FastDiv {
  unsigned long long m;
  int d;
  __device__ __forceinline__ int q(int t) const {
    return (int)(((unsigned long long)(unsigned)t * m) >> 32);
  }
};
inline FastDiv make_div(int d) {
  return FastDiv{(1ull << 32) / (unsigned long long)d + 1ull, d};
}

// Elements per thread of the compile-time plans.
constexpr int kP2E = 8;

struct FftPlan {
  int n;
  int nst;
  int E;  // kP2E: compile-time plan (lengths 2^LOGN below), 0: run-time plan
  int rad[kMaxStages];
  FastDiv dn;               // by n
  FastDiv dnb[kMaxStages];  // by n / rad[s]
  FastDiv dns[kMaxStages];  // by the stage's span ns (product of earlier radices)
};

// Elements per thread the run-time plan's workgroups are sized for: a stage
// of radix R gives every thread ceil(kGenE / R) butterflies (some idle when R
// does not divide kGenE). Threads used to hold whole multiples of
// lcm(radices) elements instead: 24 for a 192-point line (radices 8, 8, 3),
// 64 threads per 12 KB (FP32) of LDS, a third of the wavefronts this gives.
// Measured at 192^3, FP64, per pass: z 199 -> 97 us, y 180 / 126 -> 92 / 70,
// x + projection 225 -> 109, z inverse 153 -> 87 (FP32 92, 69 / 64, 107, 77 ->
// 53, 49 / 44, 73, 57).
constexpr int kGenE = 8;
// Register-heavy FP64 radices: 512 threads leave 256 VGPRs each.
template <typename T>
constexpr int kGenMaxThreads = sizeof(T) == 8 ? 512 : 1024;

// Threads of a workgroup that transforms ncols sequences of n.
inline int fft_threads(const FftPlan &p, int ncols) {
  if (p.E > 0) return p.n / p.E * ncols;
  return ((p.n * ncols + kGenE - 1) / kGenE + 63) / 64 * 64;
}
inline int fft_max_threads(const FftPlan &p, int tsz) {
  return p.E > 0 || tsz == 4 ? 1024 : 512;
}

// log2(n) for the lengths with compile-time plans, else 0.
inline int p2_log(int n) {
  return n == 64 ? 6 : n == 128 ? 7 : n == 256 ? 8 : n == 512 ? 9 : 0;
}

// Radices of a run-time plan, largest first: as few stages as possible (each
// is a round trip through LDS and a barrier), and among those the smallest
// largest radix (the registers of a butterfly).
inline bool gen_radices(int n, int maxr, int left, int *rad, int *nst,
                        int depth = 0) {
  static const int set[] = {16, 12, 10, 9, 8, 6, 5, 4, 3, 2};
  if (n == 1) {
    *nst = depth;
    return true;
  }
  if (left == 0) return false;
  for (int r : set)
    if (r <= maxr && n % r == 0) {
      rad[depth] = r;
      if (gen_radices(n / r, r, left - 1, rad, nst, depth + 1)) return true;
    }
  return false;
}

// Plan of n = 2^a 3^b 5^c. Lengths 64 to 512 that are powers of two take the
// compile-time plan: radix 8, then what is left. (Radix 16 there, two stages
// instead of three at 256 points, is within 3% of it in FP32 and 20% slower in
// FP64: a thread's 16 values leave half the wavefronts. A run-time plan's stage
// count decides, so 160 takes 16 x 10 and 192 takes 16 x 12.)
inline bool make_plan(int n, FftPlan *p) {
  int a = 0, m = n;
  while (m % 2 == 0) m /= 2, ++a;
  while (m % 3 == 0) m /= 3;
  while (m % 5 == 0) m /= 5;
  if (m != 1 || n < 2) return false;
  p->n = n;
  p->nst = 0;
  p->E = 0;
  if (p2_log(n)) {
    p->E = kP2E;
    while (a > 0) {
      const int l = a >= 3 ? 3 : a >= 2 ? 2 : 1;
      p->rad[p->nst++] = 1 << l;
      a -= l;
    }
  } else {
    bool ok = false;
    // at least two stages: the first reads global memory, the last writes it
    for (int st = 2; st <= kMaxStages && !ok; ++st)
      for (int maxr = 2; maxr <= 16 && !ok; ++maxr)
        ok = gen_radices(n, maxr, st, p->rad, &p->nst);
    if (!ok) return false;
  }
  p->dn = make_div(n);
  int ns = 1;
  for (int s = 0; s < p->nst; ++s) {
    p->dnb[s] = make_div(n / p->rad[s]);
    p->dns[s] = make_div(ns);
    ns *= p->rad[s];
  }
  return true;
}

// cos and sin of 2 pi k / n at compile time (Taylor series on the first
// octant, reduced exactly in integers).
constexpr double ct_series(double x, bool cosine) {
  double term = cosine ? 1.0 : x, sum = term;
  for (int i = cosine ? 1 : 2; i < 24; i += 2) {
    term = -term * x * x / (double)(i * (i + 1));
    sum += term;
  }
  return sum;
}
constexpr double ct_cos(int k, int n) {
  k = ((k % n) + n) % n;
  if (2 * k > n) k = n - k;                        // cos is even
  if (4 * k > n) return -ct_cos(n - 2 * k, 2 * n); // cos(pi - x) = -cos x
  constexpr double pi = 3.14159265358979323846264338327950288;
  if (8 * k > n) return ct_series(pi / 2 - 2 * pi * k / n, false);
  return ct_series(2 * pi * k / n, true);
}
constexpr double ct_sin(int k, int n) { return ct_cos(4 * k - n, 4 * n); }

// f(integral_constant I) for I = A .. B - 1
template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

template <typename T>
__device__ __forceinline__ cx<T> mul_mi(cx<T> a) {  // a * (-i)
  return {a.y, -a.x};
}
template <typename T>
__device__ __forceinline__ cx<T> mul_pi(cx<T> a) {  // a * (+i)
  return {-a.y, a.x};
}
template <typename T>
__device__ __forceinline__ cx<T> rot(cx<T> a, bool inv) {  // a * (-/+ i)
  return inv ? mul_pi(a) : mul_mi(a);
}

template <typename T>
__device__ __forceinline__ void dft2(cx<T> *v) {
  cx<T> a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <typename T>
__device__ __forceinline__ void dft4(cx<T> *v, bool inv) {
  cx<T> s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
  cx<T> s13 = cadd(v[1], v[3]), d13 = rot(csub(v[1], v[3]), inv);
  v[0] = cadd(s02, s13);
  v[2] = csub(s02, s13);
  v[1] = cadd(d02, d13);
  v[3] = csub(d02, d13);
}

template <typename T>
__device__ __forceinline__ void dft8(cx<T> *v, bool inv) {
  const T h = (T)0.70710678118654752440084436210485;
  cx<T> e[4] = {v[0], v[2], v[4], v[6]};
  cx<T> o[4] = {v[1], v[3], v[5], v[7]};
  dft4(e, inv);
  dft4(o, inv);
  // W8^k, forward: (1-i)/sqrt2, -i, (-1-i)/sqrt2; inverse conjugated
  cx<T> o1 = inv ? cx<T>{h * (o[1].x - o[1].y), h * (o[1].x + o[1].y)}
                 : cx<T>{h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
  cx<T> o2 = rot(o[2], inv);
  cx<T> o3 = inv ? cx<T>{-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y)}
                 : cx<T>{h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}

// 16 points as 4 x 4: DFT4 over n1 for each n2, twiddle by W16^(n2 k1),
// DFT4 over n2; natural order in and out.
template <typename T>
__device__ __forceinline__ void dft16(cx<T> *v, bool inv) {
  const T c = (T)0.92387953251128675612818318939679;  // cos(pi/8)
  const T s = (T)0.38268343236508977172845998403040;  // sin(pi/8)
  const T h = (T)0.70710678118654752440084436210485;
  const T sg = inv ? (T)1 : (T)-1;  // sign of the imaginary parts
  cx<T> y[4][4];
#pragma unroll
  for (int n2 = 0; n2 < 4; ++n2) {
    cx<T> t[4] = {v[n2], v[4 + n2], v[8 + n2], v[12 + n2]};
    dft4(t, inv);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) y[n2][k1] = t[k1];
  }
  const cx<T> w1 = {c, sg * s}, w2 = {h, sg * h}, w3 = {s, sg * c},
              w6 = {-h, sg * h}, w9 = {-c, -sg * s};
  y[1][1] = cmul(y[1][1], w1);
  y[1][2] = cmul(y[1][2], w2);
  y[1][3] = cmul(y[1][3], w3);
  y[2][1] = cmul(y[2][1], w2);
  y[2][2] = rot(y[2][2], inv);  // W16^4 = -i (forward)
  y[2][3] = cmul(y[2][3], w6);
  y[3][1] = cmul(y[3][1], w3);
  y[3][2] = cmul(y[3][2], w6);
  y[3][3] = cmul(y[3][3], w9);
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    cx<T> t[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
    dft4(t, inv);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = t[k2];
  }
}

template <typename T>
__device__ __forceinline__ void dft3(cx<T> *v, bool inv) {
  const T s3 = (T)0.86602540378443864676372317075294;
  cx<T> t1 = cadd(v[1], v[2]);
  cx<T> t2 = {v[0].x - (T)0.5 * t1.x, v[0].y - (T)0.5 * t1.y};
  cx<T> d = csub(v[1], v[2]);
  cx<T> t3 = rot(cx<T>{s3 * d.x, s3 * d.y}, inv);
  v[0] = cadd(v[0], t1);
  v[1] = cadd(t2, t3);
  v[2] = csub(t2, t3);
}

template <typename T>
__device__ __forceinline__ void dft5(cx<T> *v, bool inv) {
  const T c1 = (T)0.30901699437494742410229341718282;
  const T c2 = (T)-0.80901699437494742410229341718282;
  const T s1 = (T)0.95105651629515357211643933337938;
  const T s2 = (T)0.58778525229247312916870595463907;
  cx<T> t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
  cx<T> t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
  cx<T> a0 = v[0];
  cx<T> b1 = {a0.x + c1 * t1.x + c2 * t2.x, a0.y + c1 * t1.y + c2 * t2.y};
  cx<T> b2 = {a0.x + c2 * t1.x + c1 * t2.x, a0.y + c2 * t1.y + c1 * t2.y};
  cx<T> d1 = {s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y};
  cx<T> d2 = {s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y};
  cx<T> r1 = rot(d1, inv), r2 = rot(d2, inv);
  v[0] = {a0.x + t1.x + t2.x, a0.y + t1.y + t2.y};
  v[1] = cadd(b1, r1);
  v[4] = csub(b1, r1);
  v[2] = cadd(b2, r2);
  v[3] = csub(b2, r2);
}

template <typename T, int R>
__device__ __forceinline__ void dftR(cx<T> *v, bool inv);

// R1 R2 points: R1-point transforms over n1 of v[R2 n1 + n2], twiddles
// W^(n2 k1), R2-point transforms over n2; natural order in and out.
template <typename T, int R1, int R2>
__device__ __forceinline__ void dft_comp(cx<T> *v, bool inv) {
  constexpr int R = R1 * R2;
  cx<T> y[R2][R1];
#pragma unroll
  for (int n2 = 0; n2 < R2; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) y[n2][n1] = v[R2 * n1 + n2];
    dftR<T, R1>(y[n2], inv);
  }
  static_for<1, R2>([&](auto n2) {
    static_for<1, R1>([&](auto k1) {
      constexpr int m = n2() * k1();
      constexpr double c = ct_cos(m, R), s = ct_sin(m, R);
      y[n2()][k1()] = cmul(y[n2()][k1()], cx<T>{(T)c, inv ? (T)s : (T)-s});
    });
  });
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) {
    cx<T> u[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) u[n2] = y[n2][k1];
    dftR<T, R2>(u, inv);
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) v[k1 + R1 * k2] = u[k2];
  }
}

template <typename T, int R>
__device__ __forceinline__ void dftR(cx<T> *v, bool inv) {
  if constexpr (R == 2) dft2(v);
  if constexpr (R == 3) dft3(v, inv);
  if constexpr (R == 4) dft4(v, inv);
  if constexpr (R == 5) dft5(v, inv);
  if constexpr (R == 6) dft_comp<T, 3, 2>(v, inv);
  if constexpr (R == 8) dft8(v, inv);
  if constexpr (R == 9) dft_comp<T, 3, 3>(v, inv);
  if constexpr (R == 10) dft_comp<T, 5, 2>(v, inv);
  if constexpr (R == 12) dft_comp<T, 4, 3>(v, inv);
  if constexpr (R == 16) dft16(v, inv);
}

// Padded LDS layout for contiguous sequences: element i of a sequence sits at
// i + i / G (G = 2^FS_FFT_PAD_SHIFT elements per pad group). Early Stockham
// stages write with a lane stride of R elements (d = j*R + r); unpadded,
// 16 (FP32) or 32 (FP64) lanes of a wave would hit one bank. One pad
// element per group spreads those strided writes over the banks, and
// contiguous reads stay (nearly) conflict-free. Sequences follow each other
// at fft_padded_len(n), rounded up to FS_FFT_STRIDE_MOD modulo 32 elements
// when that is set, so that lanes reading the same position of different
// sequences do not share banks.
// The defaults were chosen with the LDS bank-conflict counter on gfx950
// (64 banks of 4 bytes; an 8-byte access serves 32 lanes per cycle, a
// 16-byte one 16): one pad per 16 elements and a stride of 18 modulo 32.
#ifndef FS_FFT_PAD_SHIFT
#define FS_FFT_PAD_SHIFT 4
#endif
#ifndef FS_FFT_STRIDE_MOD
#define FS_FFT_STRIDE_MOD 18
#endif
constexpr int kFftPadGroup = 1 << FS_FFT_PAD_SHIFT;
__host__ __device__ __forceinline__ constexpr int fft_pad(int i) {
  return i + (i >> FS_FFT_PAD_SHIFT);
}
__host__ __device__ __forceinline__ constexpr int fft_padded_len(int n) {
  int l = fft_pad(n - 1) + 1;
  if (FS_FFT_STRIDE_MOD >= 0)
    while (l % 32 != FS_FFT_STRIDE_MOD) ++l;
  return l;
}

// Threads and LDS (complex values) of an x pass workgroup of Q lines: the
// compile-time plans' threads hold the three components, the run-time plan's
// LDS does.
inline int x_threads(const FftPlan &pl, int Q) {
  return pl.E > 0 ? pl.n / pl.E * Q : fft_threads(pl, 3 * Q);
}
inline size_t x_lds_values(const FftPlan &pl, int Q) {
  return pl.n + (size_t)(pl.E > 0 ? 1 : 3) * Q * fft_padded_len(pl.n);
}

// Element-major layout (element m of every sequence in one row of sm): row
// m sits at row m + m / 8, so rows 8 apart (the lanes of a radix-8 stage's
// writes) fall on different banks.
__host__ __device__ __forceinline__ constexpr int fft_rowpad(int m) {
  return m + (m >> 3);
}
__host__ __device__ __forceinline__ constexpr int fft_rowpad_len(int n) {
  return fft_rowpad(n - 1) + 1;
}

// LDS index of element i of sequence col: sequences contiguous and padded
// (PAD, stride sc = padded length) or element-major
// (fft_rowpad(i) * sm + col * sc)
template <bool PAD>
__device__ __forceinline__ int lds_idx(int i, int col, int sm, int sc) {
  return PAD ? col * sc + fft_pad(i) : fft_rowpad(i) * sm + col * sc;
}

// Where a stage reads or writes: LdsIO is the LDS buffer (element i of
// sequence col), any other functor global memory, value ld(i, col) and
// st(i, col, value). A pass's first stage reads global memory into its
// registers and its last stage writes it, instead of staging the lines in LDS
// before and after: one LDS round trip and barrier pair less at either end
// (192^3 FP64 y pass 92 / 70 -> 64 / 59 us; 256^3 FP64 189 / 167 -> 172 / 155).
template <typename T, bool PAD>
struct LdsIO {
  cx<T> *buf;
  int sm, sc;
  __device__ __forceinline__ cx<T> operator()(int i, int col) const {
    return buf[lds_idx<PAD>(i, col, sm, sc)];
  }
  __device__ __forceinline__ void operator()(int i, int col, cx<T> v) const {
    buf[lds_idx<PAD>(i, col, sm, sc)] = v;
  }
};

// One stage of the run-time plan; blockDim.x * kGenE >= n * ncols. SYNC: a
// barrier between the reads and the writes (both of the same LDS buffer).
template <typename T, int R, bool PAD, bool INV, bool SYNC, typename LD,
          typename ST>
__device__ __forceinline__ void fft_stage(int ns, int ncols, const cx<T> *tw,
                                          FastDiv dnb, FastDiv dns, FastDiv dcols,
                                          LD ld, ST st) {
  constexpr int NB = (kGenE + R - 1) / R;
  const int nb = dnb.d;
  const int nbf = nb * ncols;
  const int twstep = dns.q(nb);  // n / (ns R)
  cx<T> v[NB * R];
  int jj[NB], cc[NB];
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int t = threadIdx.x + m * blockDim.x;
    if constexpr (PAD) {  // butterflies fastest
      cc[m] = dnb.q(t);
      jj[m] = t - cc[m] * nb;
    } else {  // columns fastest
      jj[m] = dcols.q(t);
      cc[m] = t - jj[m] * ncols;
    }
    if (t < nbf) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[m * R + r] = ld(jj[m] + r * nb, cc[m]);
    }
  }
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int t = threadIdx.x + m * blockDim.x;
    if (t < nbf) {
      const int j = jj[m], jq = dns.q(j), k = j - jq * ns;
      if (ns > 1) {
        const int kt = k * twstep;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = tw[r * kt];
          if constexpr (INV) w.y = -w.y;
          v[m * R + r] = cmul(v[m * R + r], w);
        }
      }
      dftR<T, R>(&v[m * R], INV);
      jj[m] = jq * ns * R + k;  // element of output 0
    }
  }
  if constexpr (SYNC) __syncthreads();
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int t = threadIdx.x + m * blockDim.x;
    if (t < nbf) {
#pragma unroll
      for (int r = 0; r < R; ++r) st(jj[m] + r * ns, cc[m], v[m * R + r]);
    }
  }
}

#define FS_RADICES(X) X(16) X(12) X(10) X(9) X(8) X(6) X(5) X(4) X(3) X(2)

// All stages of the run-time plan (fft_threads threads), the first reading
// from ld, the last writing to st, the others in place in LDS. Ends without a
// barrier after the last writes.
template <typename T, bool PAD, bool INV, typename LD, typename ST>
__device__ void lds_fft_plan(LdsIO<T, PAD> io, const FftPlan &pl, int ncols,
                             const cx<T> *tw, FastDiv dcols, LD ld, ST st) {
  constexpr bool same = std::is_same<LD, LdsIO<T, PAD>>::value;
  constexpr bool into = std::is_same<ST, LdsIO<T, PAD>>::value;
  int ns = 1;
  for (int s = 0; s < pl.nst; ++s) {
    const int R = pl.rad[s];
    const FastDiv a = pl.dnb[s], b = pl.dns[s];
    if (s == 0) {
      switch (R) {
#define FS_STAGE(RR)                                                           \
  case RR:                                                                     \
    fft_stage<T, RR, PAD, INV, same>(ns, ncols, tw, a, b, dcols, ld, io);      \
    break;
        FS_RADICES(FS_STAGE)
#undef FS_STAGE
      }
      __syncthreads();
    } else if (s + 1 < pl.nst) {
      switch (R) {
#define FS_STAGE(RR)                                                           \
  case RR:                                                                     \
    fft_stage<T, RR, PAD, INV, true>(ns, ncols, tw, a, b, dcols, io, io);      \
    break;
        FS_RADICES(FS_STAGE)
#undef FS_STAGE
      }
      __syncthreads();
    } else {
      switch (R) {
#define FS_STAGE(RR)                                                           \
  case RR:                                                                     \
    fft_stage<T, RR, PAD, INV, into>(ns, ncols, tw, a, b, dcols, io, st);      \
    break;
        FS_RADICES(FS_STAGE)
#undef FS_STAGE
      }
    }
    ns *= R;
  }
}

// --- n = 2^LOGN with the plan fixed at compile time ------------------------
// Same stages as make_plan (radix 8, then what is left), so the same arithmetic; spans, butterfly counts, twiddle steps
// and padded offsets are constants: divisions become shifts and masks, and
// the R addresses of a butterfly are one base plus immediate offsets.

constexpr int ilog2_c(int v) { return v <= 1 ? 0 : 1 + ilog2_c(v / 2); }

template <int LOGN, int LOGNS>
constexpr int p2_radix() {
  return LOGN - LOGNS >= 3 ? 8 : LOGN - LOGNS >= 2 ? 4 : 2;
}

template <typename T, bool PAD, bool INV, int LOGN, int LOGNS,
          typename LD, typename ST>
__device__ __forceinline__ void p2_stage(LdsIO<T, PAD> io, int ncols,
                                         const cx<T> *tw, FastDiv dcols, LD ld,
                                         ST st) {
  constexpr int R = p2_radix<LOGN, LOGNS>();
  constexpr int LOGR = ilog2_c(R);
  constexpr int NB = kP2E / R;
  constexpr int LOGNB = LOGN - LOGR;
  constexpr int nb = 1 << LOGNB;
  constexpr int ns = 1 << LOGNS;
  constexpr int LOGTW = LOGN - LOGNS - LOGR;  // twiddle step n / (ns R)
  constexpr int PN = fft_padded_len(1 << LOGN);
  constexpr bool from_lds =
      LOGNS > 0 || std::is_same<LD, LdsIO<T, PAD>>::value;
  constexpr bool to_lds =
      LOGNS + LOGR < LOGN || std::is_same<ST, LdsIO<T, PAD>>::value;
  cx<T> *buf = io.buf;
  const int sm = io.sm;
  cx<T> v[kP2E];
  int jj[NB], cc[NB];
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int t = threadIdx.x + m * blockDim.x;
    int j, col;
    if constexpr (PAD) {  // sequences contiguous: butterflies fastest
      col = t >> LOGNB;
      j = t & (nb - 1);
    } else {  // sequences interleaved (element m of column c in row m)
      j = dcols.q(t);
      col = t - j * ncols;
    }
    jj[m] = j;
    cc[m] = col;
    if constexpr (!from_lds) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[m * R + r] = ld(j + r * nb, col);
    } else if constexpr (PAD) {
      const cx<T> *src = buf + col * PN;
      const int pj = fft_pad(j);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int idx;
        if constexpr (nb % kFftPadGroup == 0)
          idx = pj + fft_pad(r * nb);
        else
          idx = fft_pad(j + r * nb);
        v[m * R + r] = src[idx];
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        v[m * R + r] = buf[fft_rowpad(j + r * nb) * sm + col];
    }
  }
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int k = jj[m] & (ns - 1);
    if constexpr (LOGNS > 0) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        cx<T> w = tw[(r * k) << LOGTW];
        if constexpr (INV) w.y = -w.y;
        v[m * R + r] = cmul(v[m * R + r], w);
      }
    }
    dftR<T, R>(&v[m * R], INV);
  }
  if constexpr (from_lds && to_lds) __syncthreads();
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int j = jj[m], col = cc[m];
    const int d = ((j >> LOGNS) << (LOGNS + LOGR)) + (j & (ns - 1));
    if constexpr (!to_lds) {
#pragma unroll
      for (int r = 0; r < R; ++r) st(d + r * ns, col, v[m * R + r]);
    } else if constexpr (PAD) {
      cx<T> *dst = buf + col * PN;
      const int pd = fft_pad(d);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int idx;
        if constexpr (ns % kFftPadGroup == 0)
          idx = pd + fft_pad(r * ns);
        else
          idx = fft_pad(d + r * ns);
        dst[idx] = v[m * R + r];
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        buf[fft_rowpad(d + r * ns) * sm + col] = v[m * R + r];
    }
  }
  if constexpr (LOGNS + LOGR < LOGN) {
    __syncthreads();
    p2_stage<T, PAD, INV, LOGN, LOGNS + LOGR>(io, ncols, tw, dcols, ld, st);
  }
}

// The transform for kernels instantiated on LOGN: LOGN > 0 takes the
// compile-time plan (n = 2^LOGN, PAD: sc = fft_padded_len(n)), LOGN = 0 the
// run-time plan pl. The first stage reads from ld, the last writes to st:
// global memory, or io for LDS. No barrier after the last writes.
template <typename T, bool PAD, bool INV, int LOGN, typename LD,
          typename ST>
__device__ __forceinline__ void lds_fft(LdsIO<T, PAD> io, const FftPlan &pl,
                                        int ncols, const cx<T> *tw, LD ld, ST st,
                                        FastDiv dcols = FastDiv{0, 0}) {
  if constexpr (LOGN > 0)
    p2_stage<T, PAD, INV, LOGN, 0>(io, ncols, tw, dcols, ld, st);
  else
    lds_fft_plan<T, PAD, INV>(io, pl, ncols, tw, dcols, ld, st);
}

}  // namespace fs
