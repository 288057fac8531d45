// fcm.hip -- Force Coupling Method mobility solve for gfx950.
//
// Replaces Fcm::mobility_solve (FCMfunctions.cpp:175-464). One solve runs
//   prepare   per-segment 1D Gaussian tables + stencil bin   (gaussian_setup,
//             FCMfunctions.cpp:549-593; GA_setup :536-547)
//   bin       counting sort of segments by the grid tile holding their
//             stencil origin (deterministic order inside a bin); on the
//             matrix-core path each tile then gets the records of the
//             segments whose stencil meets it (k_tile_lists); few segments
//             take one launch for both, without bins (k_tile_lists_direct)
//   spread    gather form of mono_and_dipole_force_distribution
//             (:596-646): one workgroup per grid tile sums, in a fixed
//             order, every segment whose stencil covers the tile, then
//             writes each grid point once (no atomics, no zeroing pass);
//             by default as per-tile matrix-core products (k_spread_mfma,
//             both precisions), else with the vector gather (k_spread)
//   fft_z_r2c real->half-complex along z, two real rows per complex FFT
//   fft_y     strided complex FFT along y (forward)
//   fft_x_prj forward FFT along x, the Stokes projection of flow_solve
//             (:648-736), inverse FFT along x -- three components resident
//             on chip, so the spectrum makes one round trip through HBM
//   fft_y     inverse along y
//   fft_z_c2r half-complex->real along z
//   interp    particle_velocities + particle_rotations (:740-808) fused:
//             on the matrix cores per tile (k_interp_mfma: the transpose
//             of the tile spread, partial sums added per segment in a
//             fixed order), else one wavefront per segment in bin order
// Grids: real R[3][nx][ny][nz], half spectrum C[3][nx][ny][nz/2+1] (complex).
// Precision: FS_FP64 runs every stage in double; FS_FP32 runs them in float
// with float accumulation (stencil offsets are formed from the FP64
// positions before rounding).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "fcm_device.hpp"
#include "fcm_impl.hpp"
#include "fft.hpp"
#include "scan.hpp"

namespace fs {

// fcm_run.hpp, instantiated per precision
template <typename T>
int group_stages(FcmGroup &G, std::vector<char> *host, hipStream_t st);
template <typename T>
int set_fft_lds_attr(const FftPlan &plx, const FftPlan &ply, const FftPlan &plz);
template <typename T>
int interp_blocks(const FcmImpl &f);

static __global__ void k_friction(const int *__restrict__ act, int n3, const double *__restrict__ F,
                           const double *__restrict__ Tq, double a1, double a2,
                           double *__restrict__ V, double *__restrict__ W) {
  if (act && !*act) return;  // batched sweep: suspension converged
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n3) {
    V[i] = a1 * F[i];
    W[i] = a2 * Tq[i];
  }
}

static bool good_size(int n) {
  if (n < 2 || n > 1024 || (n & 1)) return false;
  FftPlan p;
  return make_plan(n, &p);
}

static void twiddles_host(int n, std::vector<double> &re,
                          std::vector<double> &im) {
  re.resize(n);
  im.resize(n);
  for (int m = 0; m < n; ++m) {
    long double ang = 2.0L * (long double)kPi * (long double)m / (long double)n;
    re[m] = (double)cosl(ang);
    im[m] = -(double)sinl(ang);
  }
}

template <typename T>
static int upload_tw(dbuf &b, int n) {
  std::vector<double> re, im;
  twiddles_host(n, re, im);
  std::vector<cx<T>> h(n);
  for (int m = 0; m < n; ++m) h[m] = {(T)re[m], (T)im[m]};
  FS_TRY(b.alloc(sizeof(cx<T>) * n));
  FS_HIP(hipMemcpy(b.p, h.data(), sizeof(cx<T>) * n, hipMemcpyHostToDevice));
  return FS_OK;
}

int FcmImpl::init(const fs_fcm_params &pp, int maxnp, int prec) {
  p = pp;
  max_np = maxnp;
  precision = prec;
  FS_CHECK(prec == FS_FP64 || prec == FS_FP32, FS_ERR_ARG,
           "precision must be FS_FP64 or FS_FP32");
  FS_CHECK(good_size(p.nx) && good_size(p.ny) && good_size(p.nz), FS_ERR_ARG,
           "grid %dx%dx%d: each size must be even, <= 1024 and 2^a 3^b 5^c",
           p.nx, p.ny, p.nz);
  FS_CHECK((p.ngd == 6 || p.ngd == 8 || p.ngd == 10 || p.ngd == 12 ||
            p.ngd == 16 || p.ngd == 20 || p.ngd == 24) &&
               p.ngd + 4 <= p.nx && p.ngd + 4 <= p.ny && p.ngd + 4 <= p.nz,
           FS_ERR_ARG,
           "ngd=%d must be one of 6,8,10,12,16,20,24 and ngd+4 <= every grid "
           "size", p.ngd);
  FS_CHECK(p.dx > 0 && p.sigma > 0 && p.sigma_dip > 0 && p.mu > 0 && p.a > 0,
           FS_ERR_ARG, "dx, sigma, sigma_dip, mu, a must be positive");
  FS_CHECK(maxnp >= 1, FS_ERR_ARG, "max_np must be >= 1");
  make_plan(p.nx, &plx);
  make_plan(p.ny, &ply);
  make_plan(p.nz, &plz);
  tsz = (prec == FS_FP64) ? 8 : 4;
  const size_t N = (size_t)p.nx * p.ny * p.nz;
  const size_t NC = (size_t)p.nx * p.ny * (p.nz / 2 + 1);
  FS_TRY(R.alloc(3 * N * tsz));
  FS_TRY(C.alloc(3 * NC * 2 * tsz));
  if (prec == FS_FP64) {
    FS_TRY(upload_tw<double>(twx, p.nx));
    FS_TRY(upload_tw<double>(twy, p.ny));
    FS_TRY(upload_tw<double>(twz, p.nz));
  } else {
    FS_TRY(upload_tw<float>(twx, p.nx));
    FS_TRY(upload_tw<float>(twy, p.ny));
    FS_TRY(upload_tw<float>(twz, p.nz));
  }
  FS_TRY(tab.alloc((size_t)maxnp * 9 * p.ngd * tsz));
  FS_TRY(origin.alloc((size_t)maxnp * 3 * sizeof(int)));
  FS_TRY(coef.alloc((size_t)maxnp * kCoef * tsz));
  FS_TRY(srec.alloc((size_t)std::max(maxnp, 1) * rec_bytes(tsz)));
  FS_TRY(sorg.alloc((size_t)std::max(maxnp, 1) * sizeof(int)));
  FS_TRY(bin.alloc((size_t)maxnp * sizeof(int)));
  FS_TRY(slot.alloc((size_t)maxnp * sizeof(int)));
  FS_TRY(ids.alloc((size_t)maxnp * sizeof(int)));
  FS_TRY(sids.alloc((size_t)maxnp * sizeof(int)));
  tune.fft_batch = (prec == FS_FP64) ? 8 : 16;
  tune.spread_tile = 16;
  tune.spread_zrun = 8;
  tune.spread_mfma = 1;
  // compile-time plans: one wavefront (two lines of 256 points); run-time
  // plans, whose LDS holds the three components: 3,072 (FP32) or 2,048 (FP64)
  // complex values
  tune.fft_xlines = plx.E > 0 ? std::max(1, 64 * plx.E / p.nx)
                              : std::max(1, std::min(16, (prec == FS_FP32 ? 1024
                                                                          : 680) /
                                                             p.nx));
  FS_TRY(set_geometry());
  for (int i = 0; i < 8; ++i) FS_HIP(hipEventCreate(&ev[i]));
  for (int i = 0; i < 11; ++i) FS_HIP(hipEventCreate(&kev[i]));
  if (prec == FS_FP64)
    FS_TRY(set_fft_lds_attr<double>(plx, ply, plz));
  else
    FS_TRY(set_fft_lds_attr<float>(plx, ply, plz));
  return FS_OK;
}

static int largest_divisor_le(int n, int t) {
  for (int d = std::min(n, t); d >= 1; --d)
    if (n % d == 0) return d;
  return 1;
}

int FcmImpl::set_geometry() {
  int t = tune.spread_tile;
  FS_CHECK(t == 4 || t == 8 || t == 16, FS_ERR_ARG,
           "spread_tile must be 4, 8 or 16");
  FS_CHECK(tune.spread_zrun >= 4 && tune.spread_zrun <= 16, FS_ERR_ARG,
           "spread_zrun must be in [4, 16]");
  // tile z extent: the largest instantiated length <= spread_zrun dividing
  // nz with nz >= run + ngd
  static const int runs[] = {16, 12, 10, 8, 6, 5, 4};
  int tz = 0;
  for (int r : runs)
    if (r <= tune.spread_zrun && p.nz % r == 0 && p.nz >= r + p.ngd) {
      tz = r;
      break;
    }
  FS_CHECK(tz > 0, FS_ERR_ARG, "no spread z run divides nz=%d", p.nz);
  int tx = largest_divisor_le(p.nx, t), ty = largest_divisor_le(p.ny, t);
  // matrix-core spread: fixed 8 x 8 x 16 tiles (four 16-point MFMA rows), the
  // last ones of an axis cut off where it is no multiple. A stencil that wraps
  // over a cut tile can meet one more, and one more bin can reach a tile (5 x 5
  // x 4 at most). Both ways, spread and interpolation in us: 90^3 FP32 with
  // 1,080 segments 35 and (vector gather) 84, 150^3 FP64 with 3,000 75 and 108,
  // 250^3 FP32 with 27,000 243 and 570.
  const int rx = p.nx % 8 != 0, ry = p.ny % 8 != 0, rz = p.nz % 16 != 0;
  {
    const int h = (p.ngd - 1 + 7) / 8, h16 = (p.ngd - 1 + 15) / 16;
    mfma_spread = tune.spread_mfma == 1 && p.nz >= 16 + p.ngd &&
                  std::min(h + rx + 1, ceil_div(p.nx, 8)) *
                          std::min(h + ry + 1, ceil_div(p.ny, 8)) *
                          std::min(h16 + rz + 1, ceil_div(p.nz, 16)) <= kListBins;
  }
  if (mfma_spread) {
    tx = ty = 8;
    tz = 16;
  }
  int bins = 0;
  for (int attempt = 0; attempt < 8; ++attempt) {
    int hx = (p.ngd - 1 + tx - 1) / tx, hy = (p.ngd - 1 + ty - 1) / ty,
        hz = (p.ngd - 1 + tz - 1) / tz;
    bins = std::min(hx + 1, p.nx / tx) * std::min(hy + 1, p.ny / ty) *
           std::min(hz + 1, p.nz / tz);
    if (bins <= kMaxBinsPerTile || mfma_spread) break;
    int nx2 = largest_divisor_le(p.nx, 2 * tx), ny2 = largest_divisor_le(p.ny, 2 * ty);
    if (nx2 * ny2 > 256) break;
    tx = nx2;
    ty = ny2;
  }
  FS_CHECK(bins <= kMaxBinsPerTile && tx * ty <= 256, FS_ERR_ARG,
           "no spread tile fits grid %dx%dx%d with ngd=%d", p.nx, p.ny, p.nz,
           p.ngd);
  geom.nx = p.nx;
  geom.ny = p.ny;
  geom.nz = p.nz;
  geom.ngd = p.ngd;
  geom.tx = tx;
  geom.ty = ty;
  geom.tz = tz;
  geom.nbx = ceil_div(p.nx, tx);
  geom.nby = ceil_div(p.ny, ty);
  geom.nbz = ceil_div(p.nz, tz);
  geom.hx = (p.ngd - 1 + tx - 1) / tx;
  geom.hy = (p.ngd - 1 + ty - 1) / ty;
  geom.hz = (p.ngd - 1 + tz - 1) / tz;
  nbins = geom.nbx * geom.nby * geom.nbz;
  geom.sx = stencil_tiles(p.ngd, 8) + rx;
  geom.sy = stencil_tiles(p.ngd, 8) + ry;
  geom.sz = stencil_tiles(p.ngd, 16) + rz;
  if (mfma_spread) {
    geom.hx += rx;
    geom.hy += ry;
    geom.hz += rz;
    const size_t nslot = (size_t)geom.sx * geom.sy * geom.sz;
    FS_TRY(ipart.alloc((size_t)max_np * 6 * tsz * nslot));
    FS_TRY(tslab.alloc((size_t)nbins * kTileCap * rec_bytes(tsz)));
    FS_TRY(tcnt.alloc((size_t)nbins * sizeof(int)));
    FS_TRY(tovf.alloc((size_t)nbins * sizeof(int)));
    FS_TRY(tpool.alloc((size_t)max_np * nslot * rec_bytes(tsz)));
    grid_interp = tsz == 8 ? interp_blocks<double>(*this) : interp_blocks<float>(*this);
  }
  cut = mfma_spread && (rx || ry || rz);
  // one more counter after the bins: the tile lists' pool top
  FS_TRY(bin_count.alloc((size_t)(nbins + 1) * sizeof(int)));
  FS_HIP(hipMemset(bin_count.p, 0, (size_t)(nbins + 1) * sizeof(int)));
  FS_TRY(bin_start.alloc((size_t)(nbins + 1) * sizeof(int)));
  FS_TRY(scan_tmp.alloc((size_t)(nbins / kScanBlock + 4) * sizeof(int)));
  // FFT pass geometry: z rows per workgroup (even divisor of nx), y-pass run
  // of consecutive x, x-pass lines per workgroup; workgroups stay <= 1024
  const size_t cs = 2 * tsz, lds_max = 160 * 1024;
  // 256-byte runs of x in the spectrum (512^3 FP32: 128-byte runs cost 5% of
  // the z passes)
  zP = 0;
  for (int xb = std::min(tsz == 8 ? 16 : 32, p.nx); xb >= 2; --xb)
    if (xb % 2 == 0 && p.nx % xb == 0 && fft_threads(plz, xb / 2) <= fft_max_threads(plz, tsz) &&
        cs * (p.nz + (size_t)(xb / 2) * fft_padded_len(p.nz)) <= lds_max) {
      zP = xb / 2;
      break;
    }
  yB = largest_divisor_le(p.nx, tune.fft_batch);
  while (yB > 1 && fft_threads(ply, yB) > fft_max_threads(ply, tsz)) yB = largest_divisor_le(p.nx, yB - 1);
  xQ = largest_divisor_le(p.ny, tune.fft_xlines);
  const int x_max = plx.E > 0 ? 256 : fft_max_threads(plx, tsz);
  while (xQ > 1 && (x_threads(plx, xQ) > x_max ||
                    cs * x_lds_values(plx, xQ) > lds_max))
    xQ = largest_divisor_le(p.ny, xQ - 1);
  FS_CHECK(zP >= 1 && fft_threads(ply, yB) <= fft_max_threads(ply, tsz) &&
               x_threads(plx, xQ) <= x_max,
           FS_ERR_ARG, "no FFT workgroup shape fits %dx%dx%d", p.nx, p.ny, p.nz);
  return FS_OK;
}

// Lists without bins where every row of tiles can look at all segments. Both
// sides in us, of all launches that make the lists, binned and direct: 240
// segments on 64^3 (32 row steps) 31 and 16; 3,600 on 128^3 (512) 43 and 26;
// 2,400 on 192^3 (864) 37 and 28, growing with the row steps. The way depends on
// the solve's own segments, so that its results do not change with the
// capacity of the handle. FP32 solves round FP64 weights there and on cut grids
// (fine_weights): cut grids came from the vector gather, which does, and small
// solves with hardware exp2 were up to 1.4 times further off the 64-bit result.
// It costs 0 to 3% of a solve (96^3 with 1,350 segments 89.5 and 90.8 us), 4 to
// 6% on densely filled cut grids (50^3 with 4,000 157 and 164, 100 x 80 x 90
// with 10,000 184 and 195); at 250^3 with 27,000 853 and 862.
bool FcmImpl::lists_direct(int np) const {
  return mfma_spread && np <= kDirectMax &&
         (long)ceil_div(np, 1024) * geom.nby * geom.nbz <= kDirectRowSteps;
}

void FcmImpl::release() {
  R.release();
  C.release();
  twx.release();
  twy.release();
  twz.release();
  tab.release();
  origin.release();
  coef.release();
  bin.release();
  slot.release();
  ids.release();
  sids.release();
  srec.release();
  sorg.release();
  tslab.release();
  tcnt.release();
  tovf.release();
  tpool.release();
  ipart.release();
  bin_count.release();
  bin_start.release();
  scan_tmp.release();
  for (int i = 0; i < 8; ++i)
    if (ev[i]) (void)hipEventDestroy(ev[i]);
  for (int i = 0; i < 11; ++i)
    if (kev[i]) (void)hipEventDestroy(kev[i]);
  for (hipEvent_t e : prof_ev) (void)hipEventDestroy(e);
  prof_ev.clear();
  prof_used = 0;
}

bool fcm_same_shapes(const FcmGroupMember &ma, const FcmGroupMember &mb) {
  const FcmImpl &a = *ma.fcm, &b = *mb.fcm;
  return a.precision == b.precision && a.p.nx == b.p.nx && a.p.ny == b.p.ny &&
         a.p.nz == b.p.nz && a.p.ngd == b.p.ngd && a.mfma_spread && b.mfma_spread &&
         a.zP == b.zP && a.yB == b.yB && a.xQ == b.xQ &&
         a.grid_interp == b.grid_interp && a.nbins == b.nbins &&
         a.lists_direct(ma.np) == b.lists_direct(mb.np);
}

int FcmGroup::build() {
  FS_CHECK(!m.empty(), FS_ERR_ARG, "empty FCM group");
  for (auto &x : m)
    FS_CHECK(fcm_same_shapes(m[0], x) && x.np >= 1 &&
                 x.np <= x.fcm->max_np,
             FS_ERR_ARG, "FCM group members differ in launch shapes or sizes");
  std::vector<char> host;
  off.clear();
  int rc = m[0].fcm->precision == FS_FP64 ? group_stages<double>(*this, &host, nullptr)
                                          : group_stages<float>(*this, &host, nullptr);
  FS_TRY(rc);
  FS_TRY(tab.alloc(host.size()));
  FS_HIP(hipMemcpy(tab.p, host.data(), host.size(), hipMemcpyHostToDevice));
  return FS_OK;
}

int FcmGroup::solve(hipStream_t st) {
  FS_CHECK(tab.p && !off.empty(), FS_ERR_STATE, "FCM group not built");
  return m[0].fcm->precision == FS_FP64 ? group_stages<double>(*this, nullptr, st)
                                        : group_stages<float>(*this, nullptr, st);
}

// add the stage times of every solve since the last call into acc7
// (buckets of stage_times); the caller has synchronised the stream
int FcmImpl::prof_collect(double *acc7) {
  for (size_t k = 0; k + 7 <= prof_used; k += 7) {
    float t[6];
    for (int i = 0; i < 6; ++i)
      FS_HIP(hipEventElapsedTime(&t[i], prof_ev[k + i], prof_ev[k + i + 1]));
    acc7[1] += t[0];
    acc7[2] += t[1];
    acc7[3] += t[2];
    acc7[4] += t[3];
    acc7[5] += t[4];
    acc7[6] += t[5];
  }
  prof_used = 0;
  return FS_OK;
}

int FcmImpl::mobility(int np, const double *Y, const double *F,
                      const double *Tq, double *V, double *W, hipStream_t st) {
  FS_CHECK(np >= 0, FS_ERR_ARG, "np < 0");
  FS_CHECK(np <= max_np, FS_ERR_SIZE, "np=%d exceeds max_np=%d", np, max_np);
  FS_CHECK(np == 0 || (Y && F && Tq && V && W), FS_ERR_ARG, "null array");
  if (np == 0) return FS_OK;
  last_np = np;
  if (precision == FS_FP64) return run<double>(np, Y, F, Tq, V, W, st);
  return run<float>(np, Y, F, Tq, V, W, st);
}

int FcmImpl::friction(int np, const double *F, const double *Tq, double *V,
                      double *W, hipStream_t st) {
  FS_CHECK(np >= 0 && np <= max_np, FS_ERR_SIZE, "bad np=%d", np);
  if (np == 0) return FS_OK;
  double a1 = 1. / (6 * kPi * p.a * p.mu);
  double a2 = 1. / (8 * kPi * p.a * p.a * p.a * p.mu);
  hipLaunchKernelGGL(k_friction, dim3(ceil_div(3 * np, 256)), dim3(256), 0,
                     st, act, 3 * np, F, Tq, a1, a2, V, W);
  FS_LAUNCHED();
  return FS_OK;
}

int FcmImpl::kernel_times(float *ms10) {
  for (int i = 0; i < 10; ++i) ms10[i] = 0;
  if (!timing || !kev_used[10]) return FS_OK;
  FS_HIP(hipEventSynchronize(kev[10]));
  auto span = [&](int a, int b, float *out) -> int {
    FS_HIP(hipEventElapsedTime(out, kev[a], kev[b]));
    return FS_OK;
  };
  const int sp0 = kev_used[2] ? 2 : 1;   // spread starts after the lists
  const int ie = kev_used[9] ? 9 : 10;   // interpolation ends before its sums
  FS_TRY(span(0, 1, &ms10[0]));
  if (kev_used[2]) FS_TRY(span(1, 2, &ms10[1]));
  FS_TRY(span(sp0, 3, &ms10[2]));
  for (int k = 3; k < 8; ++k) FS_TRY(span(k, k + 1, &ms10[k]));
  FS_TRY(span(8, ie, &ms10[8]));
  if (kev_used[9]) FS_TRY(span(9, 10, &ms10[9]));
  return FS_OK;
}

int FcmImpl::stage_times(float *ms7) {
  for (int i = 0; i < 7; ++i) ms7[i] = 0;
  if (!timing) return FS_OK;
  FS_HIP(hipEventSynchronize(ev[6]));
  float t[6];
  for (int i = 0; i < 6; ++i) FS_HIP(hipEventElapsedTime(&t[i], ev[i], ev[i + 1]));
  // buckets: make-zero, gauss, spread, fft fwd, flow, fft bwd, interp
  ms7[0] = 0.f;     // no zeroing pass: the spread writes every point once
  ms7[1] = t[0];    // tables + bin sort
  ms7[2] = t[1];    // spread
  ms7[3] = t[2];    // z r2c + y forward
  ms7[4] = t[3];    // x forward + projection + x inverse (fused)
  ms7[5] = t[4];    // y inverse + z c2r
  ms7[6] = t[5];    // interpolation
  return FS_OK;
}

}  // namespace fs

// ---------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------
using fs::FcmImpl;

int FcmImpl::set_tuning(const fs_fcm_tuning &t) {
  fs_fcm_tuning old = tune;
  fs_fcm_tuning nt = old;
  if (t.fft_batch > 0) nt.fft_batch = t.fft_batch;
  if (t.spread_tile > 0) nt.spread_tile = t.spread_tile;
  if (t.spread_zrun > 0) nt.spread_zrun = t.spread_zrun;
  if (t.fft_xlines > 0) nt.fft_xlines = t.fft_xlines;
  if (t.spread_mfma >= 0) nt.spread_mfma = t.spread_mfma != 0;
  FS_CHECK(nt.fft_batch >= 1 && nt.fft_batch <= 64 && nt.fft_xlines >= 1 &&
               nt.fft_xlines <= 16,
           FS_ERR_ARG, "fft_batch must be in [1,64], fft_xlines in [1,16]");
  // LDS: y pass holds ny + B*(row-padded ny) complex, x pass nx + 3Q*(padded nx).
  // Compile-time plans keep one component there and set_geometry reduces Q to
  // their 256 threads, but take the same values: a larger Q would be no other
  // shape.
  size_t cs = (size_t)tsz * 2;
  size_t lds = std::max(cs * (p.ny + (size_t)nt.fft_batch * fft_rowpad_len(p.ny)),
                        cs * (p.nx + 3 * (size_t)nt.fft_xlines *
                                         fft_padded_len(p.nx)));
  FS_CHECK(lds <= 160 * 1024, FS_ERR_ARG, "tuning needs %zu B of LDS", lds);
  tune = nt;
  int rc = set_geometry();
  if (rc != FS_OK) {
    tune = old;
    set_geometry();
  }
  return rc;
}

// synthetic segments for the autotuner: positions uniform in the box,
// forces and torques uniform in [-1, 1] (splitmix64 of the element index)
__global__ void k_synth(int np, double Lx, double Ly, double Lz,
                        double *__restrict__ Y, double *__restrict__ F,
                        double *__restrict__ T) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 9 * np) return;
  unsigned long long z = (unsigned long long)i * 0x9E3779B97F4A7C15ull +
                         0x2545F4914F6CDD1Dull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  const double u = (double)(z >> 11) * (1.0 / 9007199254740992.0);
  const int arr = i / (3 * np), k = i - arr * 3 * np, d = k % 3;
  if (arr == 0)
    Y[k] = u * (d == 0 ? Lx : d == 1 ? Ly : Lz);
  else
    (arr == 1 ? F : T)[k] = 2.0 * u - 1.0;
}

int FcmImpl::autotune(int np, int reps, fs_fcm_tuning *best) {
  FS_CHECK(np >= 1 && np <= max_np, FS_ERR_SIZE, "np=%d outside [1, %d]", np,
           max_np);
  FS_CHECK(reps >= 1, FS_ERR_ARG, "reps must be >= 1");
  dbuf buf;
  FS_TRY(buf.alloc(sizeof(double) * 15 * (size_t)np));
  double *Y = buf.as<double>(), *F = Y + 3 * (size_t)np,
         *T = F + 3 * (size_t)np, *V = T + 3 * (size_t)np,
         *W = V + 3 * (size_t)np;
  hipStream_t st = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  FS_HIP(hipStreamCreate(&st));
  int rc = FS_OK;
  auto cleanup = [&]() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(st);
    (void)hipStreamDestroy(st);
  };
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    cleanup();
    FS_CHECK(false, FS_ERR_HIP, "event creation failed");
  }
  hipLaunchKernelGGL(k_synth, dim3(ceil_div(9 * np, 256)), dim3(256), 0, st, np,
                     p.nx * p.dx, p.ny * p.dx, p.nz * p.dx, Y, F, T);
  auto time_it = [&](float *ms) -> int {
    FS_TRY(mobility(np, Y, F, T, V, W, st));  // warm-up
    FS_HIP(hipEventRecord(e0, st));
    for (int r = 0; r < reps; ++r) FS_TRY(mobility(np, Y, F, T, V, W, st));
    FS_HIP(hipEventRecord(e1, st));
    FS_HIP(hipEventSynchronize(e1));
    FS_HIP(hipEventElapsedTime(ms, e0, e1));
    return FS_OK;
  };
  fs_fcm_tuning cur = tune;
  float tbest = 0;
  rc = time_it(&tbest);
  static const int mfma[] = {0, 1}, tiles[] = {4, 8, 16}, zruns[] = {4, 8, 16},
                   batches[] = {4, 8, 16, 32}, xlines[] = {1, 2, 4, 8};
  struct Field {
    int fs_fcm_tuning::*m;
    const int *v;
    int n;
  } fields[] = {{&fs_fcm_tuning::spread_mfma, mfma, 2},
                {&fs_fcm_tuning::spread_tile, tiles, 3},
                {&fs_fcm_tuning::spread_zrun, zruns, 3},
                {&fs_fcm_tuning::fft_batch, batches, 4},
                {&fs_fcm_tuning::fft_xlines, xlines, 4}};
  for (const Field &fd : fields) {
    if (rc != FS_OK) break;
    for (int k = 0; k < fd.n && rc == FS_OK; ++k) {
      if (fd.v[k] == cur.*fd.m) continue;
      fs_fcm_tuning trial = cur;
      trial.*fd.m = fd.v[k];
      if (set_tuning(trial) != FS_OK) continue;  // shape does not fit
      float t = 0;
      rc = time_it(&t);
      if (rc == FS_OK && t < tbest) {
        tbest = t;
        cur = tune;
      }
    }
    if (set_tuning(cur) != FS_OK) rc = FS_ERR_STATE;
  }
  cleanup();
  if (rc != FS_OK) return rc;
  if (best) *best = tune;
  set_error("");
  return FS_OK;
}

struct fs_fcm {
  FcmImpl impl;
};

extern "C" int fs_fcm_create(const fs_fcm_params *p, int max_np, int precision,
                             fs_fcm **out) {
  FS_CHECK(p && out, FS_ERR_ARG, "null argument");
  *out = nullptr;
  fs_fcm *h = new fs_fcm();
  int rc = h->impl.init(*p, max_np, precision);
  if (rc != FS_OK) {
    h->impl.release();
    delete h;
    return rc;
  }
  *out = h;
  return FS_OK;
}

extern "C" int fs_fcm_destroy(fs_fcm *h) {
  if (!h) return FS_OK;
  (void)hipDeviceSynchronize();
  h->impl.release();
  delete h;
  return FS_OK;
}

extern "C" int fs_fcm_mobility(fs_fcm *h, int np, const double *Y,
                               const double *F, const double *T, double *V,
                               double *W, void *stream) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  return h->impl.mobility(np, Y, F, T, V, W, (hipStream_t)stream);
}

extern "C" int fs_fcm_mobility_host(fs_fcm *h, int np, const double *Y,
                                    const double *F, const double *T,
                                    double *V, double *W) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  FS_CHECK(np >= 0 && np <= h->impl.max_np, FS_ERR_SIZE, "bad np=%d", np);
  if (np == 0) return FS_OK;
  fs::dbuf d;
  FS_TRY(d.alloc(sizeof(double) * 15 * (size_t)np));
  double *dY = d.as<double>(), *dF = dY + 3 * np, *dT = dF + 3 * np,
         *dV = dT + 3 * np, *dW = dV + 3 * np;
  size_t b = sizeof(double) * 3 * np;
  int rc = FS_OK;
  if (hipMemcpy(dY, Y, b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dF, F, b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dT, T, b, hipMemcpyHostToDevice) != hipSuccess) {
    fs::set_error("host to device copy failed");
    rc = FS_ERR_HIP;
  }
  if (rc == FS_OK) rc = h->impl.mobility(np, dY, dF, dT, dV, dW, nullptr);
  if (rc == FS_OK && (hipMemcpy(V, dV, b, hipMemcpyDeviceToHost) != hipSuccess ||
                      hipMemcpy(W, dW, b, hipMemcpyDeviceToHost) != hipSuccess)) {
    fs::set_error("device to host copy failed");
    rc = FS_ERR_HIP;
  }
  d.release();
  return rc;
}

extern "C" int fs_fcm_friction(fs_fcm *h, int np, const double *F,
                               const double *T, double *V, double *W,
                               void *stream) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  return h->impl.friction(np, F, T, V, W, (hipStream_t)stream);
}

extern "C" int fs_fcm_set_timing(fs_fcm *h, int on) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  h->impl.timing = on ? 1 : 0;
  return FS_OK;
}

extern "C" int fs_fcm_kernel_times(fs_fcm *h, float *ms10) {
  FS_CHECK(h && ms10, FS_ERR_ARG, "null handle or output");
  return h->impl.kernel_times(ms10);
}

extern "C" int fs_fcm_stage_times(fs_fcm *h, float *ms7) {
  FS_CHECK(h && ms7, FS_ERR_ARG, "null argument");
  return h->impl.stage_times(ms7);
}

extern "C" int fs_fcm_get_tuning(fs_fcm *h, fs_fcm_tuning *t) {
  FS_CHECK(h && t, FS_ERR_ARG, "null argument");
  *t = h->impl.tune;
  return FS_OK;
}

extern "C" int fs_fcm_set_tuning(fs_fcm *h, const fs_fcm_tuning *t) {
  FS_CHECK(h && t, FS_ERR_ARG, "null argument");
  return h->impl.set_tuning(*t);
}

extern "C" int fs_fcm_autotune(fs_fcm *h, int np, int reps, fs_fcm_tuning *best) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  return h->impl.autotune(np, reps, best);
}
