// HIP kernels (gfx950) and the C-ABI of include/kgeo.h for the analytic
// Kerr raytracer.
//
// Pipeline of one kgeo_raytrace_ana call:
//   kg_clear_flags   one wave: zero the flag page of the workspace
//   kg_setup         one lane per pixel: lambda, eta, u_+-, roots, labels,
//                    tau_tot, nmax_eq and the per-pixel constants of the
//                    theta and radial integrals -> slot-major plan [PL_N][npix];
//                    wave-ballot OR of the image-wide flags the reference's
//                    numpy code decides globally (any eta > 0, any zero step);
//                    with a side stream, as kg_setup_theta (all but the
//                    radial constants) and kg_setup_radial (side stream)
// then, on the linspace grid (kg_series_pass.hpp):
//   kg_*_heads       one lane per (pixel, head): direct evaluations (Landen
//                    ladder, Carlson duplication) of the last sample and of
//                    each block's first -> records
//   kg_series        one lane per (pixel, block of samples): Taylor series
//                    along the ray; 64 lanes write 512 contiguous bytes per
//                    output and sample
//   kg_fixup         one lane per (queued range, sample): direct evaluation
//                    of what the series leaves
// A ray's first block starts from the observer and runs on the caller's
// stream, while the per-device side stream evaluates the heads and then runs
// the other blocks.  Caller-given Mino times and grids of at most two samples
// take kg_theta / kg_radial, one combined loop per coordinate.  The work is
// FP64 VALU (no MFMA).

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "../../include/kgeo.h"
#include "kg_counts.hpp"
#include "kg_series_pass.hpp"

using namespace kg;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, const char* a = "", long long b = 0) {
  std::snprintf(g_err, sizeof(g_err), fmt, a, b);
  return code;
}

int fail_msg(int code, const char* msg) {
  std::snprintf(g_err, sizeof(g_err), "%s", msg);
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(KGEO_E_HIP, "%s launch failed: %lld", what, static_cast<long long>(e));
  return KGEO_OK;
}

constexpr int kBlock = 256;
// The sample passes run one wave per workgroup: their waves differ widely in
// cost (radial case, refused steps), and a CU's slot is freed per workgroup,
// so a multi-wave workgroup would hold its SIMDs until its slowest wave ends.
constexpr int kPassBlock = 64;
constexpr size_t kFlagBytes = 256;

// The tile (pixels 64 t ..) of workgroup b of n along x.  From the image's
// middle outwards: the rays near the shadow take the most steps, and the long
// waves are to start first.  Workgroups go to the chip's 8 XCDs in turn and
// an image is often a multiple of 8 tiles wide, so each group of 8 is turned
// by one more place, lest an XCD hold the same columns of every row.  (512 x 512 x 500 samples:
// 3 % less time than in the order of the pixels.)
__device__ inline int64_t tile_of(unsigned b, unsigned n) {
  const unsigned g = b >> 3;
  const unsigned k = (g << 3) + 8 <= n ? (g << 3) + ((b + g) & 7u) : b;
  const int64_t mid = n / 2;
  return (k & 1u) ? mid - static_cast<int64_t>((k + 1) / 2) : mid + static_cast<int64_t>(k / 2);
}

struct DevParams {
  RayScalars<double> c;
  int64_t npix, ngeo;
  int do_phi_t;
  int north;  // th_o < pi/2 (n_equatorial_crossings' branch test)
};

DevParams make_dev(const kgeo_ray_params* p, int64_t ngeo) {
  DevParams d;
  d.c = make_scalars(p->a, p->th_o, p->r_o, p->maxtaufrac);
  d.c.a2 = p->a2;
  d.c.sin_th = p->sin_th;
  d.c.cos_th = p->cos_th;
  d.c.cos2_th = p->cos2_th;
  d.c.rplus = p->rplus;
  d.c.rminus = p->rminus;
  d.npix = p->npix;
  d.ngeo = ngeo;
  d.do_phi_t = (p->flags & KGEO_DO_PHI_T) ? 1 : 0;
  d.north = (p->th_o < kHalfPi) ? 1 : 0;
  return d;
}


__global__ void kg_clear_flags(uint32_t* flags) {
  if (threadIdx.x < kFlagBytes / sizeof(uint32_t)) flags[threadIdx.x] = 0u;
}

// Word 0 of the flag page holds the image-wide flags (kg_setup); word 1
// counts the fixup items of one sample pass.
constexpr int kFixupCount = 1;

__global__ void kg_clear_counters(uint32_t* flags) {
  if (threadIdx.x == 0) flags[kFixupCount] = 0u;
}

// Two waves per SIMD: unbounded the set-up needs about 300 VGPR+AGPR (one
// wave); held to 256 with spills it takes 0.23 instead of 0.27 ms at 512^2.
__global__ __launch_bounds__(kPassBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_setup(
    DevParams p, const double* __restrict__ alpha, const double* __restrict__ beta, double* __restrict__ plan,
    uint32_t* __restrict__ gflags, int8_t* __restrict__ rclass, int8_t* __restrict__ thclass,
    int32_t* __restrict__ nmax_eq, double* __restrict__ tau_tot, uint32_t* __restrict__ status) {
  const int64_t i = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  SetupOut so{false, false};
  if (i < p.npix)
    so = setup_pixel(p.c, p.ngeo, p.do_phi_t != 0, alpha[i], beta[i], plan, p.npix, i, rclass, thclass, nmax_eq,
                     tau_tot, status, i);
  wave_or(gflags, so.eta_pos, GF_ANY_ETA_POS);
  wave_or(gflags, so.step_zero, GF_ANY_STEP_ZERO);
}

// The plan kernel in two halves: kg_setup_theta (labels, tau_tot, flags and
// every plan slot but the radial constants) on the caller's stream, and
// kg_setup_radial (the radial constants, about two thirds of kg_setup's
// time) on the side stream, where the radial passes that read them run.
__global__ __launch_bounds__(kPassBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_setup_theta(
    DevParams p, const double* __restrict__ alpha, const double* __restrict__ beta, double* __restrict__ plan,
    uint32_t* __restrict__ gflags, int8_t* __restrict__ rclass, int8_t* __restrict__ thclass,
    int32_t* __restrict__ nmax_eq, double* __restrict__ tau_tot, uint32_t* __restrict__ status) {
  const int64_t i = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  SetupOut so{false, false};
  if (i < p.npix)
    so = setup_pixel<true>(p.c, p.ngeo, p.do_phi_t != 0, alpha[i], beta[i], plan, p.npix, i, rclass, thclass,
                           nmax_eq, tau_tot, status, i);
  wave_or(gflags, so.eta_pos, GF_ANY_ETA_POS);
  wave_or(gflags, so.step_zero, GF_ANY_STEP_ZERO);
}

__global__ __launch_bounds__(kPassBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_setup_radial(
    DevParams p, const double* __restrict__ alpha, const double* __restrict__ beta, double* __restrict__ plan) {
  const int64_t i = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  if (i < p.npix) setup_radial_pixel(p.c, p.do_phi_t != 0, alpha[i], beta[i], plan, p.npix, i);
}

// ---------------------------------------------------------------------------
// Direct sample kernels (caller-given Mino times, ngeo <= 2): grid (pixel
// blocks, sample chunks), one wave per SIMD (held to two, kg_radial spills 273
// registers: 0.23 for 0.18 ms on 150 x 140 pixels x 12 Mino times).  Bound by
// the latency of one wave's chains, and by its first pass over the code.
// kg_theta writes theta and parks G_phi, G_t in ph, t; kg_radial writes r and
// combines phi, t, sigma (kg_sample.hpp).
// ---------------------------------------------------------------------------
struct SampleArgs {
  const double* plan;
  const uint32_t* gflags;
  SampleOut out;
  uint32_t* status;
  int chunks;
};

template <bool DO_PHI_T>
__global__ __launch_bounds__(kPassBlock) void kg_theta(DevParams p, SampleArgs a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const int64_t j0 = p.ngeo * blockIdx.y / a.chunks, j1 = p.ngeo * (blockIdx.y + 1) / a.chunks;
  const uint32_t st = theta_pixel<DO_PHI_T, double, false>(a.plan, p.npix, i, a.gflags[0], a.out, i, j0, j1);
  if (a.status && st) atomicOr(&a.status[i], st);
}

template <bool DO_PHI_T>
__global__ __launch_bounds__(kPassBlock) void kg_radial(DevParams p, SampleArgs a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const int64_t j0 = p.ngeo * blockIdx.y / a.chunks, j1 = p.ngeo * (blockIdx.y + 1) / a.chunks;
  const uint32_t st = radial_pixel<DO_PHI_T, double, false>(p.c, a.plan, p.npix, i, a.gflags[0], a.out, i, j0, j1);
  if (a.status && st) atomicOr(&a.status[i], st);
}

// ---------------------------------------------------------------------------
// The linspace grid's passes.  The fixup queue holds one 64-bit item per
// queued range: walked << 63 | first sample << 32 | pixel.
// ---------------------------------------------------------------------------
struct FixupQueue {
  unsigned long long* items;
  uint32_t* count;
  unsigned long long cap;
};

struct DevPush {
  FixupQueue q;
  __device__ void operator()(int64_t i, int64_t j, bool walked) const {
    const uint32_t s = atomicAdd(q.count, 1u);
    if (s < q.cap)
      q.items[s] = (walked ? (1ull << 63) : 0ull) | (static_cast<unsigned long long>(j) << 32) |
                   static_cast<unsigned long long>(static_cast<uint32_t>(i));
  }
};

__device__ inline void unpack_item(unsigned long long e, int64_t& i, int64_t& j, bool& walked) {
  i = static_cast<int64_t>(e & 0xffffffffull);
  j = static_cast<int64_t>((e >> 32) & 0x7fffffffull);
  walked = (e >> 63) != 0ull;
}

// grid (pixel blocks, heads): the direct evaluations (head 0 the last
// sample, head b the first sample of block b)
__global__ __launch_bounds__(kPassBlock) void kg_theta_heads(DevParams p, SampleArgs a, Records rt, int64_t nb) {
  const int64_t i = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const uint32_t st = series_theta_head_pixel(a.plan, p.npix, i, a.gflags[0], a.out, i, blockIdx.y, nb, rt);
  if (a.status && st) atomicOr(&a.status[i], st);
}

__global__ __launch_bounds__(kPassBlock) void kg_radial_heads(DevParams p, SampleArgs a, Records rt, int64_t nb) {
  const int64_t i = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const uint32_t st = series_radial_head_pixel(a.plan, p.npix, i, a.gflags[0], a.out, i, blockIdx.y, nb, rt);
  if (a.status && st) atomicOr(&a.status[i], st);
}

// grid (pixel blocks, parts): one wave per workgroup, 64 neighbouring pixels
// at one part of block b of their grids (the last part, the longest, first).
// Bound by FP64 issue: a sample takes about 200 vector instructions (84
// multiply-adds of six polynomials, a logarithm, an arctangent, an arccosine,
// a reciprocal), an expansion with its share of the motion ahead about 2600,
// and a ray about 15 of them (a wave's rays take the smallest of their
// steps).  At 512 x 512 x 500 samples (t, r, theta, phi written) one block of
// all rays takes 1.02 ms; the whole call 2.03 ms, where the walk by addition
// theorems (up to three Carlson R_J per sample) took 4.95; 217 x 301 x 333
// 0.69 for 1.29, 64 x 64 x 100 0.28 for 0.55, 1000 x 250 0.26 for 0.55.
// (Expansions about the left end of their samples: 2.23, 0.77, 0.345 and 0.316.)
// Two waves per SIMD: one alone (512 registers) was slower from 217 x 301 on.
template <bool SIG, bool EARLY>
__global__ __launch_bounds__(kPassBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_series(
    DevParams p, SampleArgs a, Records rth, Records rr, int64_t b, int64_t nb, FixupQueue q) {
  const int64_t lane = tile_of(blockIdx.x, gridDim.x) * kPassBlock + threadIdx.x;
  const bool in = lane < p.npix;
  const int64_t i = in ? lane : p.npix - 1;
  __shared__ double sl[SERIES_SLOTS][kPassBlock];
  LdsSlots slots{sl, static_cast<int>(threadIdx.x)};
  DevPush push{q};
  const uint32_t st = series_block_pixel<SIG, EARLY>(p.c, a.plan, p.npix, i, a.gflags[0], a.out, i, in, b, nb,
                                                     gridDim.y - 1 - blockIdx.y, gridDim.y, rth, rr, slots, push);
  if (a.status && st) atomicOr(&a.status[i], st);
}

// one lane per (queued range, sample of the range) (grid-stride): theta, then
// r and the combination, by direct evaluation
__global__ __launch_bounds__(kPassBlock) void kg_fixup(DevParams p, SampleArgs a, FixupQueue q) {
  const unsigned long long c = *q.count;
  const unsigned long long n = (c < q.cap ? c : q.cap) * kFixupSpan;
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * kPassBlock + threadIdx.x; e < n;
       e += static_cast<unsigned long long>(gridDim.x) * kPassBlock) {
    int64_t i, j;
    bool walked;
    unpack_item(q.items[e / kFixupSpan], i, j, walked);
    const int64_t sg = static_cast<int64_t>(e % kFixupSpan);
    const int64_t end = series_fixup_end(j, p.ngeo, walked, p.c.r_o_inf != 0);
    uint32_t st = theta_fixup_sample<true>(a.plan, p.npix, i, a.gflags[0], a.out, i, j, end, sg);
    st |= radial_fixup_sample<true>(p.c, a.plan, p.npix, i, a.gflags[0], a.out, i, j, end, sg);
    if (a.status && st) atomicOr(&a.status[i], st);
  }
}

__global__ __launch_bounds__(kBlock) void kg_ellip_pi(const double* __restrict__ n, const double* __restrict__ phi,
                                                      const double* __restrict__ m, double* __restrict__ out,
                                                      int64_t count) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= count) return;
  const double nn = n[i], mm = m[i];
  Amp<double> A = amp_from_angle(phi[i]);
  LegendreBase<double> L = legendre_base(A, mm);
  double Pc = 0.0;
  if (A.j != 0.0) Pc = ellip_pi_complete(nn, mm, ellip_K(mm));
  // phi itself for |phi| <= 1e-10 (scipy_ellip_binding.py:126-128)
  out[i] = (kfabs(phi[i]) <= 1.0e-10) ? phi[i] : ellip_pi_amp(L, nn, mm, Pc);
}

// Samples a count kernel's lane loads before it works on them.  One lane per
// pixel leaves few waves (1024 for 256 x 256 pixels, one per SIMD), each with
// the pixel's elliptic integrals ahead of its samples, so the loads in flight
// are to hide the memory's latency: 256 x 256 pixels x 100 samples take 39 us
// (kg_counts) and 49 us (kg_turnings), 80 and 94 with one load at a time
// (157 and 137 MB: 31 and 27 us at the rate of a large copy).
constexpr int kCountAhead = 8;

// Calls f(offset, tau) for each sample of pixel i, kCountAhead loads at a time.
template <class F>
__device__ inline void count_samples(const double* __restrict__ tau, int64_t ntau, int64_t npix, int64_t i, F f) {
  const double* __restrict__ t = tau + i;
  int64_t j = 0;
  for (; j + kCountAhead <= ntau; j += kCountAhead) {
    double x[kCountAhead];
#pragma unroll
    for (int q = 0; q < kCountAhead; ++q) x[q] = t[(j + q) * npix];
#pragma unroll
    for (int q = 0; q < kCountAhead; ++q) f((j + q) * npix + i, x[q]);
  }
  for (; j < ntau; ++j) f(j * npix + i, t[j * npix]);
}

// Per-sample counts (kerr_raytracing_utils.py:551-684): equatorial crossings
// and poloidal orbits, one lane per pixel (kg_counts.hpp).
__global__ __launch_bounds__(kPassBlock) void kg_counts(DevParams p, const double* __restrict__ alpha,
                                                        const double* __restrict__ beta,
                                                        const double* __restrict__ tau, int64_t ntau,
                                                        double* __restrict__ n_eq, double* __restrict__ n_pol) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const double be = beta[i];
  const CountConsts k = count_consts(p.c, alpha[i], be);
  count_samples(tau, ntau, p.npix, i, [&](int64_t o, double tj) {
    if (n_eq) n_eq[o] = n_equatorial_at(k, p.north != 0, be, tj);
    if (n_pol) n_pol[o] = n_poloidal_at(k, tj);
  });
}

// Turning points passed by each Mino time (kerr_raytracing_utils.py:686-826),
// one lane per pixel: the reference's fractional n_angular_turnings, its
// floor (theta turning points) and the radial turning point (kg_counts.hpp).
__global__ __launch_bounds__(kPassBlock) void kg_turnings(DevParams p, const double* __restrict__ alpha,
                                                          const double* __restrict__ beta,
                                                          const double* __restrict__ tau, int64_t ntau,
                                                          double* __restrict__ n_ang, int32_t* __restrict__ turns_th,
                                                          int8_t* __restrict__ turns_r) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
  if (i >= p.npix) return;
  const double al = alpha[i], be = beta[i];
  const bool ang = n_ang || turns_th;
  CountConsts k{};
  if (ang) k = count_consts(p.c, al, be);
  RadialTurn rt{false, 0.0};
  if (turns_r) rt = radial_turn_consts(p.c, al, be);
  count_samples(tau, ntau, p.npix, i, [&](int64_t o, double tj) {
    if (ang) {
      const double n = n_angular_at(k, be, tj);
      if (n_ang) n_ang[o] = n;
      // NaN (eta == 0 rays) maps to INT32_MIN, as numpy's float -> int32 cast does on x86
      if (turns_th) turns_th[o] = (n == n && kfabs(n) < 2.0e9) ? static_cast<int32_t>(kfloor(n)) : INT32_MIN;
    }
    if (turns_r) turns_r[o] = static_cast<int8_t>(radial_turns_at(rt, tj));
  });
}

// Sample chunks per pixel of the direct loops (one lane each; the results do
// not depend on it).  A sample costs thousands of instructions (three Carlson
// R_J) and a lane's set-up about a hundred (its plan slots, the Landen
// ladder), so few pixels take one sample per lane, until 2^19 lanes are there
// (eight times the 1024 waves that kg_radial keeps resident); many pixels
// chunks of at least 32 samples, up to 2^21 lanes.  150 x 140 pixels x 12
// Mino times: kg_theta 94 and kg_radial 240 us with 1 chunk, 44 and 79 with
// 12; the whole call 0.36, 0.19, 0.195, 0.184 and 0.178 ms with 1, 3, 4, 6
// and 12.
int pick_chunks(int64_t npix, int64_t ngeo) {
  const int64_t np = npix > 0 ? npix : 1;
  int64_t c = (256LL * 128 * 64 + np - 1) / np;
  const int64_t max_c = ngeo / 32 > 0 ? ngeo / 32 : 1;
  if (c > max_c) c = max_c;
  int64_t few = (1LL << 19) / np;
  if (few > ngeo) few = ngeo;
  if (few > c) c = few;
  if (c < 1) c = 1;
  if (c > 65535) c = 65535;
  return static_cast<int>(c);
}

int env_chunks() {
  const char* s = std::getenv("KGEO_CHUNKS");
  return s ? std::atoi(s) : 0;
}

// Workspace: the flag page, the plan [PL_N][npix] and, for a grid of more
// than two samples, the fixup queue (series_items per pixel bounds the series'
// pushes) and the theta and radial anchor records.  The size is the
// interface's (kgeo.h), of which queue and records take a part.
struct WsLayout {
  size_t plan, threc, rrec, queue, total;
  unsigned long long qcap;
};

WsLayout ws_layout(int64_t npix, int64_t ngeo) {
  WsLayout L{};
  const size_t np = static_cast<size_t>(npix > 0 ? npix : 0);
  L.plan = kFlagBytes;
  size_t off = kFlagBytes + np * PL_N * sizeof(double);
  if (ngeo > 2) {
    const size_t tables = static_cast<size_t>(theta_records(ngeo)) * kThFields +
                          static_cast<size_t>(radial_records(ngeo)) * kRFields;
    L.qcap = static_cast<unsigned long long>(np) * static_cast<unsigned long long>(series_items(ngeo));
    L.queue = off;
    L.threc = off + static_cast<size_t>(L.qcap) * sizeof(unsigned long long);
    L.rrec = L.threc + static_cast<size_t>(kSeriesBlocks) * kThSFields * np * sizeof(double);
    off += np * sizeof(double) * (static_cast<size_t>(fixup_items(ngeo)) + tables + static_cast<size_t>(anchor_blocks(ngeo)));
  }
  L.total = off;
  return L;
}
static_assert(kSeriesMoreItems + kSeriesBlocks * (kThSFields + kRSFields) <= 4 * kThFields + 4 * kRFields,
              "the records and the queue's further items fit the tables' part of the workspace");

// The kernels always sample t, phi and sigma (as the reference's
// raytrace_ana does, kerr_raytracing_ana.py:97): the theta pass parks G_phi,
// G_t in the t and phi outputs and the plan holds the phi/t constants.  A
// request without KGEO_DO_PHI_T is refused rather than run on kernel code
// that no test has run.
int require_phi_t(const kgeo_ray_params* p) {
  if (!(p->flags & KGEO_DO_PHI_T))
    return fail_msg(KGEO_E_ARG, "KGEO_DO_PHI_T is required (t, phi and sigma are always sampled)");
  return KGEO_OK;
}

// Sizes one call handles: a fixup item packs the pixel in 32 bits and the
// sample in 31, and the queue counter is 32-bit (a call queues at most
// npix * series_items(ngeo) items; the bound leaves out the one or two more per
// pixel: at it the plan, t and phi take more memory than the GPU has).  Larger
// jobs are split over pixels.
int size_limit(int64_t npix, int64_t ngeo) {
  if (npix > 0x7fffffffLL) return fail(KGEO_E_ARG, "npix above 2^31 - 1%s (%lld): split the pixels", "", npix);
  if (ngeo > 0x7fffffffLL) return fail(KGEO_E_ARG, "ngeo above 2^31 - 1%s (%lld)", "", ngeo);
  if (npix > 0 && ngeo > 2 && npix * fixup_items(ngeo) > 0xffffffffLL)
    return fail(KGEO_E_ARG, "npix * ceil(ngeo / 8) above 2^32%s (%lld): split the pixels", "",
                npix * fixup_items(ngeo));
  return KGEO_OK;
}

int validate(const kgeo_ray_params* p, const double* alpha, const double* beta, void* ws, size_t wsb,
             int64_t ngeo) {
  if (!p) return fail_msg(KGEO_E_ARG, "params is NULL");
  if (require_phi_t(p)) return KGEO_E_ARG;
  if (p->npix < 0) return fail(KGEO_E_ARG, "npix < 0%s (%lld)", "", p->npix);
  if (size_limit(p->npix, ngeo)) return KGEO_E_ARG;
  if (p->npix > 0 && (!alpha || !beta)) return fail_msg(KGEO_E_ARG, "alpha/beta is NULL");
  if (p->npix > 0 && !ws) return fail_msg(KGEO_E_WORKSPACE, "workspace is NULL");
  const size_t need = kgeo_workspace_bytes(p->npix, ngeo);
  if (wsb < need)
    return fail(KGEO_E_WORKSPACE, "workspace too small%s: need %lld bytes", "", static_cast<long long>(need));
  if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return fail_msg(KGEO_E_WORKSPACE, "workspace not 256-byte aligned");
  return KGEO_OK;
}


// A second stream per device for the plan's radial constants, the heads and
// the blocks that start from them, beside the first blocks (which need only
// the plan's other part) on the caller's; created once per device, with the
// fork and join events.  The fork, the side stream's work and the join are
// enqueued under one lock, so calls from several host threads keep their
// own dependencies (their side work takes turns on the side stream).  Streams keep the default priority.
struct SideStream {
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  hipEvent_t planned = nullptr;  // the side stream's radial plan constants are written
  bool tried = false;
};
constexpr int kMaxDev = 64;
std::mutex g_side_mu;
SideStream g_side[kMaxDev];

// The side stream of the current device, or nullptr (the passes then run in
// order on the caller's stream): also when the caller's stream belongs to
// another device than the current one, whose side stream it cannot fork to.
// Call with g_side_mu held.
SideStream* side_stream(hipStream_t st) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return nullptr;
  if (st) {
    hipDevice_t sd = -1;
    if (hipStreamGetDevice(st, &sd) != hipSuccess || static_cast<int>(sd) != dev) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  SideStream& s = g_side[dev];
  if (!s.tried) {
    s.tried = true;
    if (hipStreamCreateWithFlags(&s.side, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s.join, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s.planned, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      s.side = nullptr;
    }
  }
  return s.side ? &s : nullptr;
}

// The caller's stream waits for the radial plan constants (run_plan).
int wait_planned(hipStream_t st) {
  std::lock_guard<std::mutex> lock(g_side_mu);
  SideStream* ss = side_stream(st);
  if (ss && hipStreamWaitEvent(st, ss->planned, 0) != hipSuccess)
    return fail_msg(KGEO_E_HIP, "wait for the plan failed");
  return KGEO_OK;
}

// The plan.  Its radial constants are left to the side stream; unless joined
// here, what follows on the caller's must wait for them (wait_planned) or for
// a pass that follows them there (run_series' join) before the call returns,
// whatever becomes of it, since the kernel reads alpha and beta and writes the
// workspace.
int run_plan(const kgeo_ray_params* p, const double* alpha, const double* beta, int8_t* rclass, int8_t* thclass,
             int32_t* nmax_eq, double* tau_tot, uint32_t* status, void* ws, hipStream_t st, bool join) {
  DevParams d = make_dev(p, p->ngeo);
  if (d.npix == 0) return KGEO_OK;
  uint32_t* gflags = static_cast<uint32_t*>(ws);
  double* plan = reinterpret_cast<double*>(static_cast<char*>(ws) + kFlagBytes);
  hipLaunchKernelGGL(kg_clear_flags, dim3(1), dim3(64), 0, st, gflags);
  int rc = check_launch("kg_clear_flags");
  if (rc) return rc;
  const unsigned nb = static_cast<unsigned>((d.npix + kPassBlock - 1) / kPassBlock);
  std::lock_guard<std::mutex> lock(g_side_mu);
  SideStream* ss = side_stream(st);
  if (!ss) {
    hipLaunchKernelGGL(kg_setup, dim3(nb), dim3(kPassBlock), 0, st, d, alpha, beta, plan, gflags, rclass, thclass,
                       nmax_eq, tau_tot, status);
    return check_launch("kg_setup");
  }
  // the radial constants on the side stream, after everything enqueued so
  // far on the caller's (an earlier sample pass may still read the plan)
  if (hipEventRecord(ss->fork, st) != hipSuccess || hipStreamWaitEvent(ss->side, ss->fork, 0) != hipSuccess)
    return fail_msg(KGEO_E_HIP, "fork to the side stream failed");
  hipLaunchKernelGGL(kg_setup_theta, dim3(nb), dim3(kPassBlock), 0, st, d, alpha, beta, plan, gflags, rclass, thclass,
                     nmax_eq, tau_tot, status);
  if ((rc = check_launch("kg_setup_theta"))) return rc;
  hipLaunchKernelGGL(kg_setup_radial, dim3(nb), dim3(kPassBlock), 0, ss->side, d, alpha, beta, plan);
  rc = check_launch("kg_setup_radial");
  if (hipEventRecord(ss->planned, ss->side) != hipSuccess) rc = fail_msg(KGEO_E_HIP, "plan event failed");
  else if (join && hipStreamWaitEvent(st, ss->planned, 0) != hipSuccess)
    rc = fail_msg(KGEO_E_HIP, "wait for the plan failed");
  return rc;
}

int run_series(const DevParams& d, const SampleArgs& a, void* ws, hipStream_t st) {
  const WsLayout L = ws_layout(d.npix, d.ngeo);
  char* base = static_cast<char*>(ws);
  uint32_t* flags = static_cast<uint32_t*>(ws);
  const Records rth{reinterpret_cast<double*>(base + L.threc), d.npix, 0};
  const Records rr{reinterpret_cast<double*>(base + L.rrec), d.npix, 0};
  unsigned long long* items = reinterpret_cast<unsigned long long*>(base + L.queue);
  const FixupQueue q{items, flags + kFixupCount, L.qcap};
  const unsigned np = static_cast<unsigned>((d.npix + kPassBlock - 1) / kPassBlock);
  const int64_t nb = series_blocks(d.ngeo);
  const unsigned parts = static_cast<unsigned>(pick_parts(d.npix, d.ngeo));
  const unsigned nbu = static_cast<unsigned>(nb);
  const unsigned long long fb = (L.qcap * kFixupSpan + kPassBlock - 1) / kPassBlock;
  const dim3 fgrid(static_cast<unsigned>(fb < 4096ull ? fb : 4096ull));
  // block 0 starts from the observer: with further blocks (which take the
  // last sample) it waits for no head, nor, above MINSPIN, for the radial plan;
  // t and sigma of an observer at infinity start from the second block's head
  const bool early = nb > 1 && !d.c.minspin && !d.c.r_o_inf;
  auto series = [&](auto kernel, hipStream_t on, int64_t b) {
    hipLaunchKernelGGL(kernel, dim3(np, parts), dim3(kPassBlock), 0, on, d, a, rth, rr, b, nb, q);
    return check_launch("kg_series");
  };
  hipLaunchKernelGGL(kg_clear_counters, dim3(1), dim3(64), 0, st, flags);
  int rc = check_launch("kg_clear_counters");
  if (rc) return rc;
  {
    std::lock_guard<std::mutex> lock(g_side_mu);
    SideStream* ss = side_stream(st);
    const hipStream_t rs = ss ? ss->side : st;
    if (ss) {
      if (hipEventRecord(ss->fork, st) != hipSuccess || hipStreamWaitEvent(rs, ss->fork, 0) != hipSuccess)
        return fail_msg(KGEO_E_HIP, "fork to the side stream failed");
    }
    // the heads and the blocks that start from them, beside block 0
    hipLaunchKernelGGL(kg_theta_heads, dim3(np, nbu), dim3(kPassBlock), 0, rs, d, a, rth, nb);
    rc = check_launch("kg_theta_heads");
    if (!rc) {
      hipLaunchKernelGGL(kg_radial_heads, dim3(np, nbu), dim3(kPassBlock), 0, rs, d, a, rr, nb);
      rc = check_launch("kg_radial_heads");
    }
    for (int64_t b = early ? 1 : 0; b < nb && !rc; ++b)
      rc = a.out.sig ? series(kg_series<true, false>, rs, b) : series(kg_series<false, false>, rs, b);
    const bool marked = !ss || hipEventRecord(ss->join, rs) == hipSuccess;
    if (early && !rc) rc = a.out.sig ? series(kg_series<true, true>, st, 0) : series(kg_series<false, true>, st, 0);
    // joined also where a launch failed: what was enqueued uses the caller's buffers
    if (ss && (!marked || hipStreamWaitEvent(st, ss->join, 0) != hipSuccess))
      return fail_msg(KGEO_E_HIP, "join failed");
    if (rc) return rc;
  }
  hipLaunchKernelGGL(kg_fixup, fgrid, dim3(kPassBlock), 0, st, d, a, q);
  return check_launch("kg_fixup");
}

// pending: run_plan's radial constants are not yet waited for on st.
int run_sample(const kgeo_ray_params* p, int64_t ngeo, const double* tau_in, double* tau, double* t, double* r,
               double* th, double* ph, double* sig, uint32_t* status, void* ws, hipStream_t st, bool pending) {
  DevParams d = make_dev(p, ngeo);
  if (d.npix == 0 || ngeo <= 0) return KGEO_OK;
  const uint32_t* gflags = static_cast<const uint32_t*>(ws);
  const double* plan = reinterpret_cast<const double*>(static_cast<const char*>(ws) + kFlagBytes);
  const unsigned nb = static_cast<unsigned>((d.npix + kPassBlock - 1) / kPassBlock);
  const int chunks = kgeo_sample_chunks(d.npix, ngeo);
  dim3 grid(nb, static_cast<unsigned>(chunks));
  SampleArgs a{plan, gflags, SampleOut{tau_in, tau, t, r, th, ph, sig, d.npix, ngeo}, status, chunks};
  // the linspace grid takes the series (heads, series, fixup); caller-given
  // Mino times and grids of at most two samples are evaluated directly
  if (!tau_in && ngeo > 2) return run_series(d, a, ws, st);
  hipLaunchKernelGGL(kg_theta<true>, grid, dim3(kPassBlock), 0, st, d, a);
  int rc = check_launch("kg_theta");
  if (rc || (pending && (rc = wait_planned(st)))) return rc;
  hipLaunchKernelGGL(kg_radial<true>, grid, dim3(kPassBlock), 0, st, d, a);
  return check_launch("kg_radial");
}

int require_outputs(int64_t npix, int64_t ngeo, const double* t, const double* ph) {
  if (npix > 0 && ngeo > 0 && (!t || !ph)) return fail_msg(KGEO_E_ARG, "t and ph outputs are required");
  return KGEO_OK;
}

// A plan and its samples in one call.  Where no sample pass ran to its end,
// the caller's stream waits for the plan here.
int plan_and_sample(const kgeo_ray_params* p, const double* alpha, const double* beta, int64_t ngeo,
                    const double* tau_in, double* tau, double* t, double* r, double* th, double* ph, double* sig,
                    int8_t* rclass, int8_t* thclass, int32_t* nmax_eq, double* tau_tot, uint32_t* status, void* ws,
                    hipStream_t st) {
  int rc = run_plan(p, alpha, beta, rclass, thclass, nmax_eq, tau_tot, status, ws, st, ngeo <= 0);
  if (!rc) rc = run_sample(p, ngeo, tau_in, tau, t, r, th, ph, sig, status, ws, st, true);
  if (rc && p->npix > 0) (void)wait_planned(st);
  return rc;
}

}  // namespace

extern "C" {

int kgeo_abi_version(void) { return KGEO_ABI_VERSION; }

const char* kgeo_last_error(void) { return g_err; }

void kgeo_fill_params(kgeo_ray_params* p) {
  if (!p) return;
  p->a2 = p->a * p->a;
  p->sin_th = std::sin(p->th_o);
  p->cos_th = std::cos(p->th_o);
  p->cos2_th = p->cos_th * p->cos_th;
  const double root = std::sqrt(1.0 - p->a2);
  p->rplus = 1.0 + root;
  p->rminus = 1.0 - root;
}

int kgeo_sample_chunks(int64_t npix, int64_t ngeo) {
  if (npix <= 0 || ngeo <= 0) return 0;
  int c = env_chunks();
  if (c <= 0) c = pick_chunks(npix, ngeo);
  if (c > ngeo) c = static_cast<int>(ngeo);
  return c;
}

size_t kgeo_workspace_bytes(int64_t npix, int64_t ngeo) {
  if (npix < 0) return 0;
  return ws_layout(npix, ngeo).total;
}

int kgeo_plan(const kgeo_ray_params* p, const double* alpha, const double* beta, int8_t* rclass, int8_t* thclass,
              int32_t* nmax_eq, double* tau_tot, uint32_t* status, void* workspace, size_t workspace_bytes,
              void* stream) {
  int rc = validate(p, alpha, beta, workspace, workspace_bytes, 0);
  if (rc) return rc;
  return run_plan(p, alpha, beta, rclass, thclass, nmax_eq, tau_tot, status, workspace,
                  static_cast<hipStream_t>(stream), true);
}

int kgeo_sample(const kgeo_ray_params* p, const double* tau_in, int64_t ntau, double* tau, double* t, double* r,
                double* th, double* ph, double* sig, uint32_t* status, void* workspace, size_t workspace_bytes,
                void* stream) {
  if (!p) return fail_msg(KGEO_E_ARG, "params is NULL");
  if (require_phi_t(p)) return KGEO_E_ARG;
  if (p->npix < 0 || ntau < 0) return fail_msg(KGEO_E_ARG, "negative size");
  if (size_limit(p->npix, tau_in ? 0 : ntau)) return KGEO_E_ARG;
  if (p->npix > 0 && !workspace) return fail_msg(KGEO_E_WORKSPACE, "workspace is NULL");
  const size_t need = kgeo_workspace_bytes(p->npix, tau_in ? 0 : ntau);
  if (workspace_bytes < need)
    return fail(KGEO_E_WORKSPACE, "workspace too small%s: need %lld bytes", "", static_cast<long long>(need));
  if (require_outputs(p->npix, ntau, t, ph)) return KGEO_E_ARG;
  return run_sample(p, ntau, tau_in, tau, t, r, th, ph, sig, status, workspace, static_cast<hipStream_t>(stream), false);
}

int kgeo_raytrace_ana(const kgeo_ray_params* p, const double* alpha, const double* beta, double* tau, double* t,
                      double* r, double* th, double* ph, double* sig, int8_t* rclass, int8_t* thclass,
                      int32_t* nmax_eq, double* tau_tot, uint32_t* status, void* workspace, size_t workspace_bytes,
                      void* stream) {
  int rc = validate(p, alpha, beta, workspace, workspace_bytes, p ? p->ngeo : 0);
  if (rc) return rc;
  if (p->ngeo < 1) return fail(KGEO_E_ARG, "ngeo < 1%s (%lld)", "", p->ngeo);
  if (require_outputs(p->npix, p->ngeo, t, ph)) return KGEO_E_ARG;
  return plan_and_sample(p, alpha, beta, p->ngeo, nullptr, tau, t, r, th, ph, sig, rclass, thclass, nmax_eq, tau_tot,
                         status, workspace, static_cast<hipStream_t>(stream));
}

int kgeo_coords_at_tau(const kgeo_ray_params* p, const double* alpha, const double* beta, const double* tau_in,
                       int64_t ntau, double* t, double* r, double* th, double* ph, double* sig, uint32_t* status,
                       void* workspace, size_t workspace_bytes, void* stream) {
  int rc = validate(p, alpha, beta, workspace, workspace_bytes, 0);
  if (rc) return rc;
  if (ntau < 0) return fail(KGEO_E_ARG, "ntau < 0%s (%lld)", "", ntau);
  if (ntau > 0 && p->npix > 0 && !tau_in) return fail_msg(KGEO_E_ARG, "tau_in is NULL");
  if (require_outputs(p->npix, ntau, t, ph)) return KGEO_E_ARG;
  return plan_and_sample(p, alpha, beta, ntau, tau_in, nullptr, t, r, th, ph, sig, nullptr, nullptr, nullptr, nullptr,
                         status, workspace, static_cast<hipStream_t>(stream));
}

int kgeo_crossings(const kgeo_ray_params* p, const double* alpha, const double* beta, const double* tau,
                   int64_t ntau, double* n_equatorial, double* n_poloidal, void* stream) {
  if (!p) return fail_msg(KGEO_E_ARG, "params is NULL");
  if (p->npix < 0 || ntau < 0) return fail_msg(KGEO_E_ARG, "negative size");
  if (p->npix == 0 || ntau == 0) return KGEO_OK;
  if (!alpha || !beta || !tau) return fail_msg(KGEO_E_ARG, "NULL array");
  DevParams d = make_dev(p, ntau);
  const unsigned nb = static_cast<unsigned>((d.npix + kPassBlock - 1) / kPassBlock);
  hipLaunchKernelGGL(kg_counts, dim3(nb), dim3(kPassBlock), 0, static_cast<hipStream_t>(stream), d, alpha, beta, tau,
                     ntau, n_equatorial, n_poloidal);
  return check_launch("kg_counts");
}

int kgeo_turnings(const kgeo_ray_params* p, const double* alpha, const double* beta, const double* tau,
                  int64_t ntau, double* n_angular, int32_t* turns_theta, int8_t* turns_r, void* stream) {
  if (!p) return fail_msg(KGEO_E_ARG, "params is NULL");
  if (p->npix < 0 || ntau < 0) return fail_msg(KGEO_E_ARG, "negative size");
  // n_angular_turnings accepts th_o in [0, pi/2] only (kerr_raytracing_utils.py:690-691)
  if ((n_angular || turns_theta) && !(p->th_o >= 0.0 && p->th_o <= kHalfPi))
    return fail_msg(KGEO_E_ARG, "th_o should be a float in range (0,pi/2]");
  if (p->npix == 0 || ntau == 0) return KGEO_OK;
  if (!alpha || !beta || !tau) return fail_msg(KGEO_E_ARG, "NULL array");
  DevParams d = make_dev(p, ntau);
  const unsigned nb = static_cast<unsigned>((d.npix + kPassBlock - 1) / kPassBlock);
  hipLaunchKernelGGL(kg_turnings, dim3(nb), dim3(kPassBlock), 0, static_cast<hipStream_t>(stream), d, alpha, beta, tau,
                     ntau, n_angular, turns_theta, turns_r);
  return check_launch("kg_turnings");
}

int kgeo_ellip_pi(const double* n, const double* phi, const double* m, double* out, int64_t count, void* stream) {
  if (count < 0) return fail(KGEO_E_ARG, "count < 0%s (%lld)", "", count);
  if (count == 0) return KGEO_OK;
  if (!n || !phi || !m || !out) return fail_msg(KGEO_E_ARG, "NULL array");
  const unsigned nb = static_cast<unsigned>((count + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(kg_ellip_pi, dim3(nb), dim3(kBlock), 0, static_cast<hipStream_t>(stream), n, phi, m, out, count);
  return check_launch("kg_ellip_pi");
}

}  // extern "C"
