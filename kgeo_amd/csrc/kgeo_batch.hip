// Batched survey: many raytrace_ana images, each with its own spin,
// inclination, resolution and ngeo, in persistent launches that are
// captured once in a HIP graph and replayed.
//
//   kg_batch_clear       zero the per-image flag words and item counters,
//                        the pass counters and the fixup-queue counters
//   kg_batch_setup       one lane per pixel slot of every image: the same
//                        per-pixel plan and labels as kg_setup.  Each image's
//                        slots are padded to a multiple of 64, so a wave never
//                        straddles two images and the image-wide predicates
//                        (any eta > 0, any zero grid step) are per-image
//                        wave ballots.
//   kg_batch_*_heads     the theta, then the radial heads of the plain kernels
//                        (kg_series_pass.hpp), items (image, 64-pixel tile,
//                        head) in strides over a fixed grid of waves;
//   kg_batch_series      the rays' blocks: a fixed grid of waves taking
//                        items (image, tile, block, part) from an atomic
//                        counter until the pass is empty; every wave leaves
//                        once the counter passes the pass's item total, so
//                        the grid always drains;
//   kg_batch_fixup       the queued ranges of all images, one lane per
//                        (range, sample), by direct evaluation (grid-stride).
// Outputs go to caller arenas: image k's [ngeo_k][npix_k] block of r, theta,
// phi, t starts at element out_off[k] (sum of npix*ngeo of the images before
// it); per-pixel inputs and labels are concatenated at pix_off[k].

#include <hip/hip_runtime.h>

#include <cstdio>
#include <new>
#include <vector>

#include "../../include/kgeo.h"
#include "kg_series_pass.hpp"

using namespace kg;

namespace {

thread_local char g_err_b[512] = "";

int bfail(int code, const char* msg, long long v = 0) {
  std::snprintf(g_err_b, sizeof(g_err_b), msg, v);
  return code;
}

int blaunch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    std::snprintf(g_err_b, sizeof(g_err_b), "%s failed: %d", what, static_cast<int>(e));
    return KGEO_E_HIP;
  }
  return KGEO_OK;
}

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int64_t kMaxItems = (1LL << 31) - (1LL << 24);  // leaves room for one exit fetch per wave

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// pass kinds and their per-tile work units
enum : int { K_HEAD = 0, K_SERIES = 1, K_N = 2 };
// counters: series items, the fixup queue
enum : int { CT_SERIES = 0, CT_QUEUE, kCounters };

struct BatchImage {
  RayScalars<double> c;
  int64_t npix, ngeo;
  int64_t pix_off;   // first pixel in the concatenated per-pixel arrays
  int64_t slot_off;  // first plan column (64-aligned)
  int64_t slots;     // padded pixel count
  int64_t out_off;   // first element of the image's [ngeo][npix] block
  int64_t item_off[K_N];  // first work item of each pass kind
  int64_t th_rec, r_rec;  // first element of the image's record tables
  int32_t units[K_N];     // per tile: heads (one per block); parts of all blocks
  int32_t do_phi_t;
};

struct BatchDev {
  const BatchImage* imgs;
  int nimg;
  int64_t total_slots;
  uint32_t total_items[K_N];
  const double* alpha;
  const double* beta;
  double* plan;       // [PL_N][total_slots]
  double* rec;        // per-image record tables
  unsigned long long* queue;
  unsigned long long qcap;
  uint32_t* flags;    // [nimg]
  uint32_t* done;     // [nimg] completed items
  uint32_t* counter;  // [kCounters]
  double *t, *r, *th, *ph;
  int8_t* rclass;
  int8_t* thclass;
  int32_t* nmax_eq;
  double* tau_tot;
  uint32_t* status;
};

// last image k with key(k) <= key (kind < 0: plan columns, else the first
// item of that pass kind); every lane of a wave searches the same key
__device__ inline int find_image(const BatchImage* imgs, int n, int64_t key, int kind) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    const int64_t off = kind < 0 ? imgs[mid].slot_off : imgs[mid].item_off[kind];
    if (off <= key) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ void kg_batch_clear(BatchDev d) {
  for (int k = threadIdx.x; k < d.nimg; k += blockDim.x) {
    d.flags[k] = 0u;
    d.done[k] = 0u;
  }
  if (threadIdx.x < kCounters) d.counter[threadIdx.x] = 0u;
}

// Two waves per SIMD: 0.94 ms for a 16-image survey (1.4 million slots), with 73
// spilled registers; 1.30 at one.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_batch_setup(BatchDev d) {
  const int64_t s = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  // total_slots is a multiple of 64: whole waves leave here together
  if (s >= d.total_slots) return;
  const int im = find_image(d.imgs, d.nimg, s, -1);
  const BatchImage& B = d.imgs[im];
  const int64_t i = s - B.slot_off;
  SetupOut so{false, false};
  if (i < B.npix) {
    const int64_t g = B.pix_off + i;
    so = setup_pixel(B.c, B.ngeo, B.do_phi_t != 0, d.alpha[g], d.beta[g], d.plan, d.total_slots, s, d.rclass,
                     d.thclass, d.nmax_eq, d.tau_tot, d.status, g);
  }
  wave_or(&d.flags[im], so.eta_pos, GF_ANY_ETA_POS);
  wave_or(&d.flags[im], so.step_zero, GF_ANY_STEP_ZERO);
}

// The work-item fetch is written so that the compiler sees it as uniform:
// every lane issues the atomic (lane 0 adds 1, the others 0; the backend
// combines them into one atomic per wave) and the value is taken with
// readfirstlane, so `item` lives in a scalar register and the exit test is
// a scalar branch.  A lane-0-only atomic followed by a lane shuffle lets the
// structurizer split the wave's lanes into two loop nests, in which the
// shuffle re-reads an inactive lane 0 and the loop never ends.
__device__ inline uint32_t fetch_item(uint32_t* counter, int lane) {
  const uint32_t got = atomicAdd(counter, lane == 0 ? 1u : 0u);
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(got)));
}

// Fixup queue item of a batch: walked << 63 | image << 51 | sample << 31 | pixel
// (images < 4096, ngeo <= 2^20, npix < 2^31: checked at plan time).
struct BatchPush {
  unsigned long long* items;
  uint32_t* count;
  unsigned long long cap;
  unsigned long long image;
  __device__ void operator()(int64_t i, int64_t j, bool walked) const {
    const uint32_t s = atomicAdd(count, 1u);
    if (s < cap)
      items[s] = (walked ? (1ull << 63) : 0ull) | (image << 51) | (static_cast<unsigned long long>(j) << 31) |
                 static_cast<unsigned long long>(i);
  }
};

__device__ inline SampleOut image_out(const BatchDev& d, const BatchImage& B) {
  return SampleOut{nullptr, nullptr, d.t + B.out_off, d.r + B.out_off, d.th + B.out_off, d.ph + B.out_off, nullptr,
                   B.npix, B.ngeo};
}

__device__ inline Records image_records(const BatchDev& d, const BatchImage& B, bool theta) {
  return Records{d.rec + (theta ? B.th_rec : B.r_rec), B.slots, B.slot_off};
}

// Item `item` (image, tile, unit) of pass KIND: f(image, its index, its pixel
// on this lane, whether there is one, unit); returns the image's index.
template <int KIND, class F> __device__ inline int batch_item(const BatchDev& d, uint32_t item, int lane, F f) {
  const int im = find_image(d.imgs, d.nimg, static_cast<int64_t>(item), KIND);
  const BatchImage& B = d.imgs[im];
  const int64_t li = static_cast<int64_t>(item) - B.item_off[KIND];
  const int64_t units = B.units[KIND];
  const int64_t i = (li / units) * kWave + lane;
  const bool in = i < B.npix;
  const uint32_t st = f(B, im, in ? i : B.npix - 1, in, li % units);
  if (in && d.status && st) atomicOr(&d.status[B.pix_off + i], st);
  return im;
}

// Heads cost alike, so the waves share them out in strides, without a counter:
// the fetches and the progress counts are atomics on a few words that all
// XCDs share, about 7 ns each, and with two per item they bounded the theta
// heads of a 16-image survey (43520 items: 0.65 ms, 0.39 now; the radial ones
// 0.85, 0.77 now).  A wave counts an image's items and adds them once.
template <bool THETA> __device__ inline void batch_heads(const BatchDev& d) {
  const int lane = __lane_id();
  const uint32_t waves = gridDim.x * (kBlock / kWave);
  uint32_t count = 0u;
  int last = 0;
  for (uint32_t item = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
           static_cast<int>(blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave)));
       item < d.total_items[K_HEAD]; item += waves) {
    const int im = batch_item<K_HEAD>(
        d, item, lane, [&](const BatchImage& B, int k, int64_t i, bool in, int64_t hd) {
          if (!in) return 0u;
          const int64_t s = B.slot_off + i;
          const SampleOut o = image_out(d, B);
          const Records rt = image_records(d, B, THETA);
          return THETA ? series_theta_head_pixel(d.plan, d.total_slots, s, d.flags[k], o, i, hd, B.units[K_HEAD], rt)
                       : series_radial_head_pixel(d.plan, d.total_slots, s, d.flags[k], o, i, hd, B.units[K_HEAD], rt);
        });
    if (im != last && count) {
      atomicAdd(&d.done[last], lane == 0 ? count : 0u);
      count = 0u;
    }
    last = im;
    ++count;
  }
  if (count) atomicAdd(&d.done[last], lane == 0 ? count : 0u);
}

// theta at two waves per SIMD (0.39 ms, 0.47 at one), r at one (0.77; with 110
// spilled registers at two 0.93)
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_batch_theta_heads(BatchDev d) {
  batch_heads<true>(d);
}

__global__ __launch_bounds__(kBlock) void kg_batch_radial_heads(BatchDev d) { batch_heads<false>(d); }

// kg_series (kgeo_raytrace.hip) over all images, two waves per SIMD as there.
// A survey of 16 images (64 .. 512 pixels a side, 50 .. 400 samples; 327 million
// samples, 10.5 GB) takes 7.6 ms, where the walk by addition theorems took 21.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void kg_batch_series(BatchDev d) {
  __shared__ double sl[kBlock / kWave][SERIES_SLOTS][kWave];
  LdsSlots slots{sl[threadIdx.x / kWave], static_cast<int>(threadIdx.x % kWave)};
  const int lane = __lane_id();
  for (;;) {
    const uint32_t item = fetch_item(d.counter + CT_SERIES, lane);
    if (item >= d.total_items[K_SERIES]) break;  // scalar branch: the whole wave leaves once the pass is empty
    const int im = batch_item<K_SERIES>(d, item, lane, [&](const BatchImage& B, int k, int64_t i, bool in, int64_t u) {
      BatchPush push{d.queue, d.counter + CT_QUEUE, d.qcap, static_cast<unsigned long long>(k)};
      const SampleOut o = image_out(d, B);
      const Records rth = image_records(d, B, true), rr = image_records(d, B, false);
      const int64_t nb = B.units[K_HEAD], parts = B.units[K_SERIES] / nb;
      return series_block_pixel<false, false>(B.c, d.plan, d.total_slots, B.slot_off + i, d.flags[k], o, i, in, u % nb,
                                              nb, parts - 1 - u / nb, parts, rth, rr, slots, push);
    });
    atomicAdd(&d.done[im], lane == 0 ? 1u : 0u);
  }
}

// one lane per (queued range, sample of the range) (grid-stride), each
// sample by direct evaluation, as the plain kg_fixup
__global__ __launch_bounds__(kBlock) void kg_batch_fixup(BatchDev d) {
  const unsigned long long c = d.counter[CT_QUEUE];
  const unsigned long long n = (c < d.qcap ? c : d.qcap) * kFixupSpan;
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * kBlock + threadIdx.x; e < n;
       e += static_cast<unsigned long long>(gridDim.x) * kBlock) {
    const unsigned long long q = d.queue[e / kFixupSpan];
    const int64_t sg = static_cast<int64_t>(e % kFixupSpan);
    const int im = static_cast<int>((q >> 51) & 0xfffull);
    const int64_t j = static_cast<int64_t>((q >> 31) & 0xfffffull);
    const int64_t i = static_cast<int64_t>(q & 0x7fffffffull);
    const bool walked = (q >> 63) != 0ull;
    const BatchImage& B = d.imgs[im];
    const int64_t s = B.slot_off + i;
    const uint32_t fl = d.flags[im];
    const SampleOut o = image_out(d, B);
    const int64_t end = series_fixup_end(j, B.ngeo, walked, B.c.r_o_inf != 0);
    uint32_t st = theta_fixup_sample<true>(d.plan, d.total_slots, s, fl, o, i, j, end, sg);
    st |= radial_fixup_sample<true>(B.c, d.plan, d.total_slots, s, fl, o, i, j, end, sg);
    if (d.status && st) atomicOr(&d.status[B.pix_off + i], st);
  }
}

RayScalars<double> scalars_of(const kgeo_ray_params& p) {
  RayScalars<double> c = make_scalars(p.a, p.th_o, p.r_o, p.maxtaufrac);
  c.a2 = p.a2;
  c.sin_th = p.sin_th;
  c.cos_th = p.cos_th;
  c.cos2_th = p.cos2_th;
  c.rplus = p.rplus;
  c.rminus = p.rminus;
  return c;
}

int check_images(const kgeo_ray_params* imgs, int32_t nimg) {
  if (!imgs || nimg <= 0) return bfail(KGEO_E_ARG, "no images (nimg = %lld)", nimg);
  if (nimg > 4096) return bfail(KGEO_E_ARG, "more than 4096 images (%lld)", nimg);
  for (int32_t k = 0; k < nimg; ++k) {
    if (imgs[k].npix < 1) return bfail(KGEO_E_ARG, "image %lld has npix < 1", k);
    if (imgs[k].npix >= (1LL << 31)) return bfail(KGEO_E_ARG, "image %lld has npix >= 2^31", k);
    if (imgs[k].ngeo < 1) return bfail(KGEO_E_ARG, "image %lld has ngeo < 1", k);
    if (imgs[k].ngeo > (1LL << 20)) return bfail(KGEO_E_ARG, "image %lld has ngeo > 2^20", k);
    // every image samples t, phi and sigma, as the plain kernels do
    if (!(imgs[k].flags & KGEO_DO_PHI_T)) return bfail(KGEO_E_ARG, "image %lld lacks KGEO_DO_PHI_T", k);
  }
  return KGEO_OK;
}

int64_t slots_of(const kgeo_ray_params& p) { return (p.npix + kWave - 1) / kWave * kWave; }

int64_t total_slots_of(const kgeo_ray_params* imgs, int32_t nimg) {
  int64_t s = 0;
  for (int32_t k = 0; k < nimg; ++k) s += slots_of(imgs[k]);
  return s;
}

// Elements of image k's theta and radial anchor records (a grid of the series
// has ngeo > 2; smaller images keep none) and of its fixup-queue share.
int64_t theta_rec_elems(const kgeo_ray_params& p) { return p.ngeo > 2 ? kSeriesBlocks * kThSFields * slots_of(p) : 0; }
int64_t radial_rec_elems(const kgeo_ray_params& p) { return p.ngeo > 2 ? kSeriesBlocks * kRSFields * slots_of(p) : 0; }
int64_t queue_elems(const kgeo_ray_params& p) { return series_items(p.ngeo) * slots_of(p); }

// Elements of the plan, and of the interface's record tables and queue (the
// workspace's size): the records and the queue above take a part of them.
struct BatchSizes {
  int64_t slots, rec, queue;
};

BatchSizes sizes_of(const kgeo_ray_params* imgs, int32_t nimg) {
  BatchSizes z{0, 0, 0};
  for (int32_t k = 0; k < nimg; ++k) {
    const kgeo_ray_params& p = imgs[k];
    z.slots += slots_of(p);
    if (p.ngeo > 2)
      z.rec += (theta_records(p.ngeo) * kThFields + radial_records(p.ngeo) * kRFields) * slots_of(p);
    z.queue += fixup_items(p.ngeo) * slots_of(p);
  }
  return z;
}
// per slot; a whole wave's slots cover the records' alignment too
static_assert(kSeriesMoreItems + kSeriesBlocks * (kThSFields + kRSFields) + 1 <= 4 * kThFields + 4 * kRFields,
              "the records and the queue's further items fit the smallest tables");

}  // namespace

struct kgeo_batch {
  BatchDev d;
  std::vector<uint32_t> items_per_image;
  hipGraph_t graph;
  hipGraphExec_t exec;
};

extern "C" {

const char* kgeo_batch_last_error(void) { return g_err_b; }

size_t kgeo_batch_workspace_bytes(const kgeo_ray_params* imgs, int32_t nimg) {
  if (check_images(imgs, nimg) != KGEO_OK) return 0;
  const BatchSizes z = sizes_of(imgs, nimg);
  return align256(sizeof(BatchImage) * static_cast<size_t>(nimg)) +
         2 * align256(sizeof(uint32_t) * static_cast<size_t>(nimg)) + 256 +
         align256(static_cast<size_t>(z.slots) * PL_N * sizeof(double)) +
         align256(static_cast<size_t>(z.rec) * sizeof(double)) +
         static_cast<size_t>(z.queue) * sizeof(unsigned long long);
}

int kgeo_batch_layout(const kgeo_ray_params* imgs, int32_t nimg, int64_t* pix_off, int64_t* out_off) {
  int rc = check_images(imgs, nimg);
  if (rc) return rc;
  int64_t p = 0, o = 0;
  for (int32_t k = 0; k < nimg; ++k) {
    if (pix_off) pix_off[k] = p;
    if (out_off) out_off[k] = o;
    p += imgs[k].npix;
    o += imgs[k].npix * imgs[k].ngeo;
  }
  if (pix_off) pix_off[nimg] = p;
  if (out_off) out_off[nimg] = o;
  return KGEO_OK;
}

int kgeo_batch_plan(const kgeo_ray_params* imgs, int32_t nimg, const kgeo_batch_tuning* tune, const double* alpha,
                    const double* beta, double* t, double* r, double* th, double* ph, int8_t* rclass,
                    int8_t* thclass, int32_t* nmax_eq, double* tau_tot, uint32_t* status, void* workspace,
                    size_t workspace_bytes, void* stream, kgeo_batch** out) {
  if (!out) return bfail(KGEO_E_ARG, "out handle is NULL");
  *out = nullptr;
  int rc = check_images(imgs, nimg);
  if (rc) return rc;
  if (!alpha || !beta || !th || !r) return bfail(KGEO_E_ARG, "alpha, beta, th and r are required");
  if (!stream) return bfail(KGEO_E_ARG, "graph capture needs a non-default stream");
  const size_t need = kgeo_batch_workspace_bytes(imgs, nimg);
  if (!workspace || workspace_bytes < need)
    return bfail(KGEO_E_WORKSPACE, "workspace too small: need %lld bytes", static_cast<long long>(need));
  if (reinterpret_cast<uintptr_t>(workspace) % 256 != 0) return bfail(KGEO_E_WORKSPACE, "workspace not 256-byte aligned");
  kgeo_batch_tuning tn{64, 8, {0, 0}};
  if (tune) tn = *tune;
  if (tn.samples_per_item < 1) return bfail(KGEO_E_ARG, "samples_per_item < 1 (%lld)", tn.samples_per_item);
  if (tn.waves_per_cu < 1 || tn.waves_per_cu > 64)
    return bfail(KGEO_E_ARG, "waves_per_cu outside 1..64 (%lld)", tn.waves_per_cu);

  std::vector<BatchImage> host(nimg);
  std::vector<uint32_t> per(nimg);
  int64_t pix = 0, slots = 0, outo = 0, rec = 0, queue = 0;
  int64_t items[K_N] = {0, 0};
  // the survey's size as its caller cut it: an item holds samples_per_item
  // samples, rounded up to whole segments
  int64_t asked = 0;
  const int64_t spi =
      (static_cast<int64_t>(tn.samples_per_item) + kAnchorEveryLong - 1) / kAnchorEveryLong * kAnchorEveryLong;
  const int64_t all_slots = total_slots_of(imgs, nimg);
  for (int32_t k = 0; k < nimg; ++k) {
    const kgeo_ray_params& p = imgs[k];
    BatchImage& B = host[k];
    B.c = scalars_of(p);
    B.npix = p.npix;
    B.ngeo = p.ngeo;
    B.pix_off = pix;
    B.slot_off = slots;
    B.slots = slots_of(p);
    B.out_off = outo;
    // an item of the series is 64 rays' part of a block: as many parts as
    // the tuning asks for, while they help to fill the chip (the results are
    // the same bits for any)
    const int64_t nb = series_blocks(p.ngeo);
    const int64_t fill = pick_parts(all_slots, p.ngeo), asks = (p.ngeo / nb + spi - 1) / spi;
    B.units[K_HEAD] = static_cast<int32_t>(nb);
    B.units[K_SERIES] = static_cast<int32_t>(nb * (asks < 1 ? 1 : (asks < fill ? asks : fill)));
    B.th_rec = rec;
    rec += theta_rec_elems(p);
    B.r_rec = rec;
    rec += radial_rec_elems(p);
    queue += queue_elems(p);
    B.do_phi_t = 1;  // required by check_images
    const int64_t tiles = B.slots / kWave;
    int64_t mine = 0;
    for (int q = 0; q < K_N; ++q) {
      B.item_off[q] = items[q];
      items[q] += tiles * B.units[q];
      mine += tiles * B.units[q];
    }
    asked += tiles * ((p.ngeo + spi - 1) / spi);
    if (asked > kMaxItems || items[K_HEAD] > kMaxItems)
      return bfail(KGEO_E_ARG, "too many work items (%lld); raise samples_per_item", asked);
    pix += p.npix;
    slots += B.slots;
    outo += p.npix * p.ngeo;
    per[k] = static_cast<uint32_t>(mine + tiles * B.units[K_HEAD]);  // theta and radial heads
  }
  if (!t || !ph) return bfail(KGEO_E_ARG, "t and ph are required");

  char* w = static_cast<char*>(workspace);
  BatchDev d;
  d.imgs = reinterpret_cast<const BatchImage*>(w);
  w += align256(sizeof(BatchImage) * static_cast<size_t>(nimg));
  d.flags = reinterpret_cast<uint32_t*>(w);
  w += align256(sizeof(uint32_t) * static_cast<size_t>(nimg));
  d.done = reinterpret_cast<uint32_t*>(w);
  w += align256(sizeof(uint32_t) * static_cast<size_t>(nimg));
  d.counter = reinterpret_cast<uint32_t*>(w);
  w += 256;
  d.plan = reinterpret_cast<double*>(w);
  w += align256(static_cast<size_t>(slots) * PL_N * sizeof(double));
  d.rec = reinterpret_cast<double*>(w);
  w += align256(static_cast<size_t>(rec) * sizeof(double));
  d.queue = reinterpret_cast<unsigned long long*>(w);
  d.qcap = static_cast<unsigned long long>(queue);
  d.nimg = nimg;
  d.total_slots = slots;
  for (int q = 0; q < K_N; ++q) d.total_items[q] = static_cast<uint32_t>(items[q]);
  d.alpha = alpha;
  d.beta = beta;
  d.t = t;
  d.r = r;
  d.th = th;
  d.ph = ph;
  d.rclass = rclass;
  d.thclass = thclass;
  d.nmax_eq = nmax_eq;
  d.tau_tot = tau_tot;
  d.status = status;

  hipStream_t st = static_cast<hipStream_t>(stream);
  // the image descriptors are uploaded once, outside the graph
  if (hipMemcpyAsync(const_cast<BatchImage*>(d.imgs), host.data(), sizeof(BatchImage) * host.size(),
                     hipMemcpyHostToDevice, st) != hipSuccess)
    return bfail(KGEO_E_HIP, "descriptor upload failed");
  if (hipStreamSynchronize(st) != hipSuccess) return bfail(KGEO_E_HIP, "descriptor upload failed (sync)");
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return bfail(KGEO_E_HIP, "hipGetDevice failed");
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return bfail(KGEO_E_HIP, "CU count query failed");
  const int waves_per_block = kBlock / kWave;
  const unsigned blocks = static_cast<unsigned>((cus * tn.waves_per_cu + waves_per_block - 1) / waves_per_block);
  const unsigned setup_blocks = static_cast<unsigned>((slots + kBlock - 1) / kBlock);

  kgeo_batch* b = new (std::nothrow) kgeo_batch;
  if (!b) return bfail(KGEO_E_ARG, "out of host memory");
  b->d = d;
  b->items_per_image = per;
  b->graph = nullptr;
  b->exec = nullptr;
  if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess) {
    delete b;
    return bfail(KGEO_E_HIP, "hipStreamBeginCapture failed");
  }
  hipLaunchKernelGGL(kg_batch_clear, dim3(1), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(kg_batch_setup, dim3(setup_blocks), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(kg_batch_theta_heads, dim3(blocks), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(kg_batch_radial_heads, dim3(blocks), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(kg_batch_series, dim3(blocks), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(kg_batch_fixup, dim3(blocks), dim3(kBlock), 0, st, d);
  const int lrc = blaunch("batch kernel launch (capture)");
  hipGraph_t g = nullptr;
  const hipError_t ce = hipStreamEndCapture(st, &g);
  if (lrc || ce != hipSuccess || !g) {
    if (g) (void)hipGraphDestroy(g);
    delete b;
    return lrc ? lrc : bfail(KGEO_E_HIP, "hipStreamEndCapture failed");
  }
  b->graph = g;
  if (hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0) != hipSuccess) {
    (void)hipGraphDestroy(g);
    delete b;
    return bfail(KGEO_E_HIP, "hipGraphInstantiate failed");
  }
  *out = b;
  return KGEO_OK;
}

int kgeo_batch_run(kgeo_batch* b, void* stream) {
  if (!b) return bfail(KGEO_E_ARG, "batch handle is NULL");
  if (hipGraphLaunch(b->exec, static_cast<hipStream_t>(stream)) != hipSuccess)
    return bfail(KGEO_E_HIP, "hipGraphLaunch failed");
  return KGEO_OK;
}

int64_t kgeo_batch_items(const kgeo_batch* b) {
  if (!b) return -1;
  return 2 * static_cast<int64_t>(b->d.total_items[K_HEAD]) + static_cast<int64_t>(b->d.total_items[K_SERIES]);
}

int kgeo_batch_progress(const kgeo_batch* b, uint32_t* done_items, uint32_t* total_items) {
  if (!b) return bfail(KGEO_E_ARG, "batch handle is NULL");
  const size_t n = static_cast<size_t>(b->d.nimg);
  if (total_items)
    for (size_t k = 0; k < n; ++k) total_items[k] = b->items_per_image[k];
  if (done_items && hipMemcpy(done_items, b->d.done, n * sizeof(uint32_t), hipMemcpyDeviceToHost) != hipSuccess)
    return bfail(KGEO_E_HIP, "progress copy failed");
  return KGEO_OK;
}

int kgeo_batch_destroy(kgeo_batch* b) {
  if (!b) return KGEO_OK;
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  delete b;
  return KGEO_OK;
}

}  // extern "C"
