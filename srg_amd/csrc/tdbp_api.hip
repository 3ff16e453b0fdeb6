// tdbp_api.hip -- C ABI of the TDBP engine: runtime helpers, the operator
// API over device buffers, the batch (persistent launch + device work queue +
// hipGraph) and the autotuner.  The drop-in azimuth_compress_ lives in
// tdbp_dropin.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "tdbp_api_internal.h"
#include "tdbp_geom.h"
#include "tdbp_internal.h"

namespace tdbp {

static thread_local char g_err[512] = "";
static int g_variant = -1;

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

int hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return TDBP_OK;
  return set_error(TDBP_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

// ------------------------------------------------ allocation-free scratch

// Scratch of tdbp_backproject_noalloc: the orbit table [t(n) | x(3n) | v(3n)]
// for up to kMaxStateVec state vectors, the aperture parabolas
// [nlines][3], then the 8 tile-queue counters of the burst kernel (32 B).
// One copy per device, held until the process ends; every call on a device
// shares it (calls that overlap on one device race).
constexpr int kNoAllocMaxLines = 16384;
constexpr size_t kScratchOrbit = 7 * (size_t)kMaxStateVec;
constexpr size_t kScratchCounters = kScratchOrbit + 3 * (size_t)kNoAllocMaxLines;
constexpr size_t kScratchDoubles = kScratchCounters + 4;
static __device__ __align__(256) double scratch[kScratchDoubles];

// Device address of `scratch` per device, taken once per device at set-up
// (ensure_device) with that device current.  Host code passes these
// addresses, never the array's name, which on the host is only a stand-in.
static std::map<int, double*> g_scratch;

// ------------------------------------------------------------ device init

static std::mutex g_init_mu;
static std::map<int, int> g_ready;  // device -> status

int ensure_device(int device) {
  std::lock_guard<std::mutex> lk(g_init_mu);
  auto it = g_ready.find(device);
  if (it != g_ready.end()) {
    if (it->second == TDBP_OK) {
      hipError_t e = hipSetDevice(device);
      if (e != hipSuccess) return hip_check(e, "hipSetDevice");
    }
    return it->second == TDBP_OK ? TDBP_OK
                                 : set_error(it->second, "device %d unusable", device);
  }
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  int st = TDBP_OK;
  if (e != hipSuccess || n <= device || device < 0) {
    st = set_error(TDBP_ERR_NODEV, "no HIP device %d (count %d, %s)", device, n,
                   hipGetErrorString(e));
  } else if ((e = hipSetDevice(device)) != hipSuccess) {
    st = hip_check(e, "hipSetDevice");
  } else {
    hipDeviceProp_t prop;
    if ((e = hipGetDeviceProperties(&prop, device)) != hipSuccess) {
      st = hip_check(e, "hipGetDeviceProperties");
    } else if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
      st = set_error(TDBP_ERR_NODEV, "device %d is %s, this build targets gfx950",
                     device, prop.gcnArchName);
    } else {
      double* p = nullptr;
      if ((e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch))) != hipSuccess)
        st = hip_check(e, "hipGetSymbolAddress(scratch)");
      else
        g_scratch[device] = p;
    }
  }
  g_ready[device] = st;
  return st;
}

// The scratch address of the current device (set up by ensure_device).
static int scratch_of_current(double** p) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_check(e, "hipGetDevice");
  std::lock_guard<std::mutex> lk(g_init_mu);
  auto it = g_scratch.find(dev);
  if (it == g_scratch.end() || !it->second)
    return set_error(TDBP_ERR_NODEV, "no scratch address for device %d", dev);
  *p = it->second;
  return TDBP_OK;
}

int current_device_ready() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  return ensure_device(dev);
}

int cu_count() {
  int dev = 0, n = 0;
  (void)hipGetDevice(&dev);
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
      hipSuccess)
    return 256;
  return n > 0 ? n : 256;
}

bool stream_captures(hipStream_t s) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  return s && (hipStreamIsCapturing(s, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone);
}

// ------------------------------------------------------------ geometry

int validate_geom(const tdbp_geom* g) {
  if (!g) return set_error(TDBP_ERR_ARG, "null geometry");
  if (g->rawdatalines < 2 || g->samples < 2)
    return set_error(TDBP_ERR_ARG, "burst %d x %d too small", g->rawdatalines,
                     g->samples);
  if (g->aperture < 0) return set_error(TDBP_ERR_ARG, "aperture %d < 0", g->aperture);
  if (g->numstatevec < 4 || g->numstatevec > kMaxStateVec)
    return set_error(TDBP_ERR_ARG, "numstatevec %d outside [4, %d]",
                     g->numstatevec, kMaxStateVec);
  if (!g->timeorbit || !g->xx || !g->vv)
    return set_error(TDBP_ERR_ARG, "orbit arrays missing");
  if (!(g->timeorbit[1] > g->timeorbit[0]))
    return set_error(TDBP_ERR_ARG, "orbit times not increasing");
  if (g->demwidth < 1 || g->nlines < 1)
    return set_error(TDBP_ERR_ARG, "window %d x %d empty", g->nlines, g->demwidth);
  if (g->firstpix < 0 || g->lastpix > g->demwidth ||
      g->lastpix - g->firstpix < 2)
    return set_error(TDBP_ERR_ARG, "pixel range [%d, %d] invalid for width %d",
                     g->firstpix, g->lastpix, g->demwidth);
  if (!(g->dmrg > 0.) || !(g->wvl > 0.) || !(g->prf > 0.))
    return set_error(TDBP_ERR_ARG, "dmrg/wvl/prf must be positive");
  if (g->semantics != TDBP_SEM_GPU && g->semantics != TDBP_SEM_CPU)
    return set_error(TDBP_ERR_ARG, "unknown semantics %d", g->semantics);
  // The gate rngstart <= R <= rngend - dmrg must keep sample r+1 inside the
  // row: (rngend - dmrg - rngstart)/dmrg <= S - 2 (+ rounding).
  const double rhi = (g->rngend - g->dmrg - g->rngstart) / g->dmrg;
  if (!(rhi <= g->samples - 2 + 1e-6))
    return set_error(TDBP_ERR_ARG,
                     "range window ends at sample %.3f beyond S-2 = %d", rhi,
                     g->samples - 2);
  return TDBP_OK;
}

void fill_burst(const tdbp_geom* g, BurstDev* b) {
  std::memset(b, 0, sizeof *b);
  b->L = g->rawdatalines;
  b->S = g->samples;
  b->A = g->aperture;
  b->W = g->demwidth;
  b->firstline = g->firstline;
  b->nlines = g->nlines;
  b->nfit = g->fit_last_line ? g->nlines : g->nlines - 1;
  b->firstpix = g->firstpix;
  b->lastpix = g->lastpix;
  b->nsv = g->numstatevec;
  b->rngstart = g->rngstart;
  b->rng_hi = g->rngend - g->dmrg;
  b->inv_dmrg = 1.0 / g->dmrg;
  b->two_over_wvl = 2.0 / g->wvl;
  b->cpu = g->semantics == TDBP_SEM_CPU;
  {
    const char* ec = std::getenv("TDBP_MIXED_CHAIN");
    b->chain = ec != nullptr && std::atoi(ec) != 0;
  }
  b->dmrg = g->dmrg;
  b->four_pi_over_wvl = 4. * kPi / g->wvl;  // sentinel/azimuth_compress_cpu.c:75
  b->r_hi = std::min((g->rngend - g->dmrg - g->rngstart) / g->dmrg,
                     (double)(g->samples - 2));
  b->firstlat = g->firstlat;
  b->firstlon = g->firstlon;
  b->deltalat = g->deltalat;
  b->deltalon = g->deltalon;
  b->tmid = g->tmid;
  b->wvl = g->wvl;
  b->angc0 = g->angc0;
  b->angc1 = g->angc1;
  b->prf = g->prf;
  for (int i = 0; i < 3; ++i) {
    b->xyz_mid[i] = g->xyz_mid[i];
    b->vel_mid[i] = g->vel_mid[i];
  }
  b->dtype = TDBP_CF32;
}

// Tile grid of a burst for a variant; returns the variant to launch.  named: the
// variant was asked for by index (in the call, by tdbp_set_variant or in the
// environment); else it is the default, and where variant 1 or 5 would leave
// most of the chip idle that is kSplitVariant.  The CPU twin's arithmetic has no
// split form: kSplitVariant is variant 5 there.
//
// A wave that has a SIMD to itself issues an instruction about every 8 cycles,
// whatever it waits for, so a burst of few tiles takes the time of one tile's
// pulses one after another.  Split over the workgroup's four waves they take a
// quarter, for four times the tiles and of the per-pixel set-up; that pays
// while the 256-pixel tiles with work are at most about one per CU.  Kernel
// times, whole and split: 51 tiles x 256 pulses 85 and 65 us (FP64 62 and 50);
// 54 tiles x 710 pulses 130 and 88 (136 and 56); 196: 176 and 128 (169 and
// 123); 288 x 200 pulses 62 and 75; 393: 186 and 180 (216 and 201); 785: 212
// and 343 (298 and 340).  The rule sees the burst alone, so a batch computes
// each of its bursts as a single launch does.
constexpr double kSplitTiles = 256;
int set_tiles(BurstDev* b, int variant, bool named) {
  // Lines with a valid aperture centre span L - A pulses of the track on the
  // ground.
  const auto norm = [](const double* x) {
    return std::sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  };
  const double step = norm(b->vel_mid) / b->prf * kWgs84A / std::max(norm(b->xyz_mid), kWgs84A);
  const double lines = std::min<double>(
      b->nlines, (b->L - b->A) * step / std::max(std::fabs(b->deltalat) * 111320.0, 1e-3));
  const double tiles = std::max(lines, 0.0) * b->W / 256.0;
  if (b->cpu) {
    if (variant == kSplitVariant) variant = 5;
  } else if (!named && (variant == 1 || variant == 5) && tiles <= kSplitTiles) {
    variant = kSplitVariant;
  }
  b->split = variant == kSplitVariant;
  const Variant& v = kVariants[variant];
  b->tiles_r = (b->nlines + wg_rows(v) - 1) / wg_rows(v);
  b->tiles_c = (b->W + wg_cols(v) - 1) / wg_cols(v);
  return variant;
}

// Orbit arrays packed [t(n) | x(3n) | v(3n)] for the device.
std::vector<double> pack_orbit(const tdbp_geom* g) {
  const int n = g->numstatevec;
  std::vector<double> o(7 * (size_t)n);
  std::memcpy(o.data(), g->timeorbit, n * sizeof(double));
  std::memcpy(o.data() + n, g->xx, 3 * n * sizeof(double));
  std::memcpy(o.data() + 4 * n, g->vv, 3 * n * sizeof(double));
  return o;
}

void point_orbit(BurstDev* b, const double* d_orbit, int n) {
  b->orb_t = d_orbit;
  b->orb_x = d_orbit + n;
  b->orb_v = d_orbit + 4 * n;
}

int check_samples(const tdbp_samples* s, int precision) {
  if (!s || !s->d_data) return set_error(TDBP_ERR_ARG, "no samples");
  if (s->dtype < TDBP_CF32 || s->dtype > TDBP_CI16)
    return set_error(TDBP_ERR_ARG, "unknown dtype %d", s->dtype);
  if (precision == TDBP_PLAIN_FP64 && s->dtype != TDBP_CF32)
    return set_error(TDBP_ERR_ARG, "the FP64 kernel reads cf32 samples only");
  if (precision != TDBP_PLAIN_FP64 && precision != TDBP_MIXED)
    return set_error(TDBP_ERR_ARG, "unknown precision %d", precision);
  if (s->dtype != TDBP_CF32 && !s->d_scale)
    return set_error(TDBP_ERR_ARG, "packed samples need per-pulse scales");
  return TDBP_OK;
}

int automatic_variant(int precision, bool* named) {
  const auto from_env = [&](const char* name, int otherwise) {
    const char* e = std::getenv(name);
    const int v = e ? std::atoi(e) : -1;
    *named = v >= 0 && v < kNumVariants;
    return *named ? v : otherwise;
  };
  if (precision == TDBP_PLAIN_FP64) {
    // Variant 1 (4 x 16 wave tiles side by side): 3.04 ms on one IW burst against
    // 2.99 (variant 0), 3.00 (5), 3.06 (6), 3.08 (4), 3.24 (2), 3.43 (7) and 9.1
    // (3): within 2 % but for the narrow tiles, so 1, the fastest of the pair by
    // pair kernel, stays.
    return from_env("TDBP_PLAIN_VARIANT", 1);
  }
  return from_env("TDBP_VARIANT", 5);
}

int default_variant(int precision, bool* named) {
  if (precision == TDBP_MIXED && g_variant >= 0) {
    *named = true;
    return g_variant;
  }
  return automatic_variant(precision, named);
}

// Whether the fit may carry the orbit in its arguments (launch_fit_arg).  Not
// while the stream is captured: the fit of a captured call stays refused, by
// the wait below, as replays would keep the orbit of the capture.
static bool orbit_in_args(const tdbp_geom* g, hipStream_t s) {
  return g->numstatevec <= kFitArgVec && !stream_captures(s);
}

// The fit on a stream.  Orbits of up to kFitArgVec vectors go with the launch
// and the call returns at once; larger ones are uploaded to stream-ordered
// temporary memory, which the call waits for (31 us of a small burst's 81).
int fit_on_stream(BurstDev& b, const tdbp_geom* g, double* d_coef,
                  hipStream_t s) {
  std::vector<double> orb = pack_orbit(g);
  if (orbit_in_args(g, s))
    return hip_check(launch_fit_arg(b, orb.data(), d_coef, s), "fit launch");
  double* d_orb = nullptr;
  int st = hip_check(hipMallocAsync((void**)&d_orb, orb.size() * 8, s),
                     "hipMallocAsync(orbit)");
  if (st) return st;
  st = hip_check(hipMemcpyAsync(d_orb, orb.data(), orb.size() * 8,
                                hipMemcpyHostToDevice, s),
                 "orbit upload");
  point_orbit(&b, d_orb, g->numstatevec);
  if (!st) st = hip_check(launch_fit_one(b, d_coef, s), "fit launch");
  // The pageable source must outlive the copy.
  if (!st) st = hip_check(hipStreamSynchronize(s), "fit sync");
  (void)hipFreeAsync(d_orb, s);
  b.orb_t = b.orb_x = b.orb_v = nullptr;
  return st;
}

// Tile-queue counters of the single-burst kernels, one set of 8 per
// (device, stream), allocated at the first launch on it and kept: launches on
// one stream run in order, so each zeroes and drains its own.
namespace {
struct CounterSet {
  int dev;
  hipStream_t stream;
  int* p;
};
std::mutex g_ctr_mu;
std::vector<CounterSet> g_ctr;

int counters_for(hipStream_t s, int** out) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(g_ctr_mu);
  for (const CounterSet& c : g_ctr)
    if (c.dev == dev && c.stream == s) {
      *out = c.p;
      return TDBP_OK;
    }
  int* p = nullptr;
  if (hipMalloc((void**)&p, 8 * sizeof(int)) != hipSuccess)
    return set_error(TDBP_ERR_NOMEM, "tile-queue counters");
  g_ctr.push_back(CounterSet{dev, s, p});
  *out = p;
  return TDBP_OK;
}
}  // namespace

int run_backproject(const tdbp_geom* g, const tdbp_samples* smp,
                    const double* d_satloc, const int16_t* d_dem,
                    const double* d_coef, void* d_out, int precision,
                    int variant, hipStream_t s) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = check_samples(smp, precision))) return st;
  if (!d_satloc || !d_dem || !d_out)
    return set_error(TDBP_ERR_ARG, "null device buffer");
  if ((st = current_device_ready())) return st;
  BurstDev b;
  fill_burst(g, &b);
  b.data = smp->d_data;
  b.scale = smp->d_scale;
  b.dtype = smp->dtype;
  b.satloc = d_satloc;
  b.dem = d_dem;
  b.out = (float2*)d_out;
  bool named = variant >= 0 && variant < kNumVariants;
  if (!named) variant = default_variant(precision, &named);
  variant = set_tiles(&b, variant, named);
  if ((st = counters_for(s, &b.counters))) return st;
  double* own = nullptr;
  if (!d_coef) {
    st = hip_check(hipMallocAsync((void**)&own, 24 * (size_t)g->nlines, s),
                   "hipMallocAsync(coef)");
    if (st) return st;
    if ((st = fit_on_stream(b, g, own, s))) {
      (void)hipFreeAsync(own, s);
      return st;
    }
    d_coef = own;
  }
  b.coef = d_coef;
  hipError_t e = precision == TDBP_PLAIN_FP64 ? launch_plain(b, variant, s)
                                              : launch_mixed(b, variant, s);
  st = hip_check(e, "backprojection launch");
  if (own) (void)hipFreeAsync(own, s);
  return st;
}

// The 80-byte headers of `nlines` device lines to (or from) host memory
// [nlines][80]: gathered (scattered) by a kernel on the device side of one
// contiguous copy, through a pinned chunk on the host side.  A pitched
// hipMemcpy2DAsync moves such rows one by one: 7.9 ms for 1200 lines; the
// gather with a copy into pageable memory took 0.10 ms, through the pinned
// chunk 0.05 ms.  Lines that are not the current device's own memory (a peer's,
// managed or host memory) still go row by row: the kernel may not reach them.
constexpr int kHeaderChunk = 4096;   // lines

// Pinned chunks (320 KB): a call holds one while it runs, so calls on different
// streams do not wait for each other; up to four idle ones are kept.
namespace {
std::mutex g_header_mu;
uint8_t* g_header_idle[4] = {};

uint8_t* take_header_chunk() {
  {
    std::lock_guard<std::mutex> lk(g_header_mu);
    for (uint8_t*& p : g_header_idle)
      if (p) return std::exchange(p, nullptr);
  }
  uint8_t* p = nullptr;
  const hipError_t e =
      hipHostMalloc((void**)&p, (size_t)kHeaderChunk * 80, hipHostMallocPortable);
  return hip_check(e, "header staging") ? nullptr : p;
}

void return_header_chunk(uint8_t* p) {
  {
    std::lock_guard<std::mutex> lk(g_header_mu);
    for (uint8_t*& q : g_header_idle)
      if (!q) {
        q = p;
        return;
      }
  }
  (void)hipHostFree(p);
}
// Whether p is memory of the current device.
bool on_current_device(const void* p) {
  int dev = 0;
  hipPointerAttribute_t a;
  if (hipGetDevice(&dev) == hipSuccess && hipPointerGetAttributes(&a, p) == hipSuccess)
    return a.type == hipMemoryTypeDevice && a.device == dev;
  (void)hipGetLastError();   // an address the runtime does not know is no failed launch
  return false;
}
}  // namespace

static int copy_headers(void* d_lines, int nlines, int stride, uint8_t* host, bool to_device,
                        void* stream) {
  if (!d_lines || !host || nlines < 1 || stride < 10)
    return set_error(TDBP_ERR_ARG, "headers: bad arguments");
  int st = current_device_ready();
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  if (!on_current_device(d_lines)) {
    const size_t pitch = (size_t)stride * 8, n = (size_t)nlines;
    st = to_device ? hip_check(hipMemcpy2DAsync(d_lines, pitch, host, 80, 80, n,
                                                hipMemcpyHostToDevice, s), "header upload")
                   : hip_check(hipMemcpy2DAsync(host, 80, d_lines, pitch, 80, n,
                                                hipMemcpyDeviceToHost, s), "header download");
    return st ? st : hip_check(hipStreamSynchronize(s), "header sync");
  }
  uint8_t* pin = take_header_chunk();
  if (!pin) return TDBP_ERR_HIP;
  void* d = nullptr;
  st = hip_check(hipMallocAsync(&d, (size_t)std::min(nlines, kHeaderChunk) * 80, s),
                 "header scratch");
  for (int l0 = 0; l0 < nlines && !st; l0 += kHeaderChunk) {
    const int n = std::min(kHeaderChunk, nlines - l0);
    const size_t bytes = (size_t)n * 80;
    char* lines = (char*)d_lines + (size_t)l0 * (size_t)stride * 8;
    if (to_device) {
      std::memcpy(pin, host + (size_t)l0 * 80, bytes);
      st = hip_check(hipMemcpyAsync(d, pin, bytes, hipMemcpyHostToDevice, s), "header upload");
      if (!st) st = hip_check(launch_headers(lines, n, stride, d, true, s), "header scatter");
    } else {
      st = hip_check(launch_headers(lines, n, stride, d, false, s), "header gather");
      if (!st)
        st = hip_check(hipMemcpyAsync(pin, d, bytes, hipMemcpyDeviceToHost, s),
                       "header download");
    }
    const int st2 = hip_check(hipStreamSynchronize(s), "header sync");
    if (!st) st = st2;
    if (!st && !to_device) std::memcpy(host + (size_t)l0 * 80, pin, bytes);
  }
  if (d) (void)hipFreeAsync(d, s);
  return_header_chunk(pin);
  return st;
}

}  // namespace tdbp

using namespace tdbp;

// ================================================================ C ABI

extern "C" {

const char* tdbp_last_error(void) { return g_err; }

int tdbp_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

int tdbp_init(int device) { return ensure_device(device); }

void* tdbp_dev_alloc(size_t bytes) {
  if (current_device_ready()) return nullptr;
  void* p = nullptr;
  if (hipMalloc(&p, bytes ? bytes : 1) != hipSuccess) {
    set_error(TDBP_ERR_NOMEM, "hipMalloc(%zu) failed", bytes);
    return nullptr;
  }
  return p;
}

int tdbp_dev_free(void* p) { return hip_check(hipFree(p), "hipFree"); }

int tdbp_memcpy_htod(void* d, const void* h, size_t n, void* s) {
  int st = hip_check(
      hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, (hipStream_t)s), "memcpy H2D");
  if (st) return st;
  return hip_check(hipStreamSynchronize((hipStream_t)s), "memcpy H2D sync");
}

int tdbp_memcpy_dtoh(void* h, const void* d, size_t n, void* s) {
  int st = hip_check(
      hipMemcpyAsync(h, d, n, hipMemcpyDeviceToHost, (hipStream_t)s), "memcpy D2H");
  if (st) return st;
  return hip_check(hipStreamSynchronize((hipStream_t)s), "memcpy D2H sync");
}

int tdbp_memcpy_dtod(void* d, const void* src, size_t n, void* s) {
  return hip_check(
      hipMemcpyAsync(d, src, n, hipMemcpyDeviceToDevice, (hipStream_t)s),
      "memcpy D2D");
}

int tdbp_merge_geo(void* d_grid, int W, int grid_lines, int firstline, int nlines,
                   const void* d_out, int semantics, void* stream) {
  if (!d_grid || !d_out || W < 1 || nlines < 1 || firstline < 0 ||
      firstline + nlines > grid_lines)
    return set_error(TDBP_ERR_ARG, "merge: rows [%d, %d) outside a %d-line grid", firstline,
                     firstline + nlines, grid_lines);
  if (semantics != TDBP_SEM_GPU && semantics != TDBP_SEM_CPU)
    return set_error(TDBP_ERR_ARG, "merge: unknown semantics %d", semantics);
  int st = current_device_ready();
  if (st) return st;
  return hip_check(launch_merge((float2*)d_grid, (const float2*)d_out, (size_t)nlines * W,
                                (size_t)firstline * W, semantics, (hipStream_t)stream),
                   "merge launch");
}

int tdbp_compare(const void* d_img, const void* d_ref, size_t n, double* sums,
                 void* stream) {
  if (!d_img || !d_ref || !sums) return set_error(TDBP_ERR_ARG, "compare: null pointer");
  int st = current_device_ready();
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  const int blocks = compare_blocks(n);
  double* part = nullptr;
  if ((st = hip_check(hipMallocAsync((void**)&part, (size_t)blocks * 5 * sizeof(double), s),
                      "compare scratch")))
    return st;
  std::vector<double> hp((size_t)blocks * 5);
  st = hip_check(launch_compare((const float2*)d_img, (const float2*)d_ref, n, part,
                                blocks, s),
                 "compare launch");
  if (!st)
    st = hip_check(hipMemcpyAsync(hp.data(), part, hp.size() * sizeof(double),
                                  hipMemcpyDeviceToHost, s),
                   "compare download");
  const int st2 = hip_check(hipFreeAsync(part, s), "compare scratch free");
  const int st3 = hip_check(hipStreamSynchronize(s), "compare sync");
  if (st) return st;
  if (st2) return st2;
  if (st3) return st3;
  for (int k = 0; k < 5; ++k) sums[k] = 0.0;
  for (int b = 0; b < blocks; ++b)
    for (int k = 0; k < 5; ++k) sums[k] += hp[(size_t)b * 5 + k];
  return TDBP_OK;
}

int tdbp_headers_dtoh(const void* d_lines, int nlines, int stride, uint8_t* host, void* stream) {
  return copy_headers(const_cast<void*>(d_lines), nlines, stride, host, false, stream);
}

int tdbp_headers_htod(void* d_lines, int nlines, int stride, const uint8_t* host,
                      void* stream) {
  return copy_headers(d_lines, nlines, stride, const_cast<uint8_t*>(host), true, stream);
}

int tdbp_dev_copy(void* d, const void* src, size_t n, void* s) {
  return hip_check(launch_copy(d, src, n, (hipStream_t)s), "copy");
}

int tdbp_dev_zero(void* d, size_t n, void* s) {
  return hip_check(launch_zero(d, n, (hipStream_t)s), "zero");
}

int tdbp_stream_create(void** s) {
  if (current_device_ready()) return TDBP_ERR_NODEV;
  return hip_check(hipStreamCreateWithFlags((hipStream_t*)s, hipStreamNonBlocking),
                   "hipStreamCreate");
}
int tdbp_stream_destroy(void* s) {
  return hip_check(hipStreamDestroy((hipStream_t)s), "hipStreamDestroy");
}
int tdbp_stream_sync(void* s) {
  return hip_check(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize");
}
int tdbp_device_sync(void) {
  return hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
}
int tdbp_event_create(void** e) {
  return hip_check(hipEventCreate((hipEvent_t*)e), "hipEventCreate");
}
int tdbp_event_destroy(void* e) {
  return hip_check(hipEventDestroy((hipEvent_t)e), "hipEventDestroy");
}
int tdbp_event_record(void* e, void* s) {
  return hip_check(hipEventRecord((hipEvent_t)e, (hipStream_t)s),
                   "hipEventRecord");
}
int tdbp_stream_wait_event(void* s, void* e) {
  return hip_check(hipStreamWaitEvent((hipStream_t)s, (hipEvent_t)e, 0), "hipStreamWaitEvent");
}

int tdbp_event_elapsed_ms(void* a, void* b, float* ms) {
  return hip_check(hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b),
                   "hipEventElapsedTime");
}
int tdbp_mem_info(size_t* f, size_t* t) {
  return hip_check(hipMemGetInfo(f, t), "hipMemGetInfo");
}

void tdbp_window(const double* latlons, double firstlat, double firstlon,
                 double deltalat, double deltalon, int demwidth, int demlength,
                 int* firstline, int* lastline, int* firstpix, int* lastpix) {
  int ll = (int)((latlons[0] - firstlat) / deltalat);
  int fl = (int)((latlons[1] - firstlat) / deltalat);
  fl = fl < 0 ? 0 : fl;
  ll = ll < 0 ? 0 : ll;
  fl = fl > demlength - 1 ? demlength - 1 : fl;
  ll = ll > demlength - 1 ? demlength - 1 : ll;
  int fp = (int)((latlons[2] - firstlon) / deltalon);
  fp = fp < 0 ? 0 : fp;
  int lp = (int)((latlons[3] - firstlon) / deltalon);
  lp = lp > demwidth ? demwidth : lp;
  *firstline = fl;
  *lastline = ll;
  *firstpix = fp;
  *lastpix = lp;
}

int tdbp_orbit_interp(const double* t, const double* x, const double* v, int n,
                      const double* times, int m, double* pos, double* vel) {
  if (!t || !x || !v || !times || n < 4 || m < 0)
    return set_error(TDBP_ERR_ARG, "orbit_interp: bad arguments");
  for (int i = 0; i < m; ++i) {
    double p[3], w[3];
    orbit_at(t, x, v, n, times[i], p, w);
    if (pos) std::memcpy(pos + 3 * i, p, sizeof p);
    if (vel) std::memcpy(vel + 3 * i, w, sizeof w);
  }
  return TDBP_OK;
}

int tdbp_setxyz(const tdbp_geom* g, const int16_t* d_dem, double* d_xyz,
                double* d_xyzfit, void* stream) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = current_device_ready())) return st;
  BurstDev b;
  fill_burst(g, &b);
  b.dem = d_dem;
  return hip_check(launch_setxyz(b, d_xyz, d_xyzfit, (hipStream_t)stream),
                   "setxyz launch");
}

int tdbp_fit_aperture(const tdbp_geom* g, const int16_t* d_dem, double* d_coef,
                      void* stream) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = current_device_ready())) return st;
  BurstDev b;
  fill_burst(g, &b);
  b.dem = d_dem;
  if ((st = fit_on_stream(b, g, d_coef, (hipStream_t)stream))) return st;
  // Callers may use the parabolas on another stream.
  return hip_check(hipStreamSynchronize((hipStream_t)stream), "fit sync");
}

int tdbp_setazoff(const tdbp_geom* g, const double* d_coef, double* d_azoff,
                  void* stream) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = current_device_ready())) return st;
  BurstDev b;
  fill_burst(g, &b);
  b.coef = d_coef;
  return hip_check(launch_setazoff(b, d_azoff, (hipStream_t)stream),
                   "setazoff launch");
}

int tdbp_pair_count(const tdbp_geom* g, const double* d_coef, int64_t* d_pairs,
                    void* stream) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = current_device_ready())) return st;
  BurstDev b;
  fill_burst(g, &b);
  b.coef = d_coef;
  return hip_check(launch_pair_count(b, d_pairs, (hipStream_t)stream),
                   "pair count launch");
}

int tdbp_pack_samples(const void* d_cf32, int L, int S, int dtype,
                      void* d_packed, float* d_scale, void* stream) {
  if (!d_cf32 || !d_packed || !d_scale || L < 1 || S < 1 ||
      (dtype != TDBP_CF16 && dtype != TDBP_CBF16 && dtype != TDBP_CI16))
    return set_error(TDBP_ERR_ARG, "pack: bad arguments");
  int st = current_device_ready();
  if (st) return st;
  return hip_check(launch_pack((const float2*)d_cf32, L, S, dtype, d_packed,
                               d_scale, (hipStream_t)stream),
                   "pack launch");
}

int tdbp_pixelint(const tdbp_geom* g, const void* d_burst,
                  const double* d_satloc, const double* d_xyz,
                  const double* d_azoff, void* d_out, void* stream) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = current_device_ready())) return st;
  if (!d_burst || !d_satloc || !d_xyz || !d_azoff || !d_out)
    return set_error(TDBP_ERR_ARG, "pixelint: null buffer");
  BurstDev b;
  fill_burst(g, &b);
  b.data = d_burst;
  b.satloc = d_satloc;
  b.out = (float2*)d_out;
  return hip_check(launch_pixelint(b, d_xyz, d_azoff, (hipStream_t)stream),
                   "pixelint launch");
}

int tdbp_backproject(const tdbp_geom* g, const tdbp_samples* s,
                     const double* d_satloc, const int16_t* d_dem,
                     const double* d_coef, void* d_out, int precision,
                     void* stream) {
  return run_backproject(g, s, d_satloc, d_dem, d_coef, d_out, precision, -1,
                         (hipStream_t)stream);
}

int tdbp_backproject_variant(const tdbp_geom* g, const tdbp_samples* s,
                             const double* d_satloc, const int16_t* d_dem,
                             const double* d_coef, void* d_out, int precision,
                             int variant, void* stream) {
  return run_backproject(g, s, d_satloc, d_dem, d_coef, d_out, precision,
                         variant, (hipStream_t)stream);
}

// tdbp_backproject with the fit's scratch in the per-device `scratch`
// array: the orbit table is copied from the caller's host arrays into it,
// the parabolas are written there by the fit, and the burst kernel reads
// them; nothing is allocated.  Limits: nlines <= kNoAllocMaxLines,
// numstatevec <= kMaxStateVec (validate_geom).  The fit writes every line's
// coefficients (lines past nfit get zeros), so no clearing is needed.
int tdbp_backproject_noalloc(const tdbp_geom* g, const tdbp_samples* smp,
                             const double* d_satloc, const int16_t* d_dem, void* d_out,
                             int precision, void* stream) {
  if (g && g->nlines > kNoAllocMaxLines)
    return set_error(TDBP_ERR_LIMIT, "noalloc: %d window lines > %d", g->nlines,
                     kNoAllocMaxLines);
  int st = validate_geom(g);
  if (st) return st;
  if ((st = check_samples(smp, precision))) return st;
  if (!d_satloc || !d_dem || !d_out) return set_error(TDBP_ERR_ARG, "null device buffer");
  if ((st = current_device_ready())) return st;
  double* sc = nullptr;
  if ((st = scratch_of_current(&sc))) return st;
  hipStream_t s = (hipStream_t)stream;
  BurstDev b;
  fill_burst(g, &b);
  b.data = smp->d_data;
  b.scale = smp->d_scale;
  b.dtype = smp->dtype;
  b.satloc = d_satloc;
  b.dem = d_dem;
  b.out = (float2*)d_out;
  bool named = false;
  int variant = default_variant(precision, &named);
  variant = set_tiles(&b, variant, named);
  const int n = g->numstatevec;
  double* coef = sc + kScratchOrbit;
  if (orbit_in_args(g, s)) {
    double orb[7 * kFitArgVec];
    std::copy(g->timeorbit, g->timeorbit + n, orb);
    std::copy(g->xx, g->xx + 3 * n, orb + n);
    std::copy(g->vv, g->vv + 3 * n, orb + 4 * n);
    if ((st = hip_check(launch_fit_arg(b, orb, coef, s), "fit launch"))) return st;
  } else {
    if ((st = hip_check(hipMemcpyAsync(sc, g->timeorbit, n * sizeof(double),
                                       hipMemcpyHostToDevice, s), "orbit times")) ||
        (st = hip_check(hipMemcpyAsync(sc + n, g->xx, 3 * n * sizeof(double),
                                       hipMemcpyHostToDevice, s), "orbit positions")) ||
        (st = hip_check(hipMemcpyAsync(sc + 4 * n, g->vv, 3 * n * sizeof(double),
                                       hipMemcpyHostToDevice, s), "orbit velocities")))
      return st;
    point_orbit(&b, sc, n);
    if ((st = hip_check(launch_fit_one(b, coef, s), "fit launch"))) return st;
  }
  b.orb_t = b.orb_x = b.orb_v = nullptr;
  b.coef = coef;
  b.counters = (int*)(sc + kScratchCounters);
  hipError_t e = precision == TDBP_PLAIN_FP64 ? launch_plain(b, variant, s)
                                              : launch_mixed(b, variant, s);
  if ((st = hip_check(e, "backprojection launch"))) return st;
  // The caller's host orbit arrays may be released when this returns.
  return hip_check(hipStreamSynchronize(s), "noalloc sync");
}

int tdbp_set_variant(int v) {
  if (v < -1 || v >= kNumVariants)
    return set_error(TDBP_ERR_ARG, "variant %d outside [-1, %d)", v, kNumVariants);
  g_variant = v;
  return TDBP_OK;
}
int tdbp_variant_count(void) { return kNumVariants; }
int tdbp_variant_info(int v, int* rows, int* cols, int* stage) {
  if (v < 0 || v >= kNumVariants) return set_error(TDBP_ERR_ARG, "variant %d", v);
  if (rows) *rows = wg_rows(kVariants[v]);
  if (cols) *cols = wg_cols(kVariants[v]);
  // pulses per stage of records; the LDS-staged variants sum in sub-stages
  // of kLdsPulses pulses whose sample windows sit in LDS
  if (stage) *stage = kVariants[v].lds ? kLdsPulses : kBlock;
  return TDBP_OK;
}

// ------------------------------------------------------------- synthetic

int tdbp_synth_clutter(void* d, int L, int S, uint64_t seed, float sigma,
                       const float* taps, int ntaps, void* stream) {
  if (!d || L < 1 || S < 1 || ntaps < 1 || ntaps > 64 || !taps)
    return set_error(TDBP_ERR_ARG, "synth_clutter: bad arguments");
  int st = current_device_ready();
  if (st) return st;
  return hip_check(launch_synth_clutter((float2*)d, L, S, seed, sigma, taps,
                                        ntaps, (hipStream_t)stream),
                   "synth_clutter launch");
}

int tdbp_synth_raw(void* d_raw, int L, int stride, const tdbp_chirp* c,
                   const uint8_t* header80, const double* delay, const double* carrier,
                   const float* amp, int ntargets, float noise, uint64_t seed, void* stream) {
  if (!d_raw || !c || !header80 || L < 1 || L > 65535 || stride < 10 + c->nsamps ||
      c->nsamps < 1 || c->npts < 1 || ntargets < 0 || (ntargets > 0 && (!delay || !carrier || !amp)))
    return set_error(TDBP_ERR_ARG, "synth_raw: bad arguments");
  int st = current_device_ready();
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  const size_t nd = (size_t)L * (ntargets > 0 ? ntargets : 1);
  double *dd = nullptr, *dc = nullptr;
  float2* da = nullptr;
  if (!(st = hip_check(hipMallocAsync((void**)&dd, nd * 8, s), "synth_raw scratch")) &&
      !(st = hip_check(hipMallocAsync((void**)&dc, nd * 8, s), "synth_raw scratch")) &&
      !(st = hip_check(hipMallocAsync((void**)&da, 8 * (ntargets > 0 ? ntargets : 1), s),
                       "synth_raw scratch")) &&
      ntargets > 0) {
    if (!(st = hip_check(hipMemcpyAsync(dd, delay, nd * 8, hipMemcpyHostToDevice, s),
                         "synth_raw upload")) &&
        !(st = hip_check(hipMemcpyAsync(dc, carrier, nd * 8, hipMemcpyHostToDevice, s),
                         "synth_raw upload")))
      st = hip_check(hipMemcpyAsync(da, amp, 8 * (size_t)ntargets, hipMemcpyHostToDevice, s),
                     "synth_raw upload");
  }
  if (!st)
    st = hip_check(launch_synth_raw((float2*)d_raw, L, stride, c->nsamps, c->npts, c->samplefreq,
                                    c->startfreq, c->ramprate, dd, dc, da, ntargets, noise, seed,
                                    header80, s),
                   "synth_raw launch");
  // Freed on every path (a null pointer is a no-op).
  if (dd) (void)hipFreeAsync(dd, s);
  if (dc) (void)hipFreeAsync(dc, s);
  if (da) (void)hipFreeAsync(da, s);
  if (!st) st = hip_check(hipStreamSynchronize(s), "synth_raw sync");
  return st;
}

int tdbp_synth_targets(void* d, const tdbp_geom* g, const double* d_satloc,
                       const double* xyz, const float* amp, int ntargets,
                       float res, int halfwidth, void* stream) {
  if (!d || !g || !d_satloc || (ntargets > 0 && (!xyz || !amp)) ||
      halfwidth < 0 || halfwidth > 511 || !(res > 0.f))
    return set_error(TDBP_ERR_ARG, "synth_targets: bad arguments");
  int st = current_device_ready();
  if (st) return st;
  BurstDev b;
  std::memset(&b, 0, sizeof b);
  b.L = g->rawdatalines;
  b.S = g->samples;
  b.rngstart = g->rngstart;
  b.inv_dmrg = 1.0 / g->dmrg;
  b.two_over_wvl = 2.0 / g->wvl;
  b.satloc = d_satloc;
  for (int k = 0; k < ntargets; ++k) {
    st = hip_check(launch_synth_target((float2*)d, b, xyz[3 * k], xyz[3 * k + 1],
                                       xyz[3 * k + 2], amp[2 * k], amp[2 * k + 1],
                                       res, halfwidth, (hipStream_t)stream),
                   "synth_target launch");
    if (st) return st;
  }
  return TDBP_OK;
}

}  // extern "C"
