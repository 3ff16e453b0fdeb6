// tdbp_range.hip -- range compression of decoded echo lines on the device,
// the matched filter of sentinel/processsub.f90:75-126:
//   * chirp parameters from the 80-byte packet header of the first line
//     (:75-86, with the header field readers in2/in3 and the sampling-rate
//     table samplefrequency of :163-212, in the reference's FP32 storage);
//   * reference function reftime(j) = exp(j phase(t_j)) / npts, t_j =
//     j / samplefreq, phase = 2 pi startfreq t + pi ramprate t^2, over the
//     npts chirp samples, transformed forward (:96-103);
//   * per line: the nsamps echo samples after the header, zero-padded to
//     32768, forward FFT, times conj(reference spectrum), inverse FFT
//     without normalisation; the first nvalid = nsamps - npts samples are the
//     compressed line (:108-123).
// Two implementations of the same correlation:
//   * fused overlap-save (chirps of up to 4096 samples, the IW case): one
//     kernel takes an 8192-sample block of a line into LDS, runs the forward
//     FFT, the product with the conjugate reference spectrum and the inverse
//     FFT there (tdbp_osfft.h), and writes the block's M = 8192 - npts + 1
//     valid outputs; the line's blocks cover its nvalid outputs.  HBM sees
//     one read of the echo (the blocks' overlaps come from L2) and one write
//     of the cf32 rows; a packed output is then made from those rows by one
//     elementwise pass (into a scratch when the caller wants no cf32 rows);
//   * rocFFT plans over batches of lines at the shortest 2-3-5 length >=
//     nsamps, with the loading, the spectrum product and the output stage as
//     kernels of this file (longer chirps, or TDBP_RC_ROCFFT=1).
// Both write the reference layout (header samples, then the compressed
// samples, cf32) and/or the backprojection input: the header samples zeroed
// (sentinel/backprojectgpusub.f90:190) and the line packed with its
// per-pulse scale, the same words tdbp_pack_samples makes.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "tdbp_api_internal.h"
#include "tdbp_fft.h"
#include "tdbp_internal.h"
#include "tdbp_osfft.h"
#include "tdbp_pack.h"

using namespace tdbp;

namespace {

constexpr int kFftLen = 32768;   // processsub.f90:39, the largest length used
constexpr int kChunk = 256;      // lines per batched transform
constexpr int kHdr = 10;         // header samples (80 bytes) per line
constexpr double kFref = 37.53472224;

// ------------------------------------------------------------ header fields

int be16(const uint8_t* b) { return (int)b[1] + 256 * (int)b[0]; }
int be24(const uint8_t* b) { return (int)b[2] + 256 * (int)b[1] + 65536 * (int)b[0]; }

// Sampling rate (MHz) per range decimation code, processsub.f90:181-212: the
// ratio is a single-precision quotient times 4 (Fortran default reals), then
// scaled by fref in double.  Codes outside the table: 0.
double sample_frequency(int code) {
  float r;
  switch (code) {
    case 0: r = 3.f / 4.f; break;
    case 1: r = 2.f / 3.f; break;
    case 3: r = 5.f / 9.f; break;
    case 4: r = 4.f / 9.f; break;
    case 5: r = 3.f / 8.f; break;
    case 6: r = 1.f / 3.f; break;
    case 7: r = 1.f / 6.f; break;
    case 8: r = 3.f / 7.f; break;
    case 9: r = 5.f / 16.f; break;
    case 10: r = 3.f / 26.f; break;
    case 11: r = 4.f / 11.f; break;
    default: return 0.0;
  }
  const float r4 = r * 4.f;
  return (double)r4 * kFref;
}

// ------------------------------------------------------------ kernels

// Reference function (processsub.f90:96-101): t in FP32 (integer over real*4),
// phase in FP64, cos/sin rounded to FP32, divided by npts in FP32; times
// gain = 32768 / n so that an n-point transform pair gives the reference's
// 32768-point output scale (1 when n = 32768).
__global__ void k_chirp(float2* __restrict__ ref, int n, int npts, float samplefreq,
                        float startfreq, float ramprate, float gain) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  float2 v = make_float2(0.f, 0.f);
  if (j < npts) {
#pragma clang fp contract(off)
    const double pi = 3.141592653589793115997963468544185161590576171875;
    const double t = (double)((float)j / samplefreq);
    const double phase = 2.0 * pi * (double)startfreq * t + pi * (double)ramprate * t * t;
    const float fn = (float)npts;
    v = make_float2((float)cos(phase) / fn * gain, (float)sin(phase) / fn * gain);
  }
  ref[j] = v;
}

// Zero-padded echo samples of lines [base, base + kChunk).
__global__ void k_rc_load(const float2* __restrict__ raw, int nlines, int stride, int nsamps,
                          int base, int n, float2* __restrict__ buf) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;   // sample
  const int i = blockIdx.y;                              // line in chunk
  if (j >= n) return;
  const int l = base + i;
  float2 v = make_float2(0.f, 0.f);
  if (l < nlines && j < nsamps) v = raw[(size_t)l * stride + kHdr + j];
  buf[(size_t)i * n + j] = v;
}

// Spectrum times conj(reference spectrum).
__global__ void k_rc_mul(float2* __restrict__ buf, const float2* __restrict__ ref, int n) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (j >= n) return;
  float2* p = buf + (size_t)i * n + j;
  const float2 a = *p, r = ref[j];
  *p = make_float2(a.x * r.x + a.y * r.y, a.y * r.x - a.x * r.y);
}

// Output stage, one block of 16 waves per line (a batch is 256 lines: one
// block per CU would leave most of each CU idle).
constexpr int kStoreBlock = 1024;
__global__ void __launch_bounds__(kStoreBlock)
k_rc_store(const float2* __restrict__ raw, int nlines, int stride, int base,
           const float2* __restrict__ buf, int n, int nvalid, float2* __restrict__ out,
           int out_stride, int zero_header, uint32_t* __restrict__ packed,
           float* __restrict__ scale, int dtype) {
  const int i = blockIdx.x;
  const int l = base + i;
  if (l >= nlines) return;
  const float2* row = buf + (size_t)i * n;
  if (out) {
    float2* o = out + (size_t)l * out_stride;
    for (int k = threadIdx.x; k < kHdr + nvalid; k += kStoreBlock)
      o[k] = k >= kHdr ? row[k - kHdr]
                       : (zero_header ? make_float2(0.f, 0.f) : raw[(size_t)l * stride + k]);
  }
  if (packed) {
    __shared__ float part[kStoreBlock / 64];
    float m = 0.f;
    for (int k = threadIdx.x; k < nvalid; k += kStoreBlock) {
      const float2 v = row[k];
      m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    float mx = part[0];
    for (int w = 1; w < kStoreBlock / 64; ++w) mx = fmaxf(mx, part[w]);
    const float sc = pulse_scale(mx, dtype);
    const float inv = pulse_inv(sc);
    if (threadIdx.x == 0) scale[l] = sc;
    uint32_t* po = packed + (size_t)l * (kHdr + nvalid);
    for (int k = threadIdx.x; k < kHdr + nvalid; k += kStoreBlock) {
      uint32_t w = 0u;
      if (k >= kHdr) {
        const float2 v = row[k - kHdr];
        w = pack_word(v.x * inv, v.y * inv, dtype);
      }
      po[k] = w;
    }
  }
}

// ------------------------------------------------- fused overlap-save

// The twiddle tables of the 8192-point transform.
__global__ void k_os_twiddles(float2* __restrict__ tw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < os_table_values(kOsN)) tw[i] = os_table_entry(kOsN, i);
}

// Forward transform of one 8192-point vector (the reference function's
// spectrum), one workgroup, in place: natural order in, digit-reversed order
// out, position 16 t + m (bin drev(16 t + m)) at [m kOsThreads + t], as the
// threads of k_rc_os (os_mid_thread) multiply their own outputs with it.
__global__ void __launch_bounds__(kOsThreads) k_os_spectrum(float2* __restrict__ v,
                                                             const float2* __restrict__ tw) {
  __shared__ float2 lds[kOsLds];
  __shared__ float2 twl[os_lds_values(kOsN)];
  const OsTwiddle w = os_twiddles_lds<kOsN>(twl, tw);
  const int t = threadIdx.x;
  float2 x[16];
  for (int m = 0; m < 16; ++m) x[m] = v[t + m * kOsThreads];
  __syncthreads();   // the twiddle tables; every read of v is done
  os_dif_regs(lds, t, w, x, [] {});
  for (int m = 0; m < 16; ++m) v[m * kOsThreads + os_mid_thread(t)] = x[m];
}

// Block b of line l: outputs k0 + k, k < M = 8192 - npts + 1, k0 = b M, of
// the linear correlation y[k] = sum_m echo[k + m] conj(ref[m]) (the
// reference's circular correlation without wrap, scale of its 32768-point
// inverse via the gain of the reference function): echo samples [k0, k0 +
// 8192) (zero past nsamps), forward FFT (DIF), times conj(REF) as conj(X)
// REF position by position (both in the DIF output order), forward FFT again
// (DIT, natural order out), conjugate.  Writes the cf32 row (block 0 also the
// header samples) and, when lmax is given, the largest |component| of the
// block's outputs into lmax[l] (FP32 bits; max as fmaxf takes it, so NaN is
// passed over as the pack kernel does).
// Two workgroups per CU (LDS 2 x 71 KB): 4 waves per SIMD.  Vector issue is 79 %
// busy (1535 instructions a wave) and LDS 51 % (105, no bank conflicts): an IW
// burst's 1500 lines in 0.21 ms (0.22 with 1950 vector instructions, 93 % busy, before
// the twiddles went into the butterflies).
__global__ void __launch_bounds__(kOsThreads)
__attribute__((amdgpu_waves_per_eu(4)))
k_rc_os(const float2* __restrict__ raw, int nlines, int stride, int nsamps, int npts, int nvalid,
        const float2* __restrict__ spec, const float2* __restrict__ tw,
        float2* __restrict__ out, int out_stride, int zero_header, unsigned* __restrict__ lmax) {
  __shared__ float2 lds[kOsLds];
  __shared__ float2 twl[os_lds_values(kOsN)];
  // Work item q = (line, block), line-major, dealt so that XCD x (blocks x,
  // x + 8, ...) takes the x-th eighth of the items in order: the blocks of a
  // line, whose echo windows overlap by npts - 1 samples, share one L2.
  const int nblk = (nvalid + kOsN - npts) / (kOsN - npts + 1);
  const int per = (int)(gridDim.x >> 3);
  const int q = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (q >= nblk * nlines) return;
  const int l = q / nblk;
  const int b = q - l * nblk;
  const int M = kOsN - npts + 1;
  const int k0 = b * M;
  const OsTwiddle w = os_twiddles_lds<kOsN>(twl, tw);
  const float2* echo = raw + (size_t)l * stride + kHdr;
  // thread t holds values t + kOsThreads m, m < 16, of the block (natural
  // order), between the transforms positions 16 t2 + m (digit-reversed order)
  const int t = threadIdx.x;
  float2 v[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const int n = t + m * kOsThreads;
    v[m] = k0 + n < nsamps ? echo[k0 + n] : make_float2(0.f, 0.f);
  }
  __syncthreads();   // the twiddle tables
  float2 sp[16];
  const int t2 = os_mid_thread(t);
  os_dif_regs(lds, t, w, v, [&] {
#pragma unroll
    for (int m = 0; m < 16; ++m) sp[m] = spec[m * kOsThreads + t2];
  });
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = c_mul(make_float2(v[m].x, -v[m].y), sp[m]);
  os_dit_regs(lds, t, w, v);
  const int kend = min(M, nvalid - k0);
  float mx = 0.f;
  float2* o = out ? out + (size_t)l * out_stride : nullptr;
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const int k = threadIdx.x + m * kOsThreads;
    if (k >= kend) break;
    const float2 y = make_float2(v[m].x, -v[m].y);
    if (o) o[kHdr + k0 + k] = y;
    mx = fmaxf(mx, fmaxf(fabsf(y.x), fabsf(y.y)));
  }
  if (o && b == 0 && threadIdx.x < kHdr)
    o[threadIdx.x] = zero_header ? make_float2(0.f, 0.f) : raw[(size_t)l * stride + threadIdx.x];
  if (lmax) {
    for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(lmax + l, __float_as_uint(mx));
  }
}

// The packed words of cf32 rows y (kHdr + nvalid samples per row, stride
// y_stride), one workgroup per line: header words zero, then the samples from
// the line's own scale own[l] to scale[l] (pack_row).  1500 x 21018 samples in
// 64 us (5.9 TB/s); 64 small workgroups a line, 8 bytes a lane and load, took
// 105 us.
template <int DT>
__global__ void __launch_bounds__(kPackBlock)
k_os_pack_rows(const float2* __restrict__ y, int y_stride, int nvalid,
               uint32_t* __restrict__ packed, const float* __restrict__ own,
               const float* __restrict__ scale) {
  const int l = blockIdx.x;
  const float so = own[l], sf = scale[l];
  const bool rescale = so > 0.f && so != sf;
  uint32_t* o = packed + (size_t)l * (kHdr + nvalid);
  if (threadIdx.x < kHdr) o[threadIdx.x] = 0u;
  pack_row<DT>(y + (size_t)l * y_stride + kHdr, nvalid, o + kHdr, pulse_inv(so), rescale,
               rescale ? so / sf : 1.f);
}

// Per line: its own scale (the pack kernel's, from the largest |component|)
// and the scale k_unify_scales leaves it (the call's largest M when the own
// scale is 0 or within its range of M; 1 for every line when M = 0).  One
// workgroup; resets lmax for the next call.
constexpr int kScaleBlock = 1024;
__global__ void __launch_bounds__(kScaleBlock)
k_os_scales(unsigned* __restrict__ lmax, int L, int dtype, float* __restrict__ own,
            float* __restrict__ scale) {
  __shared__ float part[kScaleBlock / 64];
  float m = 0.f;
  for (int l = threadIdx.x; l < L; l += kScaleBlock) {
    const float s = pulse_scale(__uint_as_float(lmax[l]), dtype);
    own[l] = s;
    lmax[l] = 0u;
    m = fmaxf(m, s);
  }
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  float M = part[0];
  for (int w = 1; w < kScaleBlock / 64; ++w) M = fmaxf(M, part[w]);
  for (int l = threadIdx.x; l < L; l += kScaleBlock)
    scale[l] = unified_scale(own[l], M, dtype);
}

__global__ void k_zero_words(unsigned* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// ------------------------------------------------------------ state

// Per (device, stream): the transform buffer of one batch of lines and the
// reference spectrum of the last chirp seen.  Calls on different streams
// have their own, so two bursts can be range-compressed concurrently (e.g.
// one burst's compression overlapping the previous burst's backprojection).
struct RcState {
  int dev = -1;
  hipStream_t stream = nullptr;
  float2* buf = nullptr;   // [kChunk][n], n <= kFftLen
  float2* ref = nullptr;   // [n] reference spectrum for ref_of at length ref_n
  int ref_n = 0;
  tdbp_chirp ref_of;
  bool ref_valid = false;
  // fused overlap-save: twiddles, the reference spectrum at 8192 points for
  // os_of (in the DIF output order), and the per-line figures of the packed
  // output (grow-only)
  float2* tw = nullptr;
  float2* os_ref = nullptr;
  tdbp_chirp os_of;
  bool os_valid = false;
  unsigned* lmax = nullptr;   // [lines_cap] largest |component| per line
  float* own = nullptr;       // [lines_cap] each line's own scale
  int lines_cap = 0;
  float2* rows = nullptr;     // cf32 rows of a packed-only call
  size_t rows_cap = 0;        // values
};

std::mutex g_rc_mu;
std::vector<RcState*> g_rc;

int state_for(int dev, hipStream_t stream, RcState** out) {
  for (RcState* r : g_rc)
    if (r->dev == dev && r->stream == stream) {
      *out = r;
      return TDBP_OK;
    }
  RcState* r = new RcState;
  r->dev = dev;
  r->stream = stream;
  if (hipMalloc((void**)&r->ref, sizeof(float2) * (size_t)kFftLen) != hipSuccess) {
    delete r;
    return set_error(TDBP_ERR_NOMEM, "range compression buffers");
  }
  if (hipMalloc((void**)&r->buf, sizeof(float2) * (size_t)kChunk * kFftLen) != hipSuccess) {
    (void)hipFree(r->ref);
    delete r;
    return set_error(TDBP_ERR_NOMEM, "range compression buffers");
  }
  g_rc.push_back(r);
  *out = r;
  return TDBP_OK;
}

bool same_chirp(const tdbp_chirp& a, const tdbp_chirp& b) {
  return std::memcmp(&a, &b, sizeof a) == 0;
}

// Transform length: the smallest 2^a 3^b 5^c >= nsamps.  The kept samples
// k < nvalid = nsamps - npts are sums over echo samples k .. k + npts - 1 <
// nsamps only, so any length >= nsamps gives the reference's 32768-point
// values; a shorter one moves fewer bytes (24576 for a 24400-sample window).
int transform_length(int nsamps) {
  for (int n = nsamps; n < kFftLen; ++n) {
    int m = n;
    for (int p : {2, 3, 5})
      while (m % p == 0) m /= p;
    if (m == 1) return n;
  }
  return kFftLen;
}

// The fused overlap-save path of tdbp_range_compress (npts <= kOsN / 2).
// cf32 only: one launch.  Packed: the first launch writes the cf32 rows (if
// asked) and the per-line maxima, k_os_scales turns them into the scales
// tdbp_pack_samples would give, and a second launch packs the rows to its
// words.
int compress_overlap_save(RcState* r, const float2* raw, int nlines, int stride,
                          const tdbp_chirp& c, float2* out, int out_stride, int flags,
                          void* packed, float* scale, int dtype, hipStream_t s) {
  int st;
  if (!r->os_ref && hipMalloc((void**)&r->os_ref, sizeof(float2) * kOsN) != hipSuccess) {
    r->os_ref = nullptr;
    return set_error(TDBP_ERR_NOMEM, "range compression: reference spectrum");
  }
  if (!r->tw) {
    float2* tw = nullptr;
    if (hipMalloc((void**)&tw, sizeof(float2) * os_table_values(kOsN)) != hipSuccess)
      return set_error(TDBP_ERR_NOMEM, "range compression: twiddles");
    hipLaunchKernelGGL(k_os_twiddles, dim3((os_table_values(kOsN) + 255) / 256), dim3(256), 0, s,
                       tw);
    if ((st = hip_check(hipGetLastError(), "twiddle launch"))) {
      (void)hipFree(tw);
      return st;
    }
    r->tw = tw;
  }
  if (!r->os_valid || !same_chirp(r->os_of, c)) {
    r->os_valid = false;   // until the new one's launches are in
    hipLaunchKernelGGL(k_chirp, dim3(kOsN / 256), dim3(256), 0, s, r->os_ref, kOsN, c.npts,
                       c.samplefreq, c.startfreq, c.ramprate, (float)((double)kFftLen / kOsN));
    if ((st = hip_check(hipGetLastError(), "chirp launch"))) return st;
    hipLaunchKernelGGL(k_os_spectrum, dim3(1), dim3(kOsThreads), 0, s, r->os_ref, r->tw);
    if ((st = hip_check(hipGetLastError(), "spectrum launch"))) return st;
    r->os_of = c;
    r->os_valid = true;
  }
  if (packed && nlines > r->lines_cap) {
    (void)hipFree(r->lmax);
    (void)hipFree(r->own);
    r->lmax = nullptr;
    r->own = nullptr;
    r->lines_cap = 0;
    if (hipMalloc((void**)&r->lmax, sizeof(unsigned) * nlines) != hipSuccess ||
        hipMalloc((void**)&r->own, sizeof(float) * nlines) != hipSuccess) {
      (void)hipFree(r->lmax);   // hipFree(nullptr) is a no-op
      r->lmax = nullptr;
      r->own = nullptr;
      return set_error(TDBP_ERR_NOMEM, "range compression: per-line scales");
    }
    r->lines_cap = nlines;
    hipLaunchKernelGGL(k_zero_words, dim3((nlines + 255) / 256), dim3(256), 0, s, r->lmax,
                       nlines);
    if ((st = hip_check(hipGetLastError(), "zero launch"))) return st;
  }
  // Packed output: the cf32 rows go to `out` when the caller asks for them
  // too, else to a grow-only scratch, and are packed from there (an
  // elementwise pass costs less than computing the transforms again).
  float2* rows = out;
  int rows_stride = out_stride;
  if (packed && !rows) {
    const size_t need = (size_t)nlines * (size_t)(kHdr + c.nvalid);
    if (need > r->rows_cap) {
      (void)hipFree(r->rows);
      r->rows_cap = 0;
      if (hipMalloc((void**)&r->rows, sizeof(float2) * need) != hipSuccess) {
        r->rows = nullptr;
        return set_error(TDBP_ERR_NOMEM, "range compression: cf32 rows for packing");
      }
      r->rows_cap = need;
    }
    rows = r->rows;
    rows_stride = kHdr + c.nvalid;
  }
  const int M = kOsN - c.npts + 1;
  const long items = (long)((c.nvalid + M - 1) / M) * nlines;
  if (items > (long)INT32_MAX - 8)
    return set_error(TDBP_ERR_ARG, "range compress: %d lines too many", nlines);
  const dim3 grid((unsigned)((items + 7) / 8 * 8));
  hipLaunchKernelGGL(k_rc_os, grid, dim3(kOsThreads), 0, s, raw, nlines, stride, c.nsamps, c.npts,
                     c.nvalid, r->os_ref, r->tw, rows, rows_stride,
                     (flags & TDBP_RC_ZERO_HEADER) ? 1 : 0, packed ? r->lmax : nullptr);
  if ((st = hip_check(hipGetLastError(), "overlap-save launch"))) return st;
  if (!packed) return TDBP_OK;
  hipLaunchKernelGGL(k_os_scales, dim3(1), dim3(kScaleBlock), 0, s, r->lmax, nlines, dtype,
                     r->own, scale);
  if ((st = hip_check(hipGetLastError(), "scale launch"))) return st;
  const auto k = dtype == TDBP_CF16   ? k_os_pack_rows<TDBP_CF16>
                 : dtype == TDBP_CI16 ? k_os_pack_rows<TDBP_CI16>
                                      : k_os_pack_rows<TDBP_CBF16>;
  hipLaunchKernelGGL(k, dim3((unsigned)nlines), dim3(kPackBlock), 0, s, rows, rows_stride,
                     c.nvalid, (uint32_t*)packed, r->own, scale);
  return hip_check(hipGetLastError(), "pack launch");
}

}  // namespace

extern "C" {

int tdbp_chirp_decode(const uint8_t* h, tdbp_chirp* c) {
  if (!h || !c) return set_error(TDBP_ERR_ARG, "chirp decode: null pointer");
  std::memset(c, 0, sizeof *c);
  c->rangedecimation = h[40];
  const double fs = sample_frequency(c->rangedecimation);
  if (fs == 0.0)
    return set_error(TDBP_ERR_ARG, "range decimation code %d has no sampling rate",
                     c->rangedecimation);
  c->samplefreq = (float)fs;
  const int w42 = be16(h + 42), w44 = be16(h + 44);
  const int sgn42 = (w42 & 32768) ? 1 : -1;   // (-1)**(1-ipolarity)
  const int sgn44 = (w44 & 32768) ? 1 : -1;
  c->ramprate = (float)((double)(sgn42 * (w42 & 32767)) * kFref * kFref / 2097152.0);
  c->startfreq = (float)((double)(c->ramprate / 4.f) / kFref +
                         (double)(sgn44 * (w44 & 32767)) * kFref / 16384.0);
  c->pulselength = (float)((double)be24(h + 46) / kFref);
  c->nsamps = be16(h + 65) * 2;
  const float np = c->pulselength * c->samplefreq;
  c->npts = (int)np;
  c->nvalid = c->nsamps - c->npts;
  return TDBP_OK;
}

int tdbp_range_compress(const void* d_raw, int nlines, int raw_stride, const tdbp_chirp* c,
                        void* d_out, int out_stride, int flags, void* d_packed,
                        float* d_scale, int dtype, void* stream) {
  if (!d_raw || !c || nlines < 1)
    return set_error(TDBP_ERR_ARG, "range compress: null input or no lines");
  if (c->nsamps < 1 || c->nsamps > kFftLen || c->nsamps > raw_stride - kHdr)
    return set_error(TDBP_ERR_ARG, "range compress: %d echo samples for lines of %d (FFT %d)",
                     c->nsamps, raw_stride, kFftLen);
  if (c->npts < 1 || c->npts > kFftLen || c->nvalid < 1)
    return set_error(TDBP_ERR_ARG, "range compress: chirp of %d samples, %d valid",
                     c->npts, c->nvalid);
  if (!d_out && !d_packed)
    return set_error(TDBP_ERR_ARG, "range compress: no output");
  if (d_out && out_stride < kHdr + c->nvalid)
    return set_error(TDBP_ERR_ARG, "range compress: output stride %d < %d", out_stride,
                     kHdr + c->nvalid);
  if (d_packed && (!d_scale || (dtype != TDBP_CF16 && dtype != TDBP_CBF16 && dtype != TDBP_CI16)))
    return set_error(TDBP_ERR_ARG,
                     "range compress: packed output needs CF16/CBF16/CI16 and scales");
  int st = current_device_ready();
  if (st) return st;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(g_rc_mu);
  RcState* r = nullptr;
  hipStream_t s = (hipStream_t)stream;
  if ((st = state_for(dev, s, &r))) return st;
  const char* er = std::getenv("TDBP_RC_ROCFFT");
  if (c->npts <= kOsN / 2 && !(er && er[0] == '1'))
    return compress_overlap_save(r, (const float2*)d_raw, nlines, raw_stride, *c,
                                 (float2*)d_out, out_stride, flags, d_packed, d_scale, dtype, s);
  const int n = transform_length(c->nsamps);
  const unsigned nb = (unsigned)((n + 255) / 256);
  if (!r->ref_valid || !same_chirp(r->ref_of, *c) || r->ref_n != n) {
    hipLaunchKernelGGL(k_chirp, dim3(nb), dim3(256), 0, s, r->ref, n, c->npts, c->samplefreq,
                       c->startfreq, c->ramprate, (float)((double)kFftLen / n));
    if ((st = hip_check(hipGetLastError(), "chirp launch")) ||
        (st = fft_run(n, 1, false, r->ref, s)))
      return st;
    r->ref_of = *c;
    r->ref_n = n;
    r->ref_valid = true;
  }
  const float2* raw = (const float2*)d_raw;
  for (int base = 0; base < nlines; base += kChunk) {
    hipLaunchKernelGGL(k_rc_load, dim3(nb, kChunk), dim3(256), 0, s, raw, nlines, raw_stride,
                       c->nsamps, base, n, r->buf);
    if ((st = hip_check(hipGetLastError(), "load launch")) ||
        (st = fft_run(n, kChunk, false, r->buf, s)))
      return st;
    hipLaunchKernelGGL(k_rc_mul, dim3(nb, kChunk), dim3(256), 0, s, r->buf, r->ref, n);
    if ((st = hip_check(hipGetLastError(), "product launch")) ||
        (st = fft_run(n, kChunk, true, r->buf, s)))
      return st;
    const int nchunk = nlines - base < kChunk ? nlines - base : kChunk;
    hipLaunchKernelGGL(k_rc_store, dim3(nchunk), dim3(kStoreBlock), 0, s, raw, nlines,
                       raw_stride, base, r->buf, n, c->nvalid, (float2*)d_out, out_stride,
                       (flags & TDBP_RC_ZERO_HEADER) ? 1 : 0, (uint32_t*)d_packed, d_scale,
                       dtype);
    if ((st = hip_check(hipGetLastError(), "store launch"))) return st;
  }
  if (d_packed)
    return hip_check(launch_unify_scales((uint32_t*)d_packed, (size_t)(kHdr + c->nvalid),
                                         nlines, d_scale, dtype, s),
                     "scale launch");
  return TDBP_OK;
}

}  // extern "C"
