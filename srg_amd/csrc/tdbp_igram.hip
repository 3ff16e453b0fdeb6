// tdbp_igram.hip -- interferogram formation on co-registered .geo images on
// the device: the programs int/crossmul.f90 and int/makecc.f90.
//
// crossmul (int/crossmul.f90:86-199), per output line of looksdn input rows:
//   * masks from the unscaled rows: per output column, the complex sum over
//     the looksdn rows and looksac columns; |sum| <= 1e-6 marks no data
//     (:110-122);
//   * each row times `scale`, zero-padded to nnn = the next power of two >= na,
//     forward FFT; the spectrum halves placed at both ends of a 2 nnn array;
//     inverse FFT; divided by nnn, then by 2: the row upsampled by two
//     (:127-148).  Computed here without the 2 nnn transform: with X the
//     spectrum of the scaled row x, the even samples of that result are x/2
//     exactly, and the odd ones the length-nnn inverse transform of X times
//     exp(j pi k/nnn) (k signed, the upper half of X at k - nnn, as the
//     placement puts it), divided by nnn and by 2;
//   * igram = up1 conj(up2), amp = (|up1|^2, |up2|^2) over the first 2 na
//     samples; adjacent pairs summed back to na columns; summed over the
//     looksdn rows, then over looksac columns; amp square-rooted per
//     component; masked outputs zero (:150-184).
// makecc (int/makecc.f90:46-60): amp = re(b) im(b), cc = |a| / amp (0 where
// amp <= 0), written as [amp row | cc row].
//
// For nnn = 1024 to 8192 (widths 513 ... 8192, the images of these bursts) one
// kernel does everything: a workgroup of two halves takes an output line, each
// half upsamples the rows of one image in LDS (the in-place pair
// of tdbp_osfft.h with the ramp between, in digit-reversed order), and products,
// looks and masks are formed there, with no upsampled rows in HBM
// (k_xmul_rows at looks 1 x 1, crossmul's default; k_xmul_looks).  Output
// lines too few for that to fill the chip take one workgroup per row instead
// (k_up_fused), and the cross product, looks and masks read the upsampled rows
// from HBM (k_xmul).  Other lengths (or TDBP_IGRAM_ROCFFT=1) upsample through
// rocFFT batches and take k_xmul too.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include <cstdlib>
#include <cstring>

#include "tdbp_api_internal.h"
#include "tdbp_fft.h"
#include "tdbp_internal.h"
#include "tdbp_osfft.h"

using namespace tdbp;

namespace {

constexpr int kRows = 512;   // rows per rocFFT batch (rounded down to whole looks)
constexpr int kMaxDev = 64;

__global__ void k_up_load(const float2* __restrict__ img, int na, int nrows, int row0,
                          int nvalid_rows, int nnn, float scale, float2* __restrict__ buf) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (j >= nnn) return;
  const int r = row0 + i;
  float2 v = make_float2(0.f, 0.f);
  if (i < nrows && r < nvalid_rows && j < na) {
    const float2 a = img[(size_t)r * na + j];
    v = make_float2(a.x * scale, a.y * scale);
  }
  buf[(size_t)i * nnn + j] = v;
}

// The half-sample delay of the spectrum: row i of buf times exp(j pi ks/nnn),
// ks = k for k < nnn/2, k - nnn above, into row i of odd.
__global__ void k_up_ramp(const float2* __restrict__ buf, int nnn, float2* __restrict__ odd) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (k >= nnn) return;
  const int ks = k < nnn / 2 ? k : k - nnn;
  float sn, cs;
  sincospif((float)ks / (float)nnn, &sn, &cs);   // ks/nnn is exact in float
  const float2 a = buf[(size_t)i * nnn + k];
  odd[(size_t)i * nnn + k] = make_float2(a.x * cs - a.y * sn, a.x * sn + a.y * cs);
}

// Transform lengths of the fused kernels and their tables, one after another on
// the device: per length N the twiddles (tdbp_osfft.h), then exp(j pi ks/N) as
// k_up_ramp computes it (bin b, ks = b, or b - N from N/2 on) for value m of
// thread t in the DIF output order, at [m N/16 + t].
constexpr int kUpMin = 1024, kUpMax = kOsN;
constexpr int up_table_values(int n) { return os_table_values(n) + n; }
constexpr int up_table_at(int n) {
  return n == kUpMin ? 0 : up_table_at(n / 2) + up_table_values(n / 2);
}
constexpr int kUpTables = up_table_at(kUpMax) + up_table_values(kUpMax);

// The tables of n points.
__global__ void k_up_tables(int n, float2* __restrict__ tab) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= up_table_values(n)) return;
  if (i < os_table_values(n)) {
    tab[i] = os_table_entry(n, i);
    return;
  }
  const int k = i - os_table_values(n), m = k / (n / 16), t = k - m * (n / 16);
  const int p = 16 * t + m, r = n / 256;
  const int b = n == kOsN
                    ? (p >> 9) + 16 * ((p >> 5) & 15) + 256 * ((p >> 1) & 15) + 4096 * (p & 1)
                    : p / (n / 16) + 16 * ((p / r) & 15) + 256 * (p & (r - 1));
  const int ks = b < n / 2 ? b : b - n;
  float s1, c1;
  sincospif((float)ks / (float)n, &s1, &c1);
  tab[i] = make_float2(c1, s1);
}

// The scaled, zero-padded image row r as N/16 threads (t their index among
// them) hold it for up_transform: u[m] = value t + (N/16) m.
template <int N>
__device__ __forceinline__ void up_load(const float2* __restrict__ img, int na, int r,
                                        float scale, int t, float2* u) {
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const int j = t + m * up_threads(N);
    u[m] = make_float2(0.f, 0.f);
    if (j < na) {
      const float2 a = img[(size_t)r * na + j];
      u[m] = make_float2(a.x * scale, a.y * scale);
    }
  }
}

// The row of up_load upsampled by its N/16 threads (every thread of the
// workgroup makes the same call): forward N-point DIF, times the ramp in
// the DIF output order, the unnormalised inverse as conj(DIT(conj(.))): u[k]
// becomes odd sample t + (N/16) k times nnn times 2 (what k_up_load + forward
// FFT + k_up_ramp + inverse FFT leave).  `ramp` is the length's own table.
// Starts with a barrier, so a second call may reuse lds at once.
template <int N>
__device__ __forceinline__ void up_transform(const OsTwiddle& w, const float2* __restrict__ ramp,
                                             float2* lds, int t, float2* u) {
  __syncthreads();   // the twiddle tables; the previous row's last LDS reads
  float2 c[16], T[8];
  const int t2 = N == kOsN ? os_mid_thread(t) : t;   // holds positions 16 t2 + m between
  const auto ramps = [&] {
#pragma unroll
    for (int m = 0; m < 16; ++m) c[m] = ramp[m * up_threads(N) + t2];
  };
  if constexpr (N == kOsN) {
    os_dif_regs(lds, t, w, u, ramps);
  } else {
    up_dif_first<N>(lds, t, u);
    os_tw_last1<N>(w, t, T);   // a stage ahead, as in os_dif_regs
    __syncthreads();
    up_mid<N, false>(lds, t, w, u);
    ramps();
    wave_sync();   // as in os_dif_regs: R threads' values
    up_dif_last<N>(lds, t, T, u);
  }
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const float2 a = u[m];
    u[m] = make_float2(a.x * c[m].x - a.y * c[m].y, -(a.x * c[m].y + a.y * c[m].x));   // conj(a c)
  }
  if constexpr (N == kOsN) {
    os_dit_regs(lds, t, w, u);
  } else {
    up_dit_first<N>(lds, t, u);
    os_tw_last2<N>(w, t, T);
    wave_sync();
    up_mid<N, true>(lds, t, w, u);
    __syncthreads();
    up_dit_last<N>(lds, t, T, u);
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) u[k].y = -u[k].y;
}

// Row i of the batch (image row row0 + i) upsampled in one workgroup, into row
// i of `up`.
template <int N>
__global__ void __launch_bounds__(up_threads(N)) __attribute__((amdgpu_waves_per_eu(4)))
k_up_fused(const float2* __restrict__ img, int na, int row0, float scale,
           const float2* __restrict__ tab, float2* __restrict__ up) {
  __shared__ float2 lds[up_lds(N)];
  __shared__ float2 twl[os_lds_values(N)];
  const OsTwiddle w = os_twiddles_lds<N>(twl, tab);
  const int t = threadIdx.x, i = blockIdx.x;
  float2 v[16];
  up_load<N>(img, na, row0 + i, scale, t, v);
  up_transform<N>(w, tab + os_table_values(N), lds, t, v);
#pragma unroll
  for (int k = 0; k < 16; ++k) up[(size_t)i * N + t + k * up_threads(N)] = v[k];
}

// Even and odd samples 2j, 2j+1 of a row upsampled by two: x_j scale / 2 and
// the odd transform divided by nnn and by 2.
__device__ __forceinline__ float2 up_odd(const float2* odd, size_t idx, float fn) {
  const float2 a = odd[idx];
  return make_float2((a.x / fn) / 2.0f, (a.y / fn) / 2.0f);
}

__global__ void k_xmul(const float2* __restrict__ up1, const float2* __restrict__ up2, int nnn,
                       const float2* __restrict__ img1, const float2* __restrict__ img2, int na,
                       float scale, int row0, int nout_lines_chunk, int out_line0, int looksac,
                       int looksdn, int mask, float2* __restrict__ igram,
                       float2* __restrict__ amp) {
  const int nw = na / looksac;
  const int oc = blockIdx.x * blockDim.x + threadIdx.x;
  const int ol = blockIdx.y;
  if (oc >= nw || ol >= nout_lines_chunk) return;
  const float fn = (float)nnn;
  float ig_r = 0.f, ig_i = 0.f, a1 = 0.f, a2 = 0.f;
  float m1r = 0.f, m1i = 0.f, m2r = 0.f, m2i = 0.f;
  for (int k = 0; k < looksac; ++k) {
    const int j = oc * looksac + k;
    float cr = 0.f, ci = 0.f, c1 = 0.f, c2 = 0.f;      // sums over the rows
    float s1r = 0.f, s1i = 0.f, s2r = 0.f, s2i = 0.f;
    for (int r = 0; r < looksdn; ++r) {
      const int il = ol * looksdn + r;                   // row in the batch
      const size_t o = (size_t)(row0 + il) * na + j;
      const float2 x1 = img1[o], x2 = img2[o];
      const float2 ua = make_float2(x1.x * scale * 0.5f, x1.y * scale * 0.5f);
      const float2 va = make_float2(x2.x * scale * 0.5f, x2.y * scale * 0.5f);
      const size_t b = (size_t)il * nnn + j;
      const float2 ub = up_odd(up1, b, fn), vb = up_odd(up2, b, fn);
      const float pr = (ua.x * va.x + ua.y * va.y) + (ub.x * vb.x + ub.y * vb.y);
      const float pi = (ua.y * va.x - ua.x * va.y) + (ub.y * vb.x - ub.x * vb.y);
      cr += pr;
      ci += pi;
      c1 += fmaf(ua.x, ua.x, ua.y * ua.y) + fmaf(ub.x, ub.x, ub.y * ub.y);   // |up1|^2
      c2 += fmaf(va.x, va.x, va.y * va.y) + fmaf(vb.x, vb.x, vb.y * vb.y);   // |up2|^2
      if (mask) {
        s1r += x1.x;
        s1i += x1.y;
        s2r += x2.x;
        s2i += x2.y;
      }
    }
    ig_r += cr;
    ig_i += ci;
    a1 += c1;
    a2 += c2;
    m1r += s1r;
    m1i += s1i;
    m2r += s2r;
    m2i += s2i;
  }
  float2 g = make_float2(ig_r, ig_i);
  float2 a = make_float2(sqrtf(a1), sqrtf(a2));
  if (mask && (hypotf(m1r, m1i) <= 1.e-6f || hypotf(m2r, m2i) <= 1.e-6f)) {
    g = make_float2(0.f, 0.f);
    a = make_float2(0.f, 0.f);
  }
  const size_t o = (size_t)(out_line0 + ol) * nw + oc;
  igram[o] = g;
  amp[o] = a;
}

// Looks 1 x 1 (crossmul's default) for nnn = N, one workgroup of two
// halves per image row r: half h reads the row of image h + 1 once and
// upsamples it (up_transform, in its own LDS area); each thread keeps the
// values and odd samples of the columns it takes and hands the other half's
// over through LDS; then per column the sum over the sample pair of
// up1 conj(up2), the amplitudes and the mask, as k_xmul computes them for one
// row and one column -- each image read once, no upsampled batch in HBM.  Vector
// issue and LDS (the transforms' butterflies and exchanges) bound it, close above
// HBM: 13500 x 4000 0.47 ms, 3.7 TB/s (0.52 ms with twiddle products apart from
// the butterflies and a barrier between all stages); 3000 x 1800 55 us and 3000 x
// 4400 235 us (366 and 840 us through rocFFT).
template <int N>
__global__ void __launch_bounds__(2 * up_threads(N)) __attribute__((amdgpu_waves_per_eu(4)))
k_xmul_rows(const float2* __restrict__ img1, const float2* __restrict__ img2, int na,
            float scale, int mask, const float2* __restrict__ tab, float2* __restrict__ igram,
            float2* __restrict__ amp) {
  constexpr int kT = up_threads(N);
  __shared__ float2 lds[2][up_lds(N)];
  __shared__ float2 twl[os_lds_values(N)];
  const OsTwiddle w = os_twiddles_lds<N>(twl, tab);
  const int T = threadIdx.x, h = T / kT, t = T % kT;   // h wave-uniform
  const int r = blockIdx.x;
  const float2* img = h ? img2 : img1;
  float2 x[16], u[16];   // the row as read; scaled, then upsampled
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const int j = t + m * kT;
    x[m] = j < na ? img[(size_t)r * na + j] : make_float2(0.f, 0.f);
    u[m] = make_float2(x[m].x * scale, x[m].y * scale);
  }
  up_transform<N>(w, tab + os_table_values(N), lds[h], t, u);
  // Thread (h, t) takes columns j = t + kT m, m = 2 k + h (j = T + 2 kT k),
  // where it holds its own image's value and odd sample; it hands the other
  // half's columns (m = 2 k + 1 - h) over through LDS.
  __syncthreads();   // up_transform's last LDS reads
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    lds[h][2 * kT * k + t] = h ? u[2 * k] : u[2 * k + 1];
    lds[h][2 * kT * k + kT + t] = h ? x[2 * k] : x[2 * k + 1];
  }
  __syncthreads();
  const float fn = (float)N;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int j = T + k * 2 * kT;
    if (j >= na) continue;
    const size_t o = (size_t)r * na + j;
    const float2 uo = h ? u[2 * k + 1] : u[2 * k], xo = h ? x[2 * k + 1] : x[2 * k];
    const float2 up = lds[1 - h][2 * kT * k + t], xp = lds[1 - h][2 * kT * k + kT + t];
    const float2 x1 = h ? xp : xo, x2 = h ? xo : xp;
    const float2 o1 = h ? up : uo, o2 = h ? uo : up;
    const float2 ua = make_float2(x1.x * scale * 0.5f, x1.y * scale * 0.5f);
    const float2 va = make_float2(x2.x * scale * 0.5f, x2.y * scale * 0.5f);
    const float2 ub = make_float2((o1.x / fn) / 2.0f, (o1.y / fn) / 2.0f);
    const float2 vb = make_float2((o2.x / fn) / 2.0f, (o2.y / fn) / 2.0f);
    const float pr = (ua.x * va.x + ua.y * va.y) + (ub.x * vb.x + ub.y * vb.y);
    const float pi = (ua.y * va.x - ua.x * va.y) + (ub.y * vb.x - ub.x * vb.y);
    const float c1 = fmaf(ua.x, ua.x, ua.y * ua.y) + fmaf(ub.x, ub.x, ub.y * ub.y);
    const float c2 = fmaf(va.x, va.x, va.y * va.y) + fmaf(vb.x, vb.x, vb.y * vb.y);
    float2 g = make_float2(pr, pi);
    float2 a = make_float2(sqrtf(c1), sqrtf(c2));
    if (mask && (hypotf(x1.x, x1.y) <= 1.e-6f || hypotf(x2.x, x2.y) <= 1.e-6f)) {
      g = make_float2(0.f, 0.f);
      a = make_float2(0.f, 0.f);
    }
    igram[o] = g;
    amp[o] = a;
  }
}

// Any other looks, nnn = N: one workgroup of two halves per output line.  Row
// after row of the line's looksdn rows, half h upsamples the row of image h +
// 1, the halves hand each other half of their odd samples through LDS, and
// thread (h, t) adds the products of the odd samples of its columns t + kT m,
// m = 2 k + h, to sums in registers (up1 conj(up2), |up1|^2, |up2|^2).  The
// sums then lie in LDS by column, and thread after thread takes an output
// column: its looksac sums, and the even samples and the mask from the image
// rows themselves (read for the second time, mostly from the caches).  The
// transforms bound it as they do k_xmul_rows: 5403 x 1789 at 4 x 2 0.105 ms, where
// rocFFT batches of 512 rows, five launches and four passes over HBM each, took
// 0.69 ms; 11000 x 4000 at 4 x 2 0.46 ms against 1.27 ms with the upsampled rows
// in HBM.
template <int N>
__global__ void __launch_bounds__(2 * up_threads(N)) __attribute__((amdgpu_waves_per_eu(4)))
k_xmul_looks(const float2* __restrict__ img1, const float2* __restrict__ img2, int na,
             float scale, int looksac, int looksdn, int mask, const float2* __restrict__ tab, float2* __restrict__ igram,
             float2* __restrict__ amp) {
  constexpr int kT = up_threads(N);
  __shared__ __align__(16) float2 lds[2][up_lds(N)];
  __shared__ float2 twl[os_lds_values(N)];
  static_assert(sizeof lds >= sizeof(float4) * N, "the columns' sums fit the transforms' LDS");
  const OsTwiddle w = os_twiddles_lds<N>(twl, tab);
  const int T = threadIdx.x, h = T / kT;   // h wave-uniform
  const int row0 = blockIdx.x * looksdn;
  const float2* img = h ? img2 : img1;
  const float fn = (float)N;
  float4 s[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) s[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int r = 0; r < looksdn; ++r) {
    // Made anew for each row: twiddles, ramps and addresses kept from row to
    // row would take 70 to 110 more registers than there are.
    const int t = os_fresh(T % kT);
    float2 u[16];
    up_load<N>(img, na, row0 + r, scale, t, u);
    up_transform<N>(w, tab + os_table_values(N), lds[h], t, u);
    __syncthreads();   // up_transform's last LDS reads
#pragma unroll
    for (int k = 0; k < 8; ++k) lds[h][kT * k + t] = h ? u[2 * k] : u[2 * k + 1];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float2 uo = h ? u[2 * k + 1] : u[2 * k], up = lds[1 - h][kT * k + t];
      const float2 o1 = h ? up : uo, o2 = h ? uo : up;
      const float2 a = make_float2((o1.x / fn) / 2.0f, (o1.y / fn) / 2.0f);
      const float2 b = make_float2((o2.x / fn) / 2.0f, (o2.y / fn) / 2.0f);
      s[k].x += a.x * b.x + a.y * b.y;
      s[k].y += a.y * b.x - a.x * b.y;
      s[k].z += fmaf(a.x, a.x, a.y * a.y);
      s[k].w += fmaf(b.x, b.x, b.y * b.y);
    }
  }
  __syncthreads();
  float4* cols = (float4*)&lds[0][0];
#pragma unroll
  for (int k = 0; k < 8; ++k) cols[T + 2 * kT * k] = s[k];
  __syncthreads();
  const int nw = na / looksac;
  const float2* p1 = img1 + (size_t)row0 * na;
  const float2* p2 = img2 + (size_t)row0 * na;
  for (int oc = T; oc < nw; oc += 2 * kT) {
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    float2 m1 = make_float2(0.f, 0.f), m2 = m1;
    for (int k = 0; k < looksac; ++k) {
      const int j = oc * looksac + k;
      float4 c = cols[j];
      float2 s1 = make_float2(0.f, 0.f), s2 = s1;   // the mask's sums, down the rows first
      for (int r = 0; r < looksdn; ++r) {
        const float2 x1 = p1[(size_t)r * na + j], x2 = p2[(size_t)r * na + j];
        const float2 a = make_float2(x1.x * scale * 0.5f, x1.y * scale * 0.5f);
        const float2 b = make_float2(x2.x * scale * 0.5f, x2.y * scale * 0.5f);
        c.x += a.x * b.x + a.y * b.y;
        c.y += a.y * b.x - a.x * b.y;
        c.z += fmaf(a.x, a.x, a.y * a.y);
        c.w += fmaf(b.x, b.x, b.y * b.y);
        s1.x += x1.x;
        s1.y += x1.y;
        s2.x += x2.x;
        s2.y += x2.y;
      }
      q.x += c.x;
      q.y += c.y;
      q.z += c.z;
      q.w += c.w;
      m1.x += s1.x;
      m1.y += s1.y;
      m2.x += s2.x;
      m2.y += s2.y;
    }
    float2 g = make_float2(q.x, q.y);
    float2 a = make_float2(sqrtf(q.z), sqrtf(q.w));
    if (mask && (hypotf(m1.x, m1.y) <= 1.e-6f || hypotf(m2.x, m2.y) <= 1.e-6f)) {
      g = make_float2(0.f, 0.f);
      a = make_float2(0.f, 0.f);
    }
    const size_t o = (size_t)blockIdx.x * nw + oc;
    igram[o] = g;
    amp[o] = a;
  }
}

// The fused kernels of a length.
struct FusedKernels {
  decltype(&k_up_fused<kUpMin>) up;
  decltype(&k_xmul_rows<kUpMin>) rows;
  decltype(&k_xmul_looks<kUpMin>) looks;
};
template <int N>
constexpr FusedKernels fused_kernels() {
  return {k_up_fused<N>, k_xmul_rows<N>, k_xmul_looks<N>};
}
FusedKernels fused_kernels(size_t nnn) {
  return nnn == 1024   ? fused_kernels<1024>()
         : nnn == 2048 ? fused_kernels<2048>()
         : nnn == 4096 ? fused_kernels<4096>()
                       : fused_kernels<8192>();
}

__global__ void k_makecc(const float2* __restrict__ ig, const float2* __restrict__ am, int npix,
                         int nlines, float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (i >= npix || l >= nlines) return;
  const float2 a = ig[(size_t)l * npix + i], b = am[(size_t)l * npix + i];
  const float amp = b.x * b.y;
  const float cc = amp > 0.f ? hypotf(a.x, a.y) / amp : 0.f;
  out[(size_t)l * 2 * npix + i] = amp;
  out[(size_t)l * 2 * npix + npix + i] = cc;
}

// Per device: the transform buffers of one batch, grown as calls need them; a
// call uses its own length nnn (rows nnn apart).  Calls take turns with them:
// each waits on its stream for the end of the last one's, whichever stream that
// was on.  A call that is being captured can neither wait for nor record that:
// its graph keeps the buffers it was captured with (never freed then), and its
// replays are the caller's to keep apart from other calls.
struct IgState {
  size_t values = 0;       // values each up buffer holds
  size_t buf_values = 0;
  float2* buf = nullptr;   // [kRows][nnn] spectra of a rocFFT batch
  float2* up1 = nullptr;   // [rows][nnn] odd samples of image 1
  float2* up2 = nullptr;
  hipEvent_t used = nullptr;  // the end of the last call that used them
  bool captured = false;      // some graph holds them
  float2* tables = nullptr;   // [kUpTables] of the fused kernels
};
std::mutex g_ig_mu;
IgState g_ig[kMaxDev];

int buffers(IgState& s, size_t values, size_t buf_values) {
  if (s.values >= values && s.buf_values >= buf_values) return TDBP_OK;
  (void)hipDeviceSynchronize();
  values = std::max(values, s.values);
  buf_values = std::max(buf_values, s.buf_values);
  for (float2* p : {s.buf, s.up1, s.up2})
    if (p && !s.captured) (void)hipFree(p);
  s.buf = s.up1 = s.up2 = nullptr;
  s.values = s.buf_values = 0;
  s.captured = false;
  if ((buf_values && hipMalloc((void**)&s.buf, sizeof(float2) * buf_values) != hipSuccess) ||
      hipMalloc((void**)&s.up1, sizeof(float2) * values) != hipSuccess ||
      hipMalloc((void**)&s.up2, sizeof(float2) * values) != hipSuccess)
    return set_error(TDBP_ERR_NOMEM, "interferogram buffers (2 x %zu values)", values);
  s.values = values;
  s.buf_values = buf_values;
  return TDBP_OK;
}

bool fused_length(size_t nnn) {
  const char* e = std::getenv("TDBP_IGRAM_ROCFFT");
  return nnn >= (size_t)kUpMin && nnn <= (size_t)kUpMax && !(e && std::strcmp(e, "1") == 0);
}

// The fused kernels' tables, made on first use on the device, on a stream of
// their own that the call waits for: calls on any stream may read them from
// then on, also where the first one's stream is being captured.
int tables(IgState& s) {
  if (s.tables) return TDBP_OK;
  float2* t = nullptr;
  hipStream_t st = nullptr;
  if (hipMalloc((void**)&t, sizeof(float2) * kUpTables) != hipSuccess)
    return set_error(TDBP_ERR_NOMEM, "interferogram tables");
  int e = hip_check(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "upsample tables");
  for (int n = kUpMin; n <= kUpMax && !e; n *= 2) {
    hipLaunchKernelGGL(k_up_tables, dim3((up_table_values(n) + 255) / 256), dim3(256), 0, st, n,
                       t + up_table_at(n));
    e = hip_check(hipGetLastError(), "upsample tables");
  }
  if (st) {
    const int e2 = hip_check(hipStreamSynchronize(st), "upsample tables");
    if (!e) e = e2;
    (void)hipStreamDestroy(st);
  }
  if (e) {
    (void)hipFree(t);
    return e;
  }
  s.tables = t;
  return TDBP_OK;
}

// Values of an upsampled image's batch in the fused kernels' two-pass form
// (64 MB a buffer); rows in it are whole output lines, 512 rows each at most.
constexpr size_t kFusedValues = (size_t)8 << 20;
static_assert(kFusedValues / kUpMax >= kRows, "an output line's rows fit a batch");

// Whether the looks are taken in one pass, one workgroup per output line
// (k_xmul_looks), or row by row first (k_up_fused, k_xmul).  The first takes
// looksdn row transforms one after another, 8.4, 10, 11.6 and 17 us each at
// 1024 to 8192 points while the lines fit the chip at once; the second takes
// about 15 us and 24 ps per value of the rows.  Below that crossing the one-pass
// kernel leaves the chip idle: 50 lines of 8 rows at 1024 points 67 us against
// 35, 125 lines of 8 rows at 2048 points 80 against 63; above it 375 lines of 8
// rows at 4096 points 198 against 383, 2701 lines of 2 rows at 2048 points 105
// against 306 (and 688 through rocFFT).
bool one_pass(int nout, int looksdn, size_t nnn) {
  const double row = 7.2 + 1.2 * (double)nnn / kUpMin;
  return 24e-6 * (double)nout * looksdn * (double)nnn + 15.0 >= looksdn * row;
}

// Rows [row0, row0 + rows) of an image through rocFFT.
int upsample_rocfft(const float2* img, int na, int rows, int row0, int nvalid_rows, size_t nnn,
                    float scale, IgState& s, float2* up, hipStream_t st) {
  hipLaunchKernelGGL(k_up_load, dim3((unsigned)((nnn + 255) / 256), kRows), dim3(256), 0, st,
                     img, na, rows, row0, nvalid_rows, (int)nnn, scale, s.buf);
  int e = hip_check(hipGetLastError(), "upsample load");
  if (!e) e = fft_run(nnn, kRows, false, s.buf, st);
  if (e) return e;
  hipLaunchKernelGGL(k_up_ramp, dim3((unsigned)((nnn + 255) / 256), kRows), dim3(256), 0, st,
                     s.buf, (int)nnn, up);
  e = hip_check(hipGetLastError(), "upsample ramp");
  if (!e) e = fft_run(nnn, kRows, true, up, st);
  return e;
}

// The two-pass form: batch after batch of output lines, rows upsampled into the
// state's buffers, then products and looks out of them.
int batches(IgState& s, const FusedKernels& k, const float2* tab, bool fused, size_t nnn,
            const float2* i1, const float2* i2, int na, int nout, int lines_per_batch,
            float scale, int looksac, int looksdn, int mask, float2* ig, float2* amp,
            hipStream_t str) {
  int st = TDBP_OK;
  for (int ol0 = 0; ol0 < nout; ol0 += lines_per_batch) {
    const int nol = nout - ol0 < lines_per_batch ? nout - ol0 : lines_per_batch;
    const int row0 = ol0 * looksdn;
    const int rows = nol * looksdn;
    // An image with itself is upsampled once.
    for (int i = 0; i < (i2 == i1 ? 1 : 2); ++i) {
      const float2* img = i ? i2 : i1;
      float2* up = i ? s.up2 : s.up1;
      if (fused) {
        hipLaunchKernelGGL(k.up, dim3((unsigned)rows), dim3((unsigned)(nnn / 16)), 0, str, img,
                           na, row0, scale, tab, up);
        st = hip_check(hipGetLastError(), "fused upsample");
      } else {
        st = upsample_rocfft(img, na, rows, row0, nout * looksdn, nnn, scale, s, up, str);
      }
      if (st) return st;
    }
    const int nw = na / looksac;
    hipLaunchKernelGGL(k_xmul, dim3((unsigned)((nw + 127) / 128), nol), dim3(128), 0, str,
                       s.up1, i2 == i1 ? s.up1 : s.up2, (int)nnn, i1, i2, na, scale, row0, nol,
                       ol0, looksac, looksdn, mask, ig, amp);
    if ((st = hip_check(hipGetLastError(), "crossmul launch"))) return st;
  }
  return TDBP_OK;
}

}  // namespace

extern "C" {

int tdbp_crossmul(const void* d_img1, const void* d_img2, int na, int nvalid, float scale,
                  int looksac, int looksdn, int mask, void* d_igram, void* d_amp,
                  void* stream) {
  if (!d_img1 || !d_img2 || !d_igram || !d_amp || na < 1 || nvalid < 1 || looksac < 1 ||
      looksdn < 1 || looksdn > kRows || na / looksac < 1 || nvalid / looksdn < 1)
    return set_error(TDBP_ERR_ARG, "crossmul: width %d, %d lines, looks %d x %d", na, nvalid,
                     looksac, looksdn);
  if (na > (1 << 24)) return set_error(TDBP_ERR_LIMIT, "crossmul: width %d", na);
  int st = current_device_ready();
  if (st) return st;
  size_t nnn = 2;
  while (nnn < (size_t)na) nnn <<= 1;   // crossmul.f90:72-76
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev < 0 || dev >= kMaxDev) return set_error(TDBP_ERR_ARG, "device %d", dev);
  std::lock_guard<std::mutex> lk(g_ig_mu);
  IgState& s = g_ig[dev];
  const bool fused = fused_length(nnn);
  hipStream_t str = (hipStream_t)stream;
  const float2* i1 = (const float2*)d_img1;
  const float2* i2 = (const float2*)d_img2;
  const int nout = nvalid / looksdn;             // output lines
  const int used_rows = nout * looksdn;
  FusedKernels k = {};
  const float2* tab = nullptr;
  if (fused) {
    if ((st = tables(s))) return st;
    k = fused_kernels(nnn);
    tab = s.tables + up_table_at((int)nnn);
    const dim3 grid((unsigned)nout), block((unsigned)(nnn / 8));
    if (looksac == 1 && looksdn == 1) {
      hipLaunchKernelGGL(k.rows, grid, block, 0, str, i1, i2, na, scale, mask ? 1 : 0, tab, (float2*)d_igram, (float2*)d_amp);
      return hip_check(hipGetLastError(), "crossmul launch");
    }
    if (one_pass(nout, looksdn, nnn)) {
      hipLaunchKernelGGL(k.looks, grid, block, 0, str, i1, i2, na, scale, looksac, looksdn,
                         mask ? 1 : 0, tab, (float2*)d_igram, (float2*)d_amp);
      return hip_check(hipGetLastError(), "crossmul launch");
    }
  }
  const int batch_rows =
      fused ? std::min((int)(kFusedValues / nnn), used_rows) : kRows;
  const int lines_per_batch = std::max(1, batch_rows / looksdn);   // output lines per batch
  if ((st = buffers(s, (size_t)std::max(batch_rows, looksdn) * nnn,
                    fused ? 0 : (size_t)kRows * nnn)))
    return st;
  const bool capturing = stream_captures(str);
  if (capturing) s.captured = true;
  else if (!s.used)
    st = hip_check(hipEventCreateWithFlags(&s.used, hipEventDisableTiming), "crossmul event");
  else
    st = hip_check(hipStreamWaitEvent(str, s.used, 0), "crossmul wait");
  if (st) return st;
  st = batches(s, k, tab, fused, nnn, i1, i2, na, nout, lines_per_batch, scale, looksac, looksdn,
               mask ? 1 : 0, (float2*)d_igram, (float2*)d_amp, str);
  // Also where a launch failed: the ones before it may be running.
  const int st2 = capturing ? TDBP_OK : hip_check(hipEventRecord(s.used, str), "crossmul event");
  return st ? st : st2;
}

int tdbp_makecc(const void* d_igram, const void* d_amp, int npix, int nlines, float* d_out,
                void* stream) {
  if (!d_igram || !d_amp || !d_out || npix < 1 || nlines < 1 || nlines > 65535)
    return set_error(TDBP_ERR_ARG, "makecc: %d x %d", npix, nlines);
  int st = current_device_ready();
  if (st) return st;
  hipLaunchKernelGGL(k_makecc, dim3((unsigned)((npix + 255) / 256), nlines), dim3(256), 0,
                     (hipStream_t)stream, (const float2*)d_igram, (const float2*)d_amp, npix,
                     nlines, d_out);
  return hip_check(hipGetLastError(), "makecc launch");
}

}  // extern "C"
