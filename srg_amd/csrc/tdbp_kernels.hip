// tdbp_kernels.hip -- gfx950 kernels of the TDBP engine.
//
// Hot path: one workgroup (4 waves of 64) owns a tile of output pixels of one
// burst.  Each lane owns one pixel: it computes the pixel's ECEF position from
// the int16 DEM and its pulse window from the line parabola (the reference's
// setxyz and setazoff, fused), then sums over its pulses.  Pulses are looped
// wave-uniformly, so per-pulse data are wave-uniform operands (scalar loads
// in the FP64 kernel, LDS broadcast reads in the mixed kernel) and only the
// range-sample gather is a per-lane memory access.
//
//  * k_plain : FP64 range, cycle-reduced FP64 phase, FP32 lerp, FP64
//              accumulator -- the drop-in and the accuracy reference.
//  * k_mixed : per workgroup, a FP64 reference point x0; per pulse (FP64,
//              once per workgroup) range R0, unit look vector u, and the
//              phase/range bases; per pixel-pulse only FP32:
//                 a  = u.d (d = x - x0),  R = R0 + a + (|d|^2 - a^2)/(2(R0+a))
//              with the linear phase split as K u_ref.d (per pixel, FP64
//              once) + K (u - u_ref).d (small, FP32), hardware sin/cos on
//              revolutions, stage-blocked FP32 sums joined by Kahan addition.
//
// Tile order is XCD-aware.  Single-burst launches of more than two rounds of
// resident workgroups are persistent: one workgroup per resident slot; the workgroups on XCD x (blockIdx % 8 = x,
// the hardware's round-robin) take the tiles of the column bands x, x + 8,
// ... (each band's row tiles in order) through counter x, then take what is
// left of the other XCDs' bands -- tiles in one column band share range
// samples, which stay in that XCD's L2, and the bands left at the end are
// shared out instead of holding one XCD busy.  The batch kernels do the same
// over (burst, band) queues; the MFMA kernel maps block b to tile
// x*q + min(x, r) + j (x = b % 8), a contiguous run per XCD.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tdbp_api_internal.h"
#include "tdbp_geom.h"
#include "tdbp_internal.h"
#include "tdbp_pack.h"

namespace tdbp {

const Variant kVariants[kNumVariants] = {
    {8, 0, 0, 0}, {4, 0, 0, 0}, {2, 0, 0, 0}, {1, 0, 0, 0}, {8, 1, 0, 0},
    {4, 1, 0, 0}, {2, 1, 0, 0}, {1, 1, 0, 0}, {4, 1, 1, 0},
    {4, 1, 0, 1}, {8, 1, 0, 1}, {4, kWavesSplit, 0, 0}};

typedef const double __attribute__((address_space(4)))* const_dptr;

// ------------------------------------------------------------------ helpers

__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, x = b & 7, j = b >> 3;
  return x * q + (x < r ? x : r) + j;
}

// kWavesSplit: the wave's quarter of a stage's pulses [p0, p1), cut out of [*qa,
// *qb).
__device__ __forceinline__ void split_stage(int p0, int p1, int* qa, int* qb) {
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int seg = (p1 - p0 + 3) >> 2;
  *qa = max(*qa, p0 + wave * seg);
  *qb = min(*qb, p0 + (wave + 1) * seg);
}
// The four waves' sums of a pixel, added in wave order (part: 512 values of LDS
// that the waves are done with); true on the wave that stores it.
template <class T>
__device__ __forceinline__ bool split_join(T* part, T* re, T* im) {
  const int tid = threadIdx.x;
  part[tid] = *re;
  part[kBlock + tid] = *im;
  __syncthreads();
  if (tid >= kWave) return false;
#pragma unroll
  for (int w = 1; w < kBlock / kWave; ++w) {
    *re += part[w * kWave + tid];
    *im += part[kBlock + w * kWave + tid];
  }
  return true;
}

// The persistent tile loop of a single-burst launch: queue x holds the row
// tiles of the column bands c = x, x + 8, ... in order (tile = c tiles_r +
// row); a workgroup drains the queue of its XCD, then the other seven in
// turn, and returns when all eight are exhausted (every workgroup does, so
// the grid drains).  F(tile) runs one tile; item is one LDS word.
template <class F>
__device__ __forceinline__ void persistent_tiles(const BurstDev& b, int* item, F&& f) {
  const int home = blockIdx.x & 7;
  const bool queue = b.counters != nullptr;   // else a workgroup per tile
  int qi = 0;
  while (qi < 8) {
    int it;
    if (queue) {
      const int qk = (home + qi) & 7;
      if (threadIdx.x == 0) {
        const int bands = qk < b.tiles_c ? ((b.tiles_c - 1 - qk) >> 3) + 1 : 0;
        const int k = atomicAdd(&b.counters[qk], 1);
        *item = k < bands * b.tiles_r ? (qk + 8 * (k / b.tiles_r)) * b.tiles_r + k % b.tiles_r
                                      : -1;
      }
      __syncthreads();
      it = *item;
      __syncthreads();
      if (it < 0) {
        ++qi;
        continue;
      }
    } else {
      it = xcd_tile(blockIdx.x, b.tiles_r * b.tiles_c);
      qi = 8;   // the only one
    }
    f(it);   // the one call: inlined twice the kernels ran 8-17 % slower
    __syncthreads();
  }
}

// A value known to be equal on every lane, moved to scalar registers.
__device__ __forceinline__ double uniform(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// Pixel owned by this thread in tile `tile` of burst b, with its window.
struct PixelCtx {
  int row, col;      // window line, DEM column
  bool inwin;        // inside the [nlines][W] output array
  bool computed;     // azoff > 0: the reference computes this pixel
  int azs, aze;      // pulse window, empty if not computed
};

// Pixels of a workgroup: wave tiles of TR x 64/TR, the four waves side by side,
// stacked along rows, or all on one wave tile with a quarter of the pulses
// each (STACK = kWavesSideBySide, kWavesStacked, kWavesSplit).
template <int TR, int STACK>
struct TileShape {
  static constexpr int TC = kWave / TR;
  static constexpr int WR = STACK == kWavesStacked ? 4 * TR : TR;
  static constexpr int WC = STACK == kWavesSideBySide ? 4 * TC : TC;
  static __device__ __forceinline__ int row(int tid) {
    return (STACK == kWavesStacked ? (tid >> 6) * TR : 0) + (tid & 63) / TC;
  }
  static __device__ __forceinline__ int col(int tid) {
    return (STACK == kWavesSideBySide ? (tid >> 6) * TC : 0) + (tid & 63) % TC;
  }
};

template <int TR, int STACK>
__device__ __forceinline__ PixelCtx pixel_of(const BurstDev& b, int tile) {
  using G = TileShape<TR, STACK>;
  const int band = tile / b.tiles_r;
  const int rt = tile - band * b.tiles_r;
  PixelCtx p;
  p.row = rt * G::WR + G::row(threadIdx.x);
  p.col = band * G::WC + G::col(threadIdx.x);
  p.inwin = p.row < b.nlines && p.col < b.W;
  p.azs = 0;
  p.aze = 0;
  p.computed = false;
  if (p.inwin && p.row < b.nfit && p.col >= b.firstpix && p.col <= b.lastpix) {
    const double* c = b.coef + 3 * p.row;
    const double az = pixel_azoff(c, p.col, b.firstpix, b.lastpix, b.A, b.L);
    if (az > 0.) {
      p.computed = true;
      pulse_window(az, b.A, b.L, &p.azs, &p.aze);
    }
  }
  return p;
}

__device__ __forceinline__ void pixel_ecef(const BurstDev& b, int row, int col,
                                           double* x) {
  const double h = b.dem[(size_t)row * b.W + col];
  dem_to_ecef(row, b.firstline, col, b.firstlat, b.deltalat, b.firstlon,
              b.deltalon, h, x);
}

// Reference GPU output: cf32(acc) * float(1/(azend-azstart))
// (sentinel/azimuth_compress.cu:78-79); the CPU twin stores cf32(acc)
// unscaled (sentinel/azimuth_compress_cpu.c:82).
__device__ __forceinline__ void store_out(const BurstDev& b, const PixelCtx& p,
                                          float re, float im) {
  if (!p.inwin) return;
  float2 o = make_float2(0.f, 0.f);
  if (p.computed) {
    if (b.cpu) {
      o = make_float2(re, im);
    } else {
      const float s = (float)(1. / (p.aze - p.azs));
      o = make_float2(re * s, im * s);
    }
  }
  b.out[(size_t)p.row * b.W + p.col] = o;
}

// ------------------------------------- FP64 pair (drop-in, accuracy reference)

// One pixel-pulse pair in FP64: range, gate, FP32 lerp of the two samples,
// phase exp(+j 4 pi R / lambda) reduced in cycles before sincospi.
// Global-address-space view of the sample rows: keeps the gather a
// global_load (scalar base + 32-bit lane offset) even when the row pointer
// comes from the burst table in memory.
typedef const char __attribute__((address_space(1)))* grow_t;
typedef uint32_t U32x2 __attribute__((ext_vector_type(2), aligned(4)));
typedef float F32x4 __attribute__((ext_vector_type(4), aligned(8)));
template <class T>
__device__ __forceinline__ T gload(grow_t p) {
  return *(const __attribute__((address_space(1))) T*)p;
}

// sqrt of a range squared (normal, ~1e12 m^2): the hardware reciprocal-root
// estimate refined by goldschmidt_sqrt.
__device__ __forceinline__ double range_sqrt(double x) {
  return goldschmidt_sqrt(x, __builtin_amdgcn_rsq(x));
}

__device__ __forceinline__ void plain_pair(const float2* __restrict__ row,
                                           const double* x, double sx,
                                           double sy, double sz,
                                           const BurstDev& b, double& ar,
                                           double& ai) {
  const double dx = x[0] - sx, dy = x[1] - sy, dz = x[2] - sz;
  const double R = range_sqrt(dx * dx + dy * dy + dz * dz);
  if (R >= b.rngstart && R <= b.rng_hi) {
    const double r = (R - b.rngstart) * b.inv_dmrg;
    const double fl = floor(r);
    int i = (int)fl;
    i = i > b.S - 2 ? b.S - 2 : i;
    const double fr = r - fl;
    const F32x4 v = gload<F32x4>((grow_t)row + (unsigned)i * 8u);   // samples i, i+1
    const float2 b0 = make_float2(v.x, v.y), b1 = make_float2(v.z, v.w);
    const float w0 = (float)(1.0 - fr), w1 = (float)fr;
    const float cr = b0.x * w0 + b1.x * w1;
    const float ci = b0.y * w0 + b1.y * w1;
    const double cyc = R * b.two_over_wvl;
    const double f = cyc - rint(cyc);
    double sn, cs;
    sincos_2pi(f, &sn, &cs);
    const double dr = cr, di = ci;
    ar = fma(dr, cs, ar);
    ar = fma(-di, sn, ar);
    ai = fma(dr, sn, ai);
    ai = fma(di, cs, ai);
  }
}

// The CPU twin's pair (sentinel/azimuth_compress_cpu.c:64-79): range index
// by division, lerp in FP64 rounded to cf32, phase 4*pi/wvl*range in FP64
// with full-range sin/cos, FP64 complex product; contraction off, so each
// step rounds as the reference's x86 build (no FMA) rounds it.
__device__ __forceinline__ void cpu_pair(const float2* __restrict__ row,
                                         const double* x, double sx, double sy,
                                         double sz, const BurstDev& b,
                                         double& ar, double& ai) {
#pragma clang fp contract(off)
  const double dx = x[0] - sx, dy = x[1] - sy, dz = x[2] - sz;
  const double R = sqrt(dx * dx + dy * dy + dz * dz);
  if (R >= b.rngstart && R <= b.rng_hi) {
    const double r = (R - b.rngstart) / b.dmrg;
    int i = (int)floor(r);
    const double fr = r - i;
    i = i > b.S - 2 ? b.S - 2 : i;
    const float2 b0 = row[i], b1 = row[i + 1];
    const double w0 = 1 - fr;
    const float cr = (float)((double)b0.x * w0 + (double)b1.x * fr);
    const float ci = (float)((double)b0.y * w0 + (double)b1.y * fr);
    const double ph = b.four_pi_over_wvl * R;
    const double pc = cos(ph), ps = sin(ph);
    const double tr = (double)cr * pc - (double)ci * ps;
    const double ti = (double)cr * ps + (double)ci * pc;
    ar = ar + tr;
    ai = ai + ti;
  }
}

// The CPU twin's tile: every pair by cpu_pair.
template <int TR, int STACK>
__device__ __forceinline__ void cpu_tile(const BurstDev& b, int tile) {
  PixelCtx p = pixel_of<TR, STACK>(b, tile);
  double x[3] = {0., 0., 0.};
  const bool live = p.aze > p.azs;
  if (live) pixel_ecef(b, p.row, p.col, x);
  const int lo = wave_min(live ? p.azs : 0x7fffffff);
  const int hi = wave_max(live ? p.aze : -1);
  double ar = 0., ai = 0.;
  const float2* base = (const float2*)b.data;
  const const_dptr sat = (const_dptr)b.satloc;
  const unsigned n = (unsigned)(p.aze - p.azs);
  for (int q = lo; q < hi; ++q) {
    const double sx = sat[3 * q], sy = sat[3 * q + 1], sz = sat[3 * q + 2];
    if ((unsigned)(q - p.azs) < n)
      cpu_pair(base + (size_t)q * b.S, x, sx, sy, sz, b, ar, ai);
  }
  store_out(b, p, (float)ar, (float)ai);
}

// ------------------------------------------------------- mixed precision

// Per-pulse record in LDS (3 x float4, written once per workgroup stage):
//   r0 = (du.x, du.y, du.z, c0)   du = u_p - u_ref, c0 = frac(2 R0/lambda)
//   r1 = (f0, i0*elem bits, 1/(2 R0), scale)  (R0 - rngstart)/dmrg = i0 + f0
//   r2 = (safe, lim, i0 bits, -)   lim: rho <= lim <=> r <= r_hi; safe != 0:
//        every pixel of the workgroup tile is inside the range gate (and, for
//        the quadratic form, its local index is at least 0)
//   r3 = (k, f0s, c0, scale)       k = q - pc, pc the central pulse of the tile
//        window; (R0 - rngstart)/dmrg = i0s + f0s with i0s fixed per stage
struct PulseRec {
  float4 r0, r1, r2, r3;
};

constexpr int kStage = kBlock;  // pulses per stage = one per thread

// Workgroup scratch of the mixed kernel besides the pulse records.
struct TileShared {
  double x0[3];      // reference point
  int key, wlo, whi;
  unsigned dmax;     // bits of max |x - x0| over live pixels (float, >= 0)
  unsigned pmax;     // bits of max |sd| of the quadratics over their windows
  int iamin, iamax;  // range of the lanes' whole-sample offsets ia (LDS staging)
  int nchain;        // live waves on the FP32 chain (LDS staging needs none)
};


// Structured-buffer view of a burst's samples (stride = one sample), so a
// gather addresses sample vindex at voffset + soffset bytes with no address
// arithmetic on the vector unit.  The base sits kSbufBias bytes below the
// samples so the per-pulse scalar offset stays non-negative.  The index is
// the local range index floor(rho) of the quadratic form, which the stage's
// safety test keeps in [1, 2047] (f0s in [pmx/dmrg + 1.5, 1024], |P/dmrg| <=
// pmx/dmrg + 1/2); num_records = kSbufIndexLimit makes the hardware return
// zeros for any index outside [0, 2048) instead of reading past it.
//
// CI16 samples are read with a format conversion: data format 16_16_16_16,
// number format SSCALED, so one load returns samples i and i + 1 as four
// exact FP32 values (re_i, im_i, re_i+1, im_i+1) and the vector unit spends
// no instruction on the int16 -> float conversion.
typedef int I32x4 __attribute__((ext_vector_type(4)));
typedef float SbufF2 __attribute__((ext_vector_type(2)));
typedef float SbufF4 __attribute__((ext_vector_type(4)));
__device__ SbufF2 sbuf_load_v2f32(I32x4 rsrc, int vindex, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.struct.buffer.load.v2f32");
__device__ SbufF4 sbuf_load_v4f32(I32x4 rsrc, int vindex, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.struct.buffer.load.v4f32");
__device__ SbufF4 sbuf_load_format_v4f32(I32x4 rsrc, int vindex, int voffset, int soffset,
                                         int aux)
    __asm("llvm.amdgcn.struct.buffer.load.format.v4f32");
constexpr long kSbufBias = 1l << 20;
constexpr int kSbufIndexLimit = 2048;
// Descriptor word 3: destination select X, Y, Z, W; number format; data format.
constexpr int kSbufWord3Raw32 = 4 << 15;                  // data format 32 (raw loads)
constexpr int kSbufWord3I16x4 = 4 | (5 << 3) | (6 << 6) | (7 << 9) |
                                (3 << 12) |               // SSCALED
                                (12 << 15);               // 16_16_16_16
constexpr int kSbufWord3F16x4 = 4 | (5 << 3) | (6 << 6) | (7 << 9) |
                                (7 << 12) |               // FLOAT
                                (12 << 15);               // 16_16_16_16

// FMT: the descriptor converts 16-bit components to FP32 (CF16: IEEE half,
// CI16: signed integer); else raw 32-bit loads (the gathers of the pair
// loops read CF16 words raw and convert them in the FMA).
template <int DT, bool FMT = (DT == TDBP_CI16)>
__device__ __forceinline__ I32x4 sample_rsrc(const void* data, int elem) {
  const unsigned long long a = (unsigned long long)data - (unsigned long long)kSbufBias;
  I32x4 r;
  r.x = __builtin_amdgcn_readfirstlane((int)(unsigned)a);
  r.y = __builtin_amdgcn_readfirstlane((int)(((unsigned)(a >> 32) & 0xffffu) |
                                             ((unsigned)elem << 16)));
  r.z = kSbufIndexLimit;
  r.w = (FMT && DT == TDBP_CI16)   ? kSbufWord3I16x4
        : (FMT && DT == TDBP_CF16) ? kSbufWord3F16x4
                                   : kSbufWord3Raw32;
  return r;
}

// CI16 word -> its two components as exact floats (the sign-extending
// conversions take one instruction each).
__device__ __forceinline__ float i16_re(uint32_t w) { return (float)(int16_t)(w & 0xffffu); }
__device__ __forceinline__ float i16_im(uint32_t w) { return (float)((int32_t)w >> 16); }

// Sample pair (i, i+1) at byte offset `off` from a uniform row base, lerped
// with weight fr and scaled by the per-pulse scale sc.  The weights carry the
// scale: sc*(1-fr), sc*fr.  For cf16, fma(b1, w1, fma(b0, w0, +0)) keeps the
// f16 operands inside v_fma_mix_f32 (an fma with +0 cannot become a multiply).
template <int DT>
__device__ __forceinline__ float2 lerp_pair(grow_t rowb, unsigned off, float fr,
                                            float sc) {
  if constexpr (DT == TDBP_CF32) {
    const F32x4 v = gload<F32x4>(rowb + off);
    return make_float2(fmaf(fr, v.z - v.x, v.x), fmaf(fr, v.w - v.y, v.y));
  } else if constexpr (DT == TDBP_CF16) {
    const U32x2 w = gload<U32x2>(rowb + off);
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 u0 = __builtin_bit_cast(h2, (uint32_t)w.x);
    const h2 u1 = __builtin_bit_cast(h2, (uint32_t)w.y);
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(fmaf((float)u1.x, w1, fmaf((float)u0.x, w0, 0.0f)),
                       fmaf((float)u1.y, w1, fmaf((float)u0.y, w0, 0.0f)));
  } else if constexpr (DT == TDBP_CI16) {
    const U32x2 w = gload<U32x2>(rowb + off);
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(fmaf(i16_re(w.y), w1, i16_re(w.x) * w0),
                       fmaf(i16_im(w.y), w1, i16_im(w.x) * w0));
  } else {
    const U32x2 w = gload<U32x2>(rowb + off);
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(
        fmaf(__uint_as_float(w.y << 16), w1, __uint_as_float(w.x << 16) * w0),
        fmaf(__uint_as_float(w.y & 0xffff0000u), w1,
             __uint_as_float(w.x & 0xffff0000u) * w0));
  }
}

template <int DT>
__device__ __forceinline__ int elem_bytes() {
  return DT == TDBP_CF32 ? 8 : 4;
}

// The two sample words of a pair as loaded (cf32: 4 floats; cf16/bf16: 2
// packed words), and the lerp of lerp_pair on them.
template <int DT>
struct RawPair {
  typedef typename std::conditional<DT == TDBP_CF32, F32x4, U32x2>::type type;
};
template <int DT>
__device__ __forceinline__ float2 lerp_raw(const typename RawPair<DT>::type v, float fr,
                                           float sc) {
  if constexpr (DT == TDBP_CF32) {
    return make_float2(fmaf(fr, v.z - v.x, v.x), fmaf(fr, v.w - v.y, v.y));
  } else if constexpr (DT == TDBP_CF16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 u0 = __builtin_bit_cast(h2, (uint32_t)v.x);
    const h2 u1 = __builtin_bit_cast(h2, (uint32_t)v.y);
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(fmaf((float)u1.x, w1, fmaf((float)u0.x, w0, 0.0f)),
                       fmaf((float)u1.y, w1, fmaf((float)u0.y, w0, 0.0f)));
  } else if constexpr (DT == TDBP_CI16) {
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(fmaf(i16_re(v.y), w1, i16_re(v.x) * w0),
                       fmaf(i16_im(v.y), w1, i16_im(v.x) * w0));
  } else {
    const float w1 = fr * sc, w0 = sc - w1;
    return make_float2(
        fmaf(__uint_as_float(v.y << 16), w1, __uint_as_float(v.x << 16) * w0),
        fmaf(__uint_as_float(v.y & 0xffff0000u), w1,
             __uint_as_float(v.x & 0xffff0000u) * w0));
  }
}

// lerp_raw for a stage whose pulses share one scale, applied to the stage's
// sum instead: u0 + fr (u1 - u0) as u0 - fr u0 + fr u1, two FMAs per
// component on the raw words (FP16 through the mixed-precision FMA).
template <int DT>
__device__ __forceinline__ float2 lerp_raw_unscaled(const typename RawPair<DT>::type v,
                                                    float fr) {
  if constexpr (DT == TDBP_CF32) {
    return make_float2(fmaf(fr, v.z - v.x, v.x), fmaf(fr, v.w - v.y, v.y));
  } else if constexpr (DT == TDBP_CF16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 u0 = __builtin_bit_cast(h2, (uint32_t)v.x);
    const h2 u1 = __builtin_bit_cast(h2, (uint32_t)v.y);
    return make_float2(fmaf(fr, (float)u1.x, fmaf(-fr, (float)u0.x, (float)u0.x)),
                       fmaf(fr, (float)u1.y, fmaf(-fr, (float)u0.y, (float)u0.y)));
  } else if constexpr (DT == TDBP_CI16) {
    const float a0 = i16_re(v.x), a1 = i16_re(v.y), b0 = i16_im(v.x), b1 = i16_im(v.y);
    return make_float2(fmaf(fr, a1, fmaf(-fr, a0, a0)), fmaf(fr, b1, fmaf(-fr, b0, b0)));
  } else {
    const float a0 = __uint_as_float(v.x << 16), a1 = __uint_as_float(v.y << 16);
    const float b0 = __uint_as_float(v.x & 0xffff0000u),
                b1 = __uint_as_float(v.y & 0xffff0000u);
    return make_float2(fmaf(fr, a1, fmaf(-fr, a0, a0)), fmaf(fr, b1, fmaf(-fr, b0, b0)));
  }
}

// Per-lane constants of the mixed pulse loop.  With d = x - x0, aref =
// u_ref.d, bb = |d|^2 and w = 1 - aref/R0 + (aref/R0)^2 (1/(R0+a) ~ w/R0):
// the range excess over R0 + aref is
//   sd = da + w (bb - a^2) / (2 R0),   a = aref + da,
// and w (bb - a^2) = t0 - (w da + t1) da with the per-pixel t0 = w (bb -
// aref^2), t1 = 2 w aref (both formed in FP64), so sd takes three FMAs.
struct MixedPixel {
  float dx, dy, dz;   // x - x0
  float t0;           // w (bb - aref^2)
  float t1;           // 2 w aref
  float arefd;        // aref / dmrg
  float w;
};

// The range excess of a pixel over its pulse window as a quadratic in the
// pulse index k = q - pc (pc: the tile window's central pulse), fitted per
// pixel in FP64 (mixed_tile).  Over one wave's window the excess is smooth
// to far below the quadratic's remainder: on IW geometry the fit is good to
// 2e-8 m, the FP32 Horner evaluation to 3e-8 m (0.006 mrad of phase).
//
// The quadratic also carries the pixel's sub-sample range offset: with
// aref/dmrg = ia + fa (ia = rint), P(k) = sd + fa dmrg, so the local range
// index is rho = P/dmrg + f0s (one FMA) and the sample index i0s + ia +
// floor(rho).  The row pointer of a pulse carries (i0s + ia_min) * elem,
// the lane (ia - ia_min) * elem; the phase fa dmrg 2/lambda that P adds is
// taken out once per pixel at the end.
//
// SD: the quadratic is sd alone and the offset fa is added to the index, one
// instruction more; the phase then takes no cycles of fa dmrg (up to 21, whose
// FP32 rounding is most of the quadratic form's error).  The split tiles, which
// are not short of issue slots, take this form.
struct PolyPixel {
  float c0, c1, c2;
  unsigned iaoff;    // (ia - ia_min) * elem
  float fa;          // SD: aref/dmrg - ia
};
template <bool SD>
__device__ __forceinline__ float poly_rho(const PolyPixel& pp, float P, float invd, float f0s) {
  const float rho = fmaf(P, invd, f0s);
  return SD ? rho + pp.fa : rho;
}

// One pair on the quadratic.  rows: row start shifted by (i0s + ia_min) *
// elem (unchecked pairs); rowq: the row start (checked pairs, which address
// by the sample index i0s + ia + floor(rho) = ibase + floor(rho)).  lim:
// rho <= lim <=> r <= r_hi.
template <int DT, bool CHECK, bool SD>
__device__ __forceinline__ void poly_pair(const PolyPixel& pp, const float4& r3, float sc,
                                          grow_t rowq, grow_t rows, float Kf, float invd,
                                          bool inwin, int ibase, unsigned smax, float lim,
                                          float& sr, float& si) {
  const float P = fmaf(fmaf(pp.c2, r3.x, pp.c1), r3.x, pp.c0);
  const float rho = poly_rho<SD>(pp, P, invd, r3.y);
  int il;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(rho));
  float2 c;
  const float fr = __builtin_amdgcn_fractf(rho);
  if constexpr (CHECK) {
    const int idx = il + ibase;
    if (!(inwin && (unsigned)idx <= smax && rho <= lim)) return;
    c = lerp_pair<DT>(rowq, (unsigned)idx * (unsigned)elem_bytes<DT>(), fr, sc);
  } else {
    c = lerp_pair<DT>(rows, (unsigned)il * (unsigned)elem_bytes<DT>() + pp.iaoff, fr, sc);
  }
  const float cyc = fmaf(Kf, P, r3.z);
  const float sn = __builtin_amdgcn_sinf(cyc), cs = __builtin_amdgcn_cosf(cyc);
  sr = fmaf(c.x, cs, sr);
  sr = fmaf(-c.y, sn, sr);
  si = fmaf(c.x, sn, si);
  si = fmaf(c.y, cs, si);
}

// One pixel-pulse pair; CHECK selects the per-lane window and gate tests.
// rowb is the uniform start of pulse row q; the lane's byte offset is
// (floor(rho) + i0) * elem, non-negative whenever the gate holds.
template <int DT, bool CHECK>
__device__ __forceinline__ void mixed_pair(const MixedPixel& m, const PulseRec& r, grow_t rowb,
                                           float Kf, float invd, bool inwin, unsigned smax,
                                           float& sr, float& si) {
  const float da = fmaf(r.r0.x, m.dx, fmaf(r.r0.y, m.dy, r.r0.z * m.dz));
  const float e = fmaf(m.w, da, m.t1);
  const float t = fmaf(-e, da, m.t0);             // w (bb - a^2)
  const float sd = fmaf(t, r.r1.z, da);           // R - R0 - aref
  const float rho = fmaf(sd, invd, r.r1.x + m.arefd);
  int il;  // floor(rho) as an integer in one instruction
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(rho));
  if constexpr (CHECK) {
    const int idx = il + __float_as_int(r.r2.z);
    if (!(inwin && (unsigned)idx <= smax && rho <= r.r2.y)) return;
  }
  const float fr = __builtin_amdgcn_fractf(rho);
  const unsigned off =
      (unsigned)il * (unsigned)elem_bytes<DT>() + (unsigned)__float_as_int(r.r1.y);
  const float2 c = lerp_pair<DT>(rowb, off, fr, r.r1.w);
  const float cyc = fmaf(Kf, sd, r.r0.w);
  const float sn = __builtin_amdgcn_sinf(cyc), cs = __builtin_amdgcn_cosf(cyc);
  sr = fmaf(c.x, cs, sr);
  sr = fmaf(-c.y, sn, sr);
  si = fmaf(c.x, sn, si);
  si = fmaf(c.y, cs, si);
}

// The test-free pair split in two for a one-pulse software pipeline: the
// front computes the range, issues the sample load and the phase argument;
// the back (a pulse later) lerps and accumulates.  Same arithmetic as
// mixed_pair<DT, false> (POLY false) or poly_pair<DT, false> (POLY true).
// What a front holds of its sample pair: the loaded words, or for CI16 on the
// quadratic form the four floats of the format-converting load.
template <int DT, bool POLY>
struct FrontWord {
  typedef typename RawPair<DT>::type type;
};
template <>
struct FrontWord<TDBP_CI16, true> {
  typedef F32x4 type;
};
template <int DT, bool POLY>
struct PairFront {
  typename FrontWord<DT, POLY>::type v;
  float fr, cyc, sc;
};
// POLY: the sample pair comes through the structured buffer `rsrc` at
// scalar offset `soff` (row start + (i0s + ia_min) * elem + kSbufBias).
template <int DT, bool POLY, bool SD>
__device__ __forceinline__ PairFront<DT, POLY> mixed_front(const MixedPixel& m,
                                                           const PolyPixel& pp,
                                                           const PulseRec& r, grow_t rowb,
                                                           const I32x4& rsrc, unsigned soff,
                                                           float Kf, float invd) {
  PairFront<DT, POLY> f;
  if constexpr (POLY) {
    const float P = fmaf(fmaf(pp.c2, r.r3.x, pp.c1), r.r3.x, pp.c0);
    const float rho = poly_rho<SD>(pp, P, invd, r.r3.y);
    int il;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(rho));
    // Measured on the 27-burst IW scene: 1.5% above the same loop with a
    // global_load (whose lane offset costs one more VALU op per pair).
    if constexpr (DT == TDBP_CF32)
      f.v = __builtin_bit_cast(F32x4, sbuf_load_v4f32(rsrc, il, (int)pp.iaoff, (int)soff, 0));
    else if constexpr (DT == TDBP_CI16)
      f.v = __builtin_bit_cast(F32x4,
                               sbuf_load_format_v4f32(rsrc, il, (int)pp.iaoff, (int)soff, 0));
    else
      f.v = __builtin_bit_cast(U32x2, sbuf_load_v2f32(rsrc, il, (int)pp.iaoff, (int)soff, 0));
    f.fr = __builtin_amdgcn_fractf(rho);
    f.cyc = fmaf(Kf, P, r.r3.z);
    f.sc = r.r3.w;
  } else {
    const float da = fmaf(r.r0.x, m.dx, fmaf(r.r0.y, m.dy, r.r0.z * m.dz));
    const float e = fmaf(m.w, da, m.t1);
    const float t = fmaf(-e, da, m.t0);
    const float sd = fmaf(t, r.r1.z, da);
    const float rho = fmaf(sd, invd, r.r1.x + m.arefd);
    int il;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(rho));
    const unsigned off =
        (unsigned)il * (unsigned)elem_bytes<DT>() + (unsigned)__float_as_int(r.r1.y);
    f.v = gload<typename RawPair<DT>::type>(rowb + off);
    f.fr = __builtin_amdgcn_fractf(rho);
    f.cyc = fmaf(Kf, sd, r.r0.w);
    f.sc = r.r1.w;
  }
  return f;
}
// U: the stage's pulses share one scale, applied to the stage sum.
template <int DT, bool U, bool POLY>
__device__ __forceinline__ void mixed_back(const PairFront<DT, POLY>& f, float& sr, float& si) {
  float2 c;
  if constexpr (DT == TDBP_CI16 && POLY) {
    if constexpr (U) {
      c = lerp_raw_unscaled<TDBP_CF32>(f.v, f.fr);
    } else {
      const float w1 = f.fr * f.sc, w0 = f.sc - w1;
      c = make_float2(fmaf(f.v.z, w1, f.v.x * w0), fmaf(f.v.w, w1, f.v.y * w0));
    }
  } else {
    c = U ? lerp_raw_unscaled<DT>(f.v, f.fr) : lerp_raw<DT>(f.v, f.fr, f.sc);
  }
  const float sn = __builtin_amdgcn_sinf(f.cyc), cs = __builtin_amdgcn_cosf(f.cyc);
  sr = fmaf(c.x, cs, sr);
  sr = fmaf(-c.y, sn, sr);
  si = fmaf(c.x, sn, si);
  si = fmaf(c.y, cs, si);
}

// The test-free core [qq, cb) of a stage on the quadratic form.  U: the
// stage's pulses share one scale, which the caller applies to the stage sum.
template <int DT, bool U, bool SD>
__device__ __forceinline__ void poly_core(const MixedPixel& m, const PolyPixel& pp,
                                          const PulseRec* rec, int p0,
                                          int qq, int cb, grow_t base, const I32x4& rsrc,
                                          size_t rowbytes, long shift, int ibase, float Kf,
                                          float invd, unsigned smax, float lim, float& sr,
                                          float& si) {
  // CF32: two pairs in flight (the 16-byte gathers bind the texture path,
  // and a third pair's registers buy no latency there): measured 1550 against
  // 1515 Gpixel-pulse/s with three on the 27-burst IW scene (variants 0 and 5).
  if constexpr (DT == TDBP_CF32) {
    if (qq < cb && ((cb - qq) & 1)) {
      const grow_t rowq = base + (size_t)qq * rowbytes;
      const float4 r3 = rec[qq - p0].r3;
      poly_pair<DT, false, SD>(pp, r3, U ? 1.f : r3.w, rowq, rowq + shift, Kf, invd, true, ibase,
                           smax, lim, sr, si);
      ++qq;
    }
    if (qq < cb) {
      grow_t rp = base + (size_t)qq * rowbytes;
      unsigned so = (unsigned)((long)qq * (long)rowbytes + shift + kSbufBias);
      const unsigned rb32 = (unsigned)rowbytes;
      const PulseRec* rr = rec + (qq - p0);
      PairFront<DT, true> fa = mixed_front<DT, true, SD>(m, pp, rr[0], rp, rsrc, so, Kf, invd);
      PairFront<DT, true> fb;
      for (; qq + 2 < cb; qq += 2) {
        fb = mixed_front<DT, true, SD>(m, pp, rr[1], rp, rsrc, so + rb32, Kf, invd);
        __builtin_amdgcn_sched_barrier(0);
        mixed_back<DT, U, true>(fa, sr, si);
        so += 2 * rb32;
        rr += 2;
        fa = mixed_front<DT, true, SD>(m, pp, rr[0], rp, rsrc, so, Kf, invd);
        __builtin_amdgcn_sched_barrier(0);
        mixed_back<DT, U, true>(fb, sr, si);
      }
      fb = mixed_front<DT, true, SD>(m, pp, rr[1], rp, rsrc, so + rb32, Kf, invd);
      mixed_back<DT, U, true>(fa, sr, si);
      mixed_back<DT, U, true>(fb, sr, si);
    }
    return;
  }
  // Packed storages: three pairs in flight: the load of pulse q + 2 is
  // issued before the back of pulse q.  (cb - ca) mod 3 plain pairs first; the
  // rest is a multiple of 3, so a loop pass (taken when >= 6 remain) reads
  // records q..q+4 inside the core.  Measured: 2.6 % above two in flight on
  // the 27-burst IW scene with cf16 (the quadratic's shorter body leaves less
  // work to cover the gather with).
  const int rem = (cb - qq) % 3;
  for (int r = 0; r < rem; ++r, ++qq) {
    const grow_t rowq = base + (size_t)qq * rowbytes;
    const float4 r3 = rec[qq - p0].r3;
    poly_pair<DT, false, SD>(pp, r3, U ? 1.f : r3.w, rowq, rowq + shift, Kf, invd, true, ibase,
                         smax, lim, sr, si);
  }
  if (qq < cb) {
    grow_t rp = base + (size_t)qq * rowbytes;
    unsigned so = (unsigned)((long)qq * (long)rowbytes + shift + kSbufBias);
    const unsigned rb32 = (unsigned)rowbytes;
    const PulseRec* rr = rec + (qq - p0);
    PairFront<DT, true> fa = mixed_front<DT, true, SD>(m, pp, rr[0], rp, rsrc, so, Kf, invd);
    PairFront<DT, true> fb = mixed_front<DT, true, SD>(m, pp, rr[1], rp, rsrc, so + rb32, Kf, invd);
    PairFront<DT, true> fc;
    for (; qq + 3 < cb; qq += 3) {
      fc = mixed_front<DT, true, SD>(m, pp, rr[2], rp, rsrc, so + 2 * rb32, Kf, invd);
      __builtin_amdgcn_sched_barrier(0);
      mixed_back<DT, U, true>(fa, sr, si);
      fa = mixed_front<DT, true, SD>(m, pp, rr[3], rp, rsrc, so + 3 * rb32, Kf, invd);
      __builtin_amdgcn_sched_barrier(0);
      mixed_back<DT, U, true>(fb, sr, si);
      fb = mixed_front<DT, true, SD>(m, pp, rr[4], rp, rsrc, so + 4 * rb32, Kf, invd);
      __builtin_amdgcn_sched_barrier(0);
      mixed_back<DT, U, true>(fc, sr, si);
      so += 3 * rb32;
      rr += 3;
    }
    fc = mixed_front<DT, true, SD>(m, pp, rr[2], rp, rsrc, so + 2 * rb32, Kf, invd);
    mixed_back<DT, U, true>(fa, sr, si);
    mixed_back<DT, U, true>(fb, sr, si);
    mixed_back<DT, U, true>(fc, sr, si);
  }
}

// One stage's pulses [qa, qb) for one wave: checked edges [qa, ea) and
// [eb, qb), the core [ca, cb) where every live lane is inside its window.
// stage_safe: every pulse of the stage keeps the whole tile inside the gate.
// POLY: the quadratic (shift = (i0s + ia_min) * elem, ibase = i0s + ia, lim
// = r_hi - i0s - ia); else the FP32 chain.
template <int DT, bool POLY, bool SD>
__device__ __forceinline__ void stage_pulses(const MixedPixel& m, const PolyPixel& pp,
                                             const PulseRec* rec, int p0, int qa, int qb,
                                             int qc0, int qc1, bool stage_safe, bool uni,
                                             grow_t base, const I32x4& rsrc, size_t rowbytes,
                                             long shift, int ibase, float lim,
                                             float Kf, float invd, int azs, unsigned n,
                                             unsigned smax, float& sr, float& si) {
  const int ea = min(qb, qc0);                      // [qa, ea): checked
  const int ca = max(qa, qc0), cb = min(qb, qc1);   // core
  const int eb = max(qa, qc1);                      // [eb, qb): checked
  auto checked = [&](int qq) {
    const grow_t rowq = base + (size_t)qq * rowbytes;
    if constexpr (POLY)
      poly_pair<DT, true, SD>(pp, rec[qq - p0].r3, uni ? 1.f : rec[qq - p0].r3.w, rowq, rowq, Kf,
                          invd, (unsigned)(qq - azs) < n,
                          ibase, smax, lim, sr, si);
    else
      mixed_pair<DT, true>(m, rec[qq - p0], rowq, Kf, invd, (unsigned)(qq - azs) < n, smax, sr,
                           si);
  };
  auto unchecked = [&](int qq) {
    const grow_t rowq = base + (size_t)qq * rowbytes;
    if constexpr (POLY)
      poly_pair<DT, false, SD>(pp, rec[qq - p0].r3, uni ? 1.f : rec[qq - p0].r3.w, rowq,
                           rowq + shift, Kf, invd, true, ibase,
                           smax, lim, sr, si);
    else
      mixed_pair<DT, false>(m, rec[qq - p0], rowq, Kf, invd, true, smax, sr, si);
  };
  for (int qq = qa; qq < ea; ++qq) checked(qq);
  if (stage_safe) {
    // No tests.  Each sample load is issued ahead of its use (the fronts keep
    // their own registers; the scheduling barrier after each front keeps the
    // load there).  An empty core (cb <= ca) does nothing.
    int qq = ca;
    if constexpr (POLY) {
      if (uni)
        poly_core<DT, true, SD>(m, pp, rec, p0, qq, cb, base, rsrc, rowbytes, shift, ibase, Kf, invd,
                            smax, lim, sr, si);
      else
        poly_core<DT, false, SD>(m, pp, rec, p0, qq, cb, base, rsrc, rowbytes, shift, ibase, Kf, invd,
                             smax, lim, sr, si);
    } else {
      // FP32 chain: two pairs in flight; an odd count starts with one plain
      // pair.  Measured: one pair in flight 1240, two 1442-1546, three 1% below
      // two Gpixel-pulse/s on the 27-burst IW scene.
      if (qq < cb && ((cb - qq) & 1)) {
        unchecked(qq);
        ++qq;
      }
      if (qq < cb) {
        grow_t rp = base + (size_t)qq * rowbytes;
        unsigned so = (unsigned)((long)qq * (long)rowbytes + shift + kSbufBias);
        const unsigned rb32 = (unsigned)rowbytes;
        const PulseRec* rr = rec + (qq - p0);
        PairFront<DT, POLY> fa = mixed_front<DT, POLY, SD>(m, pp, rr[0], rp, rsrc, so, Kf, invd);
        PairFront<DT, POLY> fb;
        for (; qq + 2 < cb; qq += 2) {
          fb = mixed_front<DT, POLY, SD>(m, pp, rr[1], rp + rowbytes, rsrc, so + rb32, Kf, invd);
          __builtin_amdgcn_sched_barrier(0);
          mixed_back<DT, false, POLY>(fa, sr, si);
          rp += 2 * rowbytes;
          so += 2 * rb32;
          rr += 2;
          fa = mixed_front<DT, POLY, SD>(m, pp, rr[0], rp, rsrc, so, Kf, invd);
          __builtin_amdgcn_sched_barrier(0);
          mixed_back<DT, false, POLY>(fb, sr, si);
        }
        fb = mixed_front<DT, POLY, SD>(m, pp, rr[1], rp + rowbytes, rsrc, so + rb32, Kf, invd);
        mixed_back<DT, false, POLY>(fa, sr, si);
        mixed_back<DT, false, POLY>(fb, sr, si);
      }
    }
  } else {
    for (int qq = ca; qq < cb; ++qq) {
      if (__builtin_amdgcn_readfirstlane(__float_as_int(rec[qq - p0].r2.x)) != 0)
        unchecked(qq);
      else
        checked(qq);
    }
  }
  for (int qq = eb; qq < qb; ++qq) checked(qq);
}

// 1/sqrt(x) in FP64 for normal x > 0: the hardware estimate and two Newton
// steps y <- y (3/2 - x/2 y^2), each squaring the relative error.
__device__ __forceinline__ double rsqrt64(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * x;
  y = y * fma(-h * y, y, 1.5);
  y = y * fma(-h * y, y, 1.5);
  return y;
}

// Lane `l`'s double, moved to scalar registers.
__device__ __forceinline__ double lane_double(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Range excess R - |x0 - s_q| - aref of pixel x0 + d at pulse q, in FP64,
// from the pulse's look vector u = (x0 - s_q)/R0 and h = 1/(2 R0): with a =
// u.d and |d|^2 = bb, R - R0 - a = (bb - a^2)/(R + R0 + a) and 1/(R + R0 +
// a) = h (1 - q + q^2) with q = 2 h a, to 1e-10 m at satellite ranges.
__device__ __forceinline__ double node_excess(double u0, double u1, double u2, double h,
                                              const double* d, double bb, double aref) {
  const double a = u0 * d[0] + u1 * d[1] + u2 * d[2];
  const double q = 2.0 * h * a;
  return (a - aref) + (bb - a * a) * fma(q, q - 1.0, 1.0) * h;
}

// One stage of pulses [p0, stage_end) of a tile whose sample windows are
// staged in LDS (every live wave on the quadratic, the stage safe, the
// tile's window <= kLdsWindow samples).  Sub-stages of kLdsPulses pulses:
// the four waves load the pulses' windows -- kLdsWindow samples from the
// absolute index in rec[].r1.y, one 16-byte load per lane and pulse,
// converted to FP32 by the descriptor for CF16/CI16, scaled when the stage's
// pulses do not share one scale -- into sbuf, then each wave sums its pulses
// reading the sample pair of a lane at slot j, local index
//   (ia - ia_min) + floor(P/dmrg + F_j),   F_j = rec[].r2.w,
// which the window construction keeps in [1, kLdsWindow - 2].  Lanes outside
// their own window (sub-stages not inside the wave's core) add nothing.
template <int DT>
__device__ __forceinline__ void staged_stage(const BurstDev& b, const PolyPixel& pp,
                                             const PulseRec* rec, F32x4* sbuf, int p0,
                                             int stage_end, int qa, int qb, int qc0, int qc1,
                                             bool wave_live, bool scale_here, int laneoffs,
                                             const I32x4& srsrc, size_t rowbytes, float Kf,
                                             float invd, int azs, unsigned n, float& sr,
                                             float& si) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int kSlot = kLdsWindow / 2;   // float4 (two samples) per pulse slot
  constexpr int kPer = kLdsPulses / 4;    // pulses each wave stages per sub-stage
  // Lanes past the window load nothing (their index is out of the
  // descriptor's range, which returns zeros).
  const int lane2 = 2 * lane + 1 < kLdsWindow ? 2 * lane : (1 << 24);
  // Byte address in LDS of this lane's sample window position 0, slot 0.
  const char* lbase = (const char*)sbuf + laneoffs * 8;
  // Issue the loads of sub-stage s0's windows for this wave's pulses
  // j = wave + 4i into v[i] (in flight while the previous sub-stage sums).
  auto issue = [&](int s0, F32x4* v) {
    const int np = min(kLdsPulses, stage_end - s0);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int j = wave + 4 * i;
      if (j < np) {
        const PulseRec& r = rec[s0 - p0 + j];
        const int base = __builtin_amdgcn_readfirstlane(__float_as_int(r.r1.y));
        // Pairs that would leave the row read zeros: the window may reach
        // past the row's ends.
        const int vidx = (unsigned)(base + lane2) <= (unsigned)(b.S - 2) ? lane2
                                                                          : kSbufIndexLimit;
        const unsigned so = (unsigned)((long)(s0 + j) * (long)rowbytes +
                                       (long)base * elem_bytes<DT>() + kSbufBias);
        if constexpr (DT == TDBP_CF32) {
          v[i] = __builtin_bit_cast(F32x4, sbuf_load_v4f32(srsrc, vidx, 0, (int)so, 0));
        } else if constexpr (DT == TDBP_CF16 || DT == TDBP_CI16) {
          v[i] = __builtin_bit_cast(F32x4, sbuf_load_format_v4f32(srsrc, vidx, 0, (int)so, 0));
        } else {
          const U32x2 w =
              __builtin_bit_cast(U32x2, sbuf_load_v2f32(srsrc, vidx, 0, (int)so, 0));
          v[i] = F32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                       __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
        }
      }
    }
  };
  // One pair from slot j: the local index floor(P/dmrg + F_j) from the
  // pulse's record, both samples read at slot offset j*kLdsWindow*8 (an
  // immediate when j is a constant), lerp, phase, MAC; MASK: lanes outside
  // their own window add nothing.
  auto pair = [&](int j, int q, const PulseRec& r, bool mask) {
    const float P = fmaf(fmaf(pp.c2, r.r3.x, pp.c1), r.r3.x, pp.c0);
    const float rho = fmaf(P, invd, r.r2.w);
    int il;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(rho));
    const float fr = __builtin_amdgcn_fractf(rho);
    const char* a = lbase + il * 8 + j * (kLdsWindow * 8);
    const float2 u0 = *(const float2*)a;
    const float2 u1 = *(const float2*)(a + 8);
    float cr = fmaf(fr, u1.x - u0.x, u0.x), ci = fmaf(fr, u1.y - u0.y, u0.y);
    if (mask && (unsigned)(q - azs) >= n) {
      cr = 0.f;
      ci = 0.f;
    }
    const float cyc = fmaf(Kf, P, r.r3.z);
    const float sn = __builtin_amdgcn_sinf(cyc), cs = __builtin_amdgcn_cosf(cyc);
    sr = fmaf(cr, cs, sr);
    sr = fmaf(-ci, sn, sr);
    si = fmaf(cr, sn, si);
    si = fmaf(ci, cs, si);
  };
  F32x4 v[kPer];
  issue(p0, v);
  for (int s0 = p0; s0 < stage_end; s0 += kLdsPulses) {
    const int np = min(kLdsPulses, stage_end - s0);
    // Store this sub-stage's windows (the loads were issued a sub-stage ago).
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int j = wave + 4 * i;
      if (j < np) {
        F32x4 w = v[i];
        if (scale_here) {
          const float sc = rec[s0 - p0 + j].r3.w;
          w = F32x4{w.x * sc, w.y * sc, w.z * sc, w.w * sc};
        }
        if (lane < kSlot) sbuf[j * kSlot + lane] = w;
      }
    }
    __syncthreads();
    if (s0 + kLdsPulses < stage_end) issue(s0 + kLdsPulses, v);
    if (wave_live) {
      const int ja = max(s0, qa) - s0, jb = min(s0 + np, qb) - s0;
      const bool full = s0 + ja >= qc0 && s0 + jb <= qc1;
      const PulseRec* rs = rec + (s0 - p0);
      if (full && ja == 0 && jb == kLdsPulses) {
        // The wave's core covers the whole sub-stage: a fixed sequence of
        // kLdsPulses pairs with no per-lane test.
#pragma unroll
        for (int j = 0; j < kLdsPulses; ++j) pair(j, s0 + j, rs[j], false);
      } else {
        for (int j = ja; j < jb; ++j) pair(j, s0 + j, rs[j], !full);
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------- FP64 tile on the range excess
//
// The FP64 kernel is bound by FP64 VALU issue (and, at full issue, by the
// clock the card holds under it): plain_pair takes 86 instructions, half of
// them for the root, the reduction and the sin/cos of a phase that changes
// smoothly from pulse to pulse.  Here a pixel's range is taken as
//   R = R0 + e,   R0 = |x0 - s_p|,   e = (2 u.d + |d|^2) / (R + R0)
// with x0 a reference pixel of the tile, u = x0 - s_p and d = x - x0.  R0, its
// phase factor T = exp(j 4 pi R0/lambda) and its range index are formed once
// per pulse and workgroup (PlainRec in LDS); the excess e of a pixel is a
// quartic in the pulse index over the tile's window, interpolated at five
// Chebyshev pulses.  Within a block of up to 2 kPlainHalf pulses the quartic
// is a quadratic to 2e-11 m, so the index advances by differences and the
// phase factor by a rotation (PlainBlock).  25 instructions per pair in a full
// block, 33 over the launch with the blocks' and tiles' set-up, all in FP64
// but the lerp, which is FP32 as in plain_pair (in FP64 a burst took 5 % longer).
//
// What the form rests on is checked: per pixel the quartic at the window's
// two ends (1e-10 m, the rounding of R itself in FP64 at 8.5e5 m) and the
// block length against its derivatives, per pulse the look vector u/R0
// against its own quartic (1e-10 m at the tile's farthest pixel: a pulse
// position that does not fit the others) and the range gate with the bound on
// e.  Waves or stages that miss a check take plain_pair pair by pair.
//
// One IW burst (1500 x 21000 samples, 4000 x 1500 pixels, 2.97e9 pairs): 3.15
// ms against 7.0 ms pair by pair, the error either way that of the
// FP32 lerp and the stored image (5.0e-8 at 64 pulses, 6.1e-8 at 720).  With z *= w, w *= v pulse after pulse instead of pairs about
// the block's centre: 3.6 ms (37 instructions per pair); blocks of 64 pulses:
// 3.25 ms; 256 pulses per stage: 3.25 ms.
constexpr int kPlainNodes = 5;    // interpolation pulses; two more check the ends
constexpr int kPlainHalf = 16;    // half the pulses of a full block
constexpr int kPlainStage = 768;  // pulses per stage of records (24 KB of LDS)
constexpr double kPlainTol = 1e-10;

struct PlainRec {
  double rb;       // (R0 - rngstart)/dmrg
  double tr, ti;   // T
  double pad;
};

struct PlainShared {
  double x0[3];
  double u[kPlainNodes + 2][3], r2[kPlainNodes + 2], R0[kPlainNodes + 2], t[kPlainNodes + 2];
  double rcp[10];                 // 1/(t_j - t_i) in the order newton4 takes them
  double look[3][kPlainNodes];    // u/R0 per component, monomials in t
  int key, wlo, whi;
  unsigned dmax, emax;            // FP32 bits of max |x - x0|, of max sum |coefficient|
};

// Quartic through (t[j], y[j]), j < 5, as monomial coefficients: Newton's
// divided differences (rcp: reciprocals of the node distances, level by
// level), then multiplied out.
__device__ __forceinline__ void newton4(const double* t, const double* rcp, const double* y,
                                        double* c) {
  double a[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) a[i] = y[i];
  int k = 0;
#pragma unroll
  for (int l = 1; l < 5; ++l) {
#pragma unroll
    for (int i = 4; i >= l; --i) a[i] = (a[i] - a[i - 1]) * rcp[k + i - l];
    k += 5 - l;
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) c[i] = 0.0;
  c[0] = a[4];
#pragma unroll
  for (int l = 3; l >= 0; --l) {   // c(t) <- c(t) (t - t_l) + a_l
#pragma unroll
    for (int i = 4; i >= 1; --i) c[i] = fma(-t[l], c[i], c[i - 1]);
    c[0] = fma(-t[l], c[0], a[l]);
  }
}

__device__ __forceinline__ double quartic(const double* c, double t) {
  return fma(fma(fma(fma(c[4], t, c[3]), t, c[2]), t, c[1]), t, c[0]);
}

// 1/x for normal x: the hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp64(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}

// exp(2 pi j c) for any c of moderate size.
__device__ __forceinline__ void cis_cycles(double c, double* re, double* im) {
  sincos_2pi(c - rint(c), im, re);
}

// One block of pulses, summed from its centre outward in pairs at k = -(j +
// 1/2) and j + 1/2 pulses from it.  With the excess e0 + a1 k + a2 k^2 the
// phase factors of a pair are z0 g u* and z0 g u, u = exp(j 4 pi/lambda a1 k)
// and g = exp(j 4 pi/lambda a2 k^2) common to both: one complex product by u
// of the sum and difference of the two samples, one by g (|phase| <= 1e-3,
// taken to second order), z0 once per block.  u advances by the three-term
// recurrence u_{j+1} = 2 cos(theta) u_j - u_{j-1}.
struct PlainBlock {
  double pp, dp, pm, dm, d2;   // excess in samples at +-k, differences outward
  double ur, ui, vr, vi, cc;   // u, the u before it, 2 cos(theta)
  double eps;                  // phase of g is eps k^2
  double ar, ai;               // the block's sum without z0
};
// What a pair holds between its loads and its use.
struct PlainFront {
  SbufF4 vp, vm;
  float fp, fm;
};

// The loads of the pair whose records are rp (k > 0) and rm, rows at byte
// offsets sp and sm; advances the index.
__device__ __forceinline__ PlainFront plain_front(PlainBlock& s, const PlainRec& rp,
                                                  const PlainRec& rm, const I32x4& rsrc,
                                                  unsigned sp, unsigned sm) {
  PlainFront f;
  const double xp = rp.rb + s.pp, xm = rm.rb + s.pm;
  f.vp = sbuf_load_v4f32(rsrc, (int)xp, 0, (int)sp, 0);   // xp >= 0: truncation is floor
  f.vm = sbuf_load_v4f32(rsrc, (int)xm, 0, (int)sm, 0);
  s.pp += s.dp;
  s.pm += s.dm;
  s.dp += s.d2;
  s.dm += s.d2;
  f.fp = (float)__builtin_amdgcn_fract(xp);
  f.fm = (float)__builtin_amdgcn_fract(xm);
  return f;
}
// The pair's sum.  inp, inm (MASK): lanes outside their window add nothing.
template <bool MASK>
__device__ __forceinline__ void plain_back(PlainBlock& s, const PlainRec& rp, const PlainRec& rm,
                                           const PlainFront& f, double k2, bool inp, bool inm) {
  // a (1 - t) + b t in two FMAs, as near the exact value as plain_pair's two
  // weights (a + t (b - a) would be 14 % further off on white samples).
  const auto lerp = [](float t, float a, float b) { return fmaf(t, b, fmaf(-t, a, a)); };
  float pr = lerp(f.fp, f.vp.x, f.vp.z), pi = lerp(f.fp, f.vp.y, f.vp.w);
  float mr = lerp(f.fm, f.vm.x, f.vm.z), mi = lerp(f.fm, f.vm.y, f.vm.w);
  if constexpr (MASK) {
    pr = inp ? pr : 0.f;
    pi = inp ? pi : 0.f;
    mr = inm ? mr : 0.f;
    mi = inm ? mi : 0.f;
  }
  const double dpr = pr, dpi = pi, dmr = mr, dmi = mi;
  const double Pr = fma(-dpi, rp.ti, dpr * rp.tr), Pi = fma(dpi, rp.tr, dpr * rp.ti);
  const double Mr = fma(-dmi, rm.ti, dmr * rm.tr), Mi = fma(dmi, rm.tr, dmr * rm.ti);
  const double Sr = Pr + Mr, Si = Pi + Mi, Dr = Pr - Mr, Di = Pi - Mi;
  // P u + M u*
  const double qr = fma(-Di, s.ui, Sr * s.ur), qi = fma(Dr, s.ui, Si * s.ur);
  const double x = s.eps * k2;
  const double g = fma(-0.5 * x, x, 1.0);
  s.ar = fma(qr, g, s.ar);
  s.ar = fma(-qi, x, s.ar);
  s.ai = fma(qi, g, s.ai);
  s.ai = fma(qr, x, s.ai);
  const double nr = fma(s.cc, s.ur, -s.vr), ni = fma(s.cc, s.ui, -s.vi);
  s.vr = s.ur;
  s.vi = s.ui;
  s.ur = nr;
  s.ui = ni;
}

// The 2 m pulses around the pair (rec[-1], rec[0]): rec points at the record
// just after the centre, so at its row's byte offset.  One pair's loads are
// in flight ahead of their use.  m = M when M > 0 (unrolled), else mm.  MASK:
// pulse q0 + i belongs to rec[i]; the lane's window is [azs, azs + na).
template <int M, bool MASK>
__device__ __forceinline__ void plain_pulses(PlainBlock& s, const PlainRec* rec, int mm,
                                             const I32x4& rsrc, unsigned so, unsigned rb32,
                                             int q0, int azs, unsigned na) {
  auto in = [&](int i) { return (unsigned)(q0 + i - azs) < na; };
  auto front = [&](int j) {
    return plain_front(s, rec[j], rec[-1 - j], rsrc, so + (unsigned)j * rb32,
                       so - (unsigned)(j + 1) * rb32);
  };
  auto back = [&](int j, const PlainFront& f) {
    plain_back<MASK>(s, rec[j], rec[-1 - j], f, (double)(j * (j + 1)) + 0.25, in(j), in(-1 - j));
  };
  PlainFront a = front(0), b;
  if constexpr (M > 0) {
#pragma unroll
    for (int j = 0; j < M; j += 2) {
      b = front(j + 1);
      __builtin_amdgcn_sched_barrier(0);
      back(j, a);
      if (j + 2 < M) a = front(j + 2);
      __builtin_amdgcn_sched_barrier(0);
      back(j + 1, b);
    }
  } else {
    int j = 0;
    for (; j + 2 < mm; j += 2) {
      b = front(j + 1);
      __builtin_amdgcn_sched_barrier(0);
      back(j, a);
      a = front(j + 2);
      __builtin_amdgcn_sched_barrier(0);
      back(j + 1, b);
    }
    if (j + 1 < mm) {
      b = front(j + 1);
      back(j, a);
      back(j + 1, b);
    } else {
      back(j, a);
    }
  }
}

// One block of n <= 2 * kPlainHalf pulses from pulse q, whose record is rec[0],
// added to (ar, ai).  core: n is even and every live lane is inside its
// window.  Else lanes are masked by theirs; an odd n takes one more pulse,
// masked on every lane (its record exists: a stage has one more than its
// pulses).
__device__ __forceinline__ void plain_block(const double* c, double dt, int wlo, int q, int n,
                                            const PlainRec* rec, const I32x4& rsrc, unsigned rb32,
                                            bool core, int azs, unsigned na, double cyc_per_m,
                                            double smp_per_m, double& ar, double& ai) {
  const int m = (n + 1) >> 1;
  const double h = m, hi = m == kPlainHalf ? 1.0 / kPlainHalf : 1.0 / m;
  // the quadratic through the quartic at the centre and m pulses to each side
  const double tc = fma((double)(q - wlo) + (m - 0.5), dt, -1.0);
  const double e0 = quartic(c, tc), em = quartic(c, fma(-h, dt, tc)),
               ep = quartic(c, fma(h, dt, tc));
  const double a1 = (ep - em) * (0.5 * hi);
  const double a2 = ((ep - e0) - (e0 - em)) * (0.5 * hi * hi);
  PlainBlock s;
  s.d2 = 2.0 * a2 * smp_per_m;
  s.pp = fma(0.5, a1, fma(0.25, a2, e0)) * smp_per_m;
  s.pm = fma(-0.5, a1, fma(0.25, a2, e0)) * smp_per_m;
  s.dp = fma(2.0, a2, a1) * smp_per_m;
  s.dm = fma(2.0, a2, -a1) * smp_per_m;
  s.eps = a2 * (cyc_per_m * 6.283185307179586);
  cis_cycles(0.5 * a1 * cyc_per_m, &s.ur, &s.ui);
  s.vr = s.ur;
  s.vi = -s.ui;
  s.cc = fma(-4.0 * s.ui, s.ui, 2.0);
  s.ar = 0.;
  s.ai = 0.;
  const unsigned so = (unsigned)(q + m) * rb32;
  if (core && n == 2 * kPlainHalf)
    plain_pulses<kPlainHalf, false>(s, rec + m, m, rsrc, so, rb32, q + m, azs, na);
  else if (core)
    plain_pulses<0, false>(s, rec + m, m, rsrc, so, rb32, q + m, azs, na);
  else
    plain_pulses<0, true>(s, rec + m, m, rsrc, so, rb32, q + m, azs,
                          (unsigned)max(0, min((int)na, q + n - azs)));
  double zr, zi;
  cis_cycles(e0 * cyc_per_m, &zr, &zi);
  ar = fma(s.ar, zr, ar);
  ar = fma(-s.ai, zi, ar);
  ai = fma(s.ar, zi, ai);
  ai = fma(s.ai, zr, ai);
}

template <int TR, int STACK>
__device__ __forceinline__ void plain_excess_tile(const BurstDev& b, int tile, PlainRec* rec,
                                                  PlainShared* sh) {
  PixelCtx p = pixel_of<TR, STACK>(b, tile);
  const int tid = threadIdx.x;
  const bool live = p.aze > p.azs;
  double x[3] = {0., 0., 0.};
  if (live) pixel_ecef(b, p.row, p.col, x);

  // Tile window and reference pixel (the live one nearest the centre).
  constexpr int WR = TileShape<TR, STACK>::WR, WC = TileShape<TR, STACK>::WC;
  const int wr = TileShape<TR, STACK>::row(tid), wc = TileShape<TR, STACK>::col(tid);
  if (tid == 0) {
    sh->key = 0x7fffffff;
    sh->wlo = 0x7fffffff;
    sh->whi = -1;
    sh->dmax = 0u;
    sh->emax = 0u;
  }
  __syncthreads();
  if (live) {
    atomicMin(&sh->key, (abs(2 * wr - WR) + abs(2 * wc - WC)) * 256 + tid);
    atomicMin(&sh->wlo, p.azs);
    atomicMax(&sh->whi, p.aze);
  }
  __syncthreads();
  const int ref = sh->key;
  if (ref == 0x7fffffff) {  // nothing to compute in this tile
    store_out(b, p, 0.f, 0.f);
    return;
  }
  const int wlo = __builtin_amdgcn_readfirstlane(sh->wlo);
  const int whi = __builtin_amdgcn_readfirstlane(sh->whi);
  if ((ref & 255) == tid) {
    sh->x0[0] = x[0];
    sh->x0[1] = x[1];
    sh->x0[2] = x[2];
  }
  __syncthreads();
  const double x0[3] = {uniform(sh->x0[0]), uniform(sh->x0[1]), uniform(sh->x0[2])};

  // The quartics need 32 pulses to have distinct nodes, the gather 32-bit
  // byte offsets into the burst.
  const unsigned rb32 = (unsigned)b.S * 8u;
  const bool quart = whi - wlo >= 32 && (size_t)b.L * b.S * 8u < (size_t)0x7fffffff;
  // t = (q - wlo) dt - 1 maps the window's pulses to [-1, 1].
  const double dt = quart ? 2.0 / (whi - 1 - wlo) : 0.0;
  double c[kPlainNodes] = {0., 0., 0., 0., 0.};
  bool fit = false;
  int half = 1;   // longest half block the lane's quartic allows
  if (quart) {
    // Threads 0..6: the node pulses (Chebyshev points, then the two ends).
    const int span = whi - 1 - wlo;
    auto node_pulse = [&](int j) {
      // (1 - cos((2 j + 1) pi / 10)) / 2
      const double g[kPlainNodes] = {0.024471741852423214, 0.20610737385376343, 0.5,
                                     0.79389262614623657, 0.97552825814757679};
      double f = j == kPlainNodes ? 0.0 : 1.0;
#pragma unroll
      for (int i = 0; i < kPlainNodes; ++i) f = j == i ? g[i] : f;
      return wlo + (int)rint(f * span);
    };
    if (tid < kPlainNodes + 2) {
      const int q = node_pulse(tid);
      const double* s = b.satloc + 3 * q;
      const double u0 = x0[0] - s[0], u1 = x0[1] - s[1], u2 = x0[2] - s[2];
      const double r2 = u0 * u0 + u1 * u1 + u2 * u2;
      sh->u[tid][0] = u0;
      sh->u[tid][1] = u1;
      sh->u[tid][2] = u2;
      sh->r2[tid] = r2;
      sh->R0[tid] = range_sqrt(r2);
      sh->t[tid] = fma((double)(q - wlo), dt, -1.0);
    }
    __syncthreads();
    if (tid < 10) {   // level l, place i: nodes i and i + l
      const int l = tid < 4 ? 1 : tid < 7 ? 2 : tid < 9 ? 3 : 4;
      const int i = tid - (l == 1 ? 0 : l == 2 ? 4 : l == 3 ? 7 : 9);
      sh->rcp[tid] = 1.0 / (sh->t[i + l] - sh->t[i]);
    }
    __syncthreads();
    if (tid < 3) {    // component tid of the look vector
      double y[kPlainNodes], l[kPlainNodes];
      for (int j = 0; j < kPlainNodes; ++j) y[j] = sh->u[j][tid] / sh->R0[j];
      newton4(sh->t, sh->rcp, y, l);
      for (int j = 0; j < kPlainNodes; ++j) sh->look[tid][j] = l[j];
    }
    if (live) {
      const double d0 = x[0] - x0[0], d1 = x[1] - x0[1], d2 = x[2] - x0[2];
      const double bb = d0 * d0 + d1 * d1 + d2 * d2;
      double y[kPlainNodes + 2];
#pragma unroll
      for (int j = 0; j < kPlainNodes + 2; ++j) {
        const double num =
            fma(2.0, fma(sh->u[j][0], d0, fma(sh->u[j][1], d1, sh->u[j][2] * d2)), bb);
        y[j] = num * rcp64(range_sqrt(sh->r2[j] + num) + sh->R0[j]);
        __builtin_amdgcn_sched_barrier(0);   // one node's operands at a time
      }
      newton4(sh->t, sh->rcp, y, c);
      const double el = fabs(quartic(c, sh->t[kPlainNodes]) - y[kPlainNodes]);
      const double eh = fabs(quartic(c, sh->t[kPlainNodes + 1]) - y[kPlainNodes + 1]);
      fit = el <= kPlainTol && eh <= kPlainTol;   // false for NaN
      // Second and third derivative over [-1, 1] per pulse: a block of half
      // length h has |eps k^2| <= 2 pi cycles c2 h^2 and leaves c3 h^3 (0.385
      // its largest value over the block) of the quartic.
      const double c2 =
          (fabs(c[2]) + 3.0 * fabs(c[3]) + 6.0 * fabs(c[4])) * dt * dt * b.two_over_wvl * 6.2832;
      const double c3 = (fabs(c[3]) + 4.0 * fabs(c[4])) * dt * dt * dt * 0.385;
      half = kPlainHalf;
      while (half > 1 && !(c2 * half * half <= 1e-3 && c3 * half * half * half <= 2e-11))
        half >>= 1;
      fit = fit && half >= 4;
      // |quartic| <= sum |c_j| on [-1, 1]; FP32 rounded up.
      const double em = fabs(c[0]) + fabs(c[1]) + fabs(c[2]) + fabs(c[3]) + fabs(c[4]);
      if (fit) atomicMax(&sh->emax, __float_as_uint((float)(em * (1.0 + 1e-6))));
      atomicMax(&sh->dmax, __float_as_uint((float)(sqrt(bb) * (1.0 + 1e-6))));
    }
    __syncthreads();
  }
  const bool wave_fit = quart && wave_min(live && !fit ? 0 : 1) == 1;
  const int blk = 2 * wave_min(live ? half : kPlainHalf);
  // Bound on the excess the recurrences can form, in samples: a block's
  // quadratic through three values of the quartic stays within 5/4 of their
  // largest, and those lie at most 1 1/2 pulses outside the window, |t| <=
  // 1.1; two samples of margin.
  const double ext =
      2.0 * (double)__uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)sh->emax)) *
          b.inv_dmrg + 2.0;
  const double dmax =
      (double)__uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)sh->dmax));

  const int qlo = wave_min(live ? p.azs : 0x7fffffff);
  const int qhi = wave_max(live ? p.aze : -1);
  const int qc0 = wave_max(live ? p.azs : -1);         // every live lane inside
  const int qc1 = wave_min(live ? p.aze : 0x7fffffff); // its window in [qc0, qc1)
  const bool wave_live = qhi > qlo;
  const unsigned na = (unsigned)(p.aze - p.azs);
  const float2* base = (const float2*)b.data;
  const const_dptr sat = (const_dptr)b.satloc;
  I32x4 rsrc;   // one record per sample; indices past S - 2 read zeros
  {
    const unsigned long long a = (unsigned long long)b.data;
    rsrc.x = __builtin_amdgcn_readfirstlane((int)(unsigned)a);
    rsrc.y = __builtin_amdgcn_readfirstlane((int)(((unsigned)(a >> 32) & 0xffffu) | (8u << 16)));
    rsrc.z = b.S - 1;
    rsrc.w = kSbufWord3Raw32;
  }

  double ar = 0., ai = 0.;
  for (int p0 = wlo; p0 < whi; p0 += kPlainStage) {
    const int p1 = min(p0 + kPlainStage, whi);
    bool safe = quart;
    for (int q = p0 + tid; quart && q < p1; q += kBlock) {
      const double* s = b.satloc + 3 * q;
      const double u0 = x0[0] - s[0], u1 = x0[1] - s[1], u2 = x0[2] - s[2];
      const double r2 = u0 * u0 + u1 * u1 + u2 * u2;
      const double R0 = range_sqrt(r2), inv = rcp64(R0);
      const double t = fma((double)(q - wlo), dt, -1.0);
      const double dev = fmax(fmax(fabs(quartic(sh->look[0], t) - u0 * inv),
                                   fabs(quartic(sh->look[1], t) - u1 * inv)),
                              fabs(quartic(sh->look[2], t) - u2 * inv));
      PlainRec r;
      r.rb = (R0 - b.rngstart) * b.inv_dmrg;
      cis_cycles(R0 * b.two_over_wvl, &r.tr, &r.ti);
      r.pad = 0.;
      rec[q - p0] = r;
      safe = safe && r.rb - ext >= 0.0 && r.rb + ext <= b.r_hi && dev * dmax <= kPlainTol;
    }
    // The masked pulse of an odd last block: an index past every row reads
    // nothing.
    if (tid == 0) rec[p1 - p0] = PlainRec{-1e9, 0., 0., 0.};
    const int stage_safe = __syncthreads_and(safe ? 1 : 0);
    if (wave_live) {
      int qa = max(p0, qlo), qb = min(p1, qhi);
      if constexpr (STACK == kWavesSplit) split_stage(p0, p1, &qa, &qb);
      if (wave_fit && stage_safe) {
        for (int q = qa; q < qb;) {
          const int ce = min(qb, qc1);
          const bool core = q >= qc0 && q + 1 < ce;
          const int n = core ? min(blk, ce - q) & ~1
                             : min(blk, (q < qc0 ? min(qb, qc0) : qb) - q);
          plain_block(c, dt, wlo, q, n, rec + (q - p0), rsrc, rb32, core, p.azs, na,
                      b.two_over_wvl, b.inv_dmrg, ar, ai);
          q += n;
        }
      } else {
        for (int q = qa; q < qb; ++q) {
          const double sx = sat[3 * q], sy = sat[3 * q + 1], sz = sat[3 * q + 2];
          if ((unsigned)(q - p.azs) < na)
            plain_pair(base + (size_t)q * b.S, x, sx, sy, sz, b, ar, ai);
        }
      }
    }
    __syncthreads();
  }
  // An infinite sample leaves an infinity or NaN in the sum; the pairs' products
  // would make NaN of every infinity, so such a lane's pulses are summed one by
  // one instead.
  const auto infinite = [](double v) { return !(fabs(v) <= 1.79769313486231571e308); };
  const bool redo = live && wave_fit && (infinite(ar) || infinite(ai));
  if (__any(redo ? 1 : 0)) {
    if (redo) ar = ai = 0.;
    for (int p0 = wlo; p0 < whi; p0 += kPlainStage) {
      const int p1 = min(p0 + kPlainStage, whi);
      int qa = max(p0, qlo), qb = min(p1, qhi);
      if constexpr (STACK == kWavesSplit) split_stage(p0, p1, &qa, &qb);
      for (int q = qa; q < qb; ++q) {
        const double sx = sat[3 * q], sy = sat[3 * q + 1], sz = sat[3 * q + 2];
        if (redo && (unsigned)(q - p.azs) < na)
          plain_pair(base + (size_t)q * b.S, x, sx, sy, sz, b, ar, ai);
      }
    }
  }
  if constexpr (STACK == kWavesSplit) {
    if (!split_join((double*)rec, &ar, &ai)) return;
  }
  store_out(b, p, (float)ar, (float)ai);
}

template <int TR, int STACK, int DT, bool LDS = false>
__device__ __forceinline__ void mixed_tile(const BurstDev& b, int tile,
                                           PulseRec* rec, TileShared* sh,
                                           F32x4* sbuf = nullptr) {
  constexpr bool SD = STACK == kWavesSplit;   // PolyPixel
  PixelCtx p = pixel_of<TR, STACK>(b, tile);
  const int tid = threadIdx.x;
  const bool live = p.aze > p.azs;
  double x[3] = {0., 0., 0.};
  if (live) pixel_ecef(b, p.row, p.col, x);

  // Workgroup window and reference pixel (the live pixel nearest the tile
  // centre, ties to the lowest thread).
  constexpr int WR = TileShape<TR, STACK>::WR, WC = TileShape<TR, STACK>::WC;
  const int wr = TileShape<TR, STACK>::row(tid), wc = TileShape<TR, STACK>::col(tid);
  const int key = (abs(2 * wr - WR) + abs(2 * wc - WC)) * 256 + tid;
  if (tid == 0) {
    sh->key = 0x7fffffff;
    sh->wlo = 0x7fffffff;
    sh->whi = -1;
    sh->dmax = 0u;
    sh->pmax = 0u;
    sh->iamin = 0x7fffffff;
    sh->iamax = -0x7fffffff;
    sh->nchain = 0;
  }
  __syncthreads();
  if (live) {
    atomicMin(&sh->key, key);
    atomicMin(&sh->wlo, p.azs);
    atomicMax(&sh->whi, p.aze);
  }
  __syncthreads();
  const int ref = sh->key;
  const int wlo = sh->wlo, whi = sh->whi;
  if (ref == 0x7fffffff) {  // nothing to compute in this tile
    store_out(b, p, 0.f, 0.f);
    return;
  }
  if ((ref & 255) == tid) {
    sh->x0[0] = x[0];
    sh->x0[1] = x[1];
    sh->x0[2] = x[2];
  }
  __syncthreads();
  const double x0[3] = {uniform(sh->x0[0]), uniform(sh->x0[1]), uniform(sh->x0[2])};

  // Unit look vector and range at the window's central pulse.
  const int pc = (wlo + whi - 1) >> 1;
  double uref[3], R0ref;
  {
    const double* s = b.satloc + 3 * pc;
    const double u[3] = {x0[0] - s[0], x0[1] - s[1], x0[2] - s[2]};
    R0ref = uniform(sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
    const double inv = 1.0 / R0ref;
    uref[0] = uniform(u[0] * inv);
    uref[1] = uniform(u[1] * inv);
    uref[2] = uniform(u[2] * inv);
  }

  // Per-pixel constants (lanes without a pixel sit on x0).
  const double d64[3] = {live ? x[0] - x0[0] : 0., live ? x[1] - x0[1] : 0.,
                         live ? x[2] - x0[2] : 0.};
  const double bb64 = d64[0] * d64[0] + d64[1] * d64[1] + d64[2] * d64[2];
  const double aref64 = uref[0] * d64[0] + uref[1] * d64[1] + uref[2] * d64[2];
  if (live) atomicMax(&sh->dmax, __float_as_uint((float)sqrt(bb64)));
  const float Kf = (float)b.two_over_wvl;
  const float invd = (float)b.inv_dmrg;

  // Wave window [qlo, qhi) and core [qc0, qc1) where every live lane of the
  // wave is inside its own window.
  const int qlo = wave_min(live ? p.azs : 0x7fffffff);
  const int qhi = wave_max(live ? p.aze : -1);
  int qc0 = wave_max(live ? p.azs : -1);
  int qc1 = wave_min(live ? p.aze : 0x7fffffff);
  if (qc1 < qc0) qc1 = qc0;
  const bool wave_live = qhi > qlo;
  const unsigned n = (unsigned)(p.aze - p.azs);
  const grow_t base = (grow_t)b.data;
  const I32x4 rsrc = sample_rsrc<DT>(b.data, elem_bytes<DT>());
  const size_t rowbytes = (size_t)b.S * elem_bytes<DT>();
  const unsigned smax = (unsigned)(b.S - 2);

  // The range excess as a quadratic in k = q - pc: interpolated at three
  // Chebyshev nodes of the wave window, checked against the exact excess at
  // the window's two ends.  A wave where a live pixel misses by more than
  // 1e-7 m (0.023 mrad of phase) keeps the FP32 chain.  Lanes without a
  // pixel sit on x0 (excess 0).
  const double arefd64 = aref64 * b.inv_dmrg;
  const int ia = (int)rint(arefd64);
  const double fad = aref64 - ia * b.dmrg;          // fa dmrg, |fa| <= 1/2
  const int ia_min = wave_min(ia);
  PolyPixel pp = {0.f, 0.f, 0.f, (unsigned)(ia - ia_min) * (unsigned)elem_bytes<DT>(), 0.f};
  bool wave_poly = false;
  if (wave_live && qhi - qlo >= 16 && !b.chain) {
    const double mid = 0.5 * (qlo + qhi - 1), hh = 0.5 * (qhi - 1 - qlo);
    const int n0 = (int)rint(mid - 0.8660254037844386 * hh);
    const int n1 = (int)rint(mid);
    const int n2 = (int)rint(mid + 0.8660254037844386 * hh);
    // Lane j < 5 forms the look vector of fit pulse j (nodes, then the
    // window's ends); every lane reads them back.
    const int lane = tid & 63;
    double gu0 = 0., gu1 = 0., gu2 = 0., gh = 0.;
    if (lane < 5) {
      const int qn = lane == 0 ? n0 : lane == 1 ? n1 : lane == 2 ? n2 : lane == 3 ? qlo : qhi - 1;
      const double* sq = b.satloc + 3 * qn;
      const double v0 = x0[0] - sq[0], v1 = x0[1] - sq[1], v2 = x0[2] - sq[2];
      const double inv = rsqrt64(v0 * v0 + v1 * v1 + v2 * v2);
      gu0 = v0 * inv;
      gu1 = v1 * inv;
      gu2 = v2 * inv;
      gh = 0.5 * inv;
    }
    double y[5];
#pragma unroll
    for (int j = 0; j < 5; ++j)
      y[j] = node_excess(lane_double(gu0, j), lane_double(gu1, j), lane_double(gu2, j),
                         lane_double(gh, j), d64, bb64, aref64);
    const double k0 = n0 - pc, k1 = n1 - pc, k2 = n2 - pc;
    const double a1 = (y[1] - y[0]) / (k1 - k0);
    const double a2 = ((y[2] - y[1]) / (k2 - k1) - a1) / (k2 - k0);
    const double c2 = a2, c1 = a1 - a2 * (k0 + k1), c0 = y[0] - k0 * (a1 - a2 * k1);
    const double kl = qlo - pc, kh = qhi - 1 - pc;
    const double el = fabs((c2 * kl + c1) * kl + c0 - y[3]);
    const double eh = fabs((c2 * kh + c1) * kh + c0 - y[4]);
    // |R_q(x) - R_q(x0)| <= |d| for any pulse position, so |sd| <= 2 |d|;
    // the quadratic must keep that bound over the whole window (ends and
    // vertex), which also bounds every index it can produce.
    double pm = fmax(fabs((c2 * kl + c1) * kl + c0),
                     fabs((c2 * kh + c1) * kh + c0));
    const double kv = c2 != 0.0 ? -c1 / (2.0 * c2) : kl;
    if (kv > kl && kv < kh) pm = fmax(pm, fabs((c2 * kv + c1) * kv + c0));
    const bool ok = el <= 1e-7 && eh <= 1e-7 &&   // false for NaN
                    pm <= 2.0 * sqrt(bb64) + 1e-3 &&
                    (size_t)b.L * rowbytes + (size_t)kSbufBias < (size_t)0x7fffffff;
    wave_poly = wave_min(ok ? 1 : 0) == 1;
    if (wave_poly && live) atomicMax(&sh->pmax, __float_as_uint((float)(pm * (1.0 + 1e-6))));
    pp.c0 = (float)(SD ? c0 : c0 + fad);
    pp.fa = (float)(arefd64 - ia);
    pp.c1 = (float)c1;
    pp.c2 = (float)c2;
  }
  // Per-pixel constants of the FP32 chain (waves without the quadratic).
  MixedPixel m = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (!wave_poly) {
    const double q = aref64 / R0ref;
    const double w64 = 1.0 - q + q * q;
    m.dx = (float)d64[0];
    m.dy = (float)d64[1];
    m.dz = (float)d64[2];
    m.t0 = (float)(w64 * (bb64 - aref64 * aref64));
    m.t1 = (float)(2.0 * w64 * aref64);
    m.arefd = (float)(aref64 * b.inv_dmrg);
    m.w = (float)w64;
  }
  // Phase taken out at the end: frac(2/lambda aref), less Kf fa dmrg on the
  // quadratic, whose cycles Kf P carry it.
  const double cp64 = aref64 * b.two_over_wvl - (wave_poly && !SD ? (double)Kf * fad : 0.0);
  const float cpix = (float)(cp64 - rint(cp64));
  if constexpr (LDS) {
    atomicMin(&sh->iamin, ia);
    atomicMax(&sh->iamax, ia);
    if (wave_live && !wave_poly && (tid & 63) == 0) atomicAdd(&sh->nchain, 1);
  }
  __syncthreads();
  // max |x - x0| over the live pixels of the tile.
  const double dmax =
      (double)__uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)sh->dmax));
  // Bound on |P| of every quadratic in use: |sd| <= pmx, |fa dmrg| <= dmrg/2.
  const double pmx =
      (double)__uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)sh->pmax)) + 1e-6;

  // Sample base of the quadratic form for the tile: 64 + pmx/dmrg samples
  // below the range of x0 at the central pulse, so f0s = rb - i0s stays >= 1
  // + pmx/dmrg + 1/2 unless the range walks by more than 62 samples over the
  // window (each pulse checks it below).
  const int i0s = __builtin_amdgcn_readfirstlane(
      (int)floor((R0ref - b.rngstart) * b.inv_dmrg) - 64 - (int)fmin(pmx * b.inv_dmrg, 4096.0));
  // Range extent of the tile about x0 in samples: R - R0 in [-dmax, dmax +
  // dmax^2/(2(R0 - dmax))], the latter <= dmax^2/R0ref for R0 >= R0ref/2 +
  // dmax (checked per pulse); one sample of margin each side.
  // LDS staging (LDS variants): every live wave on the quadratic and the
  // tile's sample window -- the lanes' whole-sample offsets plus the
  // quadratics' excursion both ways plus margins -- within kLdsWindow.
  bool lds_ok = false;
  int ia_min_wg = 0;
  if constexpr (LDS) {
    ia_min_wg = __builtin_amdgcn_readfirstlane(sh->iamin);
    const int ia_max_wg = __builtin_amdgcn_readfirstlane(sh->iamax);
    const int nchain = __builtin_amdgcn_readfirstlane(sh->nchain);
    const double ex = pmx * b.inv_dmrg;
    lds_ok = nchain == 0 && ex < 512.0 &&
             (ia_max_wg - ia_min_wg) + 2 * (int)ceil(ex) + 6 <= kLdsWindow;
  }
  const int laneoffs = ia - ia_min_wg;
  const double ext_lo = dmax * b.inv_dmrg + 1.0;
  const double ext_hi = (dmax + dmax * dmax / R0ref) * b.inv_dmrg + 1.0;
  const double r0min = 0.5 * R0ref + dmax;
  const double mq = (dmax + pmx + 1e-3) * b.inv_dmrg;

  float acc_r = 0.f, acc_i = 0.f, cmp_r = 0.f, cmp_i = 0.f;
  for (int p0 = wlo; p0 < whi; p0 += kStage) {
    // Stage prologue (FP64): one pulse per thread.
    const int qs = p0 + tid;
    bool safe_all = true, uni = true;
    // The scale of the stage's first pulse; the stage is "uniform" when every
    // pulse carries it (the pack's common scale), and then the scale is
    // applied to the stage sums rather than to each pair.
    const float sc0 = (DT == TDBP_CF32 || b.scale == nullptr) ? 1.f : b.scale[p0];
    if (qs < whi) {
      const double* s = b.satloc + 3 * qs;
      const double u0 = x0[0] - s[0], u1 = x0[1] - s[1], u2 = x0[2] - s[2];
      const double r2 = u0 * u0 + u1 * u1 + u2 * u2;
      const double inv = rsqrt64(r2);
      const double R0 = r2 * inv;
      const double c = R0 * b.two_over_wvl;
      const double rb = (R0 - b.rngstart) * b.inv_dmrg;
      const double i0 = floor(rb);
      const double rlo = rb - ext_lo;
      const double rhi = rb + ext_hi;
      const double du0 = u0 * inv - uref[0], du1 = u1 * inv - uref[1],
                   du2 = u2 * inv - uref[2];
      // Quadratic form: |P| <= pmx + dmrg/2 and |ia| <= dmax/dmrg + 1/2, so
      // the local index P/dmrg + f0s is >= 1 and the sample index i0s + ia +
      // floor(rho) (and its neighbour) lies in [0, S - 1] when these hold.
      const double f0s = rb - i0s;
      const bool safe = R0 >= r0min && rlo >= 1.0 && rhi <= b.r_hi - 1.0 &&
                        f0s - pmx * b.inv_dmrg - 1.5 >= 0.0 && f0s <= 1024.0 &&
                        rb - mq - 3.0 >= 0.0 && rb + mq + 3.0 <= b.S - 1;
      PulseRec r;
      const float cf = (float)(c - rint(c));
      r.r0 = make_float4((float)du0, (float)du1, (float)du2, cf);
      const float sc = (DT == TDBP_CF32 || b.scale == nullptr) ? 1.f : b.scale[qs];
      r.r1 = make_float4((float)(rb - i0), __int_as_float((int)i0 * elem_bytes<DT>()),
                         (float)(0.5 * inv), sc);
      r.r2 = make_float4(safe ? 1.f : 0.f, (float)(b.r_hi - i0), __int_as_float((int)i0), 0.f);
      r.r3 = make_float4((float)(qs - pc), (float)f0s, cf, sc);
      if (LDS && lds_ok) {
        // Staged window of this pulse: from i0s + ia_min + bq, bq = floor(f0s -
        // pmx/dmrg - 1/2) - 1, so a lane's local index P/dmrg + F, F = f0s - bq,
        // is >= 1 and its pair ends below (ia_max - ia_min) + 2 pmx/dmrg + 5.
        const int bq = (int)floor(f0s - pmx * b.inv_dmrg - 0.5) - 1;
        r.r1.y = __int_as_float(i0s + ia_min_wg + bq);
        r.r2.w = (float)(f0s - bq);
      }
      rec[tid] = r;
      safe_all = safe;
      uni = sc == sc0;
    }
    // Barrier that also tells whether every pulse of the stage is safe.
    const int stage_safe = __syncthreads_and(safe_all ? 1 : 0);
    const bool stage_uni = DT == TDBP_CF32 || b.scale == nullptr ||
                           __syncthreads_and(uni ? 1 : 0) != 0;
    float sr = 0.f, si = 0.f;
    if (LDS && lds_ok && stage_safe) {
      // Every wave stages and meets the barriers; only live waves sum.
      const int qa = wave_live ? max(p0, qlo) : 0, qb = wave_live ? min(p0 + kStage, qhi) : 0;
      staged_stage<DT>(b, pp, rec, sbuf, p0, min(p0 + kStage, whi), qa, qb, qc0, qc1,
                       wave_live, DT != TDBP_CF32 && !stage_uni, laneoffs,
                       sample_rsrc<DT, true>(b.data, elem_bytes<DT>()), rowbytes, Kf, invd,
                       p.azs, n, sr, si);
    } else if (wave_live) {
      // A wave without a live pixel skips the pulse loops (its window bounds
      // are sentinels and must not enter index arithmetic).
      int qa = max(p0, qlo), qb = min(p0 + kStage, qhi);
      if constexpr (STACK == kWavesSplit) split_stage(p0, min(p0 + kStage, whi), &qa, &qb);
      if (wave_poly)
        stage_pulses<DT, true, SD>(m, pp, rec, p0, qa, qb, qc0, qc1, stage_safe != 0, stage_uni,
                               base, rsrc,
                               rowbytes, (long)(i0s + ia_min) * elem_bytes<DT>(), i0s + ia,
                               (float)(b.r_hi - i0s - ia), Kf, invd, p.azs, n, smax, sr, si);
      else
        stage_pulses<DT, false, SD>(m, pp, rec, p0, qa, qb, qc0, qc1, stage_safe != 0, false,
                                base, rsrc,
                                rowbytes, 0, 0, 0.f, Kf, invd, p.azs, n, smax, sr, si);
    }
    // A uniform stage summed the quadratic form's pairs unscaled.
    if (DT != TDBP_CF32 && stage_uni && wave_poly) {
      sr *= sc0;
      si *= sc0;
    }
    // Kahan-compensated join of the stage sums.
    {
      const float yr = sr - cmp_r, tr = acc_r + yr;
      cmp_r = (tr - acc_r) - yr;
      acc_r = tr;
      const float yi = si - cmp_i, ti = acc_i + yi;
      cmp_i = (ti - acc_i) - yi;
      acc_i = ti;
    }
    __syncthreads();
  }
  // The per-pixel phase offset frac(2/lambda u_ref.d) is common to all
  // pulses: apply it once.
  float ps, pcs;
  sincospif(2.0f * cpix, &ps, &pcs);
  float fr_ = acc_r - cmp_r, fi_ = acc_i - cmp_i;
  if constexpr (STACK == kWavesSplit) {
    if (!split_join((float*)rec, &fr_, &fi_)) return;
  }
  store_out(b, p, fr_ * pcs - fi_ * ps, fr_ * ps + fi_ * pcs);
}

// ------------------------------------- mixed precision on the matrix cores
//
// The same pair arithmetic as mixed_tile, with the range chain on MFMA.  With
// da = du.d, the range index and phase of a pixel-pulse pair are
//   sd  = da + r1z t0 - r1z t1 da - r1z w da^2          (R - R0 - aref)
//   rho = f0 + arefd + sd/dmrg,      cyc = c0 + (2/lambda) sd
// -- linear forms in per-pixel features F (d_i, t0, t1 d_i, w d_i d_j, 1,
// arefd) and per-pulse weights G (du_i, r1z, -r1z du_i, -r1z du_i du_j, f0 or
// c0, 1).  Every product F G is carried by f16 pieces after a per-tile
// power-of-two balance that puts both factors near sqrt(|F G|): first-order
// terms as Fh Gh + Fh Gl + Fl Gh, the second-order ones as Fh Gh, arefd in
// three pieces.  The products are exact in the FP32 accumulator of
// v_mfma_f32_16x16x32_f16, so one MFMA per output covers 16 pulses x 16 pixels
// (K = 32 slots; rho uses 26, cyc 23, the pixel side is shared).  On an IW
// tile against FP64: rho 7.5e-7 samples RMS, cyc 6.8e-7 rad RMS, the FP32
// chain's accuracy.  Per pair the VALU keeps only the index, the gather, the
// lerp, sin/cos and the MAC.
//
// Workgroup: 16 waves, wave w on row w of a 16 x 16 pixel tile.  Lane
// l = 16 kg + n holds column n and, in each 16-pulse step, pulses 4 kg + v
// (v = 0..3) -- the MFMA's output layout -- so it has four gathers in flight.

constexpr int kMBlock = 512;    // 8 waves, two tile rows each
constexpr int kMStage = 256;    // pulses per stage
constexpr int kMRowA = 72;      // halves per pulse row in LDS: 64 used; 144 B keeps
                                // rows 16-byte aligned and, being an odd number of
                                // 16-byte units, spreads a quarter-wave's 16-byte
                                // reads over all banks
constexpr int kMRowB = 40;      // halves per pixel row in LDS (32 used, padded)

typedef _Float16 h8m __attribute__((ext_vector_type(8)));
typedef float f4m __attribute__((ext_vector_type(4)));

struct MShared {
  union {
    struct {
      _Float16 pf[256][kMRowB];       // pixel features
      int2 win[256];                  // pixel pulse window [azs, aze), empty if not live
    } tl;                             // tile set-up (read into registers before stage 0)
    struct {
      _Float16 aw[kMStage][kMRowA];   // pulse weights: rho slots 0-31, cyc 32-63
      unsigned rowoff[kMStage];       // (q S + i0) * elem: byte offset of sample i0 of row q
      float sc[kMStage];              // per-pulse sample scale
      int i0[kMStage];
    } st;
    float2 part[4][256];              // per-quarter pixel sums (tile end)
  } u;
  double x0[3];
  double uref[3], R0ref, U;           // tile-uniform, computed once by thread 0
  double fsc[4], kr[4], kc[4];        // term scales (F side) and weight constants
  int key, wlo, whi;
  unsigned dmax;
};

// f16 pieces are made with v_cvt_pkrtz_f16_f32 (two floats -> two halves,
// round toward zero, one instruction).  A split x = h + l keeps l = x - h
// exactly in FP32, so the truncation only moves error into l.
__device__ __forceinline__ unsigned mpk(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(a, b));
}
__device__ __forceinline__ float mhi(float x) {   // x truncated to f16, as float
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return (float)__builtin_bit_cast(h2, mpk(x, 0.f)).x;
}

// Exponent e of the power of two 2^e that balances a product: mF 2^e ~ mG
// 2^-e (within a factor of 2: only magnitudes matter).
__device__ __forceinline__ int mbalance(double mF, double mG) {
  return (ilogb(fmax(mG, 1e-300)) - ilogb(fmax(mF, 1e-300))) / 2;
}

// F-side scales of the four term families (the G side takes their inverses).
struct MScale {
  double da, t0, t1, q;
};

// K-slot layout (32 slots = 16 words, pixel side F / pulse side G):
//   0-7   first-order terms T = da_x, da_y, da_z, t0: F (Fh, Fh), G (Gh, Gl)
//   8-11  the same terms:                               F Fl,       G Gh
//   12-14 t1 d_i r1z du_i                               F Fh,       G Gh
//   15-20 w d_i d_j r1z du_i du_j (xx yy zz xy xz yz)   F Fh,       G Gh
//   21-22 f0 (rho) or c0 (cyc):                         F 1, 1,     G Gh, Gl
//   23-25 arefd (rho only):                             F Fh Fm Fl, G 1, 1, 1 (cyc 0)
//   26-31 zero
__device__ __forceinline__ void mfma_pixel_features(const double* d, double t0, double t1,
                                                    double w, double arefd, const MScale& s,
                                                    unsigned* f) {
  const float x[4] = {(float)(d[0] * s.da), (float)(d[1] * s.da), (float)(d[2] * s.da),
                      (float)(t0 * s.t0)};
  float lo[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float h = mhi(x[t]);
    lo[t] = x[t] - h;
    f[t] = mpk(x[t], x[t]);
  }
  f[4] = mpk(lo[0], lo[1]);
  f[5] = mpk(lo[2], lo[3]);
  const double t1s = t1 * s.t1, ws = w * s.q;
  f[6] = mpk((float)(t1s * d[0]), (float)(t1s * d[1]));
  f[7] = mpk((float)(t1s * d[2]), (float)(ws * d[0] * d[0]));
  f[8] = mpk((float)(ws * d[1] * d[1]), (float)(ws * d[2] * d[2]));
  f[9] = mpk((float)(ws * d[0] * d[1]), (float)(ws * d[0] * d[2]));
  f[10] = mpk((float)(ws * d[1] * d[2]), 1.f);
  // arefd in three pieces from FP64 (it needs ~1e-6 sample of ~60)
  const float ah = mhi((float)arefd);
  const double ar = arefd - (double)ah;
  const float am = mhi((float)ar);
  f[11] = mpk(1.f, ah);
  f[12] = mpk(am, (float)(ar - (double)am));
  f[13] = 0u;
  f[14] = 0u;
  f[15] = 0u;
}

// Weights of one output: k = c / scale per term family (c = 1/dmrg for rho,
// 2/lambda for cyc), each formed in FP64 and rounded once to FP32 (2^-24,
// below the 2^-22 the split keeps).
struct MWeightK {
  double da, t0, t1, q;
};
__device__ __forceinline__ void mfma_pulse_weights(const double* du, double r1z, double k0,
                                                   const MWeightK& k, bool rho,
                                                   unsigned* g) {
  const float x[4] = {(float)(du[0] * k.da), (float)(du[1] * k.da), (float)(du[2] * k.da),
                      (float)(r1z * k.t0)};
#pragma unroll
  for (int t = 0; t < 4; ++t) g[t] = mpk(x[t], x[t] - mhi(x[t]));
  g[4] = mpk(x[0], x[1]);
  g[5] = mpk(x[2], x[3]);
  const double r1 = -r1z * k.t1, rq = -r1z * k.q;
  g[6] = mpk((float)(r1 * du[0]), (float)(r1 * du[1]));
  g[7] = mpk((float)(r1 * du[2]), (float)(rq * du[0] * du[0]));
  g[8] = mpk((float)(rq * du[1] * du[1]), (float)(rq * du[2] * du[2]));
  g[9] = mpk((float)(2.0 * rq * du[0] * du[1]), (float)(2.0 * rq * du[0] * du[2]));
  const float kf = (float)k0;
  g[10] = mpk((float)(2.0 * rq * du[1] * du[2]), kf);
  const float one = rho ? 1.f : 0.f;
  g[11] = mpk(kf - mhi(kf), one);
  g[12] = mpk(one, one);
  g[13] = 0u;
  g[14] = 0u;
  g[15] = 0u;
}

template <int DT>
__device__ __forceinline__ void mfma_tile(const BurstDev& b, int tile, MShared& sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, kg = lane >> 4;
  const bool owner = tid < 256;   // owns tile pixel tid (row tid/16, column tid%16)

  PixelCtx p;
  p.inwin = false;
  p.computed = false;
  p.azs = p.aze = 0;
  p.row = p.col = 0;
  double x[3] = {0., 0., 0.};
  bool live = false;
  if (owner) {
    p = pixel_of<4, kWavesStacked>(b, tile);   // 16 x 16 tile: row tid/16, column tid%16
    live = p.aze > p.azs;
    if (live) pixel_ecef(b, p.row, p.col, x);
  }
  if (tid == 0) {
    sh.key = 0x7fffffff;
    sh.wlo = 0x7fffffff;
    sh.whi = -1;
    sh.dmax = 0u;
  }
  __syncthreads();
  if (live) {
    const int wr = tid >> 4, wc = tid & 15;
    const int key = (abs(2 * wr - 16) + abs(2 * wc - 16)) * 1024 + tid;
    atomicMin(&sh.key, key);
    atomicMin(&sh.wlo, p.azs);
    atomicMax(&sh.whi, p.aze);
  }
  if (owner) sh.u.tl.win[tid] = live ? make_int2(p.azs, p.aze) : make_int2(0, 0);
  __syncthreads();
  const int ref = sh.key;
  const int wlo = sh.wlo, whi = sh.whi;
  if (ref == 0x7fffffff) {
    if (owner) store_out(b, p, 0.f, 0.f);
    return;
  }
  if ((ref & 1023) == tid) {
    sh.x0[0] = x[0];
    sh.x0[1] = x[1];
    sh.x0[2] = x[2];
  }
  __syncthreads();
  const double x0[3] = {uniform(sh.x0[0]), uniform(sh.x0[1]), uniform(sh.x0[2])};

  // Tile-uniform set-up, once (thread 0): look vector and range at the
  // window's central pulse, |du| at the window's ends.
  if (tid == 0) {
    const int pc = (wlo + whi - 1) >> 1;
    const double* sp = b.satloc + 3 * pc;
    const double u[3] = {x0[0] - sp[0], x0[1] - sp[1], x0[2] - sp[2]};
    const double R = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double inv = 1.0 / R;
    // |du| over the window ~ half the track span over the range (a
    // magnitude for the balance only).
    const double* sl = b.satloc + 3 * wlo;
    const double* sh_ = b.satloc + 3 * (whi - 1);
    const double span = fmax(fmax(fabs(sh_[0] - sl[0]), fabs(sh_[1] - sl[1])), fabs(sh_[2] - sl[2]));
    for (int i = 0; i < 3; ++i) sh.uref[i] = u[i] * inv;
    sh.R0ref = R;
    sh.U = fmax(0.5 * span * inv, 1e-12);
  }
  __syncthreads();
  const double uref[3] = {uniform(sh.uref[0]), uniform(sh.uref[1]), uniform(sh.uref[2])};
  const double R0ref = uniform(sh.R0ref);

  // Per-pixel constants (FP64), tile radius.
  double d64[3] = {0., 0., 0.};
  double t0 = 0., t1 = 0., w64 = 1., arefd = 0.;
  float cpix = 0.f;
  if (owner) {
    if (live) {
      d64[0] = x[0] - x0[0];
      d64[1] = x[1] - x0[1];
      d64[2] = x[2] - x0[2];
    }
    const double bb = d64[0] * d64[0] + d64[1] * d64[1] + d64[2] * d64[2];
    const double aref = uref[0] * d64[0] + uref[1] * d64[1] + uref[2] * d64[2];
    const double q = aref / R0ref;
    w64 = 1.0 - q + q * q;
    t0 = w64 * (bb - aref * aref);
    t1 = 2.0 * w64 * aref;
    arefd = aref * b.inv_dmrg;
    const double cp = aref * b.two_over_wvl;
    cpix = (float)(cp - rint(cp));
    if (live) atomicMax(&sh.dmax, __float_as_uint((float)sqrt(bb)));
  }
  __syncthreads();
  const double dmax =
      (double)__uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)sh.dmax));
  // Balance of the four term families for both outputs at once (geometric
  // mean of 1/dmrg and 2/lambda): the pixel side is shared by the two MFMAs.
  // Thread 0 computes the scales and the weight constants (c over the scale).
  if (tid == 0) {
    const double D = fmax(dmax, 1.0), U = sh.U;
    const double cg = sqrt(b.inv_dmrg * b.two_over_wvl);
    const double rz = 0.5 / R0ref;
    const int e[4] = {mbalance(D, U * cg), mbalance(D * D, cg * rz),
                      mbalance(2.0 * D * D, U * cg * rz),
                      mbalance(D * D, 2.0 * U * U * cg * rz)};
    for (int i = 0; i < 4; ++i) {
      sh.fsc[i] = ldexp(1.0, e[i]);
      sh.kr[i] = ldexp(b.inv_dmrg, -e[i]);
      sh.kc[i] = ldexp(b.two_over_wvl, -e[i]);
    }
  }
  __syncthreads();
  const MScale sc = {uniform(sh.fsc[0]), uniform(sh.fsc[1]), uniform(sh.fsc[2]),
                     uniform(sh.fsc[3])};
  const MWeightK kr = {uniform(sh.kr[0]), uniform(sh.kr[1]), uniform(sh.kr[2]),
                       uniform(sh.kr[3])};
  const MWeightK kc = {uniform(sh.kc[0]), uniform(sh.kc[1]), uniform(sh.kc[2]),
                       uniform(sh.kc[3])};
  if (owner) {
    unsigned f[16];
    mfma_pixel_features(d64, t0, t1, w64, arefd, sc, f);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      *(uint4*)&sh.u.tl.pf[tid][8 * k] = make_uint4(f[4 * k], f[4 * k + 1], f[4 * k + 2],
                                                 f[4 * k + 3]);
  }
  __syncthreads();
  // This lane's pixels: column n of rows 2 wave and 2 wave + 1.
  const int px0 = (2 * wave) * 16 + n, px1 = px0 + 16;
  const h8m bf0 = *(const h8m*)&sh.u.tl.pf[px0][8 * kg];
  const h8m bf1 = *(const h8m*)&sh.u.tl.pf[px1][8 * kg];
  const int2 wn0 = sh.u.tl.win[px0], wn1 = sh.u.tl.win[px1];
  const bool lv0 = wn0.y > wn0.x, lv1 = wn1.y > wn1.x;
  const int qlo = wave_min(min(lv0 ? wn0.x : 0x7fffffff, lv1 ? wn1.x : 0x7fffffff));
  const int qhi = wave_max(max(lv0 ? wn0.y : -1, lv1 ? wn1.y : -1));
  const int qc0 = wave_max(max(lv0 ? wn0.x : -1, lv1 ? wn1.x : -1));
  const int qc1 = wave_min(min(lv0 ? wn0.y : 0x7fffffff, lv1 ? wn1.y : 0x7fffffff));
  const bool wave_live = qhi > qlo;
  const grow_t base = (grow_t)b.data;
  const unsigned smax = (unsigned)(b.S - 2);
  const unsigned elem = (unsigned)elem_bytes<DT>();
  const double r_hi = b.r_hi;
  __syncthreads();   // the stage tables reuse the pixel-feature rows

  float acc_r[2] = {0.f, 0.f}, acc_i[2] = {0.f, 0.f}, cmp_r[2] = {0.f, 0.f},
        cmp_i[2] = {0.f, 0.f};
  for (int p0 = wlo; p0 < whi; p0 += kMStage) {
    // Stage prologue: thread t builds output t >> 8 (0 rho, 1 cyc) of pulse
    // t & 255 (FP64 geometry, FP32-rounded weights); the rho threads also
    // write the pulse's scalars and range-gate flag.
    bool safe_all = true;
    {
      const int j = tid & (kMStage - 1);
      const bool is_rho = tid < kMStage;
      const int qs = p0 + j;
      unsigned g[16];
      if (qs < whi) {
        const double* sp = b.satloc + 3 * qs;
        const double u0 = x0[0] - sp[0], u1 = x0[1] - sp[1], u2 = x0[2] - sp[2];
        const double R0 = sqrt(u0 * u0 + u1 * u1 + u2 * u2);
        const double inv = 1.0 / R0;
        const double du[3] = {u0 * inv - uref[0], u1 * inv - uref[1], u2 * inv - uref[2]};
        const double rb = (R0 - b.rngstart) * b.inv_dmrg;
        const double i0 = floor(rb);
        if (is_rho) {
          mfma_pulse_weights(du, 0.5 * inv, rb - i0, kr, true, g);
          const double rlo = rb - dmax * b.inv_dmrg - 1.0;
          const double rhi =
              rb + (dmax + dmax * dmax / (2.0 * (R0 - dmax))) * b.inv_dmrg + 1.0;
          safe_all = rlo >= 1.0 && rhi <= b.r_hi - 1.0;
          sh.u.st.rowoff[j] = (unsigned)(((size_t)qs * (size_t)b.S + (size_t)(long)i0) * elem);
          sh.u.st.sc[j] = (DT == TDBP_CF32 || b.scale == nullptr) ? 1.f : b.scale[qs];
          sh.u.st.i0[j] = (int)i0;
        } else {
          const double c = R0 * b.two_over_wvl;
          mfma_pulse_weights(du, 0.5 * inv, c - rint(c), kc, false, g);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) g[k] = 0u;
        if (is_rho) {
          sh.u.st.rowoff[j] = 0u;
          sh.u.st.sc[j] = 0.f;
          sh.u.st.i0[j] = -0x40000000;   // fails the gate test
        }
      }
      const int col = is_rho ? 0 : 32;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *(uint4*)&sh.u.st.aw[j][col + 8 * k] =
            make_uint4(g[4 * k], g[4 * k + 1], g[4 * k + 2], g[4 * k + 3]);
    }
    const int stage_safe = __syncthreads_and(safe_all ? 1 : 0);
    float sr[2] = {0.f, 0.f}, si[2] = {0.f, 0.f};
    if (wave_live) {
      const int qa = max(p0, qlo), qb = min(p0 + kMStage, qhi);
      for (int s0 = ((qa - p0) >> 4) << 4; p0 + s0 < qb; s0 += 16) {
        const int q0 = p0 + s0;
        const h8m ar = *(const h8m*)&sh.u.st.aw[s0 + n][8 * kg];
        const h8m ac = *(const h8m*)&sh.u.st.aw[s0 + n][32 + 8 * kg];
        const uint4 ro = *(const uint4*)&sh.u.st.rowoff[s0 + 4 * kg];
        const float4 s4 = *(const float4*)&sh.u.st.sc[s0 + 4 * kg];
        const unsigned rov[4] = {ro.x, ro.y, ro.z, ro.w};
        const float scv[4] = {s4.x, s4.y, s4.z, s4.w};
        const f4m z = {0.f, 0.f, 0.f, 0.f};
        const bool core = stage_safe && q0 >= qc0 && q0 + 16 <= qc1;
        int4 i4 = make_int4(0, 0, 0, 0);
        if (!core) i4 = *(const int4*)&sh.u.st.i0[s0 + 4 * kg];
        const int i0v[4] = {i4.x, i4.y, i4.z, i4.w};
        // Both groups' products first: the second pair of MFMAs runs while
        // the first group's pairs are finished on the VALU.
        const f4m drg[2] = {__builtin_amdgcn_mfma_f32_16x16x32_f16(ar, bf0, z, 0, 0, 0),
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(ar, bf1, z, 0, 0, 0)};
        const f4m dcg[2] = {__builtin_amdgcn_mfma_f32_16x16x32_f16(ac, bf0, z, 0, 0, 0),
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(ac, bf1, z, 0, 0, 0)};
        if (core) {
          // Every live lane of the wave is inside its windows for the whole
          // step and the whole tile inside the range gate: no tests.  All
          // eight gathers are issued before the first is used.
          typename RawPair<DT>::type v[2][4];
          float fr[2][4];
#pragma unroll
          for (int gi = 0; gi < 2; ++gi)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              // floor(rho) in one instruction.  The asm takes fr as an input
              // so it runs after fract, whose read of the MFMA result the
              // compiler sees and guards with the MFMA-to-VALU wait states.
              fr[gi][j] = __builtin_amdgcn_fractf(drg[gi][j]);
              int il;
              asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(il) : "v"(drg[gi][j]), "v"(fr[gi][j]));
              v[gi][j] =
                  gload<typename RawPair<DT>::type>(base + ((unsigned)il * elem + rov[j]));
            }
#pragma unroll
          for (int gi = 0; gi < 2; ++gi)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float2 c = lerp_raw<DT>(v[gi][j], fr[gi][j], scv[j]);
              const float sn = __builtin_amdgcn_sinf(dcg[gi][j]),
                          cs = __builtin_amdgcn_cosf(dcg[gi][j]);
              sr[gi] = fmaf(c.x, cs, sr[gi]);
              sr[gi] = fmaf(-c.y, sn, sr[gi]);
              si[gi] = fmaf(c.x, sn, si[gi]);
              si[gi] = fmaf(c.y, cs, si[gi]);
            }
        } else {
#pragma unroll
          for (int gi = 0; gi < 2; ++gi) {
            const f4m dr = drg[gi], dc = dcg[gi];
            const int2 wn = gi ? wn1 : wn0;
            const unsigned nwin = (unsigned)(wn.y - wn.x);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int q = q0 + 4 * kg + j;
              const float rho = dr[j];
              const int il = (int)floorf(rho);
              // gate: window, sample index in [0, S-2], r <= r_hi
              if ((unsigned)(q - wn.x) < nwin && (unsigned)(il + i0v[j]) <= smax &&
                  rho <= (float)(r_hi - (double)i0v[j])) {
                const typename RawPair<DT>::type vv =
                    gload<typename RawPair<DT>::type>(base + ((unsigned)il * elem + rov[j]));
                const float2 c = lerp_raw<DT>(vv, __builtin_amdgcn_fractf(rho), scv[j]);
                const float sn = __builtin_amdgcn_sinf(dc[j]),
                            cs = __builtin_amdgcn_cosf(dc[j]);
                sr[gi] = fmaf(c.x, cs, sr[gi]);
                sr[gi] = fmaf(-c.y, sn, sr[gi]);
                si[gi] = fmaf(c.x, sn, si[gi]);
                si[gi] = fmaf(c.y, cs, si[gi]);
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      const float yr = sr[gi] - cmp_r[gi], tr = acc_r[gi] + yr;
      cmp_r[gi] = (tr - acc_r[gi]) - yr;
      acc_r[gi] = tr;
      const float yi = si[gi] - cmp_i[gi], ti = acc_i[gi] + yi;
      cmp_i[gi] = (ti - acc_i[gi]) - yi;
      acc_i[gi] = ti;
    }
    __syncthreads();
  }
  // Quarter sums per pixel, joined by the pixel's owner, then the per-pixel
  // phase offset frac(2/lambda u_ref.d).
  sh.u.part[kg][px0] = make_float2(acc_r[0] - cmp_r[0], acc_i[0] - cmp_i[0]);
  sh.u.part[kg][px1] = make_float2(acc_r[1] - cmp_r[1], acc_i[1] - cmp_i[1]);
  __syncthreads();
  if (owner) {
    float fr_ = 0.f, fi_ = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      fr_ += sh.u.part[k][tid].x;
      fi_ += sh.u.part[k][tid].y;
    }
    float ps, pcs;
    sincospif(2.0f * cpix, &ps, &pcs);
    store_out(b, p, fr_ * pcs - fi_ * ps, fr_ * ps + fi_ * pcs);
  }
}

// ----------------------------------------------------------- kernels

// Occupancy target of the FP64 kernels: 3 waves per SIMD leave 168 VGPRs, which
// hold a block's recurrences without spills; the loads run a pair ahead, and
// the kernel keeps VALU busy 92 % of its cycles (one IW burst: 3.15 ms at 3,
// 3.2 at 4 with spills outside the loops, 3.9 at 5).
#define TDBP_PLAIN_OCC __attribute__((amdgpu_waves_per_eu(3)))

template <int TR, int STACK, bool CPU>
__global__ __launch_bounds__(kBlock) TDBP_PLAIN_OCC void k_plain(BurstDev b) {
  __shared__ int item;
  if constexpr (CPU) {
    persistent_tiles(b, &item, [&](int tile) { cpu_tile<TR, STACK>(b, tile); });
  } else {
    __shared__ PlainRec rec[kPlainStage + 1];
    __shared__ PlainShared sh;
    persistent_tiles(b, &item,
                     [&](int tile) { plain_excess_tile<TR, STACK>(b, tile, rec, &sh); });
  }
}

// Occupancy target of the mixed kernels: 8 waves per SIMD, the hardware
// maximum (<= 64 VGPRs); the pulse loop is a dependent gather, so resident
// waves hide its latency (measured: 7 -> 8 waves is +9 % on the 27-burst IW scene).
#define TDBP_MIXED_OCC __attribute__((amdgpu_waves_per_eu(8)))
// LDS-staged variants: 16 KB of pulse records and 14 KB of sample windows
// per workgroup leave room for 5 workgroups (5 waves per SIMD) in a CU's
// 160 KB, and 5 waves give each 96 VGPRs.
#define TDBP_LDS_OCC __attribute__((amdgpu_waves_per_eu(5)))

template <int TR, int STACK, int DT>
__global__ __launch_bounds__(kBlock) TDBP_MIXED_OCC void k_mixed(BurstDev b) {
  __shared__ PulseRec rec[kStage];
  __shared__ TileShared sh;
  __shared__ int item;
  persistent_tiles(b, &item, [&](int tile) { mixed_tile<TR, STACK, DT>(b, tile, rec, &sh); });
}

template <int TR, int STACK, int DT>
__global__ __launch_bounds__(kBlock) TDBP_LDS_OCC void k_mixed_lds(BurstDev b) {
  __shared__ PulseRec rec[kStage];
  __shared__ TileShared sh;
  __shared__ int item;
  __shared__ __attribute__((aligned(16))) F32x4 sbuf[kLdsPulses * kLdsWindow / 2];
  persistent_tiles(b, &item,
                   [&](int tile) { mixed_tile<TR, STACK, DT, true>(b, tile, rec, &sh, sbuf); });
}

// MFMA variant of k_mixed (512-thread workgroups, 16 x 16 pixel tiles).
template <int DT>
__global__ __launch_bounds__(kMBlock) TDBP_MIXED_OCC void k_mixed_mfma(BurstDev b) {
  __shared__ MShared sh;
  const int nb = b.tiles_r * b.tiles_c;
  mfma_tile<DT>(b, xcd_tile(blockIdx.x, nb), sh);
}

// Persistent batch kernel on the MFMA tile; same queues as k_batch_mixed.
template <int DT>
__global__ __launch_bounds__(kMBlock) TDBP_MIXED_OCC void k_batch_mfma(
    const BurstDev* __restrict__ bursts, const int2* __restrict__ items,
    const int* __restrict__ qbase, int* counters) {
  __shared__ MShared sh;
  __shared__ int item_s;
  const int home = blockIdx.x & 7;
  int qi = 0;
  while (qi < 8) {
    const int qk = (home + qi) & 7;
    if (threadIdx.x == 0) {
      const int k = atomicAdd(&counters[qk], 1);
      item_s = (k < qbase[qk + 1] - qbase[qk]) ? qbase[qk] + k : -1;
    }
    __syncthreads();
    const int it = item_s;
    __syncthreads();
    if (it < 0) {
      ++qi;
      continue;
    }
    const int2 w = items[it];
    mfma_tile<DT>(bursts[w.x], w.y, sh);
    __syncthreads();
  }
}

// Persistent batch kernel: workgroup on XCD x = blockIdx % 8 drains queue x,
// then steals from the others.  Queue k holds items [qbase[k], qbase[k+1]).
template <int PREC, int TR, int STACK, int DT, bool LDS = false, class REC, class SHARED>
__device__ __forceinline__ void batch_body(const BurstDev* __restrict__ bursts,
                                           const int2* __restrict__ items,
                                           const int* __restrict__ qbase,
                                           int* counters, REC* rec,
                                           SHARED* sh, int* item_s,
                                           F32x4* sbuf = nullptr) {
  const int home = blockIdx.x & 7;
  int qi = 0;
  while (qi < 8) {
    const int qk = (home + qi) & 7;
    if (threadIdx.x == 0) {
      const int k = atomicAdd(&counters[qk], 1);
      *item_s = (k < qbase[qk + 1] - qbase[qk]) ? qbase[qk] + k : -1;
    }
    __syncthreads();
    const int it = *item_s;
    __syncthreads();
    if (it < 0) {
      ++qi;
      continue;
    }
    const int2 w = items[it];
    const BurstDev& bd = bursts[w.x];
    if constexpr (PREC == TDBP_MIXED) {
      mixed_tile<TR, STACK, DT, LDS>(bd, w.y, rec, sh, sbuf);
    } else if (bd.cpu) {
      cpu_tile<TR, STACK>(bd, w.y);
    } else {
      plain_excess_tile<TR, STACK>(bd, w.y, rec, sh);
    }
    __syncthreads();
  }
}

template <int TR, int STACK, int DT>
__global__ __launch_bounds__(kBlock) TDBP_MIXED_OCC void k_batch_mixed(
    const BurstDev* __restrict__ bursts, const int2* __restrict__ items,
    const int* __restrict__ qbase, int* counters) {
  __shared__ PulseRec rec[kStage];
  __shared__ TileShared sh;
  __shared__ int item_s;
  batch_body<TDBP_MIXED, TR, STACK, DT>(bursts, items, qbase, counters, rec, &sh, &item_s);
}

template <int TR, int STACK, int DT>
__global__ __launch_bounds__(kBlock) TDBP_LDS_OCC void k_batch_mixed_lds(
    const BurstDev* __restrict__ bursts, const int2* __restrict__ items,
    const int* __restrict__ qbase, int* counters) {
  __shared__ PulseRec rec[kStage];
  __shared__ TileShared sh;
  __shared__ int item_s;
  __shared__ __attribute__((aligned(16))) F32x4 sbuf[kLdsPulses * kLdsWindow / 2];
  batch_body<TDBP_MIXED, TR, STACK, DT, true>(bursts, items, qbase, counters, rec, &sh,
                                              &item_s, sbuf);
}

template <int TR, int STACK>
__global__ __launch_bounds__(kBlock) TDBP_PLAIN_OCC void k_batch_plain(
    const BurstDev* __restrict__ bursts, const int2* __restrict__ items,
    const int* __restrict__ qbase, int* counters) {
  __shared__ PlainRec rec[kPlainStage + 1];
  __shared__ PlainShared sh;
  __shared__ int item_s;
  batch_body<TDBP_PLAIN_FP64, TR, STACK, TDBP_CF32>(bursts, items, qbase, counters, rec, &sh,
                                                     &item_s);
}

// The aperture fit is a latency chain (Newton steps of a 4-point Hermite
// interpolation full of divisions, bit for bit the oracle's), so a window line
// takes 16 lanes: a quad per fit node, a lane per state vector of the
// interpolation, the divisions by state-vector times through their
// reciprocals.  256 lines: 8 us; one lane per line, 60 divisions a step, took
// 80 us at any line count up to the card's width.
constexpr int kFitLanes = 16;

// Lane J's double, on every lane of its quad.
template <int J>
__device__ __forceinline__ double quad_lane(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffll), J * 0x55, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), J * 0x55, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double quad_sum(double v) {
#pragma clang fp contract(off)
  return ((0.0 + quad_lane<0>(v) + quad_lane<1>(v)) + quad_lane<2>(v)) + quad_lane<3>(v);
}

// Zero-Doppler range of ground point xyz by a quad: Newton on (x - s(t)).v(t)
// with the derivative taken as -|v|^2, at most 51 steps, stop at |dt| < 5e-9 s
// (sentinel/orbitrangetime.f90:23-69), from the state (t0, s0, v0).  The state
// vectors as orbit_at selects them.
__device__ __forceinline__ double zero_doppler_range(const double* xyz, const double* t,
                                                     const double* x, const double* v, int n,
                                                     double t0, const double* s0,
                                                     const double* v0) {
#pragma clang fp contract(off)
  const double dt = t[1] - t[0], rdt = 1.0 / dt;
  const bool plain_dt = !(fabs(rdt) < 1e100 && fabs(rdt) > 1e-100);
  double tl = t0, sx[3] = {s0[0], s0[1], s0[2]}, sv[3] = {v0[0], v0[1], v0[2]};
  double dr[3];
  HermiteNode node;
  int have = -1;
  bool split = false;
  for (int k = 0; k < 51; ++k) {
    const double tprev = tl;
    for (int i = 0; i < 3; ++i) dr[i] = xyz[i] - sx[i];
    const double fn = dot3(dr, sv);
    const double fnprime = -dot3(sv, sv) + 0.0 * fn;
    tl = tl - fn / fnprime;
    int iloc = (int)(plain_dt ? (tl - t[0]) / dt : div_by(tl - t[0], dt, rdt));
    iloc = iloc < 2 ? 2 : iloc;
    iloc = iloc > n - 2 ? n - 2 : iloc;
    const int first = iloc - 2;
    if (first != have) {   // the same on the quad's four lanes
      const bool ok =
          hermite_node(t + first, x + 3 * first, v + 3 * first, threadIdx.x & 3, &node);
      const int bad = ok ? 0 : 1;
      split = (__builtin_amdgcn_mov_dpp(bad, 0x00, 0xf, 0xf, true) |
               __builtin_amdgcn_mov_dpp(bad, 0x55, 0xf, 0xf, true) |
               __builtin_amdgcn_mov_dpp(bad, 0xaa, 0xf, 0xf, true) |
               __builtin_amdgcn_mov_dpp(bad, 0xff, 0xf, 0xf, true)) == 0;
      have = first;
    }
    if (split) {
      double p[3], w[3];
      hermite_term(node, tl, p, w);
      for (int i = 0; i < 3; ++i) {
        sx[i] = quad_sum(p[i]);
        sv[i] = quad_sum(w[i]);
      }
    } else {
      hermite4(x + 3 * first, v + 3 * first, t + first, tl, sx, sv);
    }
    if (fabs(tl - tprev) < 5.0e-9) break;
  }
  for (int i = 0; i < 3; ++i) dr[i] = xyz[i] - sx[i];
  return sqrt(dot3(dr, dr));
}

// Three zero-Doppler solves of a window line, the aperture centres, the
// parabola, by its kFitLanes lanes.  Lines at or beyond nfit get (0, 0, 0).
__device__ __forceinline__ void fit_line(const BurstDev& b, const double* orb_t,
                                         const double* orb_x, const double* orb_v, int line,
                                         double* coef) {
  double* c = coef + 3 * line;
  const int sub = threadIdx.x & (kFitLanes - 1);
  if (line >= b.nfit) {
    if (sub < 3) c[sub] = 0.;
    return;
  }
  FitParams f;
  f.tmid = b.tmid;
  f.wvl = b.wvl;
  f.angc0 = b.angc0;
  f.angc1 = b.angc1;
  f.prf = b.prf;
  f.rawdatalines = b.L;
  for (int i = 0; i < 3; ++i) {
    f.xyz_mid[i] = b.xyz_mid[i];
    f.vel_mid[i] = b.vel_mid[i];
  }
  const int node = min(sub >> 2, 2);   // the fourth quad repeats the third's
  const int pix = b.firstpix + node * fit_node_step(b.firstpix, b.lastpix);
  double xyz[3];
  pixel_ecef(b, line, pix, xyz);
  const double rng = zero_doppler_range(xyz, orb_t, orb_x, orb_v, b.nsv, f.tmid, f.xyz_mid,
                                        f.vel_mid);
  const int y = aperture_centre(xyz, rng, f);
  const int y0 = __shfl(y, 0, kFitLanes), y1 = __shfl(y, 4, kFitLanes),
            y2 = __shfl(y, 8, kFitLanes);
  if (sub == 0) parabola(y0, y1, y2, c);
}

__global__ __launch_bounds__(kWave) void k_fit(BurstDev b, double* coef) {
  const int line = (blockIdx.x * kWave + threadIdx.x) / kFitLanes;
  if (line < b.nlines) fit_line(b, b.orb_t, b.orb_x, b.orb_v, line, coef);
}

// The fit of a burst whose orbit travels with the launch: no table on the
// device, no upload, and nothing on the host to wait for.
struct FitArg {
  BurstDev b;
  double* coef;
  double orb[7 * kFitArgVec];   // [t(n) | x(3n) | v(3n)]
};
__global__ __launch_bounds__(kWave) void k_fit_arg(FitArg a) {
  // The table is indexed in the kernel's argument segment itself.
  typedef const char __attribute__((address_space(4)))* arg_t;
  const double* orb = (const double*)((arg_t)__builtin_amdgcn_kernarg_segment_ptr() +
                                      __builtin_offsetof(FitArg, orb));
  const int line = (blockIdx.x * kWave + threadIdx.x) / kFitLanes;
  if (line < a.b.nlines)
    fit_line(a.b, orb, orb + a.b.nsv, orb + 4 * a.b.nsv, line, a.coef);
}

__global__ __launch_bounds__(kWave) void k_batch_fit(const BurstDev* __restrict__ bursts) {
  const BurstDev& b = bursts[blockIdx.y];
  const int line = (blockIdx.x * kWave + threadIdx.x) / kFitLanes;
  if (line < b.nlines)
    fit_line(b, b.orb_t, b.orb_x, b.orb_v, line, const_cast<double*>(b.coef));
}

// setxyz: ECEF of [firstpix, lastpix], zero elsewhere; fit nodes per line.
__global__ void k_setxyz(BurstDev b, double* xyz, double* xyzfit) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)b.nlines * b.W;
  if (k >= total) return;
  const int row = (int)(k / b.W), col = (int)(k - (size_t)row * b.W);
  double o[3] = {0., 0., 0.};
  if (col >= b.firstpix && col <= b.lastpix) pixel_ecef(b, row, col, o);
  xyz[3 * k] = o[0];
  xyz[3 * k + 1] = o[1];
  xyz[3 * k + 2] = o[2];
  if (xyzfit && col >= b.firstpix && col <= b.lastpix) {
    const int step = fit_node_step(b.firstpix, b.lastpix);
    for (int node = 0; node < 3; ++node)
      if (col == b.firstpix + node * step)
        for (int i = 0; i < 3; ++i) xyzfit[9 * row + 3 * node + i] = o[i];
  }
}

__global__ void k_setazoff(BurstDev b, double* azoff) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)b.nlines * b.W;
  if (k >= total) return;
  const int row = (int)(k / b.W), col = (int)(k - (size_t)row * b.W);
  double a = -1.0;
  if (col >= b.firstpix && col <= b.lastpix)
    a = pixel_azoff(b.coef + 3 * row, col, b.firstpix, b.lastpix, b.A, b.L);
  azoff[k] = a;
}

// Pairs per line: one block per line.
__global__ void k_pairs(BurstDev b, int64_t* pairs) {
  __shared__ int64_t part[kBlock / kWave];
  const int row = blockIdx.x;
  int64_t acc = 0;
  if (row < b.nfit) {
    for (int col = b.firstpix + threadIdx.x; col <= b.lastpix && col < b.W;
         col += blockDim.x) {
      const double az =
          pixel_azoff(b.coef + 3 * row, col, b.firstpix, b.lastpix, b.A, b.L);
      if (az > 0.) {
        int s, e;
        pulse_window(az, b.A, b.L, &s, &e);
        if (e > s) acc += e - s;
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t t = 0;
    for (int w = 0; w < kBlock / kWave; ++w) t += part[w];
    pairs[row] = t;
  }
}

// pixelint on materialised xyz / azoff: thread per pixel, FP64 like k_plain.
__global__ void k_pixelint(BurstDev b, const double* __restrict__ xyz,
                           const double* __restrict__ azoff) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)b.nlines * b.W;
  if (k >= total) return;
  double ar = 0., ai = 0.;
  int azs = 0, aze = 0;
  const double az = azoff[k];
  if (az > 0.) {
    pulse_window(az, b.A, b.L, &azs, &aze);
    const double x[3] = {xyz[3 * k], xyz[3 * k + 1], xyz[3 * k + 2]};
    const float2* base = (const float2*)b.data;
    for (int q = azs; q < aze; ++q) {
      if (b.cpu)
        cpu_pair(base + (size_t)q * b.S, x, b.satloc[3 * q], b.satloc[3 * q + 1],
                 b.satloc[3 * q + 2], b, ar, ai);
      else
        plain_pair(base + (size_t)q * b.S, x, b.satloc[3 * q], b.satloc[3 * q + 1],
                   b.satloc[3 * q + 2], b, ar, ai);
    }
  }
  float2 o = make_float2(0.f, 0.f);
  if (b.cpu) {
    o = make_float2((float)ar, (float)ai);
  } else if (az > 0.) {
    const float s = (float)(1. / (aze - azs));
    o = make_float2((float)ar * s, (float)ai * s);
  }
  b.out[k] = o;
}

// ------------------------------------------------------------ utilities

__global__ void k_zero16(uint4* p, size_t n16, uint8_t* tail, int ntail) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
       i += stride)
    p[i] = make_uint4(0u, 0u, 0u, 0u);
  if (blockIdx.x == 0 && (int)threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

// .geo merge of one burst output into a grid.  GPU entry
// (sentinel/azimuth_compress.cu:527-531): a pixel is replaced where
// |Re(out)| > 1e-18, compared in double.  CPU twin
// (sentinel/azimuth_compress_cpu.c:386-388): abs((int)Re) > 1e-18 as the
// reference's unoptimised x86 build evaluates it -- the truncating conversion
// is nonzero for |Re| >= 1 and gives INT_MIN (whose abs stays negative) for
// |Re| >= 2^31 and NaN -- so 1 <= |Re| < 2^31.
__global__ void k_merge(float2* __restrict__ grid, const float2* __restrict__ out,
                        size_t n, size_t grid_off, int cpu) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float2 v = out[i];
    const float a = fabsf(v.x);
    const bool take = cpu ? (a >= 1.f && a < 2147483648.f) : (fabs((double)v.x) > 1.e-18);
    if (take) grid[grid_off + i] = v;
  }
}

// Error sums of an image g against a reference o over the pixels where o is
// nonzero: [0] sum |o|^2 arg(g conj o)^2, [1] sum |o|^2, [2] sum (|g|-|o|)^2,
// [3] count, [4] pixels where o is zero and g is not.  One double partial per
// block and sum; the host adds the blocks.
constexpr int kCmpBlock = 256;
__global__ void __launch_bounds__(kCmpBlock)
k_compare(const float2* __restrict__ g, const float2* __restrict__ o, size_t n,
          double* __restrict__ part) {
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float2 a = g[i], b = o[i];
    const double ox = b.x, oy = b.y, gx = a.x, gy = a.y;
    if (ox != 0.0 || oy != 0.0) {
      const double w = ox * ox + oy * oy;
      const double ph = atan2(gy * ox - gx * oy, gx * ox + gy * oy);
      const double da = sqrt(gx * gx + gy * gy) - sqrt(w);
      acc[0] += w * ph * ph;
      acc[1] += w;
      acc[2] += da * da;
      acc[3] += 1.0;
    } else if (gx != 0.0 || gy != 0.0) {
      acc[4] += 1.0;
    }
  }
  __shared__ double red[5][kCmpBlock];
  for (int k = 0; k < 5; ++k) red[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int h = kCmpBlock / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
      for (int k = 0; k < 5; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x < 5) part[(size_t)blockIdx.x * 5 + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void k_copy16(uint4* __restrict__ d, const uint4* __restrict__ s, size_t n16,
                         uint8_t* dt, const uint8_t* st, int ntail) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
    d[i] = s[i];
  if (blockIdx.x == 0 && (int)threadIdx.x < ntail) dt[threadIdx.x] = st[threadIdx.x];
}

__global__ void k_copy1(uint8_t* __restrict__ d, const uint8_t* __restrict__ s, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    d[i] = s[i];
}

// Headers of lines `line_words` 4-byte words apart to (to_lines: from) rows of
// 20 words.
__global__ void k_headers(uint32_t* lines, size_t line_words, uint32_t* rows, size_t words,
                          bool to_lines) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= words) return;
  uint32_t* w = lines + (i / 20) * line_words + i % 20;
  if (to_lines)
    *w = rows[i];
  else
    rows[i] = *w;
}

__global__ void k_zero1(uint8_t* p, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride)
    p[i] = 0;
}

// Packing in two passes, one workgroup per pulse each: every pulse's own scale,
// then its words at the call's scale, so that the words are written once.  (One
// workgroup of 256 per pulse for own scale and words, and k_unify_scales over
// the words after it, took 110 + 45 us for 1363 x 18011 samples; now 36 + 49
// us, 5.4 and 6.0 TB/s, part of the second read from the last-level cache.)
__global__ void __launch_bounds__(kPackBlock)
k_pack_scale(const float2* __restrict__ in, int S, int dtype, float* __restrict__ scale) {
  __shared__ float part[kPackBlock / kWave];
  const int p = blockIdx.x;
  const float mx = row_max(in + (size_t)p * S, S, part);
  if (threadIdx.x == 0) scale[p] = pulse_scale(mx, dtype);
}

// scale: k_pack_scale's on entry, the pulses' final ones on return.  Every
// workgroup finds the same largest scale, whichever of the others have
// rewritten theirs (a rewritten one becomes the largest, or stays 0 ... 0 -> 1
// when all are 0, where no word depends on it).
template <int DT>
__global__ void __launch_bounds__(kPackBlock)
k_pack(const float2* __restrict__ in, int S, int L, uint32_t* __restrict__ out,
       float* __restrict__ scale) {
  __shared__ float part[kPackBlock / kWave];
  const int p = blockIdx.x;
  const float own = load_scale(scale + p);
  float m = 0.f;
  for (int i = threadIdx.x; i < L; i += kPackBlock) m = fmaxf(m, load_scale(scale + i));
  const float s = unified_scale(own, block_max(m, part), DT);   // barrier: scale[p] is read
  const bool rescale = own > 0.f && own != s;
  pack_row<DT>(in + (size_t)p * S, S, out + (size_t)p * S, pulse_inv(own), rescale,
               rescale ? own / s : 1.f);
  if (threadIdx.x == 0) store_scale(scale + p, s);
}

// One block per pulse, after the packing range-compression store:
// M = the largest scale of the L pulses; a pulse whose scale s is within
// [M 2^-16, M) (CF16/CBF16) or [M 2^-4, M) (CI16) has its words multiplied by
// s/M and takes M -- a power of two: exact for CF16/CBF16 unless the result
// is subnormal, rounded to the nearest integer (ties to even) for CI16 -- an
// all-zero pulse (s = 0) takes M, a pulse further below keeps its own scale.
// Every block reads the same M: the scales it rewrites become M, which leaves
// the maximum unchanged (all-zero input: M = 0, every scale becomes 1).
__global__ void k_unify_scales(uint32_t* __restrict__ packed, size_t rowwords, int L,
                               float* __restrict__ scale, int dtype) {
  __shared__ float part[kBlock / kWave];
  const int p = blockIdx.x;
  float m = 0.f;
  for (int i = threadIdx.x; i < L; i += blockDim.x) m = fmaxf(m, load_scale(scale + i));
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  float M = part[0];
  for (int w = 1; w < kBlock / kWave; ++w) M = fmaxf(M, part[w]);
  const float s = load_scale(scale + p);
  __syncthreads();  // every thread has read scale[p] before it changes
  if (M == 0.f) {
    if (threadIdx.x == 0) store_scale(scale + p, 1.f);
    return;
  }
  const float lowest = dtype == TDBP_CI16 ? M * (1.0f / (1 << kI16Unify)) : M * (1.0f / 65536.0f);
  if (s == M || (s > 0.f && s < lowest)) return;
  if (s > 0.f) {
    const float f = s / M;
    uint32_t* row = packed + (size_t)p * rowwords;
    for (size_t i = threadIdx.x; i < rowwords; i += blockDim.x) {
      float re, im;
      word_components(row[i], dtype, &re, &im);
      row[i] = pack_word(re * f, im * f, dtype);
    }
  }
  if (threadIdx.x == 0) store_scale(scale + p, M);
}

// Counter-based normal pair (splitmix64 hash -> Box-Muller).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ float2 gauss2(uint64_t seed, uint64_t k) {
  const uint64_t h = mix64(seed ^ mix64(k));
  const float u1 = ((uint32_t)(h >> 40) + 0.5f) * (1.0f / 16777216.0f);
  const float u2 = ((uint32_t)(h & 0xffffffu) + 0.5f) * (1.0f / 16777216.0f);
  const float r = sqrtf(-2.0f * logf(u1));
  float s, c;
  sincospif(2.0f * u2, &s, &c);
  return make_float2(r * c, r * s);
}

// Decoded echo lines: the packet header in samples [0, 10), then nsamps echo
// samples: per target, the transmitted chirp delayed by delay[p][t] samples
// with carrier exp(-j 2 pi carrier[p][t]) and amplitude amp[t], plus white
// circular Gaussian noise of standard deviation `noise`; zero beyond nsamps.
struct RawHeader {
  float2 w[10];
};

__global__ void k_synth_raw(float2* __restrict__ d, int L, int stride, int nsamps, int npts,
                            float sf, float f0, float ramp, const double* __restrict__ delay,
                            const double* __restrict__ carrier, const float2* __restrict__ amp,
                            int ntargets, float noise, uint64_t seed, RawHeader hdr) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int p = blockIdx.y;
  if (n >= stride || p >= L) return;
  float2 v = make_float2(0.f, 0.f);
  if (n < 10) {
    v = hdr.w[n];
  } else if (n - 10 < nsamps) {
    const int k = n - 10;
    double re = 0.0, im = 0.0;
    for (int t = 0; t < ntargets; ++t) {
      const double u = (double)k - delay[(size_t)p * ntargets + t];
      if (u >= 0.0 && u < (double)npts) {
        const double tt = u / (double)sf;
        const double ph = 2.0 * 3.141592653589793 * ((double)f0 * tt + 0.5 * (double)ramp * tt * tt -
                                                    carrier[(size_t)p * ntargets + t]);
        double sn, cs;
        sincos(ph, &sn, &cs);
        const float2 a = amp[t];
        re += a.x * cs - a.y * sn;
        im += a.x * sn + a.y * cs;
      }
    }
    if (noise > 0.f) {
      const float2 g = gauss2(seed, (uint64_t)p * (uint64_t)stride + (uint64_t)n);
      const float s = noise * 0.70710678f;
      re += s * g.x;
      im += s * g.y;
    }
    v = make_float2((float)re, (float)im);
  }
  d[(size_t)p * stride + n] = v;
}

struct Taps {
  float h[64];
};

__global__ void k_synth_clutter(float2* d, int L, int S, uint64_t seed,
                                float sigma, Taps taps, int ntaps) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (size_t)L * S) return;
  const int p = (int)(k / S), s = (int)(k - (size_t)p * S);
  const int half = ntaps / 2;
  float re = 0.f, im = 0.f;
  const float g = sigma * 0.70710678118654752f;
  for (int t = 0; t < ntaps; ++t) {
    const int j = s - t + half;
    if (j < 0 || j >= S) continue;
    const float2 n = gauss2(seed, (uint64_t)p * (uint64_t)S + (uint64_t)j);
    re = fmaf(taps.h[t], n.x, re);
    im = fmaf(taps.h[t], n.y, im);
  }
  d[k] = make_float2(g * re, g * im);
}

__global__ void k_synth_target(float2* d, BurstDev b, double tx, double ty,
                               double tz, float ar, float ai, float res,
                               int halfwidth) {
  const int p = blockIdx.x;
  const int j = (int)threadIdx.x - halfwidth;
  if (p >= b.L || j > halfwidth) return;
  const double* s = b.satloc + 3 * p;
  const double dx = tx - s[0], dy = ty - s[1], dz = tz - s[2];
  const double R = sqrt(dx * dx + dy * dy + dz * dz);
  const double r = (R - b.rngstart) * b.inv_dmrg;
  const int i = (int)rint(r) + j;
  if (i < 0 || i >= b.S) return;
  const double cyc = R * b.two_over_wvl;
  const double f = cyc - rint(cyc);
  double sn, cs;
  sincospi(2.0 * f, &sn, &cs);
  const double xarg = (i - r) / res;
  const double snc = fabs(xarg) < 1e-12 ? 1.0 : sinpi(xarg) / (kPi * xarg);
  // amplitude * sinc * exp(-j 2 pi f)
  const double er = (ar * cs + ai * sn) * snc;
  const double ei = (ai * cs - ar * sn) * snc;
  float2* o = d + (size_t)p * b.S + i;
  o->x += (float)er;
  o->y += (float)ei;
}

// ------------------------------------------------------------ launchers

namespace {
inline unsigned blocks_for(size_t n, int bs) {
  return (unsigned)((n + bs - 1) / bs);
}

// Launch of a burst's tiles.  Up to two rounds of resident workgroups: one
// workgroup per tile, no queue (b.counters null).  Beyond: persistent, the
// resident workgroups of `kernel` on every CU, the tile-queue counters zeroed
// first (a fill kernel on the same stream).  The queue keeps a band's tiles on
// their XCD and evens out the end, but its counters cost a burst of few tiles
// more than they give: 1400 x 12000 samples onto 400 x 800 pixels 0.31 -> 0.25
// ms, 800 x 800 (1.2 rounds) 0.66 -> 0.52 ms, 600 x 1600 (1.9) 0.69 -> 0.67
// ms without it; FP64 on 800 x 800 (3.4 rounds) 0.56 with, 0.64 without.  Split
// tiles never take it: most of them hold no work, and an empty one costs an
// atomic of 0.2 us on its counter (1200 x 2638 samples onto 737 x 409 pixels,
// 4810 tiles: 0.31 -> 0.12 ms).
template <void (*K)(BurstDev)>
hipError_t persistent_launch(const BurstDev& b, hipStream_t s) {
  if (!b.counters) return hipErrorInvalidValue;
  static int occ = 0;   // of this kernel; the same on every gfx950 device
  if (occ <= 0 &&
      (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, K, kBlock, 0) != hipSuccess ||
       occ <= 0))
    occ = 1;
  const long nb = (long)b.tiles_r * b.tiles_c;
  const long room = (long)cu_count() * occ;
  if (nb <= 0) return hipSuccess;
  if (nb <= 2 * room || b.split) {
    BurstDev d = b;
    d.counters = nullptr;
    hipLaunchKernelGGL(K, dim3((unsigned)nb), dim3(kBlock), 0, s, d);
    return hipGetLastError();
  }
  const hipError_t e = launch_zero(b.counters, 8 * sizeof(int), s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(K, dim3((unsigned)std::min(nb, room)), dim3(kBlock), 0, s, b);
  return hipGetLastError();
}

template <int TR, int STACK>
hipError_t plain_launch(const BurstDev& b, hipStream_t s) {
  if (b.cpu) return persistent_launch<k_plain<TR, STACK, true>>(b, s);
  return persistent_launch<k_plain<TR, STACK, false>>(b, s);
}

template <int TR, int STACK, int DT, bool LDS>
hipError_t mixed_launch(const BurstDev& b, hipStream_t s) {
  if constexpr (LDS) return persistent_launch<k_mixed_lds<TR, STACK, DT>>(b, s);
  else return persistent_launch<k_mixed<TR, STACK, DT>>(b, s);
}

template <int TR, int STACK, bool LDS = false>
hipError_t mixed_dt(const BurstDev& b, hipStream_t s) {
  switch (b.dtype) {
    case TDBP_CF32: return mixed_launch<TR, STACK, TDBP_CF32, LDS>(b, s);
    case TDBP_CF16: return mixed_launch<TR, STACK, TDBP_CF16, LDS>(b, s);
    case TDBP_CI16: return mixed_launch<TR, STACK, TDBP_CI16, LDS>(b, s);
    default: return mixed_launch<TR, STACK, TDBP_CBF16, LDS>(b, s);
  }
}

template <int PREC, int TR, int STACK, int DT, bool LDS>
hipError_t batch_launch(const BurstDev* d, const int2* it, const int* qb,
                        int* ctr, int grid, hipStream_t s) {
  if constexpr (PREC == TDBP_MIXED && LDS)
    hipLaunchKernelGGL((k_batch_mixed_lds<TR, STACK, DT>), dim3(grid), dim3(kBlock), 0, s,
                       d, it, qb, ctr);
  else if constexpr (PREC == TDBP_MIXED)
    hipLaunchKernelGGL((k_batch_mixed<TR, STACK, DT>), dim3(grid), dim3(kBlock), 0, s,
                       d, it, qb, ctr);
  else
    hipLaunchKernelGGL((k_batch_plain<TR, STACK>), dim3(grid), dim3(kBlock), 0, s, d,
                       it, qb, ctr);
  return hipGetLastError();
}

template <int PREC, int TR, int STACK, int DT, bool LDS>
int occupancy() {
  int n = 0;
  hipError_t e;
  if constexpr (PREC == TDBP_MIXED && LDS)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_batch_mixed_lds<TR, STACK, DT>,
                                                     kBlock, 0);
  else if constexpr (PREC == TDBP_MIXED)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_batch_mixed<TR, STACK, DT>,
                                                     kBlock, 0);
  else
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_batch_plain<TR, STACK>,
                                                     kBlock, 0);
  if (e != hipSuccess) return 1;
  return n > 0 ? n : 1;
}

// Dispatch (precision, variant, dtype) to a template instance.  Variants
// 9 and 10 are the LDS-staged kernels on the tiles of variants 5 and 4 (the
// FP64 kernel has no staged form and runs those tiles unstaged).
template <template <int, int, int, int, bool> class F, typename... Args>
auto dispatch(int prec, int variant, int dt, Args... args) {
#define TDBP_V(TR, ST, LDS)                                                     \
  if (prec == TDBP_PLAIN_FP64) return F<TDBP_PLAIN_FP64, TR, ST, TDBP_CF32, false>::run(args...); \
  if (dt == TDBP_CF32) return F<TDBP_MIXED, TR, ST, TDBP_CF32, LDS>::run(args...); \
  if (dt == TDBP_CF16) return F<TDBP_MIXED, TR, ST, TDBP_CF16, LDS>::run(args...); \
  if (dt == TDBP_CI16) return F<TDBP_MIXED, TR, ST, TDBP_CI16, LDS>::run(args...); \
  return F<TDBP_MIXED, TR, ST, TDBP_CBF16, LDS>::run(args...);
  switch (variant) {
    case 0: { TDBP_V(8, kWavesSideBySide, false) }
    case 1: { TDBP_V(4, kWavesSideBySide, false) }
    case 2: { TDBP_V(2, kWavesSideBySide, false) }
    case 3: { TDBP_V(1, kWavesSideBySide, false) }
    case 4: { TDBP_V(8, kWavesStacked, false) }
    case 5: { TDBP_V(4, kWavesStacked, false) }
    case 6: { TDBP_V(2, kWavesStacked, false) }
    case kSplitVariant: { TDBP_V(4, kWavesSplit, false) }
    case 9: { TDBP_V(4, kWavesStacked, true) }
    case 10: { TDBP_V(8, kWavesStacked, true) }
    default: { TDBP_V(1, kWavesStacked, false) }
  }
#undef TDBP_V
}

template <int PREC, int TR, int STACK, int DT, bool LDS>
struct BatchRun {
  static hipError_t run(const BurstDev* d, const int2* it, const int* qb,
                        int* ctr, int grid, hipStream_t s) {
    return batch_launch<PREC, TR, STACK, DT, LDS>(d, it, qb, ctr, grid, s);
  }
};
template <int PREC, int TR, int STACK, int DT, bool LDS>
struct OccRun {
  static int run() { return occupancy<PREC, TR, STACK, DT, LDS>(); }
};
}  // namespace

hipError_t launch_plain(const BurstDev& b, int variant, hipStream_t s) {
  switch (variant) {
    case 8: return plain_launch<4, kWavesStacked>(b, s);   // same tile as the MFMA variant
    case 9: return plain_launch<4, kWavesStacked>(b, s);   // tiles of the LDS-staged variants
    case 10: return plain_launch<8, kWavesStacked>(b, s);
    case 0: return plain_launch<8, kWavesSideBySide>(b, s);
    case 1: return plain_launch<4, kWavesSideBySide>(b, s);
    case 2: return plain_launch<2, kWavesSideBySide>(b, s);
    case 3: return plain_launch<1, kWavesSideBySide>(b, s);
    case 4: return plain_launch<8, kWavesStacked>(b, s);
    case 5: return plain_launch<4, kWavesStacked>(b, s);
    case 6: return plain_launch<2, kWavesStacked>(b, s);
    case kSplitVariant: return persistent_launch<k_plain<4, kWavesSplit, false>>(b, s);
    default: return plain_launch<1, kWavesStacked>(b, s);
  }
}

template <int DT>
hipError_t mfma_launch(const BurstDev& b, hipStream_t s) {
  const int nb = b.tiles_r * b.tiles_c;
  hipLaunchKernelGGL((k_mixed_mfma<DT>), dim3(nb), dim3(kMBlock), 0, s, b);
  return hipGetLastError();
}

hipError_t launch_mixed(const BurstDev& b, int variant, hipStream_t s) {
  if (variant == 8) {
    if (!mfma_fits(b)) return mixed_dt<4, kWavesStacked>(b, s);   // same tile shape
    if (b.dtype == TDBP_CF32) return mfma_launch<TDBP_CF32>(b, s);
    if (b.dtype == TDBP_CF16) return mfma_launch<TDBP_CF16>(b, s);
    if (b.dtype == TDBP_CI16) return mfma_launch<TDBP_CI16>(b, s);
    return mfma_launch<TDBP_CBF16>(b, s);
  }
  switch (variant) {
    case 0: return mixed_dt<8, kWavesSideBySide>(b, s);
    case 1: return mixed_dt<4, kWavesSideBySide>(b, s);
    case 2: return mixed_dt<2, kWavesSideBySide>(b, s);
    case 3: return mixed_dt<1, kWavesSideBySide>(b, s);
    case 4: return mixed_dt<8, kWavesStacked>(b, s);
    case 5: return mixed_dt<4, kWavesStacked>(b, s);
    case 6: return mixed_dt<2, kWavesStacked>(b, s);
    case kSplitVariant: return mixed_dt<4, kWavesSplit>(b, s);
    case 9: return mixed_dt<4, kWavesStacked, true>(b, s);
    case 10: return mixed_dt<8, kWavesStacked, true>(b, s);
    default: return mixed_dt<1, kWavesStacked>(b, s);
  }
}

template <int DT>
int mfma_occupancy() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_batch_mfma<DT>, kMBlock, 0) !=
      hipSuccess)
    return 1;
  return n > 0 ? n : 1;
}

int batch_blocks_per_cu(int precision, int variant, int dtype) {
  if (variant == 8 && precision == TDBP_MIXED) {
    if (dtype == TDBP_CF32) return mfma_occupancy<TDBP_CF32>();
    if (dtype == TDBP_CF16) return mfma_occupancy<TDBP_CF16>();
    if (dtype == TDBP_CI16) return mfma_occupancy<TDBP_CI16>();
    return mfma_occupancy<TDBP_CBF16>();
  }
  return dispatch<OccRun>(precision, variant == 8 ? 5 : variant, dtype);
}

hipError_t launch_batch(const BurstDev* d_bursts, const int2* d_items,
                        const int* d_qbase, int* d_counters, int precision,
                        int variant, int dtype, int grid, hipStream_t s) {
  if (variant == 8 && precision == TDBP_MIXED) {
#define TDBP_M(DT)                                                                    \
  hipLaunchKernelGGL((k_batch_mfma<DT>), dim3(grid), dim3(kMBlock), 0, s, d_bursts, \
                     d_items, d_qbase, d_counters);                                  \
  return hipGetLastError();
    if (dtype == TDBP_CF32) { TDBP_M(TDBP_CF32) }
    if (dtype == TDBP_CF16) { TDBP_M(TDBP_CF16) }
    if (dtype == TDBP_CI16) { TDBP_M(TDBP_CI16) }
    TDBP_M(TDBP_CBF16)
#undef TDBP_M
  }
  return dispatch<BatchRun>(precision, variant == 8 ? 5 : variant, dtype, d_bursts, d_items,
                            d_qbase, d_counters, grid, s);
}

hipError_t launch_batch_fit(const BurstDev* d_bursts, int nbursts,
                            int max_lines, hipStream_t s) {
  dim3 grid(blocks_for((size_t)max_lines * kFitLanes, kWave), nbursts);
  hipLaunchKernelGGL(k_batch_fit, grid, dim3(kWave), 0, s, d_bursts);
  return hipGetLastError();
}

hipError_t launch_fit_one(const BurstDev& b, double* coef, hipStream_t s) {
  hipLaunchKernelGGL(k_fit, dim3(blocks_for((size_t)b.nlines * kFitLanes, kWave)), dim3(kWave), 0,
                     s, b, coef);
  return hipGetLastError();
}

hipError_t launch_fit_arg(const BurstDev& b, const double* orbit, double* coef, hipStream_t s) {
  if (b.nsv > kFitArgVec) return hipErrorInvalidValue;
  FitArg a;
  a.b = b;
  a.coef = coef;
  std::copy(orbit, orbit + 7 * (size_t)b.nsv, a.orb);
  std::fill(a.orb + 7 * (size_t)b.nsv, a.orb + 7 * kFitArgVec, 0.0);
  hipLaunchKernelGGL(k_fit_arg, dim3(blocks_for((size_t)b.nlines * kFitLanes, kWave)),
                     dim3(kWave), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_setxyz(const BurstDev& b, double* xyz, double* xyzfit,
                         hipStream_t s) {
  const size_t n = (size_t)b.nlines * b.W;
  hipLaunchKernelGGL(k_setxyz, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s,
                     b, xyz, xyzfit);
  return hipGetLastError();
}

hipError_t launch_setazoff(const BurstDev& b, double* azoff, hipStream_t s) {
  const size_t n = (size_t)b.nlines * b.W;
  hipLaunchKernelGGL(k_setazoff, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0,
                     s, b, azoff);
  return hipGetLastError();
}

hipError_t launch_pair_count(const BurstDev& b, int64_t* pairs, hipStream_t s) {
  hipLaunchKernelGGL(k_pairs, dim3(b.nlines), dim3(kBlock), 0, s, b, pairs);
  return hipGetLastError();
}

hipError_t launch_pixelint(const BurstDev& b, const double* xyz,
                           const double* azoff, hipStream_t s) {
  const size_t n = (size_t)b.nlines * b.W;
  hipLaunchKernelGGL(k_pixelint, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0,
                     s, b, xyz, azoff);
  return hipGetLastError();
}

hipError_t launch_zero(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if ((uintptr_t)p % 16 != 0) {
    size_t g = blocks_for(bytes, kBlock);
    hipLaunchKernelGGL(k_zero1, dim3((unsigned)(g < 65535 ? g : 65535)),
                       dim3(kBlock), 0, s, (uint8_t*)p, bytes);
    return hipGetLastError();
  }
  const size_t n16 = bytes / 16;
  const int ntail = (int)(bytes - n16 * 16);
  size_t g = blocks_for(n16, kBlock);
  g = g == 0 ? 1 : (g < 65535 ? g : 65535);
  hipLaunchKernelGGL(k_zero16, dim3((unsigned)g), dim3(kBlock), 0, s,
                     (uint4*)p, n16, (uint8_t*)p + n16 * 16, ntail);
  return hipGetLastError();
}

hipError_t launch_merge(float2* grid, const float2* out, size_t n, size_t grid_off,
                        int semantics, hipStream_t s) {
  if (n == 0) return hipSuccess;
  size_t g = blocks_for(n, kBlock);
  g = g < 16384 ? g : 16384;
  hipLaunchKernelGGL(k_merge, dim3((unsigned)g), dim3(kBlock), 0, s, grid, out, n, grid_off,
                     semantics == TDBP_SEM_CPU ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_headers(void* lines, int nlines, int stride, void* rows, bool to_lines,
                          hipStream_t s) {
  const size_t words = (size_t)nlines * 20;
  hipLaunchKernelGGL(k_headers, dim3(blocks_for(words, kBlock)), dim3(kBlock), 0, s,
                     (uint32_t*)lines, 2 * (size_t)stride, (uint32_t*)rows, words, to_lines);
  return hipGetLastError();
}

int compare_blocks(size_t n) {
  const size_t g = blocks_for(n ? n : 1, kCmpBlock);
  return (int)(g < 4096 ? g : 4096);
}

hipError_t launch_compare(const float2* g, const float2* o, size_t n, double* part,
                          int blocks, hipStream_t s) {
  hipLaunchKernelGGL(k_compare, dim3(blocks), dim3(kCmpBlock), 0, s, g, o, n, part);
  return hipGetLastError();
}

hipError_t launch_copy(void* d, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if ((uintptr_t)d % 16 != 0 || (uintptr_t)src % 16 != 0) {
    size_t g = blocks_for(bytes, kBlock);
    hipLaunchKernelGGL(k_copy1, dim3((unsigned)(g < 65535 ? g : 65535)), dim3(kBlock), 0,
                       s, (uint8_t*)d, (const uint8_t*)src, bytes);
    return hipGetLastError();
  }
  const size_t n16 = bytes / 16;
  const int ntail = (int)(bytes - n16 * 16);
  size_t g = blocks_for(n16, kBlock);
  g = g == 0 ? 1 : (g < 65535 ? g : 65535);
  hipLaunchKernelGGL(k_copy16, dim3((unsigned)g), dim3(kBlock), 0, s, (uint4*)d,
                     (const uint4*)src, n16, (uint8_t*)d + n16 * 16,
                     (const uint8_t*)src + n16 * 16, ntail);
  return hipGetLastError();
}

hipError_t launch_pack(const float2* in, int L, int S, int dtype, void* out,
                       float* scale, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_scale, dim3(L), dim3(kPackBlock), 0, s, in, S, dtype, scale);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const auto k = dtype == TDBP_CF16   ? k_pack<TDBP_CF16>
                 : dtype == TDBP_CI16 ? k_pack<TDBP_CI16>
                                      : k_pack<TDBP_CBF16>;
  hipLaunchKernelGGL(k, dim3(L), dim3(kPackBlock), 0, s, in, S, L, (uint32_t*)out, scale);
  return hipGetLastError();
}

hipError_t launch_unify_scales(uint32_t* packed, size_t rowwords, int L, float* scale,
                               int dtype, hipStream_t s) {
  hipLaunchKernelGGL(k_unify_scales, dim3(L), dim3(kBlock), 0, s, packed, rowwords, L, scale,
                     dtype);
  return hipGetLastError();
}

hipError_t launch_synth_clutter(float2* d, int L, int S, uint64_t seed,
                                float sigma, const float* taps, int ntaps,
                                hipStream_t s) {
  Taps t;
  for (int i = 0; i < 64; ++i) t.h[i] = i < ntaps ? taps[i] : 0.f;
  const size_t n = (size_t)L * S;
  hipLaunchKernelGGL(k_synth_clutter, dim3(blocks_for(n, kBlock)), dim3(kBlock),
                     0, s, d, L, S, seed, sigma, t, ntaps);
  return hipGetLastError();
}

hipError_t launch_synth_raw(float2* d, int L, int stride, int nsamps, int npts, float sf,
                            float f0, float ramp, const double* delay, const double* carrier,
                            const float2* amp, int ntargets, float noise, uint64_t seed,
                            const void* header80, hipStream_t s) {
  RawHeader h;
  __builtin_memcpy(&h, header80, sizeof h);
  hipLaunchKernelGGL(k_synth_raw, dim3(blocks_for((size_t)stride, kBlock), L), dim3(kBlock), 0,
                     s, d, L, stride, nsamps, npts, sf, f0, ramp, delay, carrier, amp,
                     ntargets, noise, seed, h);
  return hipGetLastError();
}

hipError_t launch_synth_target(float2* d, const BurstDev& b, double tx,
                               double ty, double tz, float ar, float ai,
                               float res, int halfwidth, hipStream_t s) {
  hipLaunchKernelGGL(k_synth_target, dim3(b.L), dim3(2 * halfwidth + 1), 0, s,
                     d, b, tx, ty, tz, ar, ai, res, halfwidth);
  return hipGetLastError();
}

}  // namespace tdbp
