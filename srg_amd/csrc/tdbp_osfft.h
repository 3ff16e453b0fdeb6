// tdbp_osfft.h -- the 8192-point complex FP32 FFT pair of the fused range
// compression (overlap-save blocks of one echo line, tdbp_range.hip), shared
// by the device kernels and a host check.
//
// In place, mixed radix 16 x 16 x 16 x 2.  The forward transform of a block
// runs decimation in frequency (DIF): stage (R, s) with L = R s takes, in
// every L-point sub-block at base b and for j < s, the values b + j + s r (r
// < R), an R-point DFT, times w^((N/L) j k) (w = e^{-2 pi i/N}), back to b +
// j + s k.  Stages (16, 512), (16, 32), (16, 2), (2, 1) leave X[drev(p)] at
// position p, drev(p) = d0 + 16 d1 + 256 d2 + 4096 d3 for p = 512 d0 + 32 d1
// + 2 d2 + d3.  The second transform runs decimation in time (DIT) on that
// order: the same stages in reverse, each twiddling its inputs by
// w^((N/L) j r) before the DFT, from values in digit-reversed order to the
// forward transform in natural order.  A product of two DIF outputs position
// by position is the product of the spectra, so a convolution needs no
// reordering at all.  Forward sign e^{-2 pi i nk/N}; the unnormalised
// inverse of y is conj(FFT(conj(y))).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "tdbp_geom.h"   // TDBP_HD

namespace tdbp {

constexpr int kOsN = 8192;          // transform length
// Threads of the device transforms: one radix-16 butterfly per thread and
// stage; thread t holds values t + kOsThreads m (m < 16) of the block in
// natural order, or positions 2 (t + kOsThreads h) + e (m = 2 h + e) in the
// DIF output order.  Two ~70 KB workgroups fill a CU's LDS: 4 waves per SIMD.
// (1024 threads, radix 8: 0.45 ms per IW burst against 0.40 ms at 512 --
// spills at 64 VGPRs, and every barrier waits for 16 waves.)
constexpr int kOsThreads = kOsN / 16;

TDBP_HD float2 c_add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
TDBP_HD float2 c_sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
TDBP_HD float2 c_mul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a times -i, and times e^{-i pi/4}, e^{-3 i pi/4}
TDBP_HD float2 c_mni(float2 a) { return make_float2(a.y, -a.x); }
TDBP_HD float2 c_w8(float2 a) {
  const float h = 0.70710678118654752f;
  return make_float2((a.x + a.y) * h, (a.y - a.x) * h);
}
TDBP_HD float2 c_w8_3(float2 a) {
  const float h = 0.70710678118654752f;
  return make_float2((a.y - a.x) * h, -(a.x + a.y) * h);
}

// In-register forward DFT of 4 points, in place.
TDBP_HD void dft4(float2& a, float2& b, float2& c, float2& d) {
  const float2 t0 = c_add(a, c), t1 = c_sub(a, c), t2 = c_add(b, d), t3 = c_mni(c_sub(b, d));
  a = c_add(t0, t2);
  c = c_sub(t0, t2);
  b = c_add(t1, t3);
  d = c_sub(t1, t3);
}

// In-register forward DFT of 16 points, natural order in and out: with n =
// 4 n1 + n2 and k = k1 + 4 k2, four 4-point DFTs over n1, the products by
// w16^(n2 k1), four 4-point DFTs over n2.
TDBP_HD void dft16(float2* x) {
#pragma unroll
  for (int n2 = 0; n2 < 4; ++n2) dft4(x[n2], x[4 + n2], x[8 + n2], x[12 + n2]);
  // x[4 k1 + n2] now holds the n2-th sub-DFT at k1
  const float c1 = 0.92387953251128676f, s1 = 0.38268343236508977f;
  x[5] = c_mul(x[5], make_float2(c1, -s1));    // n2 = 1: w16^1, ^2, ^3
  x[9] = c_w8(x[9]);
  x[13] = c_mul(x[13], make_float2(s1, -c1));
  x[6] = c_w8(x[6]);                           // n2 = 2: w16^2, ^4, ^6
  x[10] = c_mni(x[10]);
  x[14] = c_w8_3(x[14]);
  x[7] = c_mul(x[7], make_float2(s1, -c1));    // n2 = 3: w16^3, ^6, ^9
  x[11] = c_w8_3(x[11]);
  x[15] = c_mul(x[15], make_float2(-c1, s1));
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) dft4(x[4 * k1], x[4 * k1 + 1], x[4 * k1 + 2], x[4 * k1 + 3]);
  // X[k1 + 4 k2] is at x[4 k1 + k2]: transpose the 4 x 4 block
  float2 y[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) y[k] = x[4 * (k & 3) + (k >> 2)];
#pragma unroll
  for (int k = 0; k < 16; ++k) x[k] = y[k];
}

// LDS layout: position p at os_pad(p) = p + 2 floor(p / 32), two values of
// padding per 32.  Every access of the transforms touches each pair of the
// 64 LDS banks once per half-wave (the 16-byte reads and writes of stage (2,
// 1) twice, their minimum): stage (16, 512) 32 consecutive positions,
// (16, 32) 32 consecutive, (16, 2) pairs 32 apart, (2, 1) 16-byte pairs.  The
// values of one butterfly sit a compile-time distance apart (544, 34 and 2
// values; the pairs of (2, 1) 1088 apart across a thread's eight
// butterflies), so every LDS address is a base plus an immediate.
constexpr int kOsLds = kOsN + 2 * (kOsN / 32);
TDBP_HD constexpr int os_pad(int p) { return p + 2 * (p >> 5); }

// Twiddles come from tables, every one of them rounded once from FP64: the
// table of an L-point stage (16, L/16) holds w_L^(j k) at [k L/16 + j] (k < 16,
// j < L/16), so the lanes of a wave read it in order.  The first stage's table
// (L = N, 8 N bytes) stays in global memory, where the caches keep it; those of
// the stages after it (N/16 values, for 8192 points 512 + 32) go to LDS.
// Fifteen twiddles built as products of four lookups took 60 of a stage's 270
// vector instructions, and their roundings were the pair's largest error.
TDBP_HD constexpr int os_mid_values(int n) { return n == kOsN ? n / 16 + n / 256 : n / 16; }
TDBP_HD constexpr int os_table_values(int n) { return n + os_mid_values(n); }
struct OsTwiddle {
  const float2* first;
  const float2* mid;   // 8192 points: the stage (16, 2) at mid + 512
};
// Entry i of a length's tables (first, then mid) is w_N^m, m the return value.
TDBP_HD int os_table_power(int n, int i) {
  int step = 1, L = n;   // w_L = w_N^step
  while (i >= L) {
    i -= L;
    L /= 16;
    step *= 16;
  }
  return step * ((i / (L / 16)) * (i % (L / 16)));
}

// v[k] times the twiddles of butterfly j of an L-point stage: all fifteen from
// the table (FULL), or six and the other nine as products of two of them.  FULL
// is the more exact (1.6e-7 against 1.8e-7 over a 1024-point round trip, 2.2e-7
// with four lookups) and about 5 % slower: its loads cost the caches and LDS
// more than the products cost the vector units.
template <int L, bool FULL = false>
TDBP_HD void os_apply(const float2* tab, int j, float2* v) {
  if constexpr (FULL) {
#pragma unroll
    for (int k = 1; k < 16; ++k) v[k] = c_mul(v[k], tab[k * (L / 16) + j]);
    return;
  }
  float2 lo[4], hi[4];
#pragma unroll
  for (int r = 1; r < 4; ++r) {
    lo[r] = tab[r * (L / 16) + j];
    hi[r] = tab[4 * r * (L / 16) + j];
  }
#pragma unroll
  for (int k = 1; k < 16; ++k) {
    const int q = k >> 2, r = k & 3;
    v[k] = c_mul(v[k], q == 0 ? lo[r] : r == 0 ? hi[q] : c_mul(hi[q], lo[r]));
  }
}

// A radix-16 stage of butterfly j (twiddles of an L-point stage) whose values
// sit at lds[a0 + STEP r]: read, [DIT: twiddle], DFT, [DIF: twiddle], write back
// in place.
template <int L, int STEP, bool DIT, bool FULL>
TDBP_HD void os_stage16(float2* lds, int a0, int j, const float2* tab, float2* v) {
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = lds[a0 + STEP * r];
  if constexpr (DIT) os_apply<L, FULL>(tab, j, v);
  dft16(v);
  if constexpr (!DIT) os_apply<L, FULL>(tab, j, v);
#pragma unroll
  for (int k = 0; k < 16; ++k) lds[a0 + STEP * k] = v[k];
}

// The stages of thread t.  Stage (16, 512): butterfly t, values t + 512 r,
// which the thread holds in registers (DIF: from registers; DIT: into them).
// Stage (16, 32): butterfly j = t mod 32 of sub-block t / 32.  Stage (16, 2):
// butterfly t mod 2 of sub-block t / 2.  Stage (2, 1): the eight pairs at
// positions 2 (t + 512 h), held in registers as v[2h], v[2h + 1].
template <bool FULL = false>
TDBP_HD void os_dif_first(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  dft16(v);
  os_apply<kOsN, FULL>(tw.first, t, v);
  float2* q = lds + os_pad(t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[544 * k] = v[k];
}
template <bool FULL = false>
TDBP_HD void os_dif_mid1(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  os_stage16<512, 34, false, FULL>(lds, 544 * (t >> 5) + (t & 31), t & 31, tw.mid, v);
}
template <bool FULL = false>
TDBP_HD void os_dif_mid2(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  os_stage16<32, 2, false, FULL>(lds, 34 * (t >> 1) + (t & 1), t & 1, tw.mid + 512, v);
}
TDBP_HD void os_dif_last(const float2* lds, int t, float2* v) {
  const float2* q = lds + os_pad(2 * t);
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    const float2 a = q[1088 * h], b = q[1088 * h + 1];
    v[2 * h] = c_add(a, b);
    v[2 * h + 1] = c_sub(a, b);
  }
}
TDBP_HD void os_dit_first(float2* lds, int t, const float2* v) {
  float2* q = lds + os_pad(2 * t);
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    q[1088 * h] = c_add(v[2 * h], v[2 * h + 1]);
    q[1088 * h + 1] = c_sub(v[2 * h], v[2 * h + 1]);
  }
}
template <bool FULL = false>
TDBP_HD void os_dit_mid1(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  os_stage16<32, 2, true, FULL>(lds, 34 * (t >> 1) + (t & 1), t & 1, tw.mid + 512, v);
}
template <bool FULL = false>
TDBP_HD void os_dit_mid2(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  os_stage16<512, 34, true, FULL>(lds, 544 * (t >> 5) + (t & 31), t & 31, tw.mid, v);
}
template <bool FULL = false>
TDBP_HD void os_dit_last(const float2* lds, int t, const OsTwiddle& tw, float2* v) {
  const float2* q = lds + os_pad(t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[544 * r];
  os_apply<kOsN, FULL>(tw.first, t, v);
  dft16(v);
}

// Host transforms (the check of the device code): the same stages, layout
// and registers, thread after thread, a stage loop in place of each barrier.
// os_dif_host: data in natural order -> data[p] = X[drev(p)].
// os_dit_host: data[p] = Y[drev(p)] -> data in natural order, the forward
// transform of Y.
template <int N>
struct OsHostTables {
  float2 v[os_table_values(N)];
  explicit OsHostTables(const float2* table) {   // w^m of 8192 points
    for (int i = 0; i < os_table_values(N); ++i) v[i] = table[kOsN / N * os_table_power(N, i)];
  }
  OsTwiddle tw() const { return OsTwiddle{v, v + N}; }
};
inline void os_dif_host(float2* data, const float2* table) {
  const OsHostTables<kOsN> tb(table);
  const OsTwiddle tw = tb.tw();
  float2* lds = new float2[kOsLds];
  float2 v[16];
  for (int t = 0; t < kOsThreads; ++t) {
    for (int r = 0; r < 16; ++r) v[r] = data[t + kOsThreads * r];
    os_dif_first(lds, t, tw, v);
  }
  for (int t = 0; t < kOsThreads; ++t) os_dif_mid1(lds, t, tw, v);
  for (int t = 0; t < kOsThreads; ++t) os_dif_mid2(lds, t, tw, v);
  for (int t = 0; t < kOsThreads; ++t) {
    os_dif_last(lds, t, v);
    for (int m = 0; m < 16; ++m) data[2 * (t + kOsThreads * (m >> 1)) + (m & 1)] = v[m];
  }
  delete[] lds;
}
inline void os_dit_host(float2* data, const float2* table) {
  const OsHostTables<kOsN> tb(table);
  const OsTwiddle tw = tb.tw();
  float2* lds = new float2[kOsLds];
  float2 v[16];
  for (int t = 0; t < kOsThreads; ++t) {
    for (int m = 0; m < 16; ++m) v[m] = data[2 * (t + kOsThreads * (m >> 1)) + (m & 1)];
    os_dit_first(lds, t, v);
  }
  for (int t = 0; t < kOsThreads; ++t) os_dit_mid1(lds, t, tw, v);
  for (int t = 0; t < kOsThreads; ++t) os_dit_mid2(lds, t, tw, v);
  for (int t = 0; t < kOsThreads; ++t) {
    os_dit_last(lds, t, tw, v);
    for (int k = 0; k < 16; ++k) data[t + kOsThreads * k] = v[k];
  }
  delete[] lds;
}

// ------------------------------------------------- 1024, 2048, 4096
// The N-point pairs of the interferograms' upsampling (int/crossmul.f90), the
// same scheme with N/16 threads and stages (16, N/16), (16, R), (R, 1), R =
// N/256 = 4, 8 or 16: position p = (N/16) d0 + R d1 + d2 holds bin d0 + 16 d1
// + 256 d2 after the DIF; thread t holds values t + (N/16) m in natural order
// and positions 16 t + m in the DIF order (16/R whole sub-blocks of the last
// stage).  Layout: position p at up_pad(p) = p + floor(p/32), so the values of a
// butterfly sit (N/16)(33/32) k, R r + floor(R r/32) and r apart; stages
// (16, N/16) and (R, 1) touch each bank pair once per half-wave, stage (16, R)
// twice (no additive padding clears all three, a host simulation shows).
constexpr int kUpN = 4096;
// Lengths with every twiddle from the table: those where the interferograms'
// errors would else exceed a library transform's (2048 points, looks 4 x 2:
// 1.1e-7 against 1.0e-7).
TDBP_HD constexpr bool up_full(int n) { return n != kUpN; }
TDBP_HD constexpr int up_threads(int n) { return n / 16; }
TDBP_HD constexpr int up_lds(int n) { return n == kOsN ? kOsLds : n + n / 32; }
TDBP_HD constexpr int up_pad(int p) { return p + (p >> 5); }

// In-register forward DFT of 8 points, natural order in and out (n = 2 n1 +
// n2, k = k1 + 4 k2).
TDBP_HD void dft8(float2* x) {
  float2 a0 = x[0], a1 = x[2], a2 = x[4], a3 = x[6];
  float2 b0 = x[1], b1 = x[3], b2 = x[5], b3 = x[7];
  dft4(a0, a1, a2, a3);
  dft4(b0, b1, b2, b3);
  b1 = c_w8(b1);
  b2 = c_mni(b2);
  b3 = c_w8_3(b3);
  x[0] = c_add(a0, b0);
  x[1] = c_add(a1, b1);
  x[2] = c_add(a2, b2);
  x[3] = c_add(a3, b3);
  x[4] = c_sub(a0, b0);
  x[5] = c_sub(a1, b1);
  x[6] = c_sub(a2, b2);
  x[7] = c_sub(a3, b3);
}

// The R-point DFTs of the 16/R sub-blocks in v.
template <int R>
TDBP_HD void up_dft_last(float2* v) {
  if constexpr (R == 16) {
    dft16(v);
  } else {
#pragma unroll
    for (int q = 0; q < 16; q += R) {
      if constexpr (R == 8) dft8(v + q);
      else dft4(v[q], v[q + 1], v[q + 2], v[q + 3]);
    }
  }
}

template <int N>
TDBP_HD void up_dif_first(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  dft16(v);
  os_apply<N, up_full(N)>(tw.first, t, v);
  float2* q = lds + up_pad(t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[up_pad(N / 16) * k] = v[k];
}
// Stage (16, R) of butterfly t mod R of sub-block t / R.
template <int N, bool DIT>
TDBP_HD void up_mid(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  constexpr int R = N / 256;
  const int j = t & (R - 1);
  float2* q = lds + up_pad(N / 16) * (t / R) + j;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[up_pad(R * r)];
  if constexpr (DIT) os_apply<N / 16, up_full(N)>(tw.mid, j, v);
  dft16(v);
  if constexpr (!DIT) os_apply<N / 16, up_full(N)>(tw.mid, j, v);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[up_pad(R * k)] = v[k];
}
template <int N>
TDBP_HD void up_dif_last(const float2* lds, int t, float2* v) {
  const float2* q = lds + up_pad(16 * t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[r];
  up_dft_last<N / 256>(v);
}
template <int N>
TDBP_HD void up_dit_first(float2* lds, int t, float2* v) {
  up_dft_last<N / 256>(v);
  float2* q = lds + up_pad(16 * t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[k] = v[k];
}
template <int N>
TDBP_HD void up_dit_last(const float2* lds, int t, const OsTwiddle& tw, float2* v) {
  const float2* q = lds + up_pad(t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[up_pad(N / 16) * r];
  os_apply<N, up_full(N)>(tw.first, t, v);
  dft16(v);
}

// Host transforms of these lengths, as os_dif_host / os_dit_host.
template <int N = kUpN>
inline void up_dif_host(float2* data, const float2* table) {
  const OsHostTables<N> tb(table);
  const OsTwiddle tw = tb.tw();
  constexpr int kT = up_threads(N);
  float2* lds = new float2[up_lds(N)];
  float2 v[16];
  for (int t = 0; t < kT; ++t) {
    for (int r = 0; r < 16; ++r) v[r] = data[t + kT * r];
    up_dif_first<N>(lds, t, tw, v);
  }
  for (int t = 0; t < kT; ++t) up_mid<N, false>(lds, t, tw, v);
  for (int t = 0; t < kT; ++t) {
    up_dif_last<N>(lds, t, v);
    for (int m = 0; m < 16; ++m) data[16 * t + m] = v[m];
  }
  delete[] lds;
}
template <int N = kUpN>
inline void up_dit_host(float2* data, const float2* table) {
  const OsHostTables<N> tb(table);
  const OsTwiddle tw = tb.tw();
  constexpr int kT = up_threads(N);
  float2* lds = new float2[up_lds(N)];
  float2 v[16];
  for (int t = 0; t < kT; ++t) {
    for (int m = 0; m < 16; ++m) v[m] = data[16 * t + m];
    up_dit_first<N>(lds, t, v);
  }
  for (int t = 0; t < kT; ++t) up_mid<N, true>(lds, t, tw, v);
  for (int t = 0; t < kT; ++t) {
    up_dit_last<N>(lds, t, tw, v);
    for (int k = 0; k < 16; ++k) data[t + kT * k] = v[k];
  }
  delete[] lds;
}

// The tables of N points on the device (os_table_values(N) values), and the ones
// that go to LDS copied into `twl` (os_mid_values(N) values); a barrier must
// follow before any transform reads them.
template <int N>
__device__ __forceinline__ OsTwiddle os_twiddles_lds(float2* twl, const float2* __restrict__ table) {
  for (int i = threadIdx.x; i < os_mid_values(N); i += blockDim.x) twl[i] = table[N + i];
  return OsTwiddle{table, twl};
}

// Entry i of the tables of n points.
__device__ __forceinline__ float2 os_table_entry(int n, int i) {
  const double pi = 3.141592653589793115997963468544185161590576171875;
  double sn, cs;
  sincos(-2.0 * pi * (double)os_table_power(n, i) / n, &sn, &cs);
  return make_float2((float)cs, (float)sn);
}

// The index again, as a value the compiler cannot connect with the first: the
// last stage's twiddles are the first's, and keeping them in 30 registers from
// one to the other would spill what the stages between need.
__device__ __forceinline__ int os_fresh(int t) {
  asm volatile("" : "+v"(t));
  return t;
}

// Device DIF by kOsThreads threads, t their index: v[m] holds value t +
// kOsThreads m of the block on entry and position 2 (t + kOsThreads (m / 2)) +
// m mod 2 of the output on return.  The twiddle tables must be ordered
// before the call.  On return every thread's remaining LDS positions are its
// own (os_dit_regs may follow without a barrier).
template <bool FULL = false>
__device__ __forceinline__ void os_dif_regs(float2* lds, int t, const OsTwiddle& tw,
                                            float2* v) {
  os_dif_first<FULL>(lds, t, tw, v);
  __syncthreads();
  os_dif_mid1<FULL>(lds, t, tw, v);
  __syncthreads();
  os_dif_mid2<FULL>(lds, t, tw, v);
  __syncthreads();
  os_dif_last(lds, t, v);
}

// Device DIT: v in the DIF output order on entry, value t + kOsThreads m of the forward transform on return.  LDS positions other
// threads may still read must not be needed by the caller afterwards.
template <bool FULL = false>
__device__ __forceinline__ void os_dit_regs(float2* lds, int t, const OsTwiddle& tw,
                                            float2* v) {
  os_dit_first(lds, t, v);
  t = os_fresh(t);
  __syncthreads();
  os_dit_mid1<FULL>(lds, t, tw, v);
  __syncthreads();
  os_dit_mid2<FULL>(lds, t, tw, v);
  __syncthreads();
  os_dit_last<FULL>(lds, t, tw, v);
}

}  // namespace tdbp
