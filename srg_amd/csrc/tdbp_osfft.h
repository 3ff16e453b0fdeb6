// tdbp_osfft.h -- the 8192-point complex FP32 FFT pair of the fused range
// compression (overlap-save blocks of one echo line, tdbp_range.hip), shared
// by the device kernels and a host check.
//
// In place, mixed radix 16 x 16 x 16 x 2.  Stage (R, s) takes, in every
// sub-block of R s values at base b and for j < s, the values b + j + s r (r <
// R) times t^r, an R-point DFT, back to b + j + s k.
// The first transform of a block (natural order in) runs stages (16, 512),
// (16, 32), (16, 2), (2, 1).  It splits the polynomial of the values, modulo
// x^N - 1 at first, into its remainders: a sub-block whose digits so far are d0,
// d1 .. stands for the bins K = d0 + 16 d1 + .. modulo 16^stage, and t = w^(s K)
// (w = e^{-2 pi i/N}), the same for all its butterflies, 1 in the first stage.
// Position p = 512 d0 + 32 d1 + 2 d2 + d3 ends with bin drev(p) = d0 + 16 d1 +
// 256 d2 + 4096 d3.  (This order out of natural order in is that of decimation
// in frequency, whose twiddles follow the butterflies; here they precede them.)
// The second transform runs decimation in time (DIT) on that order: the same
// stages in reverse with t = w^(N/(R s) j), from values in digit-reversed order
// to the forward transform in natural order.  A product of two outputs of the
// first, position by position, is the product of the spectra, so a convolution
// needs no reordering at all.  Forward sign e^{-2 pi i nk/N}; the unnormalised
// inverse of y is conj(FFT(conj(y))).
// Twiddles before the butterflies go into them: a + u b is two FMAs a component
// and a - u b = 2 a - (a + u b) a third, so a radix-16 stage is 32 butterflies of
// six FMAs, 192 instructions, where the DFT and then (or first) fifteen twiddle
// products, nine of them formed as products, took 272; the first stage of either
// transform has none.  (k_rc_os: vector issue 79 % busy, 93 % with the products.)
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "tdbp_geom.h"   // TDBP_HD

namespace tdbp {

constexpr int kOsN = 8192;          // transform length
// Threads of the device transforms: one radix-16 butterfly per thread and
// stage; thread t holds values t + kOsThreads m (m < 16) of the block in
// natural order, or positions 16 t + m in digit-reversed order.  Two ~70 KB
// workgroups fill a CU's LDS: 4 waves per SIMD.
// (1024 threads and radix 8, in an earlier form of the kernel, were slower by an
// eighth: spills at 64 VGPRs, and every barrier waits for 16 waves.)
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

// LDS layout: position p at os_pad(p) = p + floor(p / 32).  Every access of the
// transforms then touches each pair of the 64 LDS banks once per half-wave: stages
// (16, 512) and (16, 32) 32 consecutive positions, (16, 2) 32 positions 32 apart.
// The values of one butterfly sit a compile-time distance apart (528, 33 and 2
// values), so every LDS address is a base plus an immediate.
constexpr int kOsLds = kOsN + kOsN / 32;
TDBP_HD constexpr int os_pad(int p) { return p + (p >> 5); }

// a + u b and a - u b, in place; MI: u times -i in the place of u.
template <bool MI>
TDBP_HD void bfly(float2& a, float2& b, float2 u) {
  const float2 p = MI ? make_float2(fmaf(u.y, b.x, fmaf(u.x, b.y, a.x)),
                                    fmaf(u.y, b.y, fmaf(-u.x, b.x, a.y)))
                      : make_float2(fmaf(-u.y, b.y, fmaf(u.x, b.x, a.x)),
                                    fmaf(u.y, b.x, fmaf(u.x, b.y, a.y)));
  b = make_float2(fmaf(2.f, a.x, -p.x), fmaf(2.f, a.y, -p.y));
  a = p;
}

// In-register forward DFT of R values x_r t^r (R = 2, 4, 8, 16), natural order in
// and out, from R/2 twiddles T: the powers t^(R/2), .., t^2, t, the last three
// with their multiples by w8 (t^2) and w16^k, k < 4 (t) -- w16^(k + 4) = -i w16^k
// and the like need none.  Level by level, the DFTs of 2, 4, .. values.
template <int R>
TDBP_HD void dft_tw(float2* x, const float2* T) {
  if constexpr (R == 2) {
    bfly<false>(x[0], x[1], T[0]);
  } else {
    // DFTs of the even and of the odd values, at t^2; then both together at t.
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int r = 0; r < R / 2; ++r) {
      e[r] = x[2 * r];
      o[r] = x[2 * r + 1];
    }
    dft_tw<R / 2>(e, T);
    dft_tw<R / 2>(o, T);
    const float2* u = T + R / 4;
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      if (k < R / 4) bfly<false>(e[k], o[k], u[k]);
      else bfly<true>(e[k], o[k], u[k - R / 4]);
      x[k] = e[k];
      x[k + R / 2] = o[k];
    }
  }
}
// T[i] of dft_tw<R> for t = w_N^e is w_N^m, m the return value: R/2 values, the
// last R/4 (1 for R = 2) for t itself, those before them for t^2, ..
TDBP_HD int dft_tw_power(int n, int e, int R, int i) {
  while (R > 2 && i < R / 4) {
    e *= 2;
    R /= 2;
  }
  const int k = R > 2 ? i - R / 4 : 0;
  return (e + k * (n / R)) % n;
}

// The twiddles of a stage as [i][index], i < 8, so that the lanes of a wave read
// them in order, every one rounded once from FP64.  Per length N: in global
// memory (the caches keep them) the last stages of the first transform [8][N/16]
// (by thread) and of the second [8][N/16] (by j), for 8192 points the third of
// the first [8][256] (by sub-block); in LDS the second stage of the first [8][16]
// (by sub-block), stage (16, N/256) of the second (by j), for 8192 points its
// stage (16, 2) (by j).
TDBP_HD constexpr int os_at_last2(int n) { return n / 2; }
TDBP_HD constexpr int os_at_third(int n) { return n; }
TDBP_HD constexpr int os_at_lds(int n) { return n == kOsN ? n + 2048 : n; }
constexpr int kOsMid2 = 128;   // in the LDS part: the second transform's stages
TDBP_HD constexpr int os_at_two(int n) { return kOsMid2 + n / 32; }
TDBP_HD constexpr int os_lds_values(int n) { return os_at_two(n) + (n == kOsN ? 16 : 0); }
TDBP_HD constexpr int os_table_values(int n) { return os_at_lds(n) + os_lds_values(n); }
struct OsTwiddle {
  const float2* g;   // the length's whole table
  const float2* s;   // its LDS part
};
// Bins (modulo 256, 4096) of the sub-blocks after two and three stages.
TDBP_HD int os_bin2(int b) { return (b >> 4) + 16 * (b & 15); }
TDBP_HD int os_bin3(int b) { return (b >> 8) + 16 * ((b >> 4) & 15) + 256 * (b & 15); }
// Entry i of a length's tables is w_n^m, m the return value.
TDBP_HD int os_table_power(int n, int i) {
  const int q = n / 16, r = n / 256;   // threads, radix of the last stage
  if (i < n / 2) {   // the first transform's last stage
    const int k = i / q, t = i % q;
    if (n == kOsN) return os_bin3(8 * t + k) % n;   // radix 2
    const int h = r / 2;                            // twiddles of one butterfly
    return dft_tw_power(n, os_bin2((16 / r) * t + k / h), r, k % h);
  }
  i -= n / 2;
  if (i < n / 2) return dft_tw_power(n, i % q, 16, i / q);
  i -= n / 2;
  if (n == kOsN) {
    if (i < 2048) return dft_tw_power(n, 2 * os_bin2(i % 256), 16, i / 256);
    i -= 2048;
  }
  if (i < kOsMid2) return dft_tw_power(n, r * (i % 16), 16, i / 16);
  i -= kOsMid2;
  if (i < 8 * r) return dft_tw_power(n, 16 * (i % r), 16, i / r);
  i -= 8 * r;
  return dft_tw_power(n, 256 * (i % 2), 16, i / 2);
}

// The eight twiddles tab[i N + j].
template <int N>
TDBP_HD void os_load_tw(const float2* tab, int j, float2* T) {
#pragma unroll
  for (int i = 0; i < 8; ++i) T[i] = tab[i * N + j];
}

// The values of a radix-16 stage, at lds[a0 + STEP r].
template <int STEP>
TDBP_HD void os_read16(const float2* lds, int a0, float2* v) {
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = lds[a0 + STEP * r];
}
template <int STEP>
TDBP_HD void os_write16(float2* lds, int a0, const float2* v) {
#pragma unroll
  for (int k = 0; k < 16; ++k) lds[a0 + STEP * k] = v[k];
}
// The stage: read, DFT with the twiddles T, write back in place.
template <int STEP>
TDBP_HD void os_stage16(float2* lds, int a0, const float2* T, float2* v) {
  os_read16<STEP>(lds, a0, v);
  dft_tw<16>(v, T);
  os_write16<STEP>(lds, a0, v);
}

// The twiddles from global memory of thread t: the first transform's third and
// last stage, the second's last.
TDBP_HD void os_tw_third(const OsTwiddle& tw, int t, float2* T) {
  os_load_tw<256>(tw.g + os_at_third(kOsN), t >> 1, T);
}
template <int N>
TDBP_HD void os_tw_last1(const OsTwiddle& tw, int t, float2* T) {
  os_load_tw<N / 16>(tw.g, t, T);
}
template <int N>
TDBP_HD void os_tw_last2(const OsTwiddle& tw, int t, float2* T) {
  os_load_tw<N / 16>(tw.g + os_at_last2(N), t, T);
}

// The stages of thread t.  Stage (16, 512): butterfly t, values t + 512 r,
// which the thread holds in registers (first transform: from registers; second:
// into them).  Stage (16, 32): butterfly j = t mod 32 of sub-block t / 32.
// Stage (16, 2): butterfly t mod 2 of sub-block t / 2.  Stage (2, 1): the eight
// pairs at positions 16 t + 2 h, held in registers as v[2h], v[2h + 1].  All but
// the first of these stay within the 1024 positions of a wave (stages (16, 2) and
// (2, 1) with their threads in another order there, os_mid_thread), so that only
// stage (16, 512) needs the workgroup's barrier on its other side.
TDBP_HD void os_dif_first(float2* lds, int t, float2* v) {
  dft16(v);
  float2* q = lds + os_pad(t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[528 * k] = v[k];
}
TDBP_HD void os_dif_mid1(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  float2 T[8];
  os_load_tw<16>(tw.s, t >> 5, T);
  os_stage16<33>(lds, 528 * (t >> 5) + (t & 31), T, v);
}
TDBP_HD void os_dif_mid2(const float2* lds, int t2, const float2* T, float2* v) {
  os_read16<2>(lds, 33 * (t2 >> 1) + (t2 & 1), v);
  dft_tw<16>(v, T);
}
TDBP_HD void os_dif_pairs(const float2* T, float2* v) {
#pragma unroll
  for (int h = 0; h < 8; ++h) bfly<false>(v[2 * h], v[2 * h + 1], T[h]);
}
TDBP_HD void os_dit_pairs(float2* v) {
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    const float2 a = v[2 * h], b = v[2 * h + 1];
    v[2 * h] = c_add(a, b);
    v[2 * h + 1] = c_sub(a, b);
  }
}
TDBP_HD void os_dit_mid1(int t2, const OsTwiddle& tw, float2* v) {
  float2 T[8];
  os_load_tw<2>(tw.s + os_at_two(kOsN), t2 & 1, T);
  dft_tw<16>(v, T);
}
TDBP_HD void os_dit_write(float2* lds, int t2, const float2* v) {
  os_write16<2>(lds, 33 * (t2 >> 1) + (t2 & 1), v);
}
TDBP_HD void os_dit_mid2(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  float2 T[8];
  os_load_tw<32>(tw.s + kOsMid2, t & 31, T);
  os_stage16<33>(lds, 528 * (t >> 5) + (t & 31), T, v);
}
TDBP_HD void os_dit_last(const float2* lds, int t, const float2* T, float2* v) {
  const float2* q = lds + os_pad(t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[528 * r];
  dft_tw<16>(v, T);
}

// The thread of stages (16, 2) and (2, 1) that thread t is: lanes r and r + 32 of
// a wave are a pair 2 q, 2 q + 1.
TDBP_HD int os_mid_thread(int t) { return (t & ~63) | ((t & 31) << 1) | ((t >> 5) & 1); }
// Between those stages the values change hands within the pairs, position 32 q +
// j + 2 k of thread 2 q + j as v[k] against 32 q + 16 j + m as v[m]: the second
// half of the lower lane's values against the first half of the upper's, which
// v_permlane32_swap does for two registers at once, in the place of an LDS write
// and read (a third of the transforms' LDS cycles).  swap(a, b): the upper
// lane's a for the lower lane's b.
template <class V, class S>
TDBP_HD void pairs_gather(V* v, const S& swap) {
  V w[16];
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    w[2 * h] = v[h];
    w[2 * h + 1] = v[h + 8];
    swap(w[2 * h], w[2 * h + 1]);
  }
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = w[m];
}
template <class V, class S>
TDBP_HD void pairs_scatter(V* v, const S& swap) {
  V w[16];
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    w[h] = v[2 * h];
    w[h + 8] = v[2 * h + 1];
    swap(w[h], w[h + 8]);
  }
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = w[m];
}

// Host transforms (the check of the device code): the same stages, layout
// and per-thread registers, thread by thread, the pairs of stages (16, 2) and
// (2, 1) exchanged as the device's lanes do.
// os_dif_host: data in natural order -> data[p] = X[drev(p)].
// os_dit_host: data[p] = Y[drev(p)] -> data in natural order, the forward
// transform of Y.
template <int N>
struct OsHostTables {
  float2 v[os_table_values(N)];
  explicit OsHostTables(const float2* table) {   // w^m of 8192 points
    for (int i = 0; i < os_table_values(N); ++i) v[i] = table[kOsN / N * os_table_power(N, i)];
  }
  OsTwiddle tw() const { return OsTwiddle{v, v + os_at_lds(N)}; }
};
struct OsLanes {   // a register of lanes r and r + 32
  float2 lane[2];
};
struct OsHostSwap {
  void operator()(OsLanes& a, OsLanes& b) const {
    const float2 upper = a.lane[1];
    a.lane[1] = b.lane[0];
    b.lane[0] = upper;
  }
};
template <class F>
inline void os_host_pairs(float2 (*v)[16], F&& exchange) {   // v: all threads' registers
  for (int t = 0; t < kOsThreads; ++t) {
    if (t & 32) continue;
    OsLanes w[16];
    for (int m = 0; m < 16; ++m) w[m] = OsLanes{{v[t][m], v[t + 32][m]}};
    exchange(w);
    for (int m = 0; m < 16; ++m) {
      v[t][m] = w[m].lane[0];
      v[t + 32][m] = w[m].lane[1];
    }
  }
}
inline void os_dif_host(float2* data, const float2* table) {
  const OsHostTables<kOsN> tb(table);
  const OsTwiddle tw = tb.tw();
  float2* lds = new float2[kOsLds];
  float2(*v)[16] = new float2[kOsThreads][16];
  float2 T[8];
  for (int t = 0; t < kOsThreads; ++t) {
    for (int r = 0; r < 16; ++r) v[t][r] = data[t + kOsThreads * r];
    os_dif_first(lds, t, v[t]);
  }
  for (int t = 0; t < kOsThreads; ++t) os_dif_mid1(lds, t, tw, v[t]);
  for (int t = 0; t < kOsThreads; ++t) {
    const int t2 = os_mid_thread(t);
    os_tw_third(tw, t2, T);
    os_dif_mid2(lds, t2, T, v[t]);
  }
  os_host_pairs(v, [](OsLanes* w) { pairs_gather(w, OsHostSwap()); });
  for (int t = 0; t < kOsThreads; ++t) {
    const int t2 = os_mid_thread(t);
    os_tw_last1<kOsN>(tw, t2, T);
    os_dif_pairs(T, v[t]);
    for (int m = 0; m < 16; ++m) data[16 * t2 + m] = v[t][m];
  }
  delete[] v;
  delete[] lds;
}
inline void os_dit_host(float2* data, const float2* table) {
  const OsHostTables<kOsN> tb(table);
  const OsTwiddle tw = tb.tw();
  float2* lds = new float2[kOsLds];
  float2(*v)[16] = new float2[kOsThreads][16];
  float2 T[8];
  for (int t = 0; t < kOsThreads; ++t) {
    for (int m = 0; m < 16; ++m) v[t][m] = data[16 * os_mid_thread(t) + m];
    os_dit_pairs(v[t]);
  }
  os_host_pairs(v, [](OsLanes* w) { pairs_scatter(w, OsHostSwap()); });
  for (int t = 0; t < kOsThreads; ++t) {
    os_dit_mid1(os_mid_thread(t), tw, v[t]);
    os_dit_write(lds, os_mid_thread(t), v[t]);
  }
  for (int t = 0; t < kOsThreads; ++t) os_dit_mid2(lds, t, tw, v[t]);
  for (int t = 0; t < kOsThreads; ++t) {
    os_tw_last2<kOsN>(tw, t, T);
    os_dit_last(lds, t, T, v[t]);
    for (int k = 0; k < 16; ++k) data[t + kOsThreads * k] = v[t][k];
  }
  delete[] v;
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
TDBP_HD constexpr int up_threads(int n) { return n / 16; }
TDBP_HD constexpr int up_lds(int n) { return n == kOsN ? kOsLds : n + n / 32; }
TDBP_HD constexpr int up_pad(int p) { return p + (p >> 5); }

// The plain R-point DFTs of the 16/R sub-blocks in v.
template <int R>
TDBP_HD void up_dft_plain(float2* v) {
  if constexpr (R == 16) {
    dft16(v);
  } else if constexpr (R == 4) {
#pragma unroll
    for (int q = 0; q < 16; q += 4) dft4(v[q], v[q + 1], v[q + 2], v[q + 3]);
  } else {   // 8 points: n = 2 n1 + n2, k = k1 + 4 k2
#pragma unroll
    for (int q = 0; q < 16; q += 8) {
      float2* x = v + q;
      float2 a[4], b[4];
      for (int k = 0; k < 4; ++k) {
        a[k] = x[2 * k];
        b[k] = x[2 * k + 1];
      }
      dft4(a[0], a[1], a[2], a[3]);
      dft4(b[0], b[1], b[2], b[3]);
      b[1] = c_w8(b[1]);
      b[2] = c_mni(b[2]);
      b[3] = c_w8_3(b[3]);
      for (int k = 0; k < 4; ++k) {
        x[k] = c_add(a[k], b[k]);
        x[k + 4] = c_sub(a[k], b[k]);
      }
    }
  }
}

template <int N>
TDBP_HD void up_dif_first(float2* lds, int t, float2* v) {
  dft16(v);
  float2* q = lds + up_pad(t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[up_pad(N / 16) * k] = v[k];
}
// Stage (16, R) of butterfly t mod R of sub-block t / R, of the second transform
// (DIT) or the first.
template <int N, bool DIT>
TDBP_HD void up_mid(float2* lds, int t, const OsTwiddle& tw, float2* v) {
  constexpr int R = N / 256;
  const int j = t & (R - 1), b = t / R;
  float2* q = lds + up_pad(N / 16) * b + j;
  float2 T[8];
  if constexpr (DIT) os_load_tw<R>(tw.s + kOsMid2, j, T);
  else os_load_tw<16>(tw.s, b, T);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[up_pad(R * r)];
  dft_tw<16>(v, T);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[up_pad(R * k)] = v[k];
}
template <int N>
TDBP_HD void up_dif_last(const float2* lds, int t, const float2* T, float2* v) {
  constexpr int R = N / 256;
  const float2* q = lds + up_pad(16 * t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[r];
#pragma unroll
  for (int k = 0; k < 16 / R; ++k) dft_tw<R>(v + R * k, T + R / 2 * k);
}
template <int N>
TDBP_HD void up_dit_first(float2* lds, int t, float2* v) {
  up_dft_plain<N / 256>(v);
  float2* q = lds + up_pad(16 * t);
#pragma unroll
  for (int k = 0; k < 16; ++k) q[k] = v[k];
}
template <int N>
TDBP_HD void up_dit_last(const float2* lds, int t, const float2* T, float2* v) {
  const float2* q = lds + up_pad(t);
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = q[up_pad(N / 16) * r];
  dft_tw<16>(v, T);
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
    up_dif_first<N>(lds, t, v);
  }
  for (int t = 0; t < kT; ++t) up_mid<N, false>(lds, t, tw, v);
  for (int t = 0; t < kT; ++t) {
    float2 T[8];
    os_tw_last1<N>(tw, t, T);
    up_dif_last<N>(lds, t, T, v);
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
    float2 T[8];
    os_tw_last2<N>(tw, t, T);
    up_dit_last<N>(lds, t, T, v);
    for (int k = 0; k < 16; ++k) data[t + kT * k] = v[k];
  }
  delete[] lds;
}

// The tables of N points on the device (os_table_values(N) values), and the ones
// that go to LDS copied into `twl` (os_lds_values(N) values); a barrier must
// follow before any transform reads them.
template <int N>
__device__ __forceinline__ OsTwiddle os_twiddles_lds(float2* twl, const float2* __restrict__ table) {
  for (int i = threadIdx.x; i < os_lds_values(N); i += blockDim.x)
    twl[i] = table[os_at_lds(N) + i];
  return OsTwiddle{table, twl};
}

// Entry i of the tables of n points.
__device__ __forceinline__ float2 os_table_entry(int n, int i) {
  const double pi = 3.141592653589793115997963468544185161590576171875;
  double sn, cs;
  sincos(-2.0 * pi * (double)os_table_power(n, i) / n, &sn, &cs);
  return make_float2((float)cs, (float)sn);
}

// Orders the LDS accesses of a wave's lanes (which the hardware executes in
// order): between stages whose values stay within a wave.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v_permlane32_swap of the two components.
struct LaneSwap {
  static __device__ __forceinline__ void one(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  }
  __device__ __forceinline__ void operator()(float2& a, float2& b) const {
    one(a.x, b.x);
    one(a.y, b.y);
  }
};

// Device, first transform by kOsThreads threads, t their index (whole waves from
// a multiple of 64 on): v[m] holds value t + kOsThreads m of the block on entry
// and position 16 os_mid_thread(t) + m of the output on return.  The LDS twiddles
// must be ordered before the call.  Twiddles from global memory are loaded a stage
// ahead; so is what `ahead` loads for the caller, before the last stage.  On return
// every LDS position is free for the wave that os_dit_regs writes it from (which
// may follow without a barrier).
template <class F>
__device__ __forceinline__ void os_dif_regs(float2* lds, int t, const OsTwiddle& tw, float2* v,
                                            F&& ahead) {
  const int t2 = os_mid_thread(t);
  float2 T[8], U[8];
  os_dif_first(lds, t, v);
  os_tw_third(tw, t2, T);
  __syncthreads();
  os_dif_mid1(lds, t, tw, v);
  os_tw_last1<kOsN>(tw, t2, U);
  wave_sync();
  os_dif_mid2(lds, t2, T, v);
  ahead();
  pairs_gather(v, LaneSwap());
  os_dif_pairs(U, v);
}

// Device, second transform (DIT): v in the first's output order on entry, value
// t + kOsThreads m of the forward transform on return.  LDS positions other
// threads may still read must not be needed by the caller afterwards.
__device__ __forceinline__ void os_dit_regs(float2* lds, int t, const OsTwiddle& tw,
                                            float2* v) {
  const int t2 = os_mid_thread(t);
  float2 T[8];
  os_dit_pairs(v);
  pairs_scatter(v, LaneSwap());
  os_dit_mid1(t2, tw, v);
  wave_sync();
  os_dit_write(lds, t2, v);
  os_tw_last2<kOsN>(tw, t, T);
  wave_sync();
  os_dit_mid2(lds, t, tw, v);
  __syncthreads();
  os_dit_last(lds, t, T, v);
}

// An index as a value the compiler cannot connect with the one it was made from:
// what is computed from it is not kept from one use to another.
__device__ __forceinline__ int os_fresh(int t) {
  asm volatile("" : "+v"(t));
  return t;
}

}  // namespace tdbp
