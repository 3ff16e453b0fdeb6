// tdbp_pack.h -- the storage conversion of range-compressed samples shared by
// the pack kernel and the fused range-compression store.  Per pulse, scale =
// the power of two 2^e with max |component| / scale in [8192, 16384) for
// CF16/CBF16 and in [16384, 32768) for CI16 (0 for an all-zero pulse); each
// component is multiplied by 1/scale (exact) and rounded to FP16 (hardware
// conversion, nearest even), BF16 (nearest even on the FP32 bits) or int16
// (nearest, ties to even, held to [-32767, 32767]).  k_unify_scales then
// gives every pulse close to the largest scale of the call that largest
// scale (CF16/CBF16: within 2^16, an exact power-of-two rescale of its words;
// CI16: within 2^4, words multiplied by the power of two and rounded again;
// all-zero pulses just take it), so the pulses of a burst normally share one
// scale and the backprojection applies it once per stage of pulses instead
// of once per pixel-pulse pair.
//
// Why CI16: FP16 keeps 11 significant bits of every sample, which leaves
// ~1.3e-4 RMS relative amplitude error on distributed clutter; block
// floating point with a 16-bit significand for the pulse's largest samples
// keeps the absolute error at scale/sqrt(12), ~4x below FP16 on such data,
// at the same 4 bytes per sample.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/tdbp.h"

namespace tdbp {

// Largest stored magnitude of CI16 (symmetric, so negation never overflows).
constexpr float kI16Max = 32767.f;
// Pulses whose scale is at least M / 2^kI16Unify join the call's largest M.
constexpr int kI16Unify = 4;

__device__ __forceinline__ float pulse_scale(float maxabs, int dtype) {
  if (!(maxabs > 0.f)) return 0.f;
  const int E = (int)((__float_as_uint(maxabs) >> 23) & 0xffu);
  if (E == 0xff) return 1.f;                      // inf/NaN: no scaling
  return __uint_as_float((unsigned)max(E - (dtype == TDBP_CI16 ? 14 : 13), 1) << 23);
}
// 1/scale (exact for a power of two); 0 for the zero scale of an all-zero pulse.
__device__ __forceinline__ float pulse_inv(float sc) { return sc > 0.f ? 1.0f / sc : 0.f; }

__device__ __forceinline__ uint32_t pack_word(float re, float im, int dtype) {
  uint32_t w;
  if (dtype == TDBP_CF16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 h;
    h.x = (_Float16)re;
    h.y = (_Float16)im;
    __builtin_memcpy(&w, &h, 4);
  } else if (dtype == TDBP_CI16) {
    const float r = fminf(fmaxf(rintf(re), -kI16Max), kI16Max);
    const float i = fminf(fmaxf(rintf(im), -kI16Max), kI16Max);
    w = ((uint32_t)(int)r & 0xffffu) | ((uint32_t)(int)i << 16);
  } else {
    uint32_t a = __float_as_uint(re), c = __float_as_uint(im);
    a = (a + 0x7fffu + ((a >> 16) & 1u)) >> 16;
    c = (c + 0x7fffu + ((c >> 16) & 1u)) >> 16;
    w = (a & 0xffffu) | (c << 16);
  }
  return w;
}

// The two components of a stored word, as FP32 (exact for every format).
__device__ __forceinline__ void word_components(uint32_t w, int dtype, float* re, float* im) {
  if (dtype == TDBP_CF16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 h = __builtin_bit_cast(h2, w);
    *re = (float)h.x;
    *im = (float)h.y;
  } else if (dtype == TDBP_CI16) {
    *re = (float)(int16_t)(w & 0xffffu);
    *im = (float)((int32_t)w >> 16);
  } else {
    *re = __uint_as_float(w << 16);
    *im = __uint_as_float(w & 0xffff0000u);
  }
}

// A pulse's n samples by one workgroup: the largest |component| (NaN passed
// over, as fmaxf does), and the words: each sample at the pulse's own scale
// (inv = 1/own), then, where k_unify_scales would move the pulse to another
// scale, multiplied by f and rounded again as it does (rescale).  Two samples a
// lane and load, four loads in flight: HBM bounds both.  Rows start anywhere a
// sample (8 bytes in, 4 out) may, hence the alignment of the types.
constexpr int kPackBlock = 1024;
typedef float PackF4 __attribute__((ext_vector_type(4), aligned(8)));
typedef uint32_t PackU2 __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ float pack_max(float m, float a, float b) {
  return fmaxf(m, fmaxf(fabsf(a), fabsf(b)));
}

// The workgroup's value for every thread; `part` holds one float per wave.
__device__ __forceinline__ float block_max(float m, float* part) {
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  m = part[0];
  for (int w = 1; w < kPackBlock / 64; ++w) m = fmaxf(m, part[w]);
  return m;
}

__device__ __forceinline__ float row_max(const float2* __restrict__ y, int n, float* part) {
  const PackF4* y2 = (const PackF4*)y;
  const int n2 = n >> 1;
  float m = 0.f;
  int i = threadIdx.x;
  for (; i + 3 * kPackBlock < n2; i += 4 * kPackBlock) {
    PackF4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = y2[i + k * kPackBlock];
#pragma unroll
    for (int k = 0; k < 4; ++k) m = pack_max(pack_max(m, v[k].x, v[k].y), v[k].z, v[k].w);
  }
  for (; i < n2; i += kPackBlock) {
    const PackF4 v = y2[i];
    m = pack_max(pack_max(m, v.x, v.y), v.z, v.w);
  }
  if ((n & 1) && threadIdx.x == 0) m = pack_max(m, y[n - 1].x, y[n - 1].y);
  return block_max(m, part);
}

template <int DT>
__device__ __forceinline__ uint32_t pack_sample(float re, float im, float inv, bool rescale,
                                                float f) {
  uint32_t w = pack_word(re * inv, im * inv, DT);
  if (rescale) {
    word_components(w, DT, &re, &im);
    w = pack_word(re * f, im * f, DT);
  }
  return w;
}

template <int DT>
__device__ __forceinline__ void pack_row(const float2* __restrict__ y, int n,
                                         uint32_t* __restrict__ o, float inv, bool rescale,
                                         float f) {
  const PackF4* y2 = (const PackF4*)y;
  PackU2* o2 = (PackU2*)o;
  const int n2 = n >> 1;
  auto pair = [&](const PackF4& v) {
    return PackU2{pack_sample<DT>(v.x, v.y, inv, rescale, f),
                  pack_sample<DT>(v.z, v.w, inv, rescale, f)};
  };
  int i = threadIdx.x;
  for (; i + 3 * kPackBlock < n2; i += 4 * kPackBlock) {
    PackF4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = y2[i + k * kPackBlock];
#pragma unroll
    for (int k = 0; k < 4; ++k) o2[i + k * kPackBlock] = pair(v[k]);
  }
  for (; i < n2; i += kPackBlock) o2[i] = pair(y2[i]);
  if ((n & 1) && threadIdx.x == 0)
    o[n - 1] = pack_sample<DT>(y[n - 1].x, y[n - 1].y, inv, rescale, f);
}

// Scales that other workgroups of the same launch may be rewriting (k_pack,
// k_unify_scales): the old value and the new one do equally (unified_scale), so
// each access is one whole load or store and need not see past the caches.  (At
// device scope the loads passed by L2: k_pack on 1363 pulses 8 us slower.)
__device__ __forceinline__ float load_scale(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void store_scale(float* p, float s) {
  __hip_atomic_store(p, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The scale k_unify_scales leaves a pulse of scale s in a call whose largest
// is M.  With any of the call's scales already replaced by theirs the largest,
// and so every other pulse's, comes out the same, but for a call of zeros alone:
// there M may be 0 or 1, and the scale is 1 either way.
__host__ __device__ inline float unified_scale(float s, float M, int dtype) {
  const float lowest = dtype == TDBP_CI16 ? M * (1.0f / (1 << kI16Unify)) : M * (1.0f / 65536.0f);
  return M == 0.f ? 1.f : (s == M || (s > 0.f && s < lowest)) ? s : M;
}

}  // namespace tdbp
