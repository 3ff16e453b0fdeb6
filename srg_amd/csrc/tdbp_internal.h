// tdbp_internal.h -- device-side burst descriptor and launcher interface
// shared by the kernel and API translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/tdbp.h"

namespace tdbp {

constexpr int kWave = 64;        // CDNA wavefront
constexpr int kBlock = 256;      // 4 waves per workgroup
constexpr int kMaxStateVec = 1000;  // reference arrays timeorbit(1000)

// Everything one burst needs on the device.  Built on the host from a
// tdbp_geom; lives in kernel arguments (per-burst launch) or in a device
// array indexed by the work queue (batch).
struct BurstDev {
  const void* data;        // samples [L][S] of `dtype`
  const float* scale;      // per-pulse scale (CF16/CBF16) or nullptr
  const double* satloc;    // [L][3]
  const int16_t* dem;      // [nlines][W]
  const double* coef;      // [nlines][3]
  float2* out;             // [nlines][W]
  const double* orb_t;     // orbit arrays on device ([n], [n][3], [n][3])
  const double* orb_x;
  const double* orb_v;
  int L, S, A, W;
  int firstline, nlines, nfit, firstpix, lastpix;
  int dtype, nsv;
  int tiles_r, tiles_c;    // tile grid of this burst for the chosen variant
  int split;               // 1: the tiles are those of kSplitVariant (set_tiles)
  int* counters;           // single-burst launches: 8 tile-queue counters on the
                           //    device, zeroed by the launcher before each launch
  int cpu;                 // 1: CPU-twin arithmetic (TDBP_SEM_CPU)
  int chain;               // 1: the mixed kernel keeps the FP32 range chain
                           //    (TDBP_MIXED_CHAIN=1; default: the quadratic form)
  double rngstart, rng_hi, inv_dmrg, two_over_wvl, r_hi;
  double dmrg, four_pi_over_wvl;  // CPU twin: (R - rngstart)/dmrg, 4 pi/wvl * R
  double firstlat, firstlon, deltalat, deltalon;
  double tmid, wvl, angc0, angc1, prf;
  double xyz_mid[3], vel_mid[3];
};

// Mixed-kernel variants: per-wave pixel tile rows (cols = 64 / rows) and
// how the 4 waves of a workgroup are stacked.
constexpr int kWavesSideBySide = 0, kWavesStacked = 1, kWavesSplit = 2;
struct Variant {
  int tile_rows;     // rows of a wave tile
  int stack;         // the workgroup's waves: side by side, stacked along rows,
                     //    or all on one wave tile, each with a quarter of the
                     //    pulses
  int mfma;          // 1: the MFMA kernel (16 waves on a 16 x 16 tile; the
                     //    tile shape is that of tile_rows 4, stacked)
  int lds;           // 1: the pulse windows of the samples staged in LDS
                     //    (kLdsPulses pulses of kLdsWindow samples at a time)
};
constexpr int kNumVariants = 12;
// The tile that launches by default take instead of variants 1 and 5 (4-row
// wave tiles) for a burst with too few pixels to fill the chip (set_tiles).
constexpr int kSplitVariant = 11;
// LDS staging of the sample windows: pulses per sub-stage and samples per
// pulse window (FP32 complex in LDS: 16 x 112 x 8 B = 14 KB per workgroup,
// which with the 16 KB of pulse records leaves room for 5 workgroups in a
// CU's 160 KB; at 32 KB per workgroup only 4 were resident).
constexpr int kLdsPulses = 16;
constexpr int kLdsWindow = 112;
// The MFMA kernel addresses a burst's samples with 32-bit byte offsets.
inline bool mfma_fits(const BurstDev& b) {
  return (size_t)b.L * (size_t)b.S * (b.dtype == TDBP_CF32 ? 8u : 4u) < (size_t)0xffffffffu;
}
extern const Variant kVariants[kNumVariants];

inline int wg_rows(const Variant& v) {
  return v.stack == kWavesStacked ? 4 * v.tile_rows : v.tile_rows;
}
inline int wg_cols(const Variant& v) {
  return (v.stack == kWavesSideBySide ? 4 : 1) * (kWave / v.tile_rows);
}

// Launchers (tdbp_kernels.hip).  All return hipError_t of the launch.
hipError_t launch_fit_one(const BurstDev& b, double* coef, hipStream_t s);
// The same with the orbit table [t(n) | x(3n) | v(3n)] (host memory, read before
// the call returns) in the kernel's arguments: b.nsv <= kFitArgVec.
constexpr int kFitArgVec = 32;   // 1.8 KB; orbit files hold 11 to 17 vectors
hipError_t launch_fit_arg(const BurstDev& b, const double* orbit, double* coef, hipStream_t s);
hipError_t launch_setxyz(const BurstDev& b, double* xyz, double* xyzfit,
                         hipStream_t s);
hipError_t launch_setazoff(const BurstDev& b, double* azoff, hipStream_t s);
hipError_t launch_pair_count(const BurstDev& b, int64_t* pairs, hipStream_t s);
hipError_t launch_pixelint(const BurstDev& b, const double* xyz,
                           const double* azoff, hipStream_t s);
// variant: the one set_tiles returned for the burst.
hipError_t launch_plain(const BurstDev& b, int variant, hipStream_t s);
hipError_t launch_mixed(const BurstDev& b, int variant, hipStream_t s);
hipError_t launch_batch(const BurstDev* d_bursts, const int2* d_items,
                        const int* d_qbase, int* d_counters, int precision,
                        int variant, int dtype, int grid, hipStream_t s);
hipError_t launch_batch_fit(const BurstDev* d_bursts, int nbursts,
                            int max_lines, hipStream_t s);
hipError_t launch_zero(void* p, size_t bytes, hipStream_t s);
hipError_t launch_copy(void* d, const void* src, size_t bytes, hipStream_t s);
// The 80 header bytes of cf32 lines (`stride` samples apart) to or from
// contiguous rows on the device.
hipError_t launch_headers(void* lines, int nlines, int stride, void* rows, bool to_lines,
                          hipStream_t s);
int compare_blocks(size_t n);
hipError_t launch_compare(const float2* g, const float2* o, size_t n, double* part,
                          int blocks, hipStream_t s);
// semantics: TDBP_SEM_GPU or TDBP_SEM_CPU merge rule.
hipError_t launch_merge(float2* grid, const float2* out, size_t n, size_t grid_off,
                        int semantics, hipStream_t s);
hipError_t launch_pack(const float2* in, int L, int S, int dtype, void* out,
                       float* scale, hipStream_t s);
// Common power-of-two scale for the pulses of one packed call (k_unify_scales).
hipError_t launch_unify_scales(uint32_t* packed, size_t rowwords, int L, float* scale,
                               int dtype, hipStream_t s);
hipError_t launch_synth_clutter(float2* d, int L, int S, uint64_t seed,
                                float sigma, const float* taps, int ntaps,
                                hipStream_t s);
hipError_t launch_synth_raw(float2* d, int L, int stride, int nsamps, int npts, float sf,
                            float f0, float ramp, const double* delay, const double* carrier,
                            const float2* amp, int ntargets, float noise, uint64_t seed,
                            const void* header80, hipStream_t s);
hipError_t launch_synth_target(float2* d, const BurstDev& b, double tx,
                               double ty, double tz, float ar, float ai,
                               float res, int halfwidth, hipStream_t s);

// Blocks per CU the batch kernel keeps resident.
int batch_blocks_per_cu(int precision, int variant, int dtype);

}  // namespace tdbp
