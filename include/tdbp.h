/*
 * tdbp.h -- C ABI of the MI355X time-domain backprojection (TDBP) engine.
 *
 * Library: srg_amd/libsrg_tdbp.so (HIP, gfx950).  All entry points are
 * extern "C" with plain pointers and sizes.  "d_" arguments are device
 * pointers (HBM), everything else is host memory.  Streams are hipStream_t
 * passed as void* (NULL = the null stream).
 *
 * Three layers:
 *   1. The drop-in: azimuth_compress_, the symbol the reference Fortran
 *      burst driver calls (by-reference arguments, host buffers, fds).
 *   2. The operator API: the reference's device stages (setxyz, the aperture
 *      fit, setazoff, pixelint) on device buffers, plus the fused burst
 *      backprojection in FP64 ("plain") or mixed precision.
 *   3. The batch API: many uneven bursts in one persistent launch with a
 *      device work queue, captured in a hipGraph.
 * Errors: every int-returning call returns a tdbp_status; the message of the
 * last failure on the calling thread is tdbp_last_error().
 */
#ifndef SRG_TDBP_H
#define SRG_TDBP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum {
  TDBP_OK = 0,
  TDBP_ERR_ARG = 1,     /* invalid argument or geometry            */
  TDBP_ERR_HIP = 2,     /* HIP runtime error                        */
  TDBP_ERR_NODEV = 3,   /* no usable gfx950 device                  */
  TDBP_ERR_IO = 4,      /* DEM / .geo file read or write failed     */
  TDBP_ERR_NOMEM = 5,   /* device or host allocation failed         */
  TDBP_ERR_LIMIT = 6    /* request exceeds a documented size limit  */
} tdbp_status;

/* Precision of the per-burst kernel. */
typedef enum {
  TDBP_PLAIN_FP64 = 0,  /* FP64 range, phase and accumulator; FP32 lerp    */
  TDBP_MIXED = 1        /* FP64 per-tile reference, FP32 differential range */
} tdbp_precision;

/* Storage type of range-compressed samples. */
typedef enum {
  TDBP_CF32 = 0,        /* complex float, 8 B/sample                       */
  TDBP_CF16 = 1,        /* complex IEEE half + FP32 scale per pulse, 4 B   */
  TDBP_CBF16 = 2,       /* complex bfloat16 + FP32 scale per pulse, 4 B    */
  TDBP_CI16 = 3         /* complex int16 (two's complement, re in the low
                           half) + FP32 scale per pulse, 4 B: block floating
                           point, max |component| / scale in [2^14, 2^15),
                           a 16-bit significand for the largest samples   */
} tdbp_dtype;

/* Which reference entry's arithmetic a burst follows.  The two reference
 * implementations of the path differ in three places:
 *   GPU entry (sentinel/azimuth_compress.cu:61-79): FP32 lerp weights and
 *     products, output multiplied by float(1/(azend-azstart)); .geo pixel
 *     replaced where fabs((double)Re) > 1e-18 (:527-531).
 *   CPU twin (sentinel/azimuth_compress_cpu.c:68-82): lerp in FP64 rounded to
 *     cf32, phase 4*pi/wvl*range in FP64, no scaling; .geo pixel replaced
 *     where abs((int)Re) > 1e-18 (:386-388), which for the reference's own
 *     build (gcc without -O, build_proc:10) means 1 <= |Re| < 2^31 (x86's
 *     truncating conversion gives INT_MIN beyond that, and abs keeps it
 *     negative).  A window of one line is skipped (:254-257). */
typedef enum {
  TDBP_SEM_GPU = 0,
  TDBP_SEM_CPU = 1
} tdbp_semantics;

/*
 * Burst geometry: the scalars the reference driver derives per burst
 * (sentinel/backprojectgpusub.f90:193-235) and the DEM window the entry
 * point derives from latlons (sentinel/azimuth_compress.cu:295-301, :378-379).
 */
typedef struct tdbp_geom {
  int32_t rawdatalines;   /* L: pulses in the burst                        */
  int32_t samples;        /* S: samples per pulse (row stride)             */
  int32_t aperture;       /* A: integration length in pulses               */
  int32_t numstatevec;    /* orbit state vectors (>= 4)                    */
  double rngstart, rngend, dmrg, wvl, prf, angc0, angc1, tmid;
  double xyz_mid[3], vel_mid[3];
  const double *timeorbit;   /* host [numstatevec]                         */
  const double *xx, *vv;     /* host [numstatevec][3] (Fortran xx(3,n))    */
  int32_t demwidth;       /* W: DEM row length                             */
  int32_t firstline;      /* first DEM line of the window                  */
  int32_t nlines;         /* window lines                                  */
  int32_t firstpix, lastpix;  /* pixel range (lastpix may equal W)         */
  double firstlat, firstlon, deltalat, deltalon;
  int32_t fit_last_line;  /* 0: like the reference loop, the last window
                             line gets no aperture fit and stays zero; 1:
                             fit it like the others                       */
  int32_t semantics;      /* tdbp_semantics: output scale and lerp of the
                             GPU entry (0) or of the CPU twin (1)         */
} tdbp_geom;

/* ---------------------------------------------------------------- drop-in */

/* Replaces sentinel/azimuth_compress.cu:181-214 (called from
 * sentinel/backprojectgpusub.f90:244-247).  Same 33 by-reference arguments,
 * same effect: backproject one burst onto DEM lines derived from latlons and
 * merge into the .geo file behind *fdout (pixel replaced where
 * |Re| > 1e-18).  Unused, as in the reference: tstart, tend, t, dtaz,
 * iaperture.  Environment: TDBP_PRECISION=fp64|mixed_i16|mixed_fp16|mixed_bf16|mixed_cf32
 * (default fp64), TDBP_FIT_LAST_LINE=0|1 (default 0).  void like the
 * reference; failures are reported on stderr and leave the .geo unchanged. */
void azimuth_compress_(void *burstdata, double *satloc, int *rawdatalines,
                       int *samplesPerBurst, int *demwidth, int *demlength,
                       int *fdout, int *fddem, double *deltalat,
                       double *deltalon, double *firstlat, double *firstlon,
                       double *latlons, double *timeorbit, double *xx,
                       double *vv, int *numstatevec, double *rngstart,
                       double *rngend, double *tstart, double *tend,
                       double *tmid, double *xyz_mid, double *vel_mid,
                       double *t, double *dtaz, double *dmrg, double *wvl,
                       int *aperture, int *iaperture, double *angc0,
                       double *angc1, double *prf);

/* Replaces the CPU twin sentinel/azimuth_compress_cpu.c:178-213 (called
 * from sentinel/backprojectcpusub.f90:243-246) with the same 33 arguments:
 * the sum runs on the device with the CPU twin's arithmetic
 * (TDBP_SEM_CPU: FP64 lerp rounded to cf32, no 1/(azend-azstart) scale), the
 * .geo merge keeps its integer-abs rule (1 <= |Re| < 2^31), and a burst whose
 * DEM window is one line is skipped with the reference's message.  Same
 * environment knobs and status calls as azimuth_compress_. */
void azimuth_compress_cpu_(void *burstdata, double *satloc, int *rawdatalines,
                           int *samplesPerBurst, int *demwidth, int *demlength,
                           int *fdout, int *fddem, double *deltalat,
                           double *deltalon, double *firstlat, double *firstlon,
                           double *latlons, double *timeorbit, double *xx,
                           double *vv, int *numstatevec, double *rngstart,
                           double *rngend, double *tstart, double *tend,
                           double *tmid, double *xyz_mid, double *vel_mid,
                           double *t, double *dtaz, double *dmrg, double *wvl,
                           int *aperture, int *iaperture, double *angc0,
                           double *angc1, double *prf);

/* Status of the last azimuth_compress_ / azimuth_compress_cpu_ call on this thread (the reference
 * entry returns nothing). */
int tdbp_dropin_status(void);

/* With TDBP_DROPIN_ASYNC=1, azimuth_compress_ returns once the burst is on the
 * device and its sum is enqueued; the .geo read-merge-write of each burst
 * runs on a worker thread in call order, overlapping the next call's upload.
 * With TDBP_BATCH=1 (the deferred mode of the batched extension) a call only
 * stages its burst on the device; the staged bursts run as one batch (one
 * persistent launch, the .geo merges on the device in call order, one
 * read-merge-write of the rows they cover) when tdbp_dropin_flush is called,
 * before a call for another .geo file (device and inode of fdout), DEM
 * width, entry or precision or a call without TDBP_BATCH=1, and when the
 * staged bytes would pass TDBP_BATCH_BYTES (default half the free device
 * memory).  The .geo ends as the per-call read-merge-writes would leave it.
 * The caller must call tdbp_dropin_flush before the process ends: bursts
 * still staged at exit are reported on stderr and not written.
 * tdbp_dropin_flush runs the deferred bursts, waits until every queued burst
 * is written and returns the first error among them (0 = all written), then
 * clears it.  The queue is also drained when the process exits.  No
 * reference counterpart. */
int tdbp_dropin_flush(void);

/* Phase times (ms) of the last azimuth_compress_ call: [0] total, [1] DEM
 * read, [2] DEM + satloc + burst upload, [3] device compute (pack, fit,
 * sum), [4] .geo read (overlaps [3]), [5] .geo merge after the sum (with
 * what the rows' upload, which overlaps [3], has left), [6] .geo download
 * and write from the first piece's arrival (eight pieces, each written
 * while the next comes down).  Fills min(n, 7) values, returns 7.  No reference
 * counterpart (the reference prints its timers when enabled,
 * sentinel/azimuth_compress.cu:492-505, commented out). */
int tdbp_dropin_timing(double *ms, int n);

/* ------------------------------------------------------------- runtime */

const char *tdbp_last_error(void);
/* Number of visible HIP devices (sentinel/howmanygpus.cu:1-9). */
int tdbp_device_count(void);
/* Select the device and check it is gfx950; idempotent. */
int tdbp_init(int device);

void *tdbp_dev_alloc(size_t bytes);
int tdbp_dev_free(void *d_ptr);
int tdbp_memcpy_htod(void *d_dst, const void *src, size_t bytes, void *stream);
/* Host (pageable) to device through the library's two pinned 32 MB staging
 * chunks: copy threads fill one chunk while the DMA engine drains the other
 * (~50 GB/s, where a copy from pageable memory through the runtime's own
 * staging ran at 20-30 GB/s).  Returns once every byte has left `src`, which
 * the caller may then reuse; the last DMAs may still run, ordered before
 * later work on `stream`.  Calls from several threads take turns.  No
 * reference counterpart (the reference's upload is one cudaMemcpy per
 * burst, sentinel/azimuth_compress.cu:367-368). */
int tdbp_memcpy_htod_staged(void *d_dst, const void *src, size_t bytes, void *stream);
int tdbp_memcpy_dtoh(void *dst, const void *d_src, size_t bytes, void *stream);
int tdbp_memcpy_dtod(void *d_dst, const void *d_src, size_t bytes, void *stream);
/* Device-to-device copy with a copy kernel (graph-capture safe). */
int tdbp_dev_copy(void *d_dst, const void *d_src, size_t bytes, void *stream);
/* Zero device memory with a fill kernel (graph-capture safe). */
int tdbp_dev_zero(void *d_ptr, size_t bytes, void *stream);
int tdbp_stream_create(void **stream);
int tdbp_stream_destroy(void *stream);
int tdbp_stream_sync(void *stream);
int tdbp_device_sync(void);
int tdbp_event_create(void **event);
int tdbp_event_destroy(void *event);
int tdbp_event_record(void *event, void *stream);
int tdbp_event_elapsed_ms(void *start, void *stop, float *ms);
/* Later work on `stream` waits for `event` (recorded on another stream). */
int tdbp_stream_wait_event(void *stream, void *event);
/* HBM bytes free / total on the current device. */
int tdbp_mem_info(size_t *free_bytes, size_t *total_bytes);

/* Window derivation of the entry point: sentinel/azimuth_compress.cu:295-301
 * (lines) and :378-379 (pixels). */
void tdbp_window(const double *latlons, double firstlat, double firstlon,
                 double deltalat, double deltalon, int demwidth, int demlength,
                 int *firstline, int *lastline, int *firstpix, int *lastpix);

/* Host Hermite orbit interpolation at m times (sentinel/intp_orbit.f90:6-20
 * per time, as sentinel/sentineltimingsub.f90:59-65 builds per-pulse
 * positions).  pos, vel: [m][3]; either may be NULL. */
int tdbp_orbit_interp(const double *timeorbit, const double *xx,
                      const double *vv, int numstatevec, const double *times,
                      int m, double *pos, double *vel);

/* ---------------------------------------------------- operator API */

/* setxyz (sentinel/azimuth_compress.cu:85-151): ECEF of window pixels
 * [firstpix, lastpix] (zero elsewhere, like the CPU twin) and the three fit
 * nodes per line.  d_dem: int16 [nlines][W]; d_xyz: f64 [nlines][W][3];
 * d_xyzfit: f64 [nlines][9] (may be NULL). */
int tdbp_setxyz(const tdbp_geom *g, const int16_t *d_dem, double *d_xyz,
                double *d_xyzfit, void *stream);

/* Aperture-centre parabola per window line (the host loop of
 * sentinel/azimuth_compress.cu:438-481 with orbitrangetime_), computed on
 * the device.  d_coef: f64 [nlines][3].  Lines beyond the fit (the last
 * line when fit_last_line == 0) get coefficients (0, 0, 0), which setazoff
 * maps to -1. */
int tdbp_fit_aperture(const tdbp_geom *g, const int16_t *d_dem, double *d_coef,
                      void *stream);

/* setazoff (sentinel/azimuth_compress.cu:154-178).  d_azoff: f64
 * [nlines][W], -1 outside [firstpix, lastpix] and outside the valid band. */
int tdbp_setazoff(const tdbp_geom *g, const double *d_coef, double *d_azoff,
                  void *stream);

/* Pixel-pulse pairs visited per window line (sum of azend-azstart over
 * pixels with azoff > 0): the work measure.  d_pairs: int64 [nlines]. */
int tdbp_pair_count(const tdbp_geom *g, const double *d_coef, int64_t *d_pairs,
                    void *stream);

/* Range-compressed samples of one burst on the device. */
typedef struct tdbp_samples {
  const void *d_data;     /* [L][S] of the dtype                          */
  const float *d_scale;   /* [L] per-pulse scale (CF16/CBF16/CI16), else
                             NULL                                         */
  int32_t dtype;          /* tdbp_dtype                                   */
} tdbp_samples;

/* Convert cf32 samples to CF16/CBF16/CI16 with a per-pulse FP32 scale
 * (value = stored * scale).  Each pulse first gets the power of two with
 * max |component| / scale in [2^13, 2^14) (CF16/CBF16, rounded to nearest
 * even) or [2^14, 2^15) (CI16: each component rounded to the nearest
 * integer, ties to even, and held to [-32767, 32767]).  Then every pulse
 * whose scale is within 2^16 (CF16/CBF16) or 2^4 (CI16) of the call's
 * largest M, and every all-zero pulse, takes M: CF16/CBF16 words are rescaled
 * exactly by the power of two, CI16 words are multiplied by it and rounded
 * again (ties to even), dropping at most 4 low bits of a pulse 2^4 below M.
 * All-zero input: scale 1.  A burst's pulses thus normally share one scale,
 * which the backprojection applies per stage of pulses; any per-pulse scales
 * are accepted as input. */
int tdbp_pack_samples(const void *d_cf32, int L, int S, int dtype,
                      void *d_packed, float *d_scale, void *stream);

/* pixelint on materialised inputs (sentinel/azimuth_compress.cu:33-82, or
 * sentinel/azimuth_compress_cpu.c:40-86 when g->semantics is TDBP_SEM_CPU):
 * d_xyz f64 [nlines][W][3], d_azoff f64 [nlines][W], cf32 samples,
 * d_satloc f64 [L][3]; d_out cf32 [nlines][W].  FP64 range and phase; GPU
 * entry: FP32 lerp, output scaled by 1/(azend-azstart); CPU twin: FP64 lerp
 * rounded to cf32, unscaled. */
int tdbp_pixelint(const tdbp_geom *g, const void *d_burst,
                  const double *d_satloc, const double *d_xyz,
                  const double *d_azoff, void *d_out, void *stream);

/* The fused burst backprojection: DEM -> ECEF -> aperture window -> pulse
 * sum, one launch after the fit.  d_coef: from tdbp_fit_aperture (NULL: fit
 * here).  d_out: cf32 [nlines][W]; pixels outside [firstpix, lastpix] or
 * with no valid window are written 0.  Output scaled by 1/(azend-azstart)
 * as the reference GPU kernel does, unscaled under TDBP_SEM_CPU. */
int tdbp_backproject(const tdbp_geom *g, const tdbp_samples *s,
                     const double *d_satloc, const int16_t *d_dem,
                     const double *d_coef, void *d_out, int precision,
                     void *stream);

/* tdbp_backproject with d_coef = NULL that allocates nothing: the aperture
 * fit's scratch (the orbit table copied from g->timeorbit/xx/vv, and the
 * parabolas) lives in a file-scope device array of the library, one per GPU,
 * held until the process ends.  No counterpart in the reference: for callers
 * that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  Limits: g->nlines <=
 * 16384 window lines (else TDBP_ERR_LIMIT) and numstatevec <= 1000; the
 * scratch is 0.44 MB per GPU.  Every call on a GPU shares that GPU's scratch:
 * calls that overlap on one device race.  Returns after the launch has
 * completed on `stream` (the orbit copies read the caller's host arrays). */
int tdbp_backproject_noalloc(const tdbp_geom *g, const tdbp_samples *s,
                             const double *d_satloc, const int16_t *d_dem, void *d_out,
                             int precision, void *stream);

/* tdbp_backproject with an explicit kernel variant (0 .. count-1). */
int tdbp_backproject_variant(const tdbp_geom *g, const tdbp_samples *s,
                             const double *d_satloc, const int16_t *d_dem,
                             const double *d_coef, void *d_out, int precision,
                             int variant, void *stream);

/* Autotuner: time every VALU kernel variant on this burst (reps launches
 * each, after one warm-up), return the fastest in *best and, for TDBP_MIXED,
 * make it the default of later launches (the default stays automatic where it
 * already is that variant on this burst).  ms (optional, [count]) gets the
 * mean milliseconds per launch of each variant (0 for the MFMA variant 8,
 * which runs only when asked for by index).  Overwrites d_out. */
int tdbp_autotune(const tdbp_geom *g, const tdbp_samples *s,
                  const double *d_satloc, const int16_t *d_dem, void *d_out,
                  int precision, int reps, float *ms, int *best);

/* Kernel variant for TDBP_MIXED launches (autotuner output); -1 = auto: the
 * TDBP_VARIANT of the environment, else variant 5, or, for a burst of at most
 * about one 256-pixel tile per CU, variant 11: variant 5's wave tiles with a
 * workgroup's four waves sharing one tile's pulses.  A variant named here, in the environment or
 * in a call runs as it is on every burst. */
int tdbp_set_variant(int variant);
int tdbp_variant_count(void);
/* Describe variant v: rows x cols of the workgroup's pixel tile and pulses
 * per stage (variants 9 and 10, the LDS-staged kernels on the tiles of
 * variants 5 and 4: pulses per LDS sub-stage). */
int tdbp_variant_info(int v, int *tile_rows, int *tile_cols, int *stage);

/* ---------------------------------------------------------- batch API */

typedef struct tdbp_batch tdbp_batch;

/* A batch runs every added burst in one persistent launch (plus one fit
 * launch) fed by a device work queue of (burst, tile) items; the whole
 * sequence is captured once in a hipGraph and replayed by tdbp_batch_run. */
tdbp_batch *tdbp_batch_create(int precision, int variant);
/* Add a burst.  The geometry is copied; device buffers are borrowed and
 * must stay valid until tdbp_batch_destroy.  Returns the burst index >= 0
 * or -tdbp_status. */
int tdbp_batch_add(tdbp_batch *b, const tdbp_geom *g, const tdbp_samples *s,
                   const double *d_satloc, const int16_t *d_dem, void *d_out);
/* Merge burst `burst`'s output (its [nlines][W] rows) into rows
 * [firstline, firstline+nlines) of a device grid [grid_lines][grid_width]
 * (grid_width must equal the burst's demwidth) after every run, in burst
 * order, with the .geo rule of the burst's semantics (GPU entry:
 * sentinel/azimuth_compress.cu:527-531, pixel replaced where |Re| > 1e-18;
 * CPU twin: sentinel/azimuth_compress_cpu.c:386-388, 1 <= |Re| < 2^31).
 * Set before the first run.  Replaces the
 * per-burst .geo read-modify-write of sentinel/azimuth_compress.cu:513-536. */
int tdbp_batch_set_merge(tdbp_batch *b, int burst, void *d_grid, int grid_lines,
                         int grid_width, int firstline);
/* Run (first call builds the queue and captures the graph). */
int tdbp_batch_run(tdbp_batch *b, void *stream);
/* Variant the batch runs (resolved at the first run). */
int tdbp_batch_variant(const tdbp_batch *b);
/* Time every VALU variant (0-7, 9-11) on this batch's own bursts -- reps graph
 * launches each after a warm-up -- and keep the fastest for this batch only
 * (the process-wide default is unchanged; pass *best to tdbp_set_variant to
 * make it the default of later TDBP_MIXED launches).  ms (optional,
 * [tdbp_variant_count()]) gets the mean milliseconds per launch of each
 * variant (0 for the MFMA variant 8).  On a batch in which the automatic
 * choice gives some bursts variant 11 and others another, it is timed as well,
 * and *best is -1 where it is the fastest.  Overwrites the outputs and re-applies
 * the merges (an overwrite, so the grid ends as after one run).  No
 * counterpart in the reference: the batched path is new. */
int tdbp_batch_autotune(tdbp_batch *b, int reps, float *ms, int *best);
/* Pairs visited by one run (valid after the first run). */
int64_t tdbp_batch_pairs(const tdbp_batch *b);
/* Device memory held by the batch itself (queue, descriptors, coef). */
size_t tdbp_batch_device_bytes(const tdbp_batch *b);
void tdbp_batch_destroy(tdbp_batch *b);

/* The .geo merge on the device: burst output d_out [nlines][W] into rows
 * [firstline, firstline+nlines) of d_grid [grid_lines][W].  semantics
 * TDBP_SEM_GPU replaces a pixel where |Re(out)| > 1e-18
 * (sentinel/azimuth_compress.cu:527-531); TDBP_SEM_CPU where
 * 1 <= |Re(out)| < 2^31 (sentinel/azimuth_compress_cpu.c:386-388 as the
 * reference builds it). */
int tdbp_merge_geo(void *d_grid, int W, int grid_lines, int firstline, int nlines,
                   const void *d_out, int semantics, void *stream);

/* Error sums of a cf32 image against a cf32 reference, n pixels, over the
 * pixels where the reference is nonzero: sums[0] = sum |ref|^2 dphi^2,
 * sums[1] = sum |ref|^2, sums[2] = sum (|img| - |ref|)^2, sums[3] = count,
 * sums[4] = pixels where ref is zero and img is not.  RMS phase =
 * sqrt(sums[0]/sums[1]); RMS relative amplitude = sqrt(sums[2]/sums[1]).
 * Synchronises the stream.  No reference counterpart: this is the per-config
 * precision report of the mixed path against the FP64 path. */
int tdbp_compare(const void *d_img, const void *d_ref, size_t n, double *sums,
                 void *stream);

/* ------------------------------------------- burst set-up (the caller side) */

/* Burst parameters from the first line's 80-byte header
 * (sentinel/backprojectgpusub.f90:406-439, burstparams): start time (bytes
 * 68-75, native double), PRF, sampling rate (Hz), PRI (s), range window
 * start time SWST (s), rank, range0 = c/2 (rank PRI + SWST) + 60 m, and the
 * wavelength literal 0.05546576 as the caller stores it (FP32-rounded). */
typedef struct tdbp_burst_params {
  double starttime, prf, samplefreq, pri, swst, range0, wvl;
  int32_t rangedecimation, rank;
} tdbp_burst_params;

int tdbp_burst_decode(const uint8_t *header80, tdbp_burst_params *p);

/* TOPS steering coefficients (fdopcoefs + linfit,
 * sentinel/backprojectgpusub.f90:262-300, :355-383): least-squares line of
 * the azimuth beam angle against time over lines 21..lines-20.  headers:
 * `lines` headers of 80 bytes, stride_bytes apart (a decoded line is
 * 30000 x 8 bytes).  Outputs the FP32 coefficients the reference keeps. */
int tdbp_steering_fit(const uint8_t *headers, size_t stride_bytes, int lines,
                      double *angc0, double *angc1);

/* Integration length of sentinel/backprojectgpusub.f90:193-209 from the
 * satellite velocity at the burst's middle line (satvel(:, lines/2)). */
int tdbp_aperture(const double *vel_mid_burst, double range0, double wvl, double prf,
                  double angc1);

/* Ground footprint of a burst (sentinel/bounds.f90): min/max latitude and
 * longitude (degrees) of the four corners at heights -100 m and 2000 m for
 * times [startime, endtime] and ranges [startr, endr]; the driver calls it
 * with tstart - 2 s, tend + 2 s (:232). */
int tdbp_bounds(double startime, double endtime, double startr, double endr,
                const double *timeorbit, const double *xx, const double *vv, int nsv,
                double *latlons);

/* The driver's per-burst set-up (sentinel/backprojectgpusub.f90:140-247)
 * from the burst's line headers (`lines` headers, header_stride bytes apart;
 * the first line's header gives the burst parameters), the satellite
 * velocity of line lines/2 (1-based, as the driver takes it from the position
 * file), the orbit state vectors and the DEM grid: fills g (integration
 * length, range window rngstart = (2 range0 / c) c / 2, rngend, dmrg, wvl,
 * prf, steering coefficients, tmid and the orbit at tmid, the DEM window from
 * the footprint) and latlons; *in_scene = 0 where the driver skips the burst
 * (|latlons| > 1000, :231-232).  The state-vector arrays are referenced by
 * g, not copied. */
int tdbp_burst_setup(const uint8_t *headers, size_t header_stride, int lines,
                     int rangesamples, const double *satvel_mid, const double *timeorbit,
                     const double *xx, const double *vv, int nsv, int demwidth,
                     int demlength, double firstlat, double firstlon, double deltalat,
                     double deltalon, tdbp_geom *g, double *latlons, int *in_scene);

/* The 80 header bytes of each of nlines decoded lines on the device (cf32
 * rows of `stride` samples) into host memory [nlines][80].  Synchronises. */
int tdbp_headers_dtoh(const void *d_lines, int nlines, int stride, uint8_t *host,
                      void *stream);

/* Host headers [nlines][80] into the first 80 bytes of each device line. */
int tdbp_headers_htod(void *d_lines, int nlines, int stride, const uint8_t *host,
                      void *stream);

/* Per-pulse satellite positions and velocities of decoded lines on the
 * device (sentinel/sentineltimingsub.f90:55-66): each line's time from its
 * header bytes 68-75, 4-point Hermite on the state vectors from
 * int((t - t1)/dt) - 1 (1-based).  d_lines: cf32 [nlines][stride] on the
 * device; outputs d_satloc, d_satvel f64 [nlines][3], d_times f64 [nlines].
 * quantize != 0 rounds positions to 1e-7 m and velocities to 1e-8 m/s, the
 * values the driver reads back from the f16.7 / f14.8 position file.  A
 * line time outside the state vectors' interpolation range is an error.
 * Synchronises the stream. */
int tdbp_pulse_orbit(const void *d_lines, int nlines, int stride, const double *timeorbit,
                     const double *xx, const double *vv, int nsv, int quantize,
                     double *d_satloc, double *d_satvel, double *d_times, void *stream);

/* ------------------------------------------------- range compression */

/* Chirp and echo-window parameters of a swath, decoded from the 80-byte
 * packet header of its first decoded line (sentinel/processsub.f90:75-86;
 * big-endian header fields as in2/in3 of :163-173; sampling rate table of
 * :181-212).  Stored in FP32 as the reference stores them. */
typedef struct tdbp_chirp {
  int32_t rangedecimation; /* header byte 40 */
  int32_t nsamps;          /* echo samples per line, 2 x bytes 65-66 */
  int32_t npts;            /* chirp samples, int(pulselength * samplefreq) */
  int32_t nvalid;          /* nsamps - npts: compressed samples kept */
  float samplefreq;        /* MHz */
  float ramprate;          /* MHz/us, bytes 42-43 (sign bit + 15 bits) */
  float startfreq;         /* MHz, bytes 44-45 (sign bit + 15 bits) */
  float pulselength;       /* us, bytes 46-48 */
} tdbp_chirp;

int tdbp_chirp_decode(const uint8_t *header80, tdbp_chirp *c);

/* Range compression of nlines decoded echo lines on the device, replacing
 * the per-line FFTW loop of sentinel/processsub.f90:96-126.  d_raw: cf32
 * [nlines][raw_stride], each line's first 10 samples the packet header
 * (raw_stride 30000 in the reference), nsamps echo samples after it.
 * Outputs (either or both):
 *   d_out     cf32 [nlines][out_stride >= nvalid + 10]: the header samples,
 *             then nvalid compressed samples (the reference rangeprocdata
 *             layout, :121-122); with flags & TDBP_RC_ZERO_HEADER the header
 *             samples are written as zero, as the burst driver leaves them
 *             before backprojection (sentinel/backprojectgpusub.f90:190);
 *   d_packed  CF16/CBF16/CI16 words [nlines][nvalid + 10] and d_scale [nlines]:
 *             the backprojection input (header samples zero, as
 *             sentinel/backprojectgpusub.f90:190 leaves them) in the storage
 *             of tdbp_pack_samples (scales made common over the nlines).
 * The values are the reference's: 32768-point forward FFT of the zero-padded
 * echo, times conj(FFT(reference chirp / npts)), inverse FFT without
 * normalisation, in FP32.  The kept samples are a linear correlation of the
 * echo window, so the device need not transform 32768 points: for chirps of
 * up to 4096 samples (every IW/EW/SM chirp) one fused kernel correlates
 * overlap-save blocks of 8192 samples in LDS, writing each output once (the
 * packed output is then made from the cf32 rows by one elementwise pass; a
 * call without d_out keeps those rows in a device scratch of the library,
 * 8 (nvalid + 10) B per line, grow-only); longer chirps, or TDBP_RC_ROCFFT=1 in the
 * environment, use batched rocFFT transforms at the shortest 2^a 3^b 5^c
 * length >= nsamps.  Both carry the 32768-point output scale. */
enum { TDBP_RC_ZERO_HEADER = 1 };
int tdbp_range_compress(const void *d_raw, int nlines, int raw_stride,
                        const tdbp_chirp *c, void *d_out, int out_stride, int flags,
                        void *d_packed, float *d_scale, int dtype, void *stream);

/* ------------------------------------------ interferograms (.geo stacks) */

/* int/crossmul.f90 on device images: d_img1, d_img2 cf32 [>= nvalid][na]
 * (the same pointer for an image with itself); uses the first
 * (nvalid / looksdn) * looksdn rows.  Outputs cf32 [nvalid / looksdn]
 * [na / looksac]: d_igram = looked sum of up1 conj(up2) of the two-times
 * upsampled rows, d_amp = (sqrt(sum |up1|^2), sqrt(sum |up2|^2)); rows
 * scaled by `scale` before upsampling; mask != 0 zeroes outputs whose
 * unscaled input sum is <= 1e-6 in either image (crossmul.f90:110-122, the
 * reference default).  Upsampling: zero-pad to nnn = next power of two >= na,
 * forward FFT, spectrum halves to both ends of 2 nnn, inverse FFT, / nnn / 2
 * (:127-148).  looksdn <= 512.  Calls may overlap on several streams and
 * threads; replays of a captured call must not overlap other calls on its
 * device (they share one batch of upsampled rows). */
int tdbp_crossmul(const void *d_img1, const void *d_img2, int na, int nvalid, float scale,
                  int looksac, int looksdn, int mask, void *d_igram, void *d_amp,
                  void *stream);

/* int/makecc.f90 on device arrays: d_igram, d_amp cf32 [nlines][npix] ->
 * d_out f32 [nlines][2 npix]: per line the amplitude row re(amp) im(amp),
 * then the correlation row |igram| / amplitude (0 where amplitude <= 0). */
int tdbp_makecc(const void *d_igram, const void *d_amp, int npix, int nlines, float *d_out,
                void *stream);

/* ------------------------------------------- synthetic data (bench/tests) */

/* Band-limited complex Gaussian clutter: white CN(0, sigma^2) from a
 * counter-based hash of (seed, pulse, sample), convolved along range with
 * the real FIR taps (host array, ntaps <= 64). */
int tdbp_synth_clutter(void *d_cf32, int L, int S, uint64_t seed, float sigma,
                       const float *taps, int ntaps, void *stream);

/* Add point-target echoes: for each target k at ECEF xyz[k] with complex
 * amplitude (amp[2k], amp[2k+1]), every pulse p gets
 * a * sinc((r - r_k(p)) / res) * exp(-j 4 pi R_k(p) / wvl) on the samples
 * r within +-halfwidth of r_k(p) = (R_k(p) - rngstart) / dmrg.  Host
 * arrays; d_satloc f64 [L][3]. */
/* Decoded echo lines cf32 [L][stride]: samples 0-9 the 80 header bytes,
 * then c->nsamps samples holding, per target t, the chirp of c delayed by
 * delay[p*ntargets+t] samples (host array) with carrier
 * exp(-j 2 pi carrier[p*ntargets+t]) and amplitude amp[2t] + j amp[2t+1],
 * plus white circular Gaussian noise (std `noise`); zero after.  Host arrays
 * are copied before the call returns (it synchronises the stream). */
int tdbp_synth_raw(void *d_raw, int L, int stride, const tdbp_chirp *c,
                   const uint8_t *header80, const double *delay, const double *carrier,
                   const float *amp, int ntargets, float noise, uint64_t seed,
                   void *stream);
int tdbp_synth_targets(void *d_cf32, const tdbp_geom *g, const double *d_satloc,
                       const double *xyz, const float *amp, int ntargets,
                       float res, int halfwidth, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* SRG_TDBP_H */
