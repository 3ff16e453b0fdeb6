// tdbp_batch.hip -- many bursts in one persistent launch, and the autotuner.
//
// A batch holds one BurstDev per burst in device memory and a work queue of
// (burst, tile) items split into 8 queues, one per XCD: the (burst, column
// band) pairs are dealt round-robin to the queues and each band contributes
// its row tiles in order, so the workgroups of one XCD walk down the same
// range band and share its samples in their L2.  A workgroup drains its home
// queue (blockIdx % 8) and then steals from the others.  The launch sequence
// (zero the queue counters, fit every burst's aperture parabolas, run the
// persistent kernel) is captured once in a hipGraph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "tdbp_api_internal.h"
#include "tdbp_internal.h"

using namespace tdbp;

struct MergeTarget {
  float2* grid = nullptr;   // nullptr: no merge for this burst
  int grid_lines = 0, firstline = 0;
};

// Work queues of one launch: the bursts of one tile kind.
struct BatchQueue {
  int variant = -1;
  int2* items = nullptr;
  int* qbase = nullptr;
  int* counters = nullptr;
  int grid = 0;
};

struct tdbp_batch {
  int precision = TDBP_MIXED;
  int variant = -1;
  bool named = false;   // the variant was asked for by index (or tuned)
  int dtype = -1;
  std::vector<BurstDev> bursts;
  std::vector<MergeTarget> merges;  // per burst, applied in burst order
  std::vector<void*> owned;  // device allocations of the bursts (orbits, coefs)
  std::vector<void*> tables; // device allocations of build() (burst table, queues)
  BurstDev* d_bursts = nullptr;
  std::vector<BatchQueue> queues;   // bursts on the variant's tiles, then split ones
  int max_lines = 0;
  int64_t pairs = 0;
  size_t dev_bytes = 0, table_bytes = 0;
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  bool built = false, use_graph = true;
};

namespace {

int balloc(tdbp_batch* b, void** p, size_t bytes) {
  if (hipMalloc(p, bytes ? bytes : 1) != hipSuccess)
    return set_error(TDBP_ERR_NOMEM, "batch hipMalloc(%zu) failed", bytes);
  b->owned.push_back(*p);
  b->dev_bytes += bytes;
  return TDBP_OK;
}

int talloc(tdbp_batch* b, void** p, size_t bytes) {
  if (hipMalloc(p, bytes ? bytes : 1) != hipSuccess)
    return set_error(TDBP_ERR_NOMEM, "batch hipMalloc(%zu) failed", bytes);
  b->tables.push_back(*p);
  b->dev_bytes += bytes;
  b->table_bytes += bytes;
  return TDBP_OK;
}

// Undo build(): the graph, the stream and the per-variant tables.
void unbuild(tdbp_batch* b) {
  if (b->cap) (void)hipStreamSynchronize(b->cap);
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->cap) (void)hipStreamDestroy(b->cap);
  b->exec = nullptr;
  b->graph = nullptr;
  b->cap = nullptr;
  for (void* p : b->tables) (void)hipFree(p);
  b->tables.clear();
  b->d_bursts = nullptr;
  b->queues.clear();
  b->dev_bytes -= b->table_bytes;
  b->table_bytes = 0;
  b->built = false;
}

int enqueue(tdbp_batch* b, hipStream_t s) {
  int st;
  for (const BatchQueue& q : b->queues)
    if ((st = hip_check(launch_zero(q.counters, 8 * sizeof(int), s), "queue reset"))) return st;
  st = hip_check(launch_batch_fit(b->d_bursts, (int)b->bursts.size(),
                                  b->max_lines, s),
                 "batch fit launch");
  if (st) return st;
  for (const BatchQueue& q : b->queues)
    if ((st = hip_check(launch_batch(b->d_bursts, q.items, q.qbase, q.counters, b->precision,
                                     q.variant, b->dtype, q.grid, s),
                        "batch launch")))
      return st;
  // .geo merges in burst order: overlapping rows take the later burst, as the
  // reference's sequential read-modify-write does.
  for (size_t i = 0; i < b->bursts.size(); ++i) {
    const MergeTarget& m = b->merges[i];
    if (!m.grid) continue;
    const BurstDev& bd = b->bursts[i];
    st = hip_check(launch_merge(m.grid, bd.out, (size_t)bd.nlines * bd.W,
                                (size_t)m.firstline * bd.W,
                                bd.cpu ? TDBP_SEM_CPU : TDBP_SEM_GPU, s),
                   "merge launch");
    if (st) return st;
  }
  return TDBP_OK;
}

int build_tables(tdbp_batch* b);

// Build the batch's tables and graph; on any failure undo what was built, so
// a later run builds from scratch instead of leaking the stream or adding to
// the table list.
int build(tdbp_batch* b) {
  const int st = build_tables(b);
  if (st) unbuild(b);
  return st;
}

int build_tables(tdbp_batch* b) {
  int st;
  if (b->bursts.empty()) return set_error(TDBP_ERR_ARG, "empty batch");
  if ((st = hip_check(hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking),
                      "batch stream")))
    return st;
  if (b->variant < 0) b->variant = default_variant(b->precision, &b->named);
  if (b->variant == 8)   // the MFMA kernel needs 32-bit sample offsets in every burst
    for (auto& bd : b->bursts)
      if (!mfma_fits(bd)) b->variant = 5;
  b->max_lines = 0;
  for (auto& bd : b->bursts) {
    set_tiles(&bd, b->variant, b->named);
    b->max_lines = std::max(b->max_lines, bd.nlines);
  }
  const size_t nb = b->bursts.size();
  if ((st = talloc(b, (void**)&b->d_bursts, nb * sizeof(BurstDev)))) return st;
  if ((st = hip_check(hipMemcpy(b->d_bursts, b->bursts.data(),
                                nb * sizeof(BurstDev), hipMemcpyHostToDevice),
                      "burst table upload")))
    return st;

  // Fit once eagerly to count the pairs of the work.
  if ((st = hip_check(launch_batch_fit(b->d_bursts, (int)nb, b->max_lines, b->cap),
                      "batch fit launch")))
    return st;
  size_t tot_lines = 0;
  for (auto& bd : b->bursts) tot_lines += bd.nlines;
  int64_t* d_pairs = nullptr;
  if ((st = talloc(b, (void**)&d_pairs, tot_lines * sizeof(int64_t)))) return st;
  size_t off = 0;
  for (auto& bd : b->bursts) {
    if ((st = hip_check(launch_pair_count(bd, d_pairs + off, b->cap),
                        "pair count launch")))
      return st;
    off += bd.nlines;
  }
  std::vector<int64_t> hp(tot_lines);
  if ((st = hip_check(hipMemcpyAsync(hp.data(), d_pairs, tot_lines * 8,
                                     hipMemcpyDeviceToHost, b->cap),
                      "pair download")) ||
      (st = hip_check(hipStreamSynchronize(b->cap), "pair sync")))
    return st;
  b->pairs = 0;
  for (int64_t v : hp) b->pairs += v;

  // Work queues, one set per tile kind (kSplitVariant's whole bursts: the CPU
  // twin's, on variant 5's tiles).
  const int whole = b->variant == kSplitVariant ? 5 : b->variant;
  for (int split = 0; split < 2; ++split) {
    std::vector<std::vector<int2>> q(8);
    int g = 0;
    for (int bi = 0; bi < (int)nb; ++bi) {
      const BurstDev& bd = b->bursts[bi];
      if (bd.split != split) continue;
      for (int band = 0; band < bd.tiles_c; ++band, ++g) {
        auto& dst = q[g & 7];
        for (int rt = 0; rt < bd.tiles_r; ++rt)
          dst.push_back(make_int2(bi, band * bd.tiles_r + rt));
      }
    }
    std::vector<int2> items;
    std::vector<int> qbase(9, 0);
    for (int k = 0; k < 8; ++k) {
      qbase[k] = (int)items.size();
      items.insert(items.end(), q[k].begin(), q[k].end());
    }
    qbase[8] = (int)items.size();
    if (items.empty()) continue;
    BatchQueue d;
    d.variant = split ? kSplitVariant : whole;
    if ((st = talloc(b, (void**)&d.items, items.size() * sizeof(int2))) ||
        (st = talloc(b, (void**)&d.qbase, 9 * sizeof(int))) ||
        (st = talloc(b, (void**)&d.counters, 8 * sizeof(int))))
      return st;
    if ((st = hip_check(hipMemcpy(d.items, items.data(), items.size() * sizeof(int2),
                                  hipMemcpyHostToDevice),
                        "item upload")) ||
        (st = hip_check(hipMemcpy(d.qbase, qbase.data(), 9 * sizeof(int), hipMemcpyHostToDevice),
                        "queue upload")))
      return st;
    d.grid = cu_count() * batch_blocks_per_cu(b->precision, d.variant, b->dtype);
    b->queues.push_back(d);
  }

  const char* eg = std::getenv("TDBP_GRAPH");
  b->use_graph = !(eg && eg[0] == '0');
  if (b->use_graph) {
    if ((st = hip_check(hipStreamBeginCapture(b->cap, hipStreamCaptureModeThreadLocal),
                        "begin capture")))
      return st;
    const int est = enqueue(b, b->cap);
    hipGraph_t gr = nullptr;
    st = hip_check(hipStreamEndCapture(b->cap, &gr), "end capture");
    if (est) return est;
    if (st) return st;
    b->graph = gr;
    if ((st = hip_check(hipGraphInstantiate(&b->exec, gr, nullptr, nullptr, 0),
                        "graph instantiate")))
      return st;
  }
  b->built = true;
  return TDBP_OK;
}

}  // namespace

extern "C" {

tdbp_batch* tdbp_batch_create(int precision, int variant) {
  if (precision != TDBP_PLAIN_FP64 && precision != TDBP_MIXED) {
    set_error(TDBP_ERR_ARG, "unknown precision %d", precision);
    return nullptr;
  }
  if (variant < -1 || variant >= kNumVariants) {
    set_error(TDBP_ERR_ARG, "variant %d", variant);
    return nullptr;
  }
  if (current_device_ready()) return nullptr;
  tdbp_batch* b = new tdbp_batch;
  b->precision = precision;
  b->variant = variant;
  b->named = variant >= 0;
  return b;
}

int tdbp_batch_add(tdbp_batch* b, const tdbp_geom* g, const tdbp_samples* s,
                   const double* d_satloc, const int16_t* d_dem, void* d_out) {
  if (!b) return -set_error(TDBP_ERR_ARG, "null batch");
  if (b->built) return -set_error(TDBP_ERR_ARG, "batch already built");
  int st = validate_geom(g);
  if (st) return -st;
  if ((st = check_samples(s, b->precision))) return -st;
  if (!d_satloc || !d_dem || !d_out)
    return -set_error(TDBP_ERR_ARG, "null device buffer");
  if (b->dtype >= 0 && s->dtype != b->dtype)
    return -set_error(TDBP_ERR_ARG, "a batch holds one sample dtype");
  b->dtype = s->dtype;
  BurstDev bd;
  fill_burst(g, &bd);
  bd.data = s->d_data;
  bd.scale = s->d_scale;
  bd.dtype = s->dtype;
  bd.satloc = d_satloc;
  bd.dem = d_dem;
  bd.out = (float2*)d_out;
  std::vector<double> orb = pack_orbit(g);
  double* d_orb = nullptr;
  double* d_coef = nullptr;
  if ((st = balloc(b, (void**)&d_orb, orb.size() * 8)) ||
      (st = balloc(b, (void**)&d_coef, 24 * (size_t)g->nlines)))
    return -st;
  if ((st = hip_check(hipMemcpy(d_orb, orb.data(), orb.size() * 8,
                                hipMemcpyHostToDevice),
                      "orbit upload")))
    return -st;
  point_orbit(&bd, d_orb, g->numstatevec);
  bd.coef = d_coef;
  b->bursts.push_back(bd);
  b->merges.push_back(MergeTarget());
  return (int)b->bursts.size() - 1;
}

int tdbp_batch_set_merge(tdbp_batch* b, int burst, void* d_grid, int grid_lines,
                         int grid_width, int firstline) {
  if (!b || burst < 0 || burst >= (int)b->bursts.size())
    return set_error(TDBP_ERR_ARG, "merge target for unknown burst %d", burst);
  if (b->built) return set_error(TDBP_ERR_ARG, "batch already built");
  const BurstDev& bd = b->bursts[burst];
  if (grid_width != bd.W)
    return set_error(TDBP_ERR_ARG, "merge grid width %d != burst DEM width %d", grid_width,
                     bd.W);
  if (!d_grid || firstline < 0 || firstline + bd.nlines > grid_lines)
    return set_error(TDBP_ERR_ARG, "merge rows [%d, %d) outside a %d-line grid", firstline,
                     firstline + bd.nlines, grid_lines);
  MergeTarget& m = b->merges[burst];
  m.grid = (float2*)d_grid;
  m.grid_lines = grid_lines;
  m.firstline = firstline;
  return TDBP_OK;
}

int tdbp_batch_run(tdbp_batch* b, void* stream) {
  if (!b) return set_error(TDBP_ERR_ARG, "null batch");
  int st = current_device_ready();
  if (st) return st;
  if (!b->built && (st = build(b))) return st;
  if (b->use_graph)
    return hip_check(hipGraphLaunch(b->exec, (hipStream_t)stream), "graph launch");
  return enqueue(b, (hipStream_t)stream);
}

int64_t tdbp_batch_pairs(const tdbp_batch* b) { return b ? b->pairs : 0; }

size_t tdbp_batch_device_bytes(const tdbp_batch* b) {
  return b ? b->dev_bytes : 0;
}

int tdbp_batch_variant(const tdbp_batch* b) { return b ? b->variant : -1; }

void tdbp_batch_destroy(tdbp_batch* b) {
  if (!b) return;
  unbuild(b);
  (void)hipDeviceSynchronize();
  for (void* p : b->owned) (void)hipFree(p);
  delete b;
}

// Time every VALU variant on the batch's own bursts and keep the fastest.  Where
// the automatic choice splits some of the bursts' tiles and not others, no
// variant by itself is that choice: it is timed too, as the last candidate.
int tdbp_batch_autotune(tdbp_batch* b, int reps, float* ms, int* best) {
  if (!b) return set_error(TDBP_ERR_ARG, "null batch");
  if (b->bursts.empty()) return set_error(TDBP_ERR_ARG, "empty batch");
  int st = current_device_ready();
  if (st) return st;
  reps = reps < 1 ? 1 : reps;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if ((st = hip_check(hipEventCreate(&e0), "event")) ||
      (st = hip_check(hipEventCreate(&e1), "event"))) {
    if (e0) (void)hipEventDestroy(e0);
    return st;
  }
  bool named = false;
  const int automatic = automatic_variant(b->precision, &named);
  size_t split = 0;
  for (BurstDev bd : b->bursts) {
    set_tiles(&bd, automatic, named);
    split += bd.split;
  }
  const bool both = !named && split > 0 && split < b->bursts.size();
  int bestv = -1;
  float bestms = 3.4e38f;
  for (int v = 0; v < kNumVariants + (both ? 1 : 0) && !st; ++v) {
    // The MFMA variant (8) runs only when asked for by index.
    if (v < kNumVariants && kVariants[v].mfma) {
      if (ms) ms[v] = 0.f;
      continue;
    }
    unbuild(b);
    b->named = v < kNumVariants;
    b->variant = b->named ? v : automatic;
    if ((st = build(b))) break;
    if ((st = tdbp_batch_run(b, b->cap))) break;   // warm-up
    (void)hipEventRecord(e0, b->cap);
    for (int r = 0; r < reps && !st; ++r) st = tdbp_batch_run(b, b->cap);
    (void)hipEventRecord(e1, b->cap);
    if (!st) st = hip_check(hipEventSynchronize(e1), "tune sync");
    float t = 0.f;
    if (!st) (void)hipEventElapsedTime(&t, e0, e1);
    t /= reps;
    if (ms && b->named) ms[v] = t;
    if (!st && t < bestms) {
      bestms = t;
      bestv = b->named ? v : -1;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  unbuild(b);
  if (st) return st;
  b->named = bestv >= 0;
  b->variant = b->named ? bestv : automatic;
  if ((st = build(b))) return st;
  if (best) *best = bestv;
  return TDBP_OK;
}

// Time every variant on one burst and keep the fastest for later TDBP_MIXED
// launches; where that is what the automatic choice runs on this burst, the
// choice stays automatic, so that it suits later bursts of other sizes.  ms (optional) gets the mean time of each variant.
int tdbp_autotune(const tdbp_geom* g, const tdbp_samples* s,
                  const double* d_satloc, const int16_t* d_dem, void* d_out,
                  int precision, int reps, float* ms, int* best) {
  int st = validate_geom(g);
  if (st) return st;
  if ((st = check_samples(s, precision))) return st;
  if ((st = current_device_ready())) return st;
  reps = reps < 1 ? 1 : reps;
  hipStream_t str = nullptr;
  if ((st = hip_check(hipStreamCreateWithFlags(&str, hipStreamNonBlocking),
                      "tune stream")))
    return st;
  double* d_coef = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int bestv = -1;
  float bestms = 3.4e38f;
  do {
    if ((st = hip_check(hipMalloc((void**)&d_coef, 24 * (size_t)g->nlines),
                        "tune coef")))
      break;
    BurstDev b;
    fill_burst(g, &b);
    b.dem = d_dem;
    if ((st = fit_on_stream(b, g, d_coef, str))) break;
    if ((st = hip_check(hipEventCreate(&e0), "event")) ||
        (st = hip_check(hipEventCreate(&e1), "event")))
      break;
    // The VALU variants only: the MFMA variant (8) is run when asked for by
    // index, never picked here (measured at par on one burst and slower
    // batched; the backprojection sum is not a dense contraction).
    for (int v = 0; v < kNumVariants && !st; ++v) {
      if (kVariants[v].mfma) {
        if (ms) ms[v] = 0.f;
        continue;
      }
      st = run_backproject(g, s, d_satloc, d_dem, d_coef, d_out, precision, v,
                           str);  // warm-up
      if (st) break;
      (void)hipEventRecord(e0, str);
      for (int r = 0; r < reps && !st; ++r)
        st = run_backproject(g, s, d_satloc, d_dem, d_coef, d_out, precision, v,
                             str);
      (void)hipEventRecord(e1, str);
      if (!st) st = hip_check(hipEventSynchronize(e1), "tune sync");
      float t = 0.f;
      if (!st) (void)hipEventElapsedTime(&t, e0, e1);
      t /= reps;
      if (ms) ms[v] = t;
      if (!st && t < bestms) {
        bestms = t;
        bestv = v;
      }
    }
  } while (0);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(str);
  if (d_coef) (void)hipFree(d_coef);
  (void)hipStreamDestroy(str);
  if (st) return st;
  if (best) *best = bestv;
  if (precision == TDBP_MIXED) {
    BurstDev b;
    fill_burst(g, &b);
    bool named = false;
    const int automatic = automatic_variant(precision, &named);
    tdbp_set_variant(set_tiles(&b, automatic, named) == bestv ? -1 : bestv);
  }
  return TDBP_OK;
}

}  // extern "C"
