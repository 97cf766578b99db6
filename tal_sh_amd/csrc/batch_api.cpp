// Batched contractions: host API (extension, include/talsh_amd.h).
//
// A batch collects many talshTensorContract-style operations on GPU-resident
// tensors and runs them as one persistent kernel launch captured in a
// hipGraph.  The first execution plans the batch (index groups, wave tiles,
// a static schedule of the work items over the kernel's waves, graph); later
// executions of an unchanged batch replay the graph.
//
// Tile shapes come from a two-stage autotuner.  Stage 1 groups contractions
// into shape classes by (log2 M, log2 N) and, for every class not tuned yet
// in this process, times each candidate wave tile on up to 32 of the class's
// own contractions (writing into scratch outputs, so user data is untouched);
// the fastest is cached per (data kind, class).  Stage 2 times whole-batch
// tile policies on one launch of the entire batch and keeps the fastest.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "batch.hpp"
#include "batch_plan.hpp"
#include "plan.hpp"
#include "runtime.hpp"
#include "talsh_amd.h"

struct talshAmdBatch {
  struct Entry {
    std::string pattern;
    talsh_tens_t *d, *l, *r;
    double ar, ai;
    int acc;
  };
  std::vector<Entry> entries;
  bool built = false;
  int g = -1, dk = NO_TYPE, nblocks = 0, ntasks = 0;
  long long total = 0;  // work items
  double flops = 0.0;
  std::vector<const void *> sig;
  std::vector<size_t> sig_bytes;  // body bytes of each sig entry
  void *dev = nullptr;
  int dev_handle = -1;
  const tal::BatchItem *d_items = nullptr;
  const int *d_qstart = nullptr;
  unsigned *d_counters = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int tuned_classes = 0, replays = 0;
  double tune_ms = 0.0;
  // Ordering state shared by every operand: the hazard entries of all its
  // tensors point at `hz`, re-recorded after each execution.  `epoch` is the
  // hazard-table epoch right after the last execution; while it is unchanged
  // nothing else has touched any operand (or moved a body) since.
  tal::EvRef hz;
  uint64_t epoch = 0;
  uint64_t images = 0;  // rt().image_epoch when `sig` was last found to hold
  int policy = 0;  // tile policy chosen by whole-batch timing
};

namespace tal {
namespace {

constexpr int kXcds = 8;  // workgroups are dispatched round-robin over the XCDs

std::map<std::pair<int, int>, WaveTile> &tuned_tiles() {
  static std::map<std::pair<int, int>, WaveTile> t;
  return t;
}

int bucket(int x) {
  int b = 0;
  while ((1 << b) < x && b < 12) ++b;
  return b;
}
int shape_class(int M, int N) { return bucket(M) * 100 + bucket(N); }

// Host description of one contraction after planning.
struct HostTask {
  BatchTaskGeom geom;
  uint64_t L = 0, R = 0, D = 0;
  uint64_t lbytes = 0, rbytes = 0, dbytes = 0;
  double alpha = 1.0;
  bool acc = false;
  int cls = 0;
  WaveTile tile{16, 16};
};

void *gpu_body(talsh_tens_t *t, int g, int *dk) {
  const int i = image_find(t, flat_gpu(g), NO_TYPE, true);
  if (i < 0) return nullptr;
  *dk = t->data_kind[i];
  return t->dev_rsc[i].gmem_p;
}

int plan_task(const talshAmdBatch::Entry &e, int g, int *dk_out, HostTask *h) {
  DigitalPattern p;
  if (parse_pattern(e.pattern.c_str(), &p) != 0) return TALSH_INVALID_ARGS;
  const talsh_tens_t *d = e.d, *l = e.l, *r = e.r;
  if (p.drank != d->shape_p->num_dim || p.lrank != l->shape_p->num_dim || p.rrank != r->shape_p->num_dim)
    return TALSH_INVALID_ARGS;
  int dk[3];
  void *D = gpu_body(e.d, g, &dk[0]), *L = gpu_body(e.l, g, &dk[1]), *R = gpu_body(e.r, g, &dk[2]);
  if (!D || !L || !R) return TALSH_NOT_AVAILABLE;
  if (dk[0] != dk[1] || dk[0] != dk[2] || (dk[0] != R4 && dk[0] != R8)) return TALSH_NOT_IMPLEMENTED;
  const int esz = dk_size(dk[0]);
  h->dbytes = shape_volume(d->shape_p) * (size_t)esz;
  h->lbytes = shape_volume(l->shape_p) * (size_t)esz;
  h->rbytes = shape_volume(r->shape_p) * (size_t)esz;
  // 32-bit buffer offsets: large contractions belong to the TTGT path
  if (h->dbytes > kBatchMaxBytes || h->lbytes > kBatchMaxBytes || h->rbytes > kBatchMaxBytes) return DEVICE_UNABLE;
  const int ge = batch_task_geometry(p, d->shape_p->dims, l->shape_p->dims, r->shape_p->dims, esz, &h->geom);
  if (ge == 1) return TALSH_INVALID_ARGS;
  if (ge != 0) return DEVICE_UNABLE;  // hyper index or more than three dims in a group
  h->L = (uint64_t)L;
  h->R = (uint64_t)R;
  h->D = (uint64_t)D;
  h->alpha = e.ar;
  h->acc = e.acc != 0;
  h->cls = shape_class(h->geom.M, h->geom.N);
  *dk_out = dk[0];
  return TALSH_SUCCESS;
}

// Smallest candidate that covers the contraction, else 64 x 64.
WaveTile fit_tile(int M, int N) { return WaveTile{M <= 32 ? 32 : 64, N <= 32 ? 32 : 64}; }

// Device image of a schedule: [queue counters][qstart (queues + 1 ints)][items, 256-byte aligned].
struct DeviceBatch {
  void *base = nullptr;
  int handle = -1;
  unsigned *counters = nullptr;
  const BatchItem *items = nullptr;
  const int *qstart = nullptr;
  long long total = 0;
};

// Workgroups of the persistent launch: as many as are resident at once.
int persistent_blocks(int g, int dk) {
  hipDeviceProp_t prop;
  int per_cu = 0;
  if (batch_blocks_per_cu(dk, &per_cu) != 0) per_cu = 2;
  if (hipGetDeviceProperties(&prop, rt().gpus[g].hip_id) != hipSuccess) return 256 * per_cu;
  return std::max(1, prop.multiProcessorCount) * per_cu;
}

// Items of `hts` (each with its tile), in kXcds work queues, copied to the device.
int upload(int g, int dk, const std::vector<HostTask> &hts, hipStream_t s, DeviceBatch *db) {
  std::vector<BatchItem> items;
  std::vector<int> task_of;
  for (size_t t = 0; t < hts.size(); ++t) {
    const HostTask &h = hts[t];
    const size_t before = items.size();
    batch_task_items(h.geom, h.L, h.R, h.D, h.lbytes, h.rbytes, h.dbytes, h.alpha, h.acc, h.tile, &items);
    task_of.insert(task_of.end(), items.size() - before, (int)t);
  }
  std::vector<BatchItem> ordered;
  std::vector<int> qstart;
  batch_queues(items, task_of, dk_size(dk), kXcds, &ordered, &qstart);
  const size_t cb = ((batch_counter_bytes(kXcds) + 255) / 256) * 256;
  const size_t sb = ((4 * qstart.size() + 255) / 256) * 256;
  const size_t bytes = cb + sb + sizeof(BatchItem) * std::max<size_t>(1, ordered.size());
  if (int e = dev_alloc(g, bytes, &db->base, &db->handle)) return e;
  char *b = (char *)db->base;
  db->counters = (unsigned *)b;
  db->qstart = (const int *)(b + cb);
  db->items = (const BatchItem *)(b + cb + sb);
  db->total = (long long)ordered.size();
  if (hipMemcpyAsync((void *)db->qstart, qstart.data(), 4 * qstart.size(), hipMemcpyHostToDevice, s) != hipSuccess ||
      (!ordered.empty() && hipMemcpyAsync((void *)db->items, ordered.data(), sizeof(BatchItem) * ordered.size(),
                                          hipMemcpyHostToDevice, s) != hipSuccess) ||
      batch_counter_reset(db->counters, kXcds, s) != 0 || hipStreamSynchronize(s) != hipSuccess) {
    dev_free(g, db->base, db->handle);
    return TALSH_FAILURE;
  }
  return TALSH_SUCCESS;
}

// Redirects every output into one scratch allocation (never into user tensors)
// and makes the contractions non-accumulative; returns the allocation.
int scratch_outputs(int g, std::vector<HostTask> *hts, void **sp, int *sh) {
  size_t scratch = 0;
  for (const auto &h : *hts) scratch += (h.dbytes + 255) / 256 * 256;
  if (int e = dev_alloc(g, std::max<size_t>(256, scratch), sp, sh)) return e;
  size_t off = 0;
  for (auto &h : *hts) {
    h.D = (uint64_t)((char *)*sp + off);
    h.acc = false;
    off += (h.dbytes + 255) / 256 * 256;
  }
  return TALSH_SUCCESS;
}

// Launch time (ms) of one schedule: the second of two launches (the first warms caches).
float time_launch(int g, int dk, const std::vector<HostTask> &hts, int nblocks, hipStream_t s, hipEvent_t e0,
                  hipEvent_t e1, int *err) {
  DeviceBatch db;
  if ((*err = upload(g, dk, hts, s, &db)) != 0) return 1e30f;
  float ms = 1e30f;
  for (int rep = 0; rep < 2; ++rep) {
    (void)hipEventRecord(e0, s);
    if (batch_launch(dk, db.items, db.qstart, db.counters, kXcds, nblocks, s) != 0) *err = TALSH_FAILURE;
    (void)hipEventRecord(e1, s);
    (void)hipEventSynchronize(e1);
    (void)hipEventElapsedTime(&ms, e0, e1);
  }
  dev_free(g, db.base, db.handle);
  return ms;
}

// Stage 1: times every candidate wave tile on up to 32 contractions of each untuned class.
int autotune(int g, int dk, const std::vector<HostTask> &hts, hipStream_t s, int *nclasses, double *ms_spent) {
  std::map<int, std::vector<int>> classes;
  for (int i = 0; i < (int)hts.size(); ++i) classes[hts[i].cls].push_back(i);
  const int nblocks = persistent_blocks(g, dk);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return TALSH_FAILURE;
  const double t0 = wall_time();
  int err = TALSH_SUCCESS;
  for (auto &kv : classes) {
    const auto key = std::make_pair(dk, kv.first);
    if (tuned_tiles().count(key)) continue;
    std::vector<HostTask> probe;
    for (int i = 0; i < (int)kv.second.size() && i < 32; ++i) probe.push_back(hts[(size_t)kv.second[(size_t)i]]);
    void *sp = nullptr;
    int sh = -1;
    if ((err = scratch_outputs(g, &probe, &sp, &sh)) != 0) break;
    float best = 1e30f;
    WaveTile pick = fit_tile(probe[0].geom.M, probe[0].geom.N);
    for (const WaveTile &c : kWaveTiles) {
      for (auto &p : probe) p.tile = c;
      const float ms = time_launch(g, dk, probe, nblocks, s, e0, e1, &err);
      if (err) break;
      if (ms < best) {
        best = ms;
        pick = c;
      }
    }
    dev_free(g, sp, sh);
    if (err) break;
    tuned_tiles()[key] = pick;
    (*nclasses)++;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *ms_spent += 1e3 * (wall_time() - t0);
  return err;
}

// Stage 2, on the whole batch: a class timed alone favours small tiles (they
// expose parallelism a 32-contraction probe lacks), while the full batch has
// items to spare and pays a fixed cost per item.  Each policy below is timed
// on one launch of the entire batch writing scratch outputs; the fastest is
// applied.  Skipped (policy 0) when the scratch outputs would not fit in a
// quarter of the free pool.
enum TilePolicy { POLICY_CLASS_TUNED = 0, POLICY_FIT = 1, POLICY_SMALL = 2, NPOLICY = 3 };

WaveTile policy_tile(int policy, int dk, const HostTask &h) {
  switch (policy) {
    case POLICY_FIT: return fit_tile(h.geom.M, h.geom.N);
    case POLICY_SMALL: return WaveTile{32, 32};
    default: {
      auto it = tuned_tiles().find(std::make_pair(dk, h.cls));
      return it != tuned_tiles().end() ? it->second : fit_tile(h.geom.M, h.geom.N);
    }
  }
}

int choose_policy(int g, int dk, std::vector<HostTask> hts, hipStream_t s, int *policy, double *ms_spent) {
  *policy = POLICY_CLASS_TUNED;
  size_t scratch = 0;
  for (auto &h : hts) scratch += (h.dbytes + 255) / 256 * 256;
  if (scratch == 0 || scratch > rt().gpus[g].arena.free_bytes() / 4) return TALSH_SUCCESS;
  void *sp = nullptr;
  int sh = -1;
  if (scratch_outputs(g, &hts, &sp, &sh) != 0) return TALSH_SUCCESS;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    dev_free(g, sp, sh);
    return TALSH_FAILURE;
  }
  const double t0 = wall_time();
  const int nblocks = persistent_blocks(g, dk);
  float best = 1e30f;
  int err = TALSH_SUCCESS;
  for (int pol = 0; pol < NPOLICY && !err; ++pol) {
    for (auto &h : hts) h.tile = policy_tile(pol, dk, h);
    const float ms = time_launch(g, dk, hts, nblocks, s, e0, e1, &err);
    if (!err && ms < best) {
      best = ms;
      *policy = pol;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  dev_free(g, sp, sh);
  *ms_spent += 1e3 * (wall_time() - t0);
  return err;
}

void release_build(talshAmdBatch *b) {
  // an asynchronous execution still reads its items and queue counters, which no hazard entry covers
  if (b->hz) (void)hipEventSynchronize(b->hz->ev);
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  if (b->dev && b->g >= 0) dev_free(b->g, b->dev, b->dev_handle);
  b->dev = nullptr;
  b->built = false;
}

std::vector<const void *> signature(const talshAmdBatch *b, int g) {
  std::vector<const void *> s;
  for (auto &e : b->entries) {
    int dk;
    s.push_back(gpu_body(e.d, g, &dk));
    s.push_back(gpu_body(e.l, g, &dk));
    s.push_back(gpu_body(e.r, g, &dk));
  }
  return s;
}

int build(talshAmdBatch *b, int g) {
  release_build(b);
  std::vector<HostTask> hts(b->entries.size());
  int dk = NO_TYPE;
  for (size_t i = 0; i < b->entries.size(); ++i) {
    int tdk = NO_TYPE;
    if (int e = plan_task(b->entries[i], g, &tdk, &hts[i])) return e;
    if (dk != NO_TYPE && tdk != dk) return TALSH_NOT_IMPLEMENTED;  // one data kind per batch
    dk = tdk;
  }
  // outputs must not overlap one another nor any input of the batch (byte ranges)
  std::vector<std::pair<uintptr_t, uintptr_t>> outs, ins;
  for (const auto &h : hts) {
    outs.emplace_back((uintptr_t)h.D, (uintptr_t)(h.D + h.dbytes));
    ins.emplace_back((uintptr_t)h.L, (uintptr_t)(h.L + h.lbytes));
    ins.emplace_back((uintptr_t)h.R, (uintptr_t)(h.R + h.rbytes));
  }
  std::sort(outs.begin(), outs.end());
  for (size_t i = 1; i < outs.size(); ++i)
    if (outs[i].first < outs[i - 1].second) return TALSH_INVALID_ARGS;
  for (const auto &in : ins) {  // the output starting last before in's end is the only candidate
    auto it = std::lower_bound(outs.begin(), outs.end(), std::make_pair(in.second, (uintptr_t)0));
    if (it != outs.begin() && std::prev(it)->second > in.first) return TALSH_INVALID_ARGS;
  }
  Device &dev = rt().gpus[g];
  hipStream_t s = dev.streams[0];
  if (int e = autotune(g, dk, hts, s, &b->tuned_classes, &b->tune_ms)) return e;
  int policy = POLICY_CLASS_TUNED;
  if (int e = choose_policy(g, dk, hts, s, &policy, &b->tune_ms)) return e;
  b->policy = policy;
  b->flops = 0;
  for (auto &h : hts) {
    h.tile = policy_tile(policy, dk, h);
    b->flops += 2.0 * h.geom.M * (double)h.geom.N * h.geom.K;
  }
  const int nblocks = persistent_blocks(g, dk);
  DeviceBatch db;
  if (int e = upload(g, dk, hts, s, &db)) return e;
  b->dev = db.base;
  b->dev_handle = db.handle;
  b->d_items = db.items;
  b->d_qstart = db.qstart;
  b->d_counters = db.counters;
  b->total = db.total;
  b->ntasks = (int)hts.size();
  b->nblocks = nblocks;
  b->g = g;
  b->dk = dk;
  // capture the persistent launch once; executions replay it
  hipStream_t cs;
  if (hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) return TALSH_FAILURE;
  int err = TALSH_SUCCESS;
  if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) err = TALSH_FAILURE;
  if (!err && batch_launch(dk, b->d_items, b->d_qstart, b->d_counters, kXcds, b->nblocks, cs)) err = TALSH_FAILURE;
  if (hipStreamEndCapture(cs, &b->graph) != hipSuccess) err = TALSH_FAILURE;
  if (!err && hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0) != hipSuccess) err = TALSH_FAILURE;
  (void)hipStreamDestroy(cs);
  if (err) {
    release_build(b);
    return err;
  }
  b->sig = signature(b, g);
  b->sig_bytes.clear();
  const size_t esz = (size_t)dk_size(dk);
  for (auto &e : b->entries)
    for (const talsh_tens_t *t : {e.d, e.l, e.r}) b->sig_bytes.push_back(shape_volume(t->shape_p) * esz);
  b->built = true;
  return TALSH_SUCCESS;
}

}  // namespace
}  // namespace tal

using namespace tal;

extern "C" {

int talshAmdBatchCreate(talshAmdBatch **batch) {
  if (!batch) return TALSH_INVALID_ARGS;
  *batch = new talshAmdBatch();
  return TALSH_SUCCESS;
}

int talshAmdBatchAdd(talshAmdBatch *b, const char *pattern, talsh_tens_t *dtens, talsh_tens_t *ltens,
                     talsh_tens_t *rtens, double scale_real, double scale_imag, int accumulative) {
  if (!b || !pattern || !dtens || !ltens || !rtens) return TALSH_INVALID_ARGS;
  if (talshTensorIsEmpty(dtens) == YEP || talshTensorIsEmpty(ltens) == YEP || talshTensorIsEmpty(rtens) == YEP)
    return TALSH_OBJECT_IS_EMPTY;
  if (scale_imag != 0.0) return TALSH_NOT_IMPLEMENTED;
  b->entries.push_back({pattern, dtens, ltens, rtens, scale_real, scale_imag, accumulative != NOPE});
  b->built = false;
  return TALSH_SUCCESS;
}

int talshAmdBatchSize(const talshAmdBatch *b) { return b ? (int)b->entries.size() : -1; }

int talshAmdBatchExecute(talshAmdBatch *b, int dev_id, int dev_kind, talsh_task_t *talsh_task) {
  std::lock_guard<std::recursive_mutex> lk(rt().mu);
  if (!rt().on) return TALSH_NOT_INITIALIZED;
  if (!b) return TALSH_INVALID_ARGS;
  if (talsh_task && talshTaskIsEmpty(talsh_task) != YEP) return TALSH_OBJECT_NOT_EMPTY;
  if (b->entries.empty()) return TALSH_SUCCESS;
  int g = -1;
  if (dev_kind == DEV_DEFAULT && dev_id == DEV_DEFAULT) g = talshDeviceBusyLeast(DEV_NVIDIA_GPU);
  else g = gpu_index(dev_kind == DEV_DEFAULT ? dev_id : talshFlatDevId(dev_kind, dev_id));
  if (g < 0) return TALSH_NOT_AVAILABLE;
  Device &dev = rt().gpus[g];
  (void)hipSetDevice(dev.hip_id);
  // Replay fast path: same GPU, graph built, hazard table unchanged since the
  // last execution, so every operand's ordering state is exactly `hz` and one
  // wait on it covers all of them (no per-tensor lookups); and no tensor gained
  // or lost an image (a caller's body leaves no trace in the hazard table when
  // its tensor is destructed).
  const bool planned = b->built && b->g == g && rt().image_epoch == b->images;
  const bool fast = planned && b->hz && rt().hazard_epoch == b->epoch;
  // Where something else ran meanwhile, the operands' bodies are still the
  // ones planned for if no image moved anywhere and no task that may hold one
  // is unfinalized (a batch of 4,096 looks 12,288 operands up otherwise: 0.3 ms).
  const bool same = planned && rt().tens_tasks.empty();
  if (!fast && !same) {
    if (!b->built || b->g != g || signature(b, g) != b->sig) {
      const int e = build(b, g);
      if (e) return e;
    }
    b->images = rt().image_epoch;
  }
  // nothing running anywhere: no operand has anything to wait for (3-4 ms of
  // per-range lookups for 12,288 operands otherwise)
  bool idle = !fast;
  for (size_t i = 0; idle && i < rt().gpus.size(); ++i) idle = !rt().gpus[i].on || device_idle((int)i);
  const bool timed = talsh_task != nullptr;
  Task *task = task_new(g, 3.0 * (double)b->entries.size() * 4096.0);
  task->timed = timed;
  hipStream_t s = task->stream;
  if (timed) (void)hipEventRecord(task->ev_start->ev, s);
  if (fast) {
    (void)hipStreamWaitEvent(s, b->hz->ev, 0);
  } else if (!idle) {
    for (size_t i = 0; i < b->entries.size(); ++i) {
      hazard_wait_write(b->sig[3 * i], b->sig_bytes[3 * i], s);
      hazard_wait_read(b->sig[3 * i + 1], b->sig_bytes[3 * i + 1], s);
      hazard_wait_read(b->sig[3 * i + 2], b->sig_bytes[3 * i + 2], s);
    }
  }
  if (timed) {
    (void)hipEventRecord(task->ev_in->ev, s);
    task->ev_mm0 = new_event(g);
    (void)hipEventRecord(task->ev_mm0->ev, s);
  }
  if (hipGraphLaunch(b->exec, s) != hipSuccess) {
    task_free(task);
    return TALSH_FAILURE;
  }
  if (timed) {
    task->ev_mm1 = new_event(g);
    (void)hipEventRecord(task->ev_mm1->ev, s);
    (void)hipEventRecord(task->ev_comp->ev, s);
  }
  (void)hipEventRecord(task->ev_done->ev, s);
  if (!fast)
    for (auto &e : b->entries) {  // other images of each output become stale
      if (e.d->ndev < 2) continue;
      const int gi = image_find(e.d, flat_gpu(g), NO_TYPE, true);
      if (gi >= 0) image_discard_other(e.d, gi);
    }
  // A blocking call ends under the runtime's lock, so nothing later has to be
  // ordered against it; entries of earlier executions keep their event.
  if (timed) {
    if (!fast) {
      if (!b->hz) b->hz = new_event(g);
      for (size_t i = 0; i < b->entries.size(); ++i) {
        hazard_set_writer(b->sig[3 * i], b->sig_bytes[3 * i], b->hz);
        hazard_add_reader(b->sig[3 * i + 1], b->sig_bytes[3 * i + 1], b->hz);
        hazard_add_reader(b->sig[3 * i + 2], b->sig_bytes[3 * i + 2], b->hz);
      }
    }
    (void)hipEventRecord(b->hz->ev, s);
    b->hz->seen_done = false;
    b->epoch = rt().hazard_epoch;
  }
  task->flops = b->flops;
  dev.tasks_submitted++;
  dev.active++;
  b->replays++;
  talsh_task_t local;
  talsh_task_t *tt = talsh_task ? talsh_task : &local;
  if (!talsh_task) talshTaskClean(&local);
  tt->task_p = task;
  tt->task_error = -1;
  tt->dev_kind = DEV_NVIDIA_GPU;
  tt->data_kind = b->dk;
  tt->coherence = 0;
  tt->num_args = 0;
  tt->flops = b->flops;
  if (talsh_task) return TALSH_SUCCESS;
  const int st = task_finalize_if_done(tt, true);
  talshTaskDestruct(tt);
  return st == TALSH_TASK_COMPLETED ? TALSH_SUCCESS : TALSH_TASK_ERROR;
}

int talshAmdBatchStats(const talshAmdBatch *b, double *flops, long long *work_items, int *tuned_classes,
                       double *tune_ms, int *executions) {
  if (!b) return TALSH_INVALID_ARGS;
  if (flops) *flops = b->flops;
  if (work_items) *work_items = b->total;
  if (tuned_classes) *tuned_classes = b->tuned_classes;
  if (tune_ms) *tune_ms = b->tune_ms;
  if (executions) *executions = b->replays;
  return TALSH_SUCCESS;
}

int talshAmdBatchDestroy(talshAmdBatch *b) {
  if (!b) return TALSH_INVALID_ARGS;
  {
    std::lock_guard<std::recursive_mutex> lk(rt().mu);
    if (b->built && rt().on && b->g >= 0) {
      for (size_t i = 0; i < b->sig.size(); ++i) hazard_drain(b->sig[i], b->sig_bytes[i]);
      release_build(b);
    }
  }
  delete b;
  return TALSH_SUCCESS;
}

}  // extern "C"
